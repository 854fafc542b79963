"""Narrow layers: the stages of whole token tiles (the dW pass at fan-in 8 over at most 1600 inputs, the
max / top-k forward over at most 2048) against the wide kernels on the same neurons.

A layer of D inputs and the same layer with unused inputs appended (zeros in X, no index reaches them)
compute the same sums in the same order, so every output must agree bit for bit; the oracle tests of
test_gpu_parity.py cover the values themselves."""
import pytest
import torch

from granulelayer_amd.autograd import Level1Runtime
from granulelayer_amd.config import LevelSpec, PhysicalPlan
from granulelayer_amd.layout import SparseLayout, init_parameters

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(D, H, G, K, B, x_dtype, w_dtype, wide):
    """(runtime factory, x, w, b) of a layer over ``wide`` inputs whose records lie in [0, D)."""
    idx, w, b = init_parameters(SparseLayout(D, H, G, K, 8, False), "cpu", w_dtype, seed=D + B, bias_std=0.3)
    gen = torch.Generator().manual_seed(B)
    x = torch.zeros(B, wide)
    x[:, :D] = torch.randn(B, D, generator=gen)
    L = SparseLayout(wide, H, G, K, 8, False)
    return L, idx.to(DEV), x.to(x_dtype).to(DEV), w.to(DEV), b.to(DEV)


# stages of 8, 4, 2 and 1 tiles at the edges of their range, whole and partial last stages, one tile,
# two token chunks of the backward (B > 1024), ragged pools, bf16 X and parameters
DW_CASES = [
    (200, 3000, 5, 36, torch.float32, torch.float32),
    (201, 3000, 5, 100, torch.float32, torch.bfloat16),
    (400, 5001, 7, 61, torch.bfloat16, torch.float32),
    (801, 5001, 7, 64, torch.float32, torch.float32),
    (1600, 4099, 16, 37, torch.float32, torch.float32),
    (1599, 900, 30, 1, torch.float32, torch.float32),
    (33, 2000, 3, 1100, torch.float32, torch.float32),
]


@pytest.mark.parametrize("act", ["relu", "identity"])
@pytest.mark.parametrize("case", DW_CASES, ids=lambda c: f"D{c[0]}B{c[3]}{str(c[4])[6:]}{str(c[5])[6:]}")
def test_narrow_dw_gives_the_bits_of_the_wide_kernel(case, act):
    D, H, G, B, xdt, wdt = case
    got = []
    for wide in (D, 1601 + D % 7):
        L, idx, x, w, b = _layer(D, H, G, 8, B, xdt, wdt, wide)
        rt = Level1Runtime(L, idx, LevelSpec("mean", activation=act), PhysicalPlan())
        out = rt.forward(x, w, b)
        dw, db = torch.zeros(L.weight_shape, device=DEV), torch.zeros(L.bias_shape, device=DEV)
        dy = torch.randn(B, G, generator=torch.Generator().manual_seed(1)).to(DEV)
        dx = rt.backward(x, w, b, dy, out, "minimal_stats", dw, db)
        got.append((out["pre"], dw, db, dx[:, :D]))
    for name, a, c in zip(("pre", "dw", "db"), got[0], got[1]):
        assert torch.equal(a, c), name
    # dX sums the same terms over other unit ranges (their number depends on D): fp32 rounding of a
    # sum of at most n = edges per input terms, sqrt(n) 2^-24 of its scale
    a, c = got[0][3].double(), got[1][3].double()
    n = H * 8 / D
    assert float((a - c).norm() / c.norm()) <= 4 * n ** 0.5 * 2.0**-24


SEL_CASES = [
    (512, 5001, 7, 61, torch.float32),   # 8 tiles per stage
    (513, 5001, 7, 64, torch.bfloat16),  # 4
    (2048, 4099, 16, 37, torch.float32),  # 2
    (2047, 3000, 5, 3, torch.float32),   # one tile in all: not staged
    (1024, 2000, 3, 130, torch.float32),
]


@pytest.mark.parametrize("pool,k", [("max", 1), ("topk_mean", 8), ("topk_mean", 16)])
@pytest.mark.parametrize("case", SEL_CASES, ids=lambda c: f"D{c[0]}B{c[3]}{str(c[4])[6:]}")
def test_narrow_selection_forward_gives_the_bits_of_the_wide_kernel(case, pool, k):
    D, H, G, B, xdt = case
    got = []
    for wide in (D, 2049 + D % 5):
        L, idx, x, w, b = _layer(D, H, G, 8, B, xdt, torch.float32, wide)
        spec = LevelSpec(pool, k=k) if pool == "topk_mean" else LevelSpec(pool)
        rt = Level1Runtime(L, idx, spec, PhysicalPlan())
        out = rt.forward(x, w, b, track_ids=True)
        got.append((out["pre"], out["winner" if pool == "max" else "topk_slot"]))
    for name, a, c in zip(("pre", "ids"), *got):
        assert torch.equal(a, c), name


# fan-in 16: two workgroups per CU over whole narrow tiles, at least 8 tiles (29 tokens on), D to 2048
@pytest.mark.parametrize("pool,kw", [("logmeanexp", {"temperature": 0.5}), ("softmax_weighted", {"beta": 1.0}),
                                     ("power_mean", {"p": 2.0}), ("topk_mean", {"k": 8})])
@pytest.mark.parametrize("D,B", [(64, 29), (255, 64), (256, 100), (2048, 33)])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_narrow_fan_in_16_forward_matches_the_wide_kernel(D, B, pool, kw, wdt):
    """The same layer with 2049 or more inputs runs the two-buffer kernel: the same z (top-k: the same
    slots and values bit for bit); the smooth states merge in the same order, their exponentials contracted
    by the compiler as it sees fit, within 8 roundings of fp32 (2^-21 of the value's scale)."""
    H, G = 3000, 7
    got = []
    for wide in (D, 2049 + D % 5):
        L, idx, x, w, b = _layer(D, H, G, 16, B, torch.float32, wdt, wide)
        rt = Level1Runtime(L, idx, LevelSpec(pool, activation="relu", **kw), PhysicalPlan())
        out = rt.forward(x, w, b, track_ids=True)
        got.append((out["pre"], out.get("topk_slot")))
    (a, ia), (c, ic) = got
    if pool == "topk_mean":
        assert torch.equal(a, c) and torch.equal(ia, ic)
    else:
        assert float((a - c).abs().max()) <= 2.0**-21 * float(c.abs().max())
