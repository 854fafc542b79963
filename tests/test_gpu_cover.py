"""Cover-TopK/16 on the GPU: the HIP selection kernel (gl_cover_select) bit-exact against the
reference's own vectors and against the CPU oracle (oracle/cover.py); the compact layer (one K16
record per 16 neurons, rec_shift 4) against the float64 oracle of the same parameters; energy
restoration; save_packed / load_packed; and the C5 shape at full size."""
from pathlib import Path

import numpy as np
import pytest
import torch

from conftest import assert_close, assert_parity, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

from granulelayer_amd import CoverTopK16Layer  # noqa: E402
from granulelayer_amd import cover_topk16 as CT  # noqa: E402
from oracle import cover as OC  # noqa: E402
from oracle import oracle as O  # noqa: E402

DEV = "cuda"
GOLDEN = Path(__file__).resolve().parent / "golden" / "cover_reference.npz"


def _golden():
    with np.load(GOLDEN) as z:
        d = {k: z[k] for k in z.files}
    names = sorted({k.split("/")[0] for k in d})
    return [(n, {k.split("/", 1)[1]: v for k, v in d.items() if k.startswith(n + "/")}) for n in names]


@pytest.mark.parametrize("name,case", _golden(), ids=lambda c: c if isinstance(c, str) else "")
def test_selection_kernel_matches_reference_vectors(name, case):
    H, G, C, seed = (int(v) for v in case["shape"])
    L = CT.EnvelopeLayout(4096, H, G, 64, C)
    w = torch.from_numpy(case["w_int"].astype(np.float32) / 4096).to(DEV)
    a = CT.feature_importance(w, L).cpu().numpy()
    assert np.array_equal(a, case["importance"]), "float64 importances differ"
    uv = case["valid_groups"]
    env0 = CT.topk_select(torch.from_numpy(case["importance"][uv]).to(DEV), 16).cpu().numpy()
    assert np.array_equal(env0, case["env_topk"])
    out = CT.cover_topk(w, L)
    assert np.array_equal(out["env"].cpu().numpy()[uv], case["env_cover"])
    rv = L.record_counts("cpu").numpy() > 0
    assert np.array_equal(out["missing0"].cpu().numpy()[rv], case["missing0"])
    assert np.array_equal(out["swaps"].cpu().numpy()[rv], case["swaps"])
    assert np.array_equal(out["loss"].cpu().numpy()[rv], case["loss"]), "energy loss (float64, swap order) differs"


def _envelope(D, H, G, C, seed, quant=None):
    L = CT.EnvelopeLayout(D, H, G, 64, C)
    gen = torch.Generator().manual_seed(seed)
    w = torch.randn(L.weight_shape, generator=gen) / 8
    if quant:  # coarse values: many importance ties
        w = torch.round(w * quant) / quant
    valid = L.valid_mask("cpu")
    w = w * valid[..., None]
    b = torch.randn(L.bias_shape, generator=gen) * 0.2 * valid
    from granulelayer_amd.layout import sample_distinct

    cand = sample_distinct(G * L.blocks_per_group, D, 64, gen, "cpu").to(torch.int32).view(L.index_shape)
    return L, w, b, cand


@pytest.mark.parametrize("C,quant", [(256, None), (64, 4), (128, 2), (16, None)])
def test_selection_kernel_matches_oracle(C, quant):
    D, G = 300, 5
    H = G * (3 * C - 5)  # two full records and a partial one whose last group is partial, per output
    L, w, b, cand = _envelope(D, H, G, C, seed=C, quant=quant)
    gpb = C // 16
    nv = L.valid_mask("cpu").reshape(-1, 16).sum(1).numpy()
    if C == 16:  # one group per record: m k < 64, infeasible for the repair
        with pytest.raises(ValueError, match="infeasible"):
            CT.cover_topk(w.to(DEV), L, cand.to(DEV))
        return
    env, a, m0, sw, lo = OC.select(w.numpy().reshape(-1, 16, 64), nv, gpb, 16, repair=True)
    out = CT.cover_topk(w.to(DEV), L, cand.to(DEV))
    valid = nv > 0
    assert np.array_equal(out["env"].cpu().numpy()[valid], env[valid])
    assert np.array_equal(out["env"].cpu().numpy()[~valid], np.tile(np.arange(16), (int((~valid).sum()), 1)))
    assert np.array_equal(out["swaps"].cpu().numpy(), sw) and np.array_equal(out["missing0"].cpu().numpy(), m0)
    assert np.array_equal(out["loss"].cpu().numpy(), lo)
    # kept global inputs and weights
    ci = cand.numpy().reshape(-1, 64).repeat(gpb, 0)
    assert np.array_equal(out["rec_idx"].cpu().numpy(), np.take_along_axis(ci, out["env"].cpu().numpy(), 1))
    wn = w.numpy().reshape(-1, 64)
    e16 = out["env"].cpu().numpy().repeat(16, 0)
    assert np.array_equal(out["W_out"].cpu().numpy(), np.take_along_axis(wn, e16, 1))


def _layer_oracle(lay, x, dy, pool="mean"):
    """Oracle forward / backward of the compact layer, its records expanded per neuron (Mode A, K 16)."""
    L = lay.layout
    S = L.slots_per_group
    idx = lay.indices.cpu().numpy().reshape(-1, 16).repeat(16, 0)  # [G S, 16]
    w = lay.weight.detach().cpu().numpy().reshape(-1, 16)
    b = lay.bias.detach().cpu().numpy().reshape(-1)
    counts = L.counts_tensor("cpu").numpy()
    want, mag = O.forward(x, idx, w, b, counts, S, "relu", pool, with_mag=True)
    dW, db, dX, bnd = O.backward(x, idx, w, b, counts, S, dy, "relu", pool, with_bounds=True)
    return want, mag, dW, db, dX, bnd


@pytest.mark.parametrize("normalization", ["none", "energy"])
def test_compact_layer_matches_oracle(normalization):
    D, G, C, B = 512, 6, 256, 70
    H = G * (C + 9 * 16 + 5)  # a full record and a partial one whose last group is partial
    L, w, b, cand = _envelope(D, H, G, C, seed=3)
    lay = CoverTopK16Layer.from_envelope(w.to(DEV), b.to(DEV), cand.to(DEV), input_dim=D, hidden_dim=H, output_dim=G,
                                         envelope_C=C, normalization=normalization)
    meta = lay.metadata
    assert meta["valid_slots"] == 16 * H and meta["executed"] == dict(K=16, C=16, records_16=int(
        L.valid_mask("cpu").reshape(-1, 16).any(1).sum()))
    # the compact parameters are the selected envelope values (scaled once with energy restoration)
    nv = L.valid_mask("cpu").reshape(-1, 16).sum(1).numpy()
    env, *_ = OC.select(w.numpy().reshape(-1, 16, 64), nv, C // 16, 16, repair=True)
    kept = np.take_along_axis(w.numpy().reshape(-1, 64), env.repeat(16, 0), 1)
    got_w = lay.weight.detach().cpu().numpy().reshape(-1, 16)
    if normalization == "none":
        assert np.array_equal(got_w, kept)
    else:
        wd = w.numpy().reshape(-1, 64).astype(np.float64)
        e, ek = (wd * wd).sum(1), (kept.astype(np.float64) ** 2).sum(1)
        with np.errstate(invalid="ignore"):  # padded neurons: 0 / 0, replaced below
            s = np.minimum(np.sqrt(e / np.maximum(ek, 1e-6 * e)), 8.0)
        s = np.where(e > 0, s, 1.0) * L.valid_mask("cpu").reshape(-1).numpy()
        assert_close(got_w, kept * s[:, None], rtol=2e-6, atol=1e-12, what="energy-restored weights")
        assert meta["normalization"]["treatment"] == "energy"
    gen = torch.Generator().manual_seed(4)
    x = torch.randn(B, D, generator=gen)
    dy = torch.randn(B, G, generator=gen)
    xd = x.to(DEV).requires_grad_(True)
    lay.enable_main_grad()
    y = lay(xd)
    y.backward(dy.to(DEV))
    want, mag, dW, db, dX, bnd = _layer_oracle(lay, x.numpy(), dy.numpy())
    (mW, mb, mX), (uW, ub, uX) = bnd["mag"], bnd["unc"]
    assert_parity(y.detach().cpu().numpy(), want, mag, what="y")
    assert_parity(xd.grad.cpu().numpy(), dX, mX, uX, what="dX")
    assert_parity(lay.weight.main_grad.cpu().numpy().reshape(-1, 16), dW, mW, uW, what="dW")
    assert_parity(lay.bias.main_grad.cpu().numpy().reshape(-1), db, mb, ub, what="db")
    assert lay.last_info["forward_backend"] == "hip"


def test_packed_round_trip(tmp_path):
    D, G, C, B = 256, 4, 128, 33
    H = G * 2 * C
    L, w, b, cand = _envelope(D, H, G, C, seed=9)
    lay = CoverTopK16Layer.from_envelope(w.to(DEV), b.to(DEV), cand.to(DEV), input_dim=D, hidden_dim=H, output_dim=G,
                                         envelope_C=C)
    x = torch.randn(B, D, device=DEV)
    y = lay(x)
    info = lay.save_packed(tmp_path / "ct16.pt")
    back = CoverTopK16Layer.load_packed(tmp_path / "ct16.pt", device=DEV)
    assert torch.equal(back(x), y)
    assert back.metadata == lay.metadata and info["fingerprints"] == back.immutable_fingerprints()
    blob = torch.load(tmp_path / "ct16.pt", weights_only=True)
    blob["state"]["indices"][0, 0, 0] += 1  # a changed support must be refused
    torch.save(blob, tmp_path / "bad.pt")
    with pytest.raises(ValueError, match="fingerprints"):
        CoverTopK16Layer.load_packed(tmp_path / "bad.pt", device=DEV)


def test_cover_topk16_at_the_c5_shape():
    """BASELINE configs[4]'s shape with Cover-TopK/16 records: N = 50,331,648 neurons in pools of
    512 (G = 98,304), D = 4096, B = 512, a C256 envelope of 64 candidates uniform in [0, 4096) with
    weights N(0, 1/16); selection of all 196,608 records, then forward and backward of the whole
    compact layer against the oracle on 12 pools (dY zero elsewhere)."""
    D, G, C, B, pool = 4096, 98_304, 256, 512, 512
    H = G * pool
    L = CT.EnvelopeLayout(D, H, G, 64, C)
    gen = torch.Generator(device=DEV).manual_seed(0)
    w = torch.randn(L.weight_shape, generator=gen, device=DEV) / 4
    b = torch.zeros(L.bias_shape, device=DEV)
    from granulelayer_amd.layout import sample_distinct

    cand = torch.empty((G * L.blocks_per_group, 64), dtype=torch.int32, device=DEV)
    for s in range(0, cand.shape[0], 1 << 16):
        e = min(s + (1 << 16), cand.shape[0])
        cand[s:e] = sample_distinct(e - s, D, 64, gen, DEV).to(torch.int32)
    lay = CoverTopK16Layer.from_envelope(w, b, cand.view(L.index_shape), input_dim=D, hidden_dim=H, output_dim=G,
                                         envelope_C=C, pooling="sum")
    del w
    st = lay.metadata["support_stats"]
    print(f"C5 Cover-TopK/16: {st}, selection {lay.metadata['construction_seconds']['selection']:.2f} s")
    assert st["swaps"] == st["missing0"] > 0
    x = torch.randn(B, D, generator=gen, device=DEV)
    pools = np.sort(np.concatenate([[0, G - 1], np.random.default_rng(0).choice(G - 2, 10, replace=False) + 1]))
    sel = torch.from_numpy(pools).to(DEV)
    dy = torch.zeros(B, G, device=DEV)
    dy[:, sel] = torch.randn(B, len(pools), generator=gen, device=DEV)
    xd = x.clone().requires_grad_(True)
    lay.enable_main_grad()
    y = lay(xd)
    y.backward(dy)
    S = lay.layout.slots_per_group
    rows = torch.cat([torch.arange(g * S // 16, (g + 1) * S // 16, device=DEV) for g in pools.tolist()])
    idx = lay.indices.view(-1, 16)[rows].cpu().numpy().repeat(16, 0)
    wk = lay.weight.detach().view(-1, 16, 16)[rows].cpu().numpy().reshape(-1, 16)
    bk = lay.bias.detach().view(-1, 16)[rows].cpu().numpy().reshape(-1)
    counts = np.full(len(pools), pool, np.int32)
    xn = x.cpu().numpy()
    want, mag = O.forward(xn, idx, wk, bk, counts, S, "relu", "sum", with_mag=True)
    assert_parity(y.detach()[:, sel].cpu().numpy(), want, mag, what="C5 Cover-TopK/16 y (sampled pools)")
    dW, db, dX, bnd = O.backward(xn, idx, wk, bk, counts, S, dy[:, sel].cpu().numpy(), "relu", "sum",
                                 with_bounds=True)
    (mW, mb, mX), (uW, ub, uX) = bnd["mag"], bnd["unc"]
    assert_parity(xd.grad.cpu().numpy(), dX, mX, uX, what="C5 Cover-TopK/16 dX")
    assert_parity(lay.weight.main_grad.view(-1, 16, 16)[rows].cpu().numpy().reshape(-1, 16), dW, mW, uW, what="dW")


# ---- the record kernels (gl_record.hip) ------------------------------------------------------------
# (D, neurons per pool, pools, B, x dtype): one token, the edges of the 64-token slices and of the dX
# slabs (64 / 128 / 256), pools of one partial record, of a partial chunk of 8 records, of chunks and a bit
RECORD_CASES = [
    (64, 5, 3, 1, torch.float32),
    (100, 16, 7, 63, torch.float32),
    (96, 130, 5, 64, torch.bfloat16),
    (33, 117, 4, 65, torch.float32),
    (512, 300, 3, 129, torch.float32),
    (40, 1040, 2, 260, torch.bfloat16),
    (64, 40, 3, 1030, torch.float32),
]


def _record_layer(D, per, G, seed=0):
    """A compact layer with random records (padded neurons' weights and biases are not zero: only the
    kernels' own masks keep them out)."""
    S = -(-per // 16) * 16
    lay = CoverTopK16Layer(D, G * per, G, S, pooling="mean", device=DEV)
    gen = torch.Generator().manual_seed(seed)
    rec = torch.stack([torch.randperm(D, generator=gen)[:16].sort().values for _ in range(G * S // 16)])
    with torch.no_grad():
        lay.indices.copy_(rec.to(torch.int32).view(lay.indices.shape))
        lay.weight.copy_(torch.randn(lay.weight.shape, generator=gen) / 4)
        lay.bias.copy_(torch.randn(lay.bias.shape, generator=gen) / 4)
    return lay


def _off_boundary(t):
    """A copy of t that starts 4 bytes past a 16-byte boundary: the per-neuron kernels take it."""
    return torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("act,pool", [("relu", "sum"), ("identity", "mean"), ("gelu", "sum")])
@pytest.mark.parametrize("case", RECORD_CASES, ids=lambda c: f"D{c[0]}n{c[1]}B{c[3]}{str(c[4])[6:]}")
def test_record_kernels_match_oracle(case, act, pool):
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    D, per, G, B, xdt = case
    lay = _record_layer(D, per, G)
    L = lay.layout
    S = L.slots_per_group
    gen = torch.Generator().manual_seed(B)
    x, dy = torch.randn(B, D, generator=gen).to(xdt), torch.randn(B, G, generator=gen)
    counts = L.counts_tensor("cpu").numpy()
    idx = lay.indices.cpu().numpy().reshape(-1, 16).repeat(16, 0)
    w, b = lay.weight.detach().cpu().numpy().reshape(-1, 16), lay.bias.detach().cpu().numpy().reshape(-1)
    xn = x.float().numpy()
    want, mag = O.forward(xn, idx, w, b, counts, S, act, pool, with_mag=True)
    rt = Level1Runtime(L, lay.indices, LevelSpec(pool, activation=act), PhysicalPlan())
    xd = x.to(DEV)
    got = rt.forward(xd, lay.weight, lay.bias)
    assert_parity(got["pre"].cpu().numpy(), want, mag, what="pre")
    dw, db = torch.zeros(L.weight_shape, device=DEV), torch.zeros(L.bias_shape, device=DEV)
    dx = rt.backward(xd, lay.weight, lay.bias, dy.to(DEV), {"pre": got["pre"]}, "minimal_stats", dw, db)
    dW, dB, dX, bnd = O.backward(xn, idx, w, b, counts, S, dy.numpy(), act, pool, with_bounds=True)
    (mW, mb, mX), (uW, ub, uX) = bnd["mag"], bnd["unc"]
    assert_parity(dw.cpu().numpy().reshape(-1, 16), dW, mW, uW, what="dW")
    assert_parity(db.cpu().numpy().reshape(-1), dB, mb, ub, what="db")
    assert_parity(dx.cpu().numpy(), dX, mX, uX, what="dX")
    valid = L.valid_mask("cpu").reshape(-1).numpy()
    assert not dw.cpu().numpy().reshape(-1, 16)[~valid].any() and not db.cpu().numpy().reshape(-1)[~valid].any()
    # views off a 16-byte boundary run the per-neuron kernels: the same z bit for bit (pools of one
    # slot show them), the same sums in another order; the backward also with an unaligned dW
    off = _off_boundary(lay.weight.detach())
    pre = rt.forward(xd, off, lay.bias)["pre"].cpu().numpy()
    assert_parity(pre, want, mag, what="pre (unaligned weights)")
    for wv, dw in ((off, torch.zeros(L.weight_shape, device=DEV)),
                   (lay.weight.detach(), _off_boundary(torch.zeros(L.weight_shape, device=DEV)))):
        db = torch.zeros(L.bias_shape, device=DEV)
        dx = rt.backward(xd, wv, lay.bias, dy.to(DEV), {"pre": got["pre"]}, "minimal_stats", dw, db)
        assert_parity(dw.cpu().numpy().reshape(-1, 16), dW, mW, uW, what="dW (unaligned)")
        assert_parity(db.cpu().numpy().reshape(-1), dB, mb, ub, what="db (unaligned)")
        assert_parity(dx.cpu().numpy(), dX, mX, uX, what="dX (unaligned)")


def test_record_z_has_the_bits_of_the_per_neuron_kernels():
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    lay = _record_layer(200, 1, 700)
    rt = Level1Runtime(lay.layout, lay.indices, LevelSpec("sum", activation="identity"), PhysicalPlan())
    x = torch.randn(70, 200, device=DEV)
    w = lay.weight.detach()
    off = torch.empty(w.numel() + 1, device=DEV)[1:].view(w.shape).copy_(w)  # not 16-byte aligned: per-neuron kernels
    assert torch.equal(rt.forward(x, w, lay.bias)["pre"], rt.forward(x, off, lay.bias)["pre"])


def test_record_forward_in_token_passes_and_without_a_workspace():
    """A part budget of 20 tokens' partials, whole batches and gl_fwd_static give the same bits: a
    token's sums do not depend on the tokens beside it."""
    import ctypes

    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd import _native as N
    from granulelayer_amd.autograd import Level1Runtime
    from granulelayer_amd.backend import _ptr, _stream

    lay = _record_layer(128, 520, 50)
    L = lay.layout
    x = torch.randn(150, 128, device=DEV)
    chunks = L.groups * -(-L.slots_per_group // 128)
    outs = []
    for budget in (None, chunks * 4 * 20, chunks * 4 * 100):
        rt = Level1Runtime(L, lay.indices, LevelSpec("sum", activation="relu"), PhysicalPlan(), None, budget)
        outs.append(rt.forward(x, lay.weight, lay.bias)["pre"])
    pre = torch.empty_like(outs[0])
    a = N.GlFwdArgs(X=_ptr(x), sxb=128, x_dtype=N.GL_DTYPE_F32, B=150, D=128, G=L.groups, S=L.slots_per_group, K=16,
                    act=N.GL_ACT["relu"], pool=N.GL_POOL["sum"], rec_shift=4, idx=_ptr(lay.indices), W=_ptr(lay.weight),
                    bias=_ptr(lay.bias), counts=_ptr(rt.counts_i32), pre=_ptr(pre))
    assert N.library().lib.gl_fwd_static(ctypes.byref(a), ctypes.c_void_p(_stream(x.device))) == 0
    for o in (*outs[1:], pre):
        assert torch.equal(o, outs[0])


# (act, D, neurons per pool, x dtype, tokens of the last per-neuron call, of the first record call): the
# record kernels pay from 28 (16 past 2048 inputs) tokens with ReLU and 20 (36) with GELU, times the share
# of a 256-slot chunk that the pool fills
@pytest.mark.parametrize("act,D,per,xdt,last,first", [
    ("relu", 64, 256, torch.float32, 28, 29),
    ("relu", 2049, 256, torch.float32, 16, 17),
    ("relu", 64, 520, torch.float32, 19, 20),       # 528 slots in 3 chunks of 256
    ("identity", 64, 16, torch.float32, 1, 2),
    ("gelu", 64, 1000, torch.float32, 19, 20),      # 1008 slots in 4 chunks
    ("gelu", 64, 256, torch.bfloat16, 36, 37),
])
def test_record_forward_from_the_tokens_it_pays_at(act, D, per, xdt, last, first):
    """Fewer tokens give the per-neuron kernels' sums bit for bit, more another order of the same terms."""
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    lay = _record_layer(D, per, 64)
    rt = Level1Runtime(lay.layout, lay.indices, LevelSpec("sum", activation=act), PhysicalPlan())
    w = lay.weight.detach()
    x = torch.randn(first, D, device=DEV).to(xdt)
    for B, rec in ((last, False), (first, True)):
        pre, per_neuron = (rt.forward(x[:B], v, lay.bias)["pre"] for v in (w, _off_boundary(w)))
        assert torch.equal(pre, per_neuron) != rec
        assert_close(pre.cpu().numpy(), per_neuron.cpu().numpy(), rtol=1e-5, atol=1e-5 * per ** 0.5)


@pytest.mark.parametrize("D,per,last,first", [(64, 512, 44, 45), (2050, 512, 32, 33), (64, 48, 16, 17)])
def test_record_dw_from_the_tokens_it_pays_at(D, per, last, first):
    """As above for the dW pass; a batch's last chunk of 1024 tokens decides for itself."""
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    lay = _record_layer(D, per, 64)
    rt = Level1Runtime(lay.layout, lay.indices, LevelSpec("sum", activation="relu"), PhysicalPlan())
    w = lay.weight.detach()
    x, dy = torch.randn(first, D, device=DEV), torch.randn(first, 64, device=DEV)
    for B, rec in ((last, False), (first, True)):
        out = []
        for v in (w, _off_boundary(w)):
            dw, db = torch.zeros_like(w), torch.zeros_like(lay.bias)
            dx = rt.backward(x[:B], v, lay.bias, dy[:B], {}, "minimal_stats", dw, db)
            out.append((dw, db, dx))
        assert torch.equal(out[0][0], out[1][0]) != rec
        assert torch.equal(out[0][2], out[1][2])  # the same mask bits
        for a, b in zip(*out):
            assert_close(a.detach().cpu().numpy(), b.detach().cpu().numpy(), rtol=1e-5, atol=2e-5)


@pytest.mark.parametrize("per,pools,rec", [(16, 400_000, True), (256, 330_000, False)])
def test_static_forward_of_record_layers_in_short_passes(per, pools, rec):
    """gl_fwd_static where fewer than 64 tokens' partials fit its scratch: passes of 36 tokens on the record
    kernels give gl_fwd's bits; where 128-slot partials leave 20 tokens a pass, the per-neuron kernels
    (256-slot partials) give their own."""
    import ctypes

    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd import _native as N
    from granulelayer_amd.autograd import Level1Runtime
    from granulelayer_amd.backend import _ptr, _stream

    D, B = 64, 70
    lay = CoverTopK16Layer(D, pools * per, pools, per, pooling="mean", device=DEV)
    L = lay.layout
    gen = torch.Generator(device=DEV).manual_seed(0)
    with torch.no_grad():
        lay.indices.random_(0, D, generator=gen)
        lay.weight.normal_(0, 0.25, generator=gen)
        lay.bias.normal_(0, 0.25, generator=gen)
    x = torch.randn(B, D, device=DEV, generator=gen)
    rt = Level1Runtime(L, lay.indices, LevelSpec("sum", activation="relu"), PhysicalPlan())
    w = lay.weight.detach()
    pre = torch.empty(B, pools, device=DEV)
    a = N.GlFwdArgs(X=_ptr(x), sxb=D, x_dtype=N.GL_DTYPE_F32, B=B, D=D, G=pools, S=per, K=16, act=N.GL_ACT["relu"],
                    pool=N.GL_POOL["sum"], rec_shift=4, idx=_ptr(lay.indices), W=_ptr(w), bias=_ptr(lay.bias),
                    counts=_ptr(rt.counts_i32), pre=_ptr(pre))
    assert N.library().lib.gl_fwd_static(ctypes.byref(a), ctypes.c_void_p(_stream(x.device))) == 0
    full = rt.forward(x, w, lay.bias)["pre"]
    per_neuron = rt.forward(x, _off_boundary(w), lay.bias)["pre"]
    assert torch.equal(pre, full if rec else per_neuron)
    assert torch.equal(full, per_neuron) is False
    err = (full - per_neuron).abs()
    assert bool((err <= 1e-5 * per_neuron.abs() + 1e-5 * per ** 0.5).all())


@pytest.mark.parametrize("act", ["relu", "identity"])
def test_record_kernels_pass_infinities_and_nan_like_the_per_neuron_kernels(act):
    """X with infinities and NaN: the same outputs and gradients are infinite or NaN (the tokens beside the
    bad ones stay out of it), the others agree.  Input 0 stays finite: the per-neuron kernels' padded
    slots read it with weight 0."""
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    D, B, G = 40, 100, 6
    lay = _record_layer(D, 37, G)  # a partial record: 11 padded slots with weights of their own
    x, dy = torch.randn(B, D, device=DEV), torch.randn(B, G, device=DEV)
    x[3, 5], x[64, 1], x[99, 7] = float("inf"), float("nan"), -float("inf")
    rt = Level1Runtime(lay.layout, lay.indices, LevelSpec("sum", activation=act), PhysicalPlan())
    out = []
    for w in (lay.weight.detach(), _off_boundary(lay.weight.detach())):
        pre = rt.forward(x, w, lay.bias)["pre"]
        dw, db = torch.zeros(lay.layout.weight_shape, device=DEV), torch.zeros(lay.layout.bias_shape, device=DEV)
        dx = rt.backward(x, w, lay.bias, dy, {}, "minimal_stats", dw, db)
        out.append((pre.detach(), dw, db, dx))
    for a, b in zip(*out):
        fin = torch.isfinite(a)
        assert torch.equal(fin, torch.isfinite(b)) and torch.equal(a.isnan(), b.isnan()) and bool(fin.any())
        assert torch.equal(a[a.isinf()], b[b.isinf()])
        assert_close(a[fin].cpu().numpy(), b[fin].cpu().numpy(), rtol=1e-5, atol=5e-5)
    assert not bool(torch.isfinite(out[0][0]).all()) and not bool(torch.isfinite(out[0][1]).all())


@pytest.mark.parametrize("act", ["identity", "gelu", "relu"])
@pytest.mark.parametrize("B", [8, 70])
def test_padded_slots_keep_finite_pools_finite(act, B):
    """An infinity or NaN reaches only the pools that have a neuron reading it: padded slots add nothing,
    in the record kernels and in the per-neuron kernels of few tokens."""
    from granulelayer_amd import LevelSpec, PhysicalPlan
    from granulelayer_amd.autograd import Level1Runtime

    D, G, per = 300, 50, 37
    lay = _record_layer(D, per, G)
    rt = Level1Runtime(lay.layout, lay.indices, LevelSpec("mean", activation=act), PhysicalPlan())
    x = torch.randn(B, D, device=DEV)
    x[2, 0], x[5, 0], x[6, 9] = float("nan"), float("inf"), -float("inf")
    idx = lay.indices.view(G, -1)  # every record has a valid neuron
    reads = {d: (idx == d).any(1) for d in (0, 9)}
    assert 0 < int(reads[0].sum()) < G and 0 < int(reads[9].sum()) < G
    finite = torch.isfinite(rt.forward(x, lay.weight.detach(), lay.bias)["pre"])
    assert bool(finite[2][~reads[0]].all()) and bool(finite[5][~reads[0]].all()) and bool(finite[6][~reads[9]].all())
    assert bool(torch.cat([finite[:2], finite[3:5], finite[7:]]).all())
    if act == "identity":
        assert not bool(finite[2][reads[0]].any())
