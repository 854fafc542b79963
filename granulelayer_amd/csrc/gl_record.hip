// Layers whose index records are shared by 16 consecutive slots (Cover-TopK/16: fan-in 16, rec_shift
// 4): sum / mean forward and dW pass on the matrix cores.
//
// The 16 neurons of a record read the same 16 inputs, so per record z = X[:, idx] W^T and dW = dz^T
// X[:, idx] are dense 16 x 16 x tokens products.  v_mfma_f32_16x16x4_f32 computes them in fp32 (fp32
// operands, fp32 accumulation: no operand is rounded) at twice the rate of scalar fp32 FMAs, and
// each gathered value of X serves 16 neurons, where the per-neuron kernels gather it 16 times.
//
// X lies in slices of 64 tokens, [slice][input][64 tokens] fp32: an input of a slice is one 256-byte
// row, and a wave loads the 16 rows of a record with four 1-KiB loads straight into the forward's MFMA
// operands (dW takes them again transposed, through LDS).  A slice of 4096 inputs is 1 MiB, so the
// slices in use stay in an XCD's L2; one of 65,536 is 16 MiB and does not, which costs 20% (4.2M neurons,
// 64 tokens: forward 158 us at 4096 inputs, 189 at 65,536; the per-neuron kernels 351 and 536).
//
// Bounds: at 12.6M neurons, 512 tokens, 4096 inputs the forward runs 2.17 ms and the dW pass 4.85 ms
// (7.47 and 10.5 in the per-neuron kernels; the products alone take 1.31 and 2.62 ms at the 157 TFLOP/s
// of fp32 MFMA).  Counted beside the MFMAs: 61 VALU per record and slice in the forward (0.62 ms of issue),
// 93 in the dW pass (0.95: dz, mask bits, db).  The dW pass with ReLU holds 224 VGPRs (2 waves per SIMD)
// and spills 44 SGPRs to VGPR lanes.  The second layout of X that dW needs (inputs, not
// tokens, across lanes) read again from memory ran 5.70 ms (4.69 then): 16-byte pieces of 64 rows per load, and
// the rows no longer in the 32-KiB L1.  Loads, not LDS, feed the products because a slice of 64
// tokens of a wide layer (1 MiB) fits no LDS, while 4 tokens (what does fit) leave 3/4 of a tile idle.
//
// A wave owns a chunk of 8 records (128 slots of one pool), holds their weights and row offsets in
// registers and walks the slices, so W is read once.  Lane l = 16 G + m; operand maps of
// v_mfma_f32_16x16x4_f32: A row m / k-slot G, B k-slot G / column m, C and D rows 4 G + q / column m.
#include <type_traits>

#include "gl_common.h"
#include "gl_internal.h"

namespace gl {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int REC_N = 16;                      // slots per record
constexpr int REC_PER_WAVE = REC_CHUNK / REC_N;  // 8 records
constexpr int REC_WAVES = 4;                   // waves per workgroup

// X rows [b0, b0 + 64 n_slices) -> slices [n_slices][D][64] fp32 (zero past B): 64 tokens x 32 inputs per
// workgroup through LDS
template <typename XT>
__global__ void __launch_bounds__(256) slice_x_kernel(const XT* __restrict__ X, long long sxb, int B, int D, int b0,
                                                      float* __restrict__ out) {
  __shared__ float tile[32][65];  // [input][token]
  const int d0 = blockIdx.x * 32, t0 = blockIdx.y * 64;
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int t = i >> 5, d = i & 31, b = b0 + t0 + t;
    tile[d][t] = b < B && d0 + d < D ? load_x(X, (long long)b * sxb + d0 + d) : 0.f;
  }
  __syncthreads();
  float* dst = out + (long long)blockIdx.y * D * 64;
  for (int i = threadIdx.x; i < 32 * 64; i += 256) {
    const int d = i >> 6, t = i & 63;
    if (d0 + d < D) dst[(long long)(d0 + d) * 64 + t] = tile[d][t];
  }
}

__device__ __forceinline__ float4 ld_row(__amdgpu_buffer_rsrc_t r, unsigned off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
  return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}
__device__ __forceinline__ float comp(const float4& v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w)); }

// sum over the 4 lanes with the same m (rows of 16 lanes), in every lane
__device__ __forceinline__ float rows_sum(float c) {
  const auto p16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(c), __float_as_uint(c), false, false);
  c = __uint_as_float(p16[0]) + __uint_as_float(p16[1]);
  const auto p32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false, false);
  return __uint_as_float(p32[0]) + __uint_as_float(p32[1]);
}

// Product j of a record takes its edges 4 j + G (k-slot G).  The MFMA adds its 4 k-slots in order,
// each as an fma, so z is the fma chain over k = 0 .. 15 from the bias that the per-neuron kernels
// run, bit for bit: the ReLU decisions are the same (edges 4 G + j, which one 16-byte load per lane
// would give, differ from it in rounding and so in the sign of a few z near 0).  The edges are loaded
// 4 per lane (k = 4 G ..) and exchanged: rec_transpose turns component j of lane (m, G) into component
// G of lane (m, j), a 4 x 4 transpose over the wave's four rows of 16 lanes.
__device__ __forceinline__ uint4 rec_transpose(uint4 v) {
  const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return make_uint4(c[0], c[1], d[0], d[1]);
}
// Orders the wave's LDS accesses on either side, in the compiler as the hardware does by itself: lanes
// exchange data through LDS that only their own wave touches, so no s_barrier is needed.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}
// the lane's weights of neuron m (w: its row + 4 G), zero for a padded slot
__device__ __forceinline__ float4 rec_weights(const float* w, bool valid) {
  uint4 v = *reinterpret_cast<const uint4*>(w);
  if (!valid) v = make_uint4(0u, 0u, 0u, 0u);
  v = rec_transpose(v);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}

// the chunk of a wave: pool g, first slot, valid slots and records
struct RecChunk {
  long long rec0;  // first record (global)
  int g, s_lo, n_g, nrec;
};
__device__ __forceinline__ RecChunk rec_chunk(long long chunk, int cpg, int S, const int32_t* counts) {
  RecChunk c;
  c.g = (int)(chunk / cpg);
  c.s_lo = (int)(chunk % cpg) * REC_CHUNK;
  c.n_g = min(counts[c.g], S);
  c.rec0 = ((long long)c.g * S + c.s_lo) / REC_N;
  const int left = (c.n_g - c.s_lo + REC_N - 1) / REC_N;
  c.nrec = c.n_g <= c.s_lo ? 0 : (left < REC_PER_WAVE ? left : REC_PER_WAVE);
  return c;
}
__device__ __forceinline__ unsigned row_off(int d, int D) { return (unsigned)(d < 0 ? 0 : (d >= D ? D - 1 : d)) * 256u; }

// f(0, a, b), f(1, b, a), ... f(7, b, a) with the record index as a constant, so every per-record array
// stays in registers; a and b hold the current and the next record's rows
template <int R, typename F, typename X>
__device__ __forceinline__ void for_records(F&& f, X& a, X& b) {
  f(std::integral_constant<int, R>{}, a, b);
  if constexpr (R + 1 < REC_PER_WAVE) for_records<R + 1>(f, b, a);
}

struct RecFwdK {
  const float* __restrict__ xs;
  const int32_t* __restrict__ idx;
  const float* __restrict__ W;
  const float* __restrict__ bias;
  const int32_t* __restrict__ counts;
  float* part;  // [n_chunks][b_pad]
  long long n_chunks;
  int D, S, cpg, n_slices, b_pad;
};

// part[chunk][token] = sum of act(z) over the chunk's valid slots.  A = W (rows: neurons), B = X
// (columns: tokens 4 m + i for component i of the loaded float4): D holds neurons 4 G + q of token
// 4 m + i, summed over q and the records in the lane, then over G across the rows.
template <int ACT>
__global__ void __launch_bounds__(REC_WAVES * 64, 2) rec_fwd_kernel(RecFwdK p) {
  const int lane = threadIdx.x & 63, m = lane & 15, G = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long chunk = (long long)blockIdx.x * REC_WAVES + wave;
  if (chunk >= p.n_chunks) return;
  const RecChunk c = rec_chunk(chunk, p.cpg, p.S, p.counts);
  float4 w[REC_PER_WAVE], bias[REC_PER_WAVE];
  unsigned off[REC_PER_WAVE][4];
#pragma unroll
  for (int r = 0; r < REC_PER_WAVE; ++r) {
    const long long rec = c.rec0 + (r < c.nrec ? r : 0);  // in bounds; records past the pool are skipped
    const int left = c.n_g - c.s_lo - r * REC_N;          // valid neurons of the record
    w[r] = rec_weights(p.W + (rec * REC_N + m) * 16 + 4 * G, m < left);
    bias[r] = *reinterpret_cast<const float4*>(p.bias + rec * REC_N + 4 * G);
    const uint4 d = rec_transpose(*reinterpret_cast<const uint4*>(p.idx + rec * 16 + 4 * G));
    off[r][0] = row_off((int)d.x, p.D) + m * 16u, off[r][1] = row_off((int)d.y, p.D) + m * 16u;
    off[r][2] = row_off((int)d.z, p.D) + m * 16u, off[r][3] = row_off((int)d.w, p.D) + m * 16u;
  }
  const int last = c.n_g - c.s_lo - (c.nrec - 1) * REC_N;  // valid neurons of the chunk's last record
  float* out = p.part + chunk * p.b_pad + 4 * m;
  for (int s = 0; s < p.n_slices; ++s) {
    const __amdgpu_buffer_rsrc_t xr = uniform_rsrc(p.xs + (long long)s * p.D * 64);
    float4 xa[4], xb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xa[j] = ld_row(xr, off[0][j]);
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
    auto record = [&](auto rc, const float4(&xc)[4], float4(&xn)[4]) {
      constexpr int r = decltype(rc)::value;
      if (r >= c.nrec) return;
      if constexpr (r + 1 < REC_PER_WAVE) {  // the next record's rows are in flight during this one's products
#pragma unroll
        for (int j = 0; j < 4; ++j) xn[j] = ld_row(xr, off[r + 1][j]);
      }
      const v4f b4 = {bias[r].x, bias[r].y, bias[r].z, bias[r].w};
      v4f z[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          z[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(comp(w[r], j), comp(xc[j], i), j == 0 ? b4 : z[i], 0, 0, 0);
      if (r == c.nrec - 1 && last < REC_N) {  // a partial record: padded slots add nothing
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[i] += 4 * G + q < last ? act_f<ACT>(z[i][q]) : 0.f;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[i] += act_f<ACT>(z[i][q]);
      }
    };
    for_records<0>(record, xa, xb);
    const float4 v = make_float4(rows_sum(sum[0]), rows_sum(sum[1]), rows_sum(sum[2]), rows_sum(sum[3]));
    if (G == 0 && s * 64 + 4 * m < p.b_pad) *reinterpret_cast<float4*>(out + s * 64) = v;  // b_pad % 4 == 0
  }
}

struct RecBwdK {
  const float* __restrict__ xs;
  const int32_t* __restrict__ idx;
  const float* __restrict__ W;
  const float* __restrict__ bias;
  const int32_t* __restrict__ counts;
  const float* __restrict__ c1t;  // [G][cap]
  float* dW;
  float* db;
  uint32_t* mask;  // [n_tc][NS][2T] (bwd_w_kernel's layout)
  long long n_chunks, NS;
  int D, S, cpg, n_slices, cap, T;
};

// z with the operands swapped (A = X: rows are the tokens 4 row + i; B = W: columns are neurons), so
// D holds tokens 16 G + 4 q + i of neuron m.  dz = c1 [z > 0] is then already the B operand of
// dW^T[k][neuron] += sum over tokens X^T[k][token] dz[token][neuron] (k-slot G = token 16 G + 4 q + i),
// whose A operand, input m of the record at those tokens, comes from the same rows through a
// transpose in the wave's own LDS (rows of 68 floats: the reads of 16 rows hit 16 residues).  Per slice
// a lane's 16 mask bits are 16 consecutive tokens of its neuron: one 16-bit store.
constexpr int REC_XROW = 68;
template <int ACT>
__global__ void __launch_bounds__(REC_WAVES * 64, 2) rec_bwd_w_kernel(RecBwdK p) {
  const int lane = threadIdx.x & 63, m = lane & 15, G = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long chunk = (long long)blockIdx.x * REC_WAVES + wave;
  if (chunk >= p.n_chunks) return;
  const RecChunk c = rec_chunk(chunk, p.cpg, p.S, p.counts);
  __shared__ __align__(16) float xls[REC_WAVES][16 * REC_XROW];
  float* const xl = xls[wave];
  float4 w[REC_PER_WAVE];
  float bias[REC_PER_WAVE], dbv[REC_PER_WAVE];
  unsigned off[REC_PER_WAVE][4];
  v4f dw[REC_PER_WAVE];
#pragma unroll
  for (int r = 0; r < REC_PER_WAVE; ++r) {
    const long long rec = c.rec0 + (r < c.nrec ? r : 0);
    const int left = c.n_g - c.s_lo - r * REC_N;
    w[r] = rec_weights(p.W + (rec * REC_N + m) * 16 + 4 * G, m < left);
    bias[r] = m < left ? p.bias[rec * REC_N + m] : 0.f;
    const uint4 d = rec_transpose(*reinterpret_cast<const uint4*>(p.idx + rec * 16 + 4 * G));
    off[r][0] = row_off((int)d.x, p.D) + m * 16u, off[r][1] = row_off((int)d.y, p.D) + m * 16u;
    off[r][2] = row_off((int)d.z, p.D) + m * 16u, off[r][3] = row_off((int)d.w, p.D) + m * 16u;
    dw[r] = v4f{0.f, 0.f, 0.f, 0.f};
    dbv[r] = 0.f;
  }
  const float* c1row = p.c1t + (long long)c.g * p.cap + 16 * G;
  for (int s = 0; s < p.n_slices; ++s) {
    const __amdgpu_buffer_rsrc_t xr = uniform_rsrc(p.xs + (long long)s * p.D * 64);
    float4 xa[4], xb[4], c1[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xa[j] = ld_row(xr, off[0][j]);
#pragma unroll
    for (int q = 0; q < 4; ++q) c1[q] = *reinterpret_cast<const float4*>(c1row + s * 64 + 4 * q);
    char* mrow = reinterpret_cast<char*>(p.mask) +
                 ((long long)(s / p.T) * p.NS + c.rec0 * REC_N + m) * (8 * p.T) + (s % p.T) * 8 + 2 * G;
    auto record = [&](auto rc, const float4(&xc)[4], float4(&xn)[4]) {
      constexpr int r = decltype(rc)::value;
      if (r >= c.nrec) return;
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<float4*>(&xl[(4 * j + G) * REC_XROW + 4 * m]) = xc[j];
      wave_lds_fence();  // the reads below take rows that other lanes wrote
      if constexpr (r + 1 < REC_PER_WAVE) {
#pragma unroll
        for (int j = 0; j < 4; ++j) xn[j] = ld_row(xr, off[r + 1][j]);
      }
      v4f z[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) z[i] = v4f{bias[r], bias[r], bias[r], bias[r]};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          z[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(comp(xc[j], i), comp(w[r], j), z[i], 0, 0, 0);
      const bool valid = m < c.n_g - c.s_lo - r * REC_N;
      unsigned bits = 0u;
      float4 xt[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) xt[q] = *reinterpret_cast<const float4*>(&xl[m * REC_XROW + 16 * G + 4 * q]);
      wave_lds_fence();  // the next record's rows overwrite them
      float dz[4][4], ds = 0.f;  // [q][i]
#pragma unroll
      for (int q = 3; q >= 0; --q)
#pragma unroll
        for (int i = 3; i >= 0; --i) {
          const bool on = ACT == GL_ACT_RELU ? z[i][q] > 0.f : valid;
          dz[q][i] = on ? comp(c1[q], i) : 0.f;
          bits = bits << 1 | (unsigned)on;
        }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          ds += dz[q][i];
          dw[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(comp(xt[q], i), dz[q][i], dw[r], 0, 0, 0);
        }
      dbv[r] += ds;
      if (valid) *reinterpret_cast<uint16_t*>(mrow + (long long)r * REC_N * (8 * p.T)) = (uint16_t)bits;
    };
    for_records<0>(record, xa, xb);
  }
#pragma unroll
  for (int r = 0; r < REC_PER_WAVE; ++r) {
    const float d = rows_sum(dbv[r]);
    if (r < c.nrec && m < c.n_g - c.s_lo - r * REC_N) {
      const long long n = (c.rec0 + r) * REC_N + m;
      float4* o = reinterpret_cast<float4*>(p.dW + n * 16 + 4 * G);
      const float4 v = *o;
      *o = make_float4(v.x + dw[r][0], v.y + dw[r][1], v.z + dw[r][2], v.w + dw[r][3]);
      if (G == 0) p.db[n] += d;
    }
  }
}

// ---- host side ---------------------------------------------------------------------------------
bool record_layer(int K, int rec_shift, int pool, int w_dtype) {
  return K == 16 && rec_shift == 4 && (pool == GL_POOL_SUM || pool == GL_POOL_MEAN) && w_dtype == GL_DTYPE_F32;
}

int launch_slice_x(const void* X, long long sxb, int x_dtype, int B, int D, int b0, int n_slices, float* xs,
                   hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(D, 32), (unsigned)n_slices);
  if (x_dtype == GL_DTYPE_F32)
    GL_LAUNCH(GL_KERNEL_TILE_X, slice_x_kernel<float>, grid, dim3(256), 0, s, (const float*)X, sxb, B, D, b0, xs);
  else
    GL_LAUNCH(GL_KERNEL_TILE_X, slice_x_kernel<__hip_bfloat16>, grid, dim3(256), 0, s, (const __hip_bfloat16*)X, sxb, B,
              D, b0, xs);
  GL_CHECK_LAUNCH();
  return 0;
}

int launch_rec_fwd(int act, const float* xs, const int32_t* idx, const float* W, const float* bias, const int32_t* counts,
                   float* part, long long n_chunks, int D, int S, int cpg, int b_pad, hipStream_t s) {
  const RecFwdK k{xs, idx, W, bias, counts, part, n_chunks, D, S, cpg, ceil_div(b_pad, 64), b_pad};
  auto fn = act == GL_ACT_RELU ? rec_fwd_kernel<GL_ACT_RELU>
                               : (act == GL_ACT_GELU ? rec_fwd_kernel<GL_ACT_GELU> : rec_fwd_kernel<GL_ACT_IDENTITY>);
  GL_LAUNCH(GL_KERNEL_FWD, fn, dim3((unsigned)ceil_div(n_chunks, REC_WAVES)), dim3(REC_WAVES * 64), 0, s, k);
  GL_CHECK_LAUNCH();
  return 0;
}

int launch_rec_bwd_w(int act, const float* xs, const int32_t* idx, const float* W, const float* bias,
                     const int32_t* counts, const float* c1t, float* dW, float* db, uint32_t* mask, int D, int G, int S,
                     int cap, int Bc, int T, hipStream_t s) {
  const int cpg = ceil_div(S, REC_CHUNK);
  const RecBwdK k{xs, idx, W, bias, counts, c1t, dW, db, mask, (long long)G * cpg, (long long)G * S,
                  D, S, cpg, ceil_div(Bc, 64), cap, T};
  auto fn = act == GL_ACT_RELU ? rec_bwd_w_kernel<GL_ACT_RELU> : rec_bwd_w_kernel<GL_ACT_IDENTITY>;
  GL_LAUNCH(GL_KERNEL_BWD_W, fn, dim3((unsigned)ceil_div(k.n_chunks, REC_WAVES)), dim3(REC_WAVES * 64), 0, s, k);
  GL_CHECK_LAUNCH();
  return 0;
}

}  // namespace gl
