// sta_dca_dec.hip -- DCA (dual chunk attention) at decode, and the rotation of new keys into the
// KV cache.
//
// Reference: the decode branch of dca_forward (dca_kernel.py:491-522).  The cache holds keys
// already rotated at j mod L (:434-435); the new token's query at cur = M - 1 is rotated three
// ways (intra at cur mod L, succ at min(cur mod L + L, s), inter at min(2L - 1, s)) and scores
// the keys [0, inter_end) inter, [inter_end, chunk_start) succ and [chunk_start, M) intra, with
// chunk_start = floor(cur / L) L and inter_end = max(0, chunk_start - L).  The reference does
// this with model-dtype matmuls and one fp32 softmax:
//   s_j = rnd(rnd(q_var . k_j) * scale)     (matmul output and the scaled scores in the dtype)
//   p_j = rnd(exp(s_j - max s) / sum exp)   (softmax in fp32, cast back to the dtype)
//   out = rnd(sum_j p_j v_j)                (matmul output in the dtype)
// rnd = rounding to the model dtype (identity for fp32); dot products and sums accumulate in
// fp32.  These kernels keep every one of those roundings.
//
// Launches: the scores (one workgroup = one kv head x 256 keys, all heads of the group; scores
// plus each block's max and sum of exp), dca_dec_pv_kernel (one workgroup = one kv head x 256
// keys, a few heads of the group: global max and sum from the block partials, weights, partial
// P.V), and dca_dec_combine_kernel (sum of the partials, rounded to the dtype).  16-bit caches
// take dca_dec_score16_kernel, which rotates the queries itself and scores on the matrix cores;
// fp32 caches take dca_dec_qrot_kernel (the three query variants of every head) and
// dca_dec_score_kernel (one key per thread, the query's products in order).
#include "sta_dca_rot.h"
#include "sta_device.h"
#include "sta_kernels.h"

namespace sta {

constexpr int DCA_DEC_BK = 256;      // keys per score / P.V workgroup
constexpr int DCA_DEC_GMAX = 16;     // heads per kv head

template <int DT>
__device__ __forceinline__ void store8(void* p, int64_t i, const float* o) {
  if constexpr (DT == DT_F32) {
    float4* q = (float4*)((float*)p + i);
    q[0] = make_float4(o[0], o[1], o[2], o[3]);
    q[1] = make_float4(o[4], o[5], o[6], o[7]);
  } else if constexpr (DT == DT_F16) {
    *(u32x4*)((uint16_t*)p + i) = pack_f16x8(o);
  } else {
    *(u32x4*)((uint16_t*)p + i) = pack_bf16x8(o);
  }
}

// ------------------------------------------------------------------------------------------
// keys of the new tokens at positions pos0 .. pos0 + N - 1, rotated at (pos mod L) into out
// (dca_kernel.py:434-435 with the cyclic key table :187-190); one thread per 8 elements
// ------------------------------------------------------------------------------------------
template <int DT, int D>
__global__ __launch_bounds__(256) void dca_rotate_keys_kernel(DcaRotArgs a) {
  constexpr int C = D / 8;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (int64_t)a.heads * a.N * C) return;
  const int c = (int)(gid % C);
  const int64_t r = gid / C;
  const int row = (int)(r % a.N);
  const int head = (int)(r / a.N);
  const int d0 = c * 8;
  const bool first = d0 < D / 2;
  const int i0 = first ? d0 : d0 - D / 2;
  float x1[8], x2[8], o[8];
  const int64_t base = (int64_t)head * a.x_head_stride + (int64_t)row * a.x_tok_stride;
  load8<DT>(a.x, base + i0, x1);
  load8<DT>(a.x, base + D / 2 + i0, x2);
  dca_rot8<DT>(x1, x2, (int)(((int64_t)a.pos0 + row) % a.L), i0, first, a.inv_freq, a.mscale, o);
  store8<DT>(a.out, (int64_t)head * a.out_head_stride + (int64_t)row * a.out_tok_stride + d0, o);
}

// ------------------------------------------------------------------------------------------
// the query's three variants (dca_kernel.py:497-517): qrot (H, 3, D) fp32 holding dtype values
// ------------------------------------------------------------------------------------------
template <int DT, int D>
__global__ __launch_bounds__(64) void dca_dec_qrot_kernel(DcaDecArgs a) {
  constexpr int C = D / 8;
  const int h = blockIdx.x;
  const int tid = threadIdx.x;
  if (tid >= 3 * C) return;
  const int var = tid / C;
  const int d0 = (tid % C) * 8;
  const int cur = a.M - 1;
  const int pid = cur % a.L;
  const int t = var == 0 ? pid : (var == 1 ? min(pid + a.L, a.chunk_size) : min(2 * a.L - 1, a.chunk_size));
  const bool first = d0 < D / 2;
  const int i0 = first ? d0 : d0 - D / 2;
  float x1[8], x2[8], o[8];
  const int64_t base = (int64_t)h * a.q_head_stride;
  load8<DT>(a.q, base + i0, x1);
  load8<DT>(a.q, base + D / 2 + i0, x2);
  dca_rot8<DT>(x1, x2, t, i0, first, a.inv_freq, a.mscale, o);
  float* dst = a.qrot + ((int64_t)h * 3 + var) * D + d0;
#pragma unroll
  for (int e = 0; e < 8; ++e) dst[e] = o[e];
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// ------------------------------------------------------------------------------------------
// scores of the keys [256 b, 256 b + 256) for every head of kv head g
// ------------------------------------------------------------------------------------------
template <int DT, int D>
__global__ __launch_bounds__(DCA_DEC_BK) void dca_dec_score_kernel(DcaDecArgs a) {
#pragma clang fp contract(off)
  __shared__ float qs[DCA_DEC_GMAX * 3 * D];
  __shared__ float red[DCA_DEC_GMAX][DCA_DEC_BK / 64];
  const int g = blockIdx.x;
  const int blk = blockIdx.y;
  const int tid = threadIdx.x;
  const int G = a.H / a.Hkv;
  for (int i = tid; i < G * 3 * D; i += DCA_DEC_BK) qs[i] = a.qrot[(int64_t)g * G * 3 * D + i];
  __syncthreads();
  const int cur = a.M - 1;
  const int chunk_start = (cur / a.L) * a.L;
  const int inter_end = max(0, chunk_start - a.L);
  const int j = blk * DCA_DEC_BK + tid;
  const bool live = j < a.M;
  // the query variant this key is scored with (:513-517, cache order inter | succ | intra)
  const int var = j < inter_end ? 2 : (j < chunk_start ? 1 : 0);
  float acc[DCA_DEC_GMAX];
#pragma unroll
  for (int u = 0; u < DCA_DEC_GMAX; ++u) acc[u] = 0.0f;
  if (live) {
    const int64_t kb = (int64_t)g * a.k_head_stride + (int64_t)j * a.k_tok_stride;
    for (int d0 = 0; d0 < D; d0 += 8) {
      float kv[8];
      load8<DT>(a.k, kb + d0, kv);
#pragma unroll
      for (int u = 0; u < DCA_DEC_GMAX; ++u) {
        if (u < G) {
          const float* qq = qs + (u * 3 + var) * D + d0;
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[u] = acc[u] + qq[e] * kv[e];
        }
      }
    }
  }
  const int lane = tid & 63, wid = tid >> 6;
  float sv[DCA_DEC_GMAX];
#pragma unroll
  for (int u = 0; u < DCA_DEC_GMAX; ++u) {
    if (u < G) {
      sv[u] = live ? round_dt<DT>(opaque_f32(round_dt<DT>(acc[u]) * a.scale)) : -INFINITY;
      if (live) a.scores[(int64_t)(g * G + u) * a.M + j] = sv[u];
      const float m = wave_max(sv[u]);
      if (lane == 0) red[u][wid] = m;
    }
  }
  __syncthreads();
  float bmax[DCA_DEC_GMAX];
#pragma unroll
  for (int u = 0; u < DCA_DEC_GMAX; ++u) {
    if (u < G) {
      float m = red[u][0];
      for (int w = 1; w < DCA_DEC_BK / 64; ++w) m = fmaxf(m, red[u][w]);
      bmax[u] = m;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < DCA_DEC_GMAX; ++u) {
    if (u < G) {
      const float e = live ? expf(sv[u] - bmax[u]) : 0.0f;
      const float s = wave_sum(e);
      if (lane == 0) red[u][wid] = s;
    }
  }
  __syncthreads();
  if (tid < G) {
    float s = 0.0f;
    for (int w = 0; w < DCA_DEC_BK / 64; ++w) s += red[tid][w];
    float m = bmax[0];
#pragma unroll
    for (int u = 0; u < DCA_DEC_GMAX; ++u)
      if (u == tid) m = bmax[u];
    const int64_t o = (int64_t)(g * G + tid) * a.nb + blk;
    a.pmax[o] = m;
    a.psum[o] = s;
  }
}

// ------------------------------------------------------------------------------------------
// scores of the keys [256 b, 256 b + 256) of a 16-bit cache for every head of kv head g.
//
// HBM-bound: the kernel reads every key row once.  Each wave takes 64 keys as four 16-row A
// operands of v_mfma_f32_16x16x32, loaded straight from the cache (a lane's 16 bytes are its 8
// contraction elements, a row's 256 bytes arrive in four 64-byte pieces), all requested before
// anything else.  The B columns are the queries of the group in their three variants, column
// var * G + u, so a key meets every variant and keeps its own: the chunk boundaries need not fall
// on tile edges.  While the keys are in flight the workgroup builds the three rows of table
// entries (one sincos a thread) and rotates its queries into LDS.  Products of 16-bit values are
// exact in fp32; only the order of the fp32 sum differs from the one-thread-per-key dot.
// 65535 keys, 32 query / 8 kv heads, D 128, bf16: 28.6 us, 4.7 TB/s (one thread a key, its row in
// strided 16-byte pieces: 143 us and a 6 us launch for the query rotation).
// ------------------------------------------------------------------------------------------
template <int DT, int D, int NC>
__global__ __launch_bounds__(DCA_DEC_BK) void dca_dec_score16_kernel(DcaDecArgs a) {
#pragma clang fp contract(off)
  constexpr int KS = D / 32;                   // contraction steps
  constexpr int QSTR = D + 8;                  // query row stride: 16 lanes' reads spread over the banks
  constexpr int W = DCA_DEC_BK / 64;
  __shared__ float2 tab[3][D / 2];
  __shared__ __align__(16) uint16_t qs[NC * 16 * QSTR];
  __shared__ float sS[DCA_DEC_GMAX][DCA_DEC_BK];
  __shared__ float redm[DCA_DEC_GMAX][W], reds[DCA_DEC_GMAX][W];
  const int g = blockIdx.x;
  const int blk = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int G = a.H / a.Hkv;
  const int r16 = lane & 15, c4 = lane >> 4;

  // this wave's keys; rows past the cache's end repeat its last row and are masked below
  u32x4 kf[4][KS];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int j = min(blk * DCA_DEC_BK + wid * 64 + t * 16 + r16, a.M - 1);
    const uint16_t* kr = (const uint16_t*)a.k + (int64_t)g * a.k_head_stride + (int64_t)j * a.k_tok_stride + 8 * c4;
#pragma unroll
    for (int s = 0; s < KS; ++s) kf[t][s] = *(const u32x4*)(kr + 32 * s);
  }

  const int cur = a.M - 1;
  const int chunk_start = (cur / a.L) * a.L;
  const int inter_end = max(0, chunk_start - a.L);
  const int pid = cur % a.L;
  for (int i = tid; i < 3 * (D / 2); i += DCA_DEC_BK) {
    const int var = i / (D / 2), f = i % (D / 2);
    const int t = var == 0 ? pid : (var == 1 ? min(pid + a.L, a.chunk_size) : min(2 * a.L - 1, a.chunk_size));
    float cs, sn;
    dca_table_entry<DT>(t, a.inv_freq[f], a.mscale, cs, sn);
    tab[var][f] = make_float2(cs, sn);
  }
  for (int i = 3 * G * QSTR + tid; i < NC * 16 * QSTR; i += DCA_DEC_BK) qs[i] = 0;   // unused columns
  __syncthreads();
  for (int i = tid; i < 3 * G * (D / 8); i += DCA_DEC_BK) {
    const int col = i / (D / 8), d0 = (i % (D / 8)) * 8;
    const int var = col / G, u = col % G;
    const bool first = d0 < D / 2;
    const int i0 = first ? d0 : d0 - D / 2;
    float x1[8], x2[8], cs[8], sn[8], o[8];
    const int64_t base = (int64_t)(g * G + u) * a.q_head_stride;
    load8<DT>(a.q, base + i0, x1);
    load8<DT>(a.q, base + D / 2 + i0, x2);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float2 t = tab[var][i0 + e];
      cs[e] = t.x;
      sn[e] = t.y;
    }
    dca_rot8_cs<DT>(x1, x2, cs, sn, first, o);
    *(u32x4*)(qs + col * QSTR + d0) = DT == DT_F16 ? pack_f16x8(o) : pack_bf16x8(o);
  }
  __syncthreads();

#pragma unroll
  for (int n = 0; n < NC; ++n) {
    const int col = n * 16 + r16;
    const int var = col / G, u = col % G;      // var >= 3: an unused column
    u32x4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *(const u32x4*)(qs + col * QSTR + 32 * s + 8 * c4);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        acc = DT == DT_F16 ? mfma16_f16(kf[t][s], qf[s], acc) : mfma16(kf[t][s], qf[s], acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = wid * 64 + t * 16 + 4 * c4 + i;
        const int j = blk * DCA_DEC_BK + key;
        if (var == (j < inter_end ? 2 : (j < chunk_start ? 1 : 0)))
          sS[u][key] = j < a.M ? round_dt<DT>(opaque_f32(round_dt<DT>(acc[i]) * a.scale)) : -INFINITY;
      }
    }
  }
  __syncthreads();
  // the block's max and sum of exp(s - max) of each head; the scores go out coalesced
  const int j = blk * DCA_DEC_BK + tid;
  for (int u = 0; u < G; ++u) {
    const float s = sS[u][tid];
    if (j < a.M) a.scores[(int64_t)(g * G + u) * a.M + j] = s;
    const float m = wave_max_f32(s);
    if (lane == 0) redm[u][wid] = m;
  }
  __syncthreads();
  for (int u = 0; u < G; ++u) {
    float m = redm[u][0];
    for (int w = 1; w < W; ++w) m = fmaxf(m, redm[u][w]);
    const float s = wave_sum(j < a.M ? expf(sS[u][tid] - m) : 0.0f);
    if (lane == 0) reds[u][wid] = s;
  }
  __syncthreads();
  if (tid < G) {
    float m = redm[tid][0], s = reds[tid][0];
    for (int w = 1; w < W; ++w) {
      m = fmaxf(m, redm[tid][w]);
      s += reds[tid][w];
    }
    const int64_t o = (int64_t)(g * G + tid) * a.nb + blk;
    a.pmax[o] = m;
    a.psum[o] = s;
  }
}

// ------------------------------------------------------------------------------------------
// softmax weights and partial P.V of GP heads of kv head g (the last workgroup of a group: those
// left) over the keys [256 b, 256 b + 256).
//
// HBM-bound: every value row is read once for GP heads, D / 8 lanes a row in 16-byte pieces.  The first PF rows of a lane are requested
// before the block partials are reduced and the weights taken, so they arrive meanwhile.  65535
// keys, 32 query / 8 kv heads, D 128, bf16: 29.5 us, 4.6 TB/s (one workgroup a query head with
// 2-byte loads: 220 us); a call 60.8 us, with all 16 rows of a lane in flight 72.6 at two workgroups
// a CU, and 197 at four, where they spill.
// ------------------------------------------------------------------------------------------
template <int DT, int D, int GP>
__global__ __launch_bounds__(DCA_DEC_BK, DT != DT_F32 ? 4 : 1) void dca_dec_pv_kernel(DcaDecArgs a) {
#pragma clang fp contract(off)
  constexpr int LPR = D / 8;                   // lanes per row
  constexpr int RPS = DCA_DEC_BK / LPR;        // rows per step of the workgroup
  constexpr int STEPS = DCA_DEC_BK / RPS;
  constexpr int PF = 8;                        // rows in flight per lane: four workgroups fit a CU
  constexpr int W = DCA_DEC_BK / 64;
  __shared__ __align__(16) float pS[DCA_DEC_BK * GP];
  __shared__ float gm[GP], gl[GP];
  __shared__ float red[W][GP][D];
  const int g = blockIdx.x;
  const int blk = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int G = a.H / a.Hkv;
  const int h0 = g * G + blockIdx.z * GP;      // this workgroup's heads: [h0, h0 + nh)
  const int nh = min(GP, G - (int)blockIdx.z * GP);
  const int c = tid % LPR, row = tid / LPR;
  const int64_t vb = (int64_t)g * a.v_head_stride + 8 * c;
  Raw8<DT> v[PF];
  auto fetch = [&](int s0) {
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      const int jv = min(blk * DCA_DEC_BK + (s0 + s) * RPS + row, a.M - 1);
      v[s].load(a.v, vb + (int64_t)jv * a.v_tok_stride);
    }
  };
  fetch(0);
  const int j = blk * DCA_DEC_BK + tid;
  float sc[GP];
#pragma unroll
  for (int u = 0; u < GP; ++u) sc[u] = u < nh && j < a.M ? a.scores[(int64_t)(h0 + u) * a.M + j] : 0.0f;
  // the global max and the sum of exp(s - max) of each head from the blocks' partials, a wave a head
  for (int u = wid; u < nh; u += W) {
    const float* pm = a.pmax + (int64_t)(h0 + u) * a.nb;
    const float* ps = a.psum + (int64_t)(h0 + u) * a.nb;
    constexpr int R = 4;                       // partials a lane holds: 256 blocks, 65536 keys
    float pr[R], sr[R], m = -INFINITY;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int b = r * 64 + lane;
      pr[r] = b < a.nb ? pm[b] : -INFINITY;
      sr[r] = b < a.nb ? ps[b] : 0.0f;
      m = fmaxf(m, pr[r]);
    }
    for (int b = R * 64 + lane; b < a.nb; b += 64) m = fmaxf(m, pm[b]);
    m = wave_max_f32(m);
    float l = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r * 64 + lane < a.nb) l += sr[r] * expf(pr[r] - m);
    for (int b = R * 64 + lane; b < a.nb; b += 64) l += ps[b] * expf(pm[b] - m);
    l = wave_sum(l);
    if (lane == 0) {
      gm[u] = m;
      gl[u] = l;
    }
  }
  __syncthreads();
  // the weights, cast to the dtype as the reference's .to(q.dtype) does (:521)
#pragma unroll
  for (int u = 0; u < GP; ++u) {
    float p = 0.0f;
    if (u < nh && j < a.M) p = round_dt<DT>(opaque_f32(expf(sc[u] - gm[u]) / gl[u]));
    pS[tid * GP + u] = p;
  }
  __syncthreads();
  float acc[GP][8];
#pragma unroll
  for (int u = 0; u < GP; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[u][e] = 0.0f;
#pragma unroll 1
  for (int s0 = 0; s0 < STEPS; s0 += PF) {
    if (s0 > 0) fetch(s0);
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      float x[8];
      if (blk * DCA_DEC_BK + (s0 + s) * RPS + row >= a.M) v[s].zero();   // 0 * inf past the end
      v[s].to_f32(x);
      const float* p = pS + ((s0 + s) * RPS + row) * GP;
#pragma unroll
      for (int u = 0; u < GP; ++u) {
        const float w = p[u];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[u][e] = fmaf(w, x[e], acc[u][e]);
      }
    }
  }
#pragma unroll
  for (int u = 0; u < GP; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float x = acc[u][e];
#pragma unroll
      for (int o = LPR; o < 64; o <<= 1) x += __shfl_xor(x, o);
      if (lane < LPR) red[wid][u][8 * c + e] = x;
    }
  __syncthreads();
  for (int i = tid; i < nh * D; i += DCA_DEC_BK) {
    const int u = i / D, d = i % D;
    float s = red[0][u][d];
#pragma unroll
    for (int w = 1; w < W; ++w) s += red[w][u][d];
    a.part[((int64_t)(h0 + u) * a.nb + blk) * D + d] = s;
  }
}

// sum of the blocks' partials: one workgroup a head and 32 dims, 16 strided segments of the blocks
// (256 blocks, 32 heads: 4.7 us; one thread a dim walking every block: 61 us)
template <int DT, int D>
__global__ __launch_bounds__(512) void dca_dec_combine_kernel(DcaDecArgs a) {
#pragma clang fp contract(off)
  __shared__ float red[16][32];
  const int h = blockIdx.x;
  const int d = blockIdx.y * 32 + (threadIdx.x & 31), seg = threadIdx.x >> 5;
  float s = 0.0f;
#pragma unroll 8
  for (int b = seg; b < a.nb; b += 16) s += a.part[((int64_t)h * a.nb + b) * D + d];
  red[seg][threadIdx.x & 31] = s;
  __syncthreads();
  if (seg != 0) return;
  s = 0.0f;
#pragma unroll
  for (int u = 0; u < 16; ++u) s += red[u][threadIdx.x];
  const int64_t oi = (int64_t)h * D + d;
  if constexpr (DT == DT_F32) ((float*)a.out)[oi] = s;
  else ((uint16_t*)a.out)[oi] = (uint16_t)(DT == DT_BF16 ? f32_to_bf16_bits(s) : f32_to_f16_bits(s));
}

// ------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------
template <int DT, int D>
static hipError_t launch_dca_rotate_keys_t(const DcaRotArgs& a, hipStream_t st) {
  const int64_t total = (int64_t)a.heads * a.N * (D / 8);
  hipLaunchKernelGGL((dca_rotate_keys_kernel<DT, D>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_dca_rotate_keys(int dtype, int D, const DcaRotArgs& a, hipStream_t st) {
#define STA_DK(DT_, D_) if (dtype == DT_ && D == D_) return launch_dca_rotate_keys_t<DT_, D_>(a, st);
  STA_DK(DT_F32, 64) STA_DK(DT_F32, 128) STA_DK(DT_BF16, 64) STA_DK(DT_BF16, 128)
  STA_DK(DT_F16, 64) STA_DK(DT_F16, 128)
#undef STA_DK
  return hipErrorInvalidValue;
}

int dca_dec_nblocks(int M) { return (M + DCA_DEC_BK - 1) / DCA_DEC_BK; }
int dca_dec_max_group() { return DCA_DEC_GMAX; }

// 3 G query variants in 16-column operands
template <int DT, int D>
static hipError_t launch_dca_scores_t(const DcaDecArgs& a, hipStream_t st) {
  const dim3 grid(a.Hkv, a.nb);
  if constexpr (DT == DT_F32) {
    hipLaunchKernelGGL((dca_dec_qrot_kernel<DT, D>), dim3(a.H), dim3(64), 0, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((dca_dec_score_kernel<DT, D>), grid, dim3(DCA_DEC_BK), 0, st, a);
  } else {
    const int nc = (3 * (a.H / a.Hkv) + 15) / 16;
    if (nc == 1) hipLaunchKernelGGL((dca_dec_score16_kernel<DT, D, 1>), grid, dim3(DCA_DEC_BK), 0, st, a);
    else if (nc == 2) hipLaunchKernelGGL((dca_dec_score16_kernel<DT, D, 2>), grid, dim3(DCA_DEC_BK), 0, st, a);
    else hipLaunchKernelGGL((dca_dec_score16_kernel<DT, D, 3>), grid, dim3(DCA_DEC_BK), 0, st, a);
  }
  return hipGetLastError();
}

template <int DT, int D>
static hipError_t launch_dca_decode_t(const DcaDecArgs& a, hipStream_t st) {
  hipError_t e = launch_dca_scores_t<DT, D>(a, st);
  if (e != hipSuccess) return e;
  const int G = a.H / a.Hkv;
  // Heads per P.V workgroup: four read a value row's bytes once and stay short; more unrolled code
  // costs a small call its fetch.  fp32, one head a workgroup below 1024 of them (16 heads / 1 kv head
  // x 100, D 64: 36.4 us a call, four 39.6, all sixteen 54.1), eight at D 128 from 4096 (32 / 4 x
  // 65535: 92 us, four 104; 16-bit 52.6 and 50.5).
  const int64_t wgs = (int64_t)a.H * a.nb;
  int gp = 4;
  if (DT == DT_F32) gp = wgs < 1024 ? 1 : (D == 128 && wgs >= 4096 ? 8 : 4);
#define STA_PV(GP_) hipLaunchKernelGGL((dca_dec_pv_kernel<DT, D, GP_>), dim3(a.Hkv, a.nb, (G + GP_ - 1) / GP_), dim3(DCA_DEC_BK), 0, st, a)
  if (gp == 1 || G == 1) STA_PV(1);
  else if (G == 2) STA_PV(2);
  else if (gp == 4 || G <= 4) STA_PV(4);
  else if constexpr (DT == DT_F32 && D == 128) STA_PV(8);
#undef STA_PV
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL((dca_dec_combine_kernel<DT, D>), dim3(a.H, D / 32), dim3(512), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_dca_decode(int dtype, int D, const DcaDecArgs& a, hipStream_t st) {
#define STA_DD(DT_, D_) if (dtype == DT_ && D == D_) return launch_dca_decode_t<DT_, D_>(a, st);
  STA_DD(DT_F32, 64) STA_DD(DT_F32, 128) STA_DD(DT_BF16, 64) STA_DD(DT_BF16, 128)
  STA_DD(DT_F16, 64) STA_DD(DT_F16, 128)
#undef STA_DD
  return hipErrorInvalidValue;
}

}  // namespace sta
