// Dense server score of the approximate pass: the mean attention probability each key receives, over
// heads and all queries (patch_attn_prob / patch_attn_prob_layermean).
//
// Nothing of size N x N is materialised:
//   stats:  for every (image, head, query) the softmax max m and sum l over all keys, in one pass over
//           the keys with a running max;
//   colsum: dense mode, for every (image, 128-query block, 128-key block) the column sums over its
//           queries of the head-mean probabilities, then the query blocks added in order; log-sum-exp
//           mode, one pass per (256-key block, head group, image) from the row LSE (the stats launch's,
//           or the attention's own), then the head groups added in order.
//
// Rounding modes (the two paths of attention.py:241-253 and triton_kernels/attention_pscore.py):
//   kDense: s = bf16(bf16(q.k) * scale), p = bf16(exp(s - m) / l) (torch softmax of a bf16 tensor;
//           formed as exp2((s - m) log2 e) times 1 / l, max and sum held apart in fp32),
//           head mean hm = bf16(sum_h p * fl(1/H)), score = bf16(sum_q hm * fl(1/N));
//   kLse:   s = (q.k) in fp32, lse = m + log(l), p = exp2(s * (scale log2e) - lse * log2e) in fp32,
//           score = bf16(sum_{q,h} p * fl(1/(H N))) -- the fused kernel's key-side sum from the row
//           log-sum-exp.
// q.k is one v_mfma_f32_32x32x16_bf16 chain (fp32 accumulation). Stats use S^T = K . Q^T so a query's
// scores sit in one lane pair (lanes l, l ^ 32); colsum uses S = Q . K^T so a key's column sits in one
// lane pair and the sum over queries is a register sum plus one exchange.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "common.hpp"

namespace oudjat {

enum { kDense = 0, kLse = 1 };

// A 16-byte operand fragment of row `row` (< rows, else zeros) at head-dim offset `d0`.
__device__ __forceinline__ bf16x8_t frag16(const uint16_t* base, int64_t row_stride, int row, int rows, int d0) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (row < rows) v = *reinterpret_cast<const uint4*>(base + (int64_t)row * row_stride + d0);
  return as_bf16x8(v);
}

// Two values rounded to bf16 (nearest even) and back to fp32 with one hardware convert.
__device__ __forceinline__ void round2_bf16(float& a, float& b) {
  typedef float f32x2v_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2v_t __attribute__((ext_vector_type(2)));
  const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v_t){a, b}, bf16x2v_t));
  a = __uint_as_float(p << 16);
  b = __uint_as_float(p & 0xffff0000u);
}

static constexpr float kLog2e = 1.4426950408889634f;

// How a kernel forms its scores from the fp32 products a = q.k (0 < scale <= 1/2 for kDenseP2):
//   kDense     s = bf16(bf16(a) * scale)
//   kDenseP2   the same for a power-of-two scale, whose second rounding changes nothing: the kernel keeps
//              v = bf16(a) and the scale moves into the exponent's factor
//   kLse       s = a * scale
// In all of them exp(s - m) = exp2((v - m) * kf) with v and m in the kernel's own units and kf = score_factor;
// `row_exp` takes it relative to the row's reference r (`row_ref`):
//   kDense, kLse  r = m: a subtraction, exact for scores near m, and a product;
//   kDenseP2      r = fl(m kf): one FMA, exp2(v kf - r), whose missing factor exp2(r - m kf), the same for every
//                 score of the row, multiplies the sum or the probabilities' 1 / l (`ref_error`). m kf must not
//                 overflow: kf <= 1 (scale <= 1/2), while kDense's kf = log2 e would from m = 2.4e38 on.
// So the exponent is rounded relative to itself and not to the row's maximum: p is off by 2e-7 (rms, before its
// bf16 rounding; 9e-7 at most) at row maxima of 1 to 16000. With m kf + log2 l folded into one float it
// was 6e-7 at a maximum of 4, 2.6e-5 at 1000 and 3e-4 at 16000. That form took 216 us for 16 x 16 heads x
// 1029^2 at scale 1/8 where this one takes 225, and 249 against 267 at scale 0.1 (kDense).
static constexpr int kDenseP2 = 2;

__host__ __device__ __forceinline__ float score_factor(int form, float scale) {
  return form == kDenseP2 ? scale * kLog2e : kLog2e;
}

template <int FORM>
__device__ __forceinline__ float row_ref(float m, float kf) {
  return FORM == kDenseP2 ? m * kf : m;
}
template <int FORM>
__device__ __forceinline__ float ref_error(float m, float kf) {
  return FORM == kDenseP2 ? __builtin_amdgcn_exp2f(-fmaf(m, kf, -m * kf)) : 1.0f;
}
template <int FORM>
__device__ __forceinline__ float row_exp(float v, float r, float kf) {
  return __builtin_amdgcn_exp2f(FORM == kDenseP2 ? fmaf(v, kf, -r) : (v - r) * kf);
}

// The scores of one 32 x 32 MFMA block in place, in the kernel's units.
template <int FORM>
__device__ __forceinline__ void block_scores(f32x16_t& acc, float scale) {
#pragma unroll
  for (int v = 0; v < 16; v += 2) {
    float a = acc[v], c = acc[v + 1];
    if (FORM != kLse) round2_bf16(a, c);
    if (FORM != kDenseP2) {
      a *= scale;
      c *= scale;
    }
    if (FORM == kDense) round2_bf16(a, c);
    acc[v] = a;
    acc[v + 1] = c;
  }
}

// Work item of workgroup `bid` among `n`: dispatch places workgroup i on XCD i % 8, so XCD x takes the
// contiguous band of items [x q + min(x, r), ...) (q = n / 8, r = n % 8) and the workgroups that share an
// image's Q and K share an L2.
__device__ __forceinline__ int xcd_band(int bid, int n) {
  const int x = bid & 7, q = n >> 3, r = n & 7;
  return x * q + min(x, r) + (bid >> 3);
}

// Row statistics: workgroup = (256 queries = 8 waves x 32, head, image). Key tiles of 64 (two 32-key
// MFMA blocks) are staged once in LDS for all waves, double-buffered through registers (16-byte chunks
// XOR-swizzled by row); S^T = K . Q^T puts a query's scores in one lane pair (lanes l, l ^ 32). One pass:
// each lane keeps the running max of its half of the keys and the sum of exp(s - max), rescaled per tile
// (the max is exact in any order; a tile's terms are summed apart and then added, which rounds less than
// one long chain); the two lanes of a query merge at the end. Bound by the VALU (one exponential per
// score): two passes over the keys with expf before, 266 -> 97 us at 16 images x 16 heads x 1029^2.
// Output: kLse the row log-sum-exp (natural log) in ref_out; dense the row's reference there and its
// ref_error / l in w_out, so that a probability is row_exp(v) * w. Waves whose queries lie past N still stage tiles and meet every
// barrier.
static constexpr int kStWaves = 8;
static constexpr int kStKeys = 64;

template <int DH, int FORM>
__global__ __launch_bounds__(kStWaves * 64) void pattn_stats_kernel(const uint16_t* __restrict__ q, int64_t qrs,
                                                                    const uint16_t* __restrict__ kv, int64_t kvb,
                                                                    int64_t kvn, int64_t kvh, int N, int H,
                                                                    float scale, float* __restrict__ ref_out,
                                                                    float* __restrict__ w_out) {
  constexpr int KS = DH / 16;
  constexpr int CPR = DH / 8;
  constexpr int CHUNKS = kStKeys * CPR;
  constexpr int NT = kStWaves * 64;
  constexpr int IT = CHUNKS / NT;
  static_assert(CHUNKS % NT == 0, "whole chunks per thread");
  __shared__ __align__(16) unsigned char kt[2][kStKeys * DH * 2];
  const int nqb = (N + 32 * kStWaves - 1) / (32 * kStWaves);
  const int item = xcd_band((int)blockIdx.x, (int)gridDim.x);
  const int qb_ = item % nqb, pair = item / nqb;
  const int h = pair % H, b = pair / H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int q0 = (qb_ * kStWaves + wave) * 32;
  const bool active = q0 < N;
  const uint16_t* qb = q + (int64_t)b * N * qrs + (int64_t)h * DH;
  const uint16_t* kb = kv + (int64_t)b * kvb + (int64_t)h * kvh;
  bf16x8_t qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = frag16(qb, qrs, q0 + l32, N, ks * 16 + 8 * g);
  const int ntiles = (N + kStKeys - 1) / kStKeys;
  const float kf = score_factor(FORM, scale);

  u32x4_t rk[IT];
  auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + i * NT;
      const int r = c / CPR, ch = c - r * CPR;
      const int key = t * kStKeys + r;
      rk[i] = u32x4_t{0, 0, 0, 0};
      if (key < N) rk[i] = *reinterpret_cast<const u32x4_t*>(kb + (int64_t)key * kvn + ch * 8);
    }
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + i * NT;
      const int r = c / CPR, ch = c - r * CPR;
      *reinterpret_cast<u32x4_t*>(&kt[buf][r * DH * 2 + ((ch ^ (r & (CPR - 1))) << 4)]) = rk[i];
    }
  };

  // A lane whose keys so far all lie past N (N <= 4: the whole half g = 1) has m = -inf and an empty sum; its
  // exponents are then taken from 0, never from the difference of two infinities.
  float m = -INFINITY, l = 0.0f;
  load(0);
  store(0);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    const int buf = t & 1;
    if (t + 1 < ntiles) load(t + 1);
    if (active) {
      f32x16_t acc[2];
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2) {
        const int r = kb2 * 32 + l32;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[kb2][v] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int ch = 2 * ks + g;
          const bf16x8_t kfr =
              as_bf16x8(*reinterpret_cast<const uint4*>(&kt[buf][r * DH * 2 + ((ch ^ (r & (CPR - 1))) << 4)]));
          acc[kb2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfr, qf[ks], acc[kb2], 0, 0, 0);
        }
        block_scores<FORM>(acc[kb2], scale);
      }
      // Keys past N exist only in the last tile: there the scores of those keys become -inf.
      if ((t + 1) * kStKeys > N) {
#pragma unroll
        for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (t * kStKeys + kb2 * 32 + 8 * (v >> 2) + 4 * g + (v & 3) >= N) acc[kb2][v] = -INFINITY;
      }
      float mx[4];
#pragma unroll
      for (int c4 = 0; c4 < 4; ++c4) {
        mx[c4] = acc[c4 >> 1][8 * (c4 & 1)];
#pragma unroll
        for (int v = 1; v < 8; ++v) mx[c4] = fmaxf(mx[c4], acc[c4 >> 1][8 * (c4 & 1) + v]);
      }
      const float m_new = fmaxf(fmaxf(m, fmaxf(mx[0], mx[1])), fmaxf(mx[2], mx[3]));
      const float mf = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = __builtin_amdgcn_exp2f((m - mf) * kf);
      const float ref = row_ref<FORM>(mf, kf);
      float ts[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
        for (int v = 0; v < 16; ++v) ts[v & 3] += row_exp<FORM>(acc[kb2][v], ref, kf);
      l = fmaf(l, alpha, ref_error<FORM>(mf, kf) * ((ts[0] + ts[1]) + (ts[2] + ts[3])));
      m = m_new;
    }
    if (t + 1 < ntiles) store(buf ^ 1);
    __syncthreads();
  }
  const float m2 = __shfl_xor(m, 32, 64), l2 = __shfl_xor(l, 32, 64);
  const float mt = fmaxf(m, m2);
  l = l * __builtin_amdgcn_exp2f((m - mt) * kf) + l2 * __builtin_amdgcn_exp2f((m2 - mt) * kf);
  const int qi = q0 + l32;
  if (active && g == 0 && qi < N) {
    const int64_t o = ((int64_t)b * H + h) * N + qi;
    ref_out[o] = FORM == kLse ? mt + logf(l) : row_ref<FORM>(mt, kf);
    if (FORM != kLse) w_out[o] = ref_error<FORM>(mt, kf) / l;
  }
}

// Dense key-side score: workgroup = (128-query block, 128-key block, image), 8 waves; wave w takes
// queries 32 (w % 4) .. + 31 and keys 64 (w / 4) .. + 63 of the tile (two 32-key MFMA blocks, S = Q . K^T
// so a key's column sits in one lane pair). For every head the Q and K tiles (128 x DH each, swizzled
// 16-byte chunks) and the 128 queries' references and weights (pattn_stats_kernel) are staged once in LDS,
// double-buffered through registers; p = bf16(row_exp(v) * w) is summed over heads per (query, key)
// in registers. After the last head each (query, key) takes bf16(sum * fl(1/H)); the tile's column sums
// over its queries (four query waves added in order in LDS) go to part[b][query block][key], and
// pattn_dense_reduce_kernel adds the query blocks in order. Waves wholly past N compute nothing
// (N = 1029 is 8 tiles and 5 rows). Bound by the VALU (one exponential and two to three bf16
// roundings per score and head): with expf and a divided quotient before, 344 -> 129 us at 16 images x 16
// heads x 1029^2.
static constexpr int kDnTile = 128;

// Two workgroups per CU at DH = 64 (LDS 66 KB each, so the registers are held to 128); one at DH = 128.
// OFF: the type of a lane's element offset from its tile's first row (uint32_t while 128 rows run forwards and
// span less).
template <int DH, int FORM, typename OFF>
__global__ __launch_bounds__(512, DH == 64 ? 4 : 2) void pattn_colsum_kernel(const uint16_t* __restrict__ q, int64_t qrs,
                                                           const uint16_t* __restrict__ kv, int64_t kvb, int64_t kvn,
                                                           int64_t kvh, int N, int H, float scale,
                                                           const float* __restrict__ ref_in,
                                                           const float* __restrict__ w_in,
                                                           float* __restrict__ part) {
  constexpr int KS = DH / 16;
  constexpr int CPR = DH / 8;
  constexpr int ROWB = DH * 2;
  constexpr int TILEB = kDnTile * ROWB;
  constexpr int CHUNKS = 2 * kDnTile * CPR;  // Q and K chunks of one head
  constexpr int NT = 512;
  constexpr int IT = CHUNKS / NT;
  static_assert(CHUNKS % NT == 0, "whole chunks per thread");
  __shared__ __align__(16) unsigned char tiles[2][2 * TILEB];
  __shared__ __align__(16) float st[2][2][kDnTile];  // row references, weights
  __shared__ float colp[4][kDnTile];
  const int nb = (N + kDnTile - 1) / kDnTile;  // query blocks = key blocks
  const int item = xcd_band((int)blockIdx.x, (int)gridDim.x);
  const int kblk = item % nb, qblk = item / nb % nb, b = item / (nb * nb);
  const int qt0 = qblk * kDnTile, kt0 = kblk * kDnTile;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int wq = 32 * (wave & 3), wk = 64 * (wave >> 2);
  const bool active = qt0 + wq < N && kt0 + wk < N;
  const float kf = score_factor(FORM, scale);

  // Rows past N repeat row N - 1: their scores reach no stored column and no counted query. Offsets are
  // relative to the tile's first row, the head's base pointers uniform.
  const uint16_t* qbase = q + ((int64_t)b * N + qt0) * qrs;
  const uint16_t* kbase = kv + (int64_t)b * kvb + (int64_t)kt0 * kvn;
  OFF off_[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = tid + (i % (IT / 2)) * NT;
    const int r = c / CPR, ch = c - r * CPR;
    off_[i] = i < IT / 2 ? (OFF)min(r, N - 1 - qt0) * (OFF)qrs + (OFF)(ch * 8)
                         : (OFF)min(r, N - 1 - kt0) * (OFF)kvn + (OFF)(ch * 8);
  }
  u32x4_t rq[IT];
  float rs = 1.0f;
  auto load = [&](int h) __attribute__((always_inline)) {
    const uint16_t* qh = qbase + (int64_t)h * DH;
    const uint16_t* kh = kbase + (int64_t)h * kvh;
#pragma unroll
    for (int i = 0; i < IT; ++i) rq[i] = *reinterpret_cast<const u32x4_t*>((i < IT / 2 ? qh : kh) + off_[i]);
    if (tid < 2 * kDnTile && qt0 + (tid & (kDnTile - 1)) < N)
      rs = (tid < kDnTile ? ref_in : w_in)[((int64_t)b * H + h) * N + qt0 + (tid & (kDnTile - 1))];
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + (i % (IT / 2)) * NT;
      const int r = c / CPR, ch = c - r * CPR;
      *reinterpret_cast<u32x4_t*>(&tiles[buf][(i < IT / 2 ? 0 : TILEB) + r * ROWB + ((ch ^ (r & (CPR - 1))) << 4)]) = rq[i];
    }
    if (tid < 2 * kDnTile) st[buf][tid / kDnTile][tid & (kDnTile - 1)] = rs;
  };

  float hs[2][16];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) hs[j][v] = 0.0f;

  load(0);
  store(0);
  __syncthreads();
  for (int h = 0; h < H; ++h) {
    const int buf = h & 1;
    if (h + 1 < H) load(h + 1);
    if (active) {
      const unsigned char* qs = tiles[buf];
      const unsigned char* ks = tiles[buf] + TILEB;
      bf16x8_t qf[KS];
      const int rq_ = wq + l32;
#pragma unroll
      for (int kstep = 0; kstep < KS; ++kstep)
        qf[kstep] = as_bf16x8(
            *reinterpret_cast<const uint4*>(qs + rq_ * ROWB + (((2 * kstep + g) ^ (rq_ & (CPR - 1))) << 4)));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        __builtin_amdgcn_sched_barrier(0);  // one block's scores in registers at a time
        f32x16_t acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
        const int rk_ = wk + 32 * j + l32;
#pragma unroll
        for (int kstep = 0; kstep < KS; ++kstep) {
          const bf16x8_t kfr = as_bf16x8(
              *reinterpret_cast<const uint4*>(ks + rk_ * ROWB + (((2 * kstep + g) ^ (rk_ & (CPR - 1))) << 4)));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[kstep], kfr, acc, 0, 0, 0);
        }
        block_scores<FORM>(acc, scale);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const float4 r4 = *reinterpret_cast<const float4*>(&st[buf][0][wq + 8 * a + 4 * g]);
          const float4 w4 = *reinterpret_cast<const float4*>(&st[buf][1][wq + 8 * a + 4 * g]);
          const float ref[4] = {r4.x, r4.y, r4.z, r4.w}, w[4] = {w4.x, w4.y, w4.z, w4.w};
          float pv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) pv[e] = row_exp<FORM>(acc[4 * a + e], ref[e], kf) * w[e];
          round2_bf16(pv[0], pv[1]);
          round2_bf16(pv[2], pv[3]);
#pragma unroll
          for (int e = 0; e < 4; ++e) hs[j][4 * a + e] += pv[e];
        }
      }
    }
    if (h + 1 < H) store(buf ^ 1);
    __syncthreads();
  }
  // bf16 head means of the valid queries, summed over this wave's queries per key.
  const float inv_h = 1.0f / (float)H;
  float col[2] = {0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int qi = qt0 + wq + 8 * (v >> 2) + 4 * g + (v & 3);
      if (qi < N) col[j] += round_bf16(hs[j][v] * inv_h);
    }
#pragma unroll
  for (int j = 0; j < 2; ++j) col[j] += __shfl_xor(col[j], 32, 64);
  if (g == 0) {
    colp[wave & 3][wk + l32] = col[0];
    colp[wave & 3][wk + 32 + l32] = col[1];
  }
  __syncthreads();
  if (tid < kDnTile && kt0 + tid < N) {
    const float t = ((colp[0][tid] + colp[1][tid]) + colp[2][tid]) + colp[3][tid];
    part[((int64_t)b * nb + qblk) * N + kt0 + tid] = t;
  }
}

// out[b, n] = bf16(fl(sum_qb part[b][qb][n]) * fl(1/N)), query blocks added in order.
__global__ void pattn_dense_reduce_kernel(const float* __restrict__ part, int B, int N, int nqb,
                                          uint16_t* __restrict__ out, int64_t osb) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)B * N) return;
  const int b = (int)(i / N), n = (int)(i - (int64_t)b * N);
  const float* p = part + (int64_t)b * nqb * N + n;
  float t = 0.0f;
  for (int qb = 0; qb < nqb; ++qb) t += p[(int64_t)qb * N];
  out[(int64_t)b * osb + n] = (uint16_t)f32_to_bf16(t * (1.0f / (float)N));
}

// Key-side score from the row log-sum-exp (mode kLse), one pass over the scores. Workgroup = (block
// of 256 keys, group of `hpg` heads, image), 8 waves of 32 keys each. For every (head, 32-query block)
// the query tile (32 x DH bf16, 16-byte chunks XOR-swizzled by row so that 16 consecutive rows read at
// one chunk cover all banks) and its 32 row LSEs (times log2 e; +inf past N) are staged once in LDS
// for all waves, double-buffered through registers; each wave keeps its keys' K fragments of the
// current head in registers, forms S = Q . K^T on v_mfma_f32_32x32x16_bf16 (a key's column in one
// lane pair) and adds exp2(s * scale log2 e - lse log2 e) over its queries in fp32 registers. Keys and
// queries past N read as zeros; their terms never reach a stored column. Partial column sums per head
// group -> part[b][group][n]; pattn_lse_reduce_kernel adds the groups in order.
static constexpr int kLseWaves = 8;
static constexpr int kLseKeys = 32 * kLseWaves;

template <int DH>
__global__ __launch_bounds__(kLseWaves * 64) void pattn_colsum_lse_kernel(
    const uint16_t* __restrict__ q, int64_t qrs, const uint16_t* __restrict__ kv, int64_t kvb, int64_t kvn,
    int64_t kvh, int N, int H, int hpg, float scale_log2, const float* __restrict__ lse, float* __restrict__ part) {
  constexpr int KS = DH / 16;          // 16-deep MFMA steps
  constexpr int CPR = DH / 8;          // 16-byte chunks per query row
  constexpr int CHUNKS = 32 * CPR;     // chunks per query tile
  constexpr int NT = kLseWaves * 64;
  constexpr int IT = (CHUNKS + NT - 1) / NT;
  __shared__ __align__(16) unsigned char qs[2][32 * DH * 2];
  __shared__ __align__(16) float ls[2][32];
  const int b = blockIdx.z, grp = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const int key = blockIdx.x * kLseKeys + wave * 32 + l32;
  const int nqb = (N + 31) / 32;
  const int h0 = grp * hpg;
  const int nh = min(H - h0, hpg);
  const int steps = nh * nqb;
  const uint16_t* qimg = q + (int64_t)b * N * qrs;
  const float* limg = lse + (int64_t)b * H * N;

  u32x4_t rq[IT];
  float rl = INFINITY;
  auto load = [&](int st) __attribute__((always_inline)) {
    const int h = h0 + st / nqb, q0 = (st % nqb) * 32;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + i * NT;
      rq[i] = u32x4_t{0, 0, 0, 0};
      if (c < CHUNKS) {
        const int r = c / CPR, ch = c - r * CPR;
        if (q0 + r < N) rq[i] = *reinterpret_cast<const u32x4_t*>(qimg + (int64_t)(q0 + r) * qrs + (int64_t)h * DH + ch * 8);
      }
    }
    if (tid < 32) rl = q0 + tid < N ? limg[(int64_t)h * N + q0 + tid] * kLog2e : INFINITY;
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + i * NT;
      if (c < CHUNKS) {
        const int r = c / CPR, ch = c - r * CPR;
        *reinterpret_cast<u32x4_t*>(&qs[buf][r * DH * 2 + ((ch ^ (r & (CPR - 1))) << 4)]) = rq[i];
      }
    }
    if (tid < 32) ls[buf][tid] = rl;
  };

  bf16x8_t kf[KS];
  auto load_k = [&](int h) {
    const uint16_t* kb = kv + (int64_t)b * kvb + (int64_t)h * kvh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (key < N) v = *reinterpret_cast<const uint4*>(kb + (int64_t)key * kvn + ks * 16 + 8 * g);
      kf[ks] = as_bf16x8(v);
    }
  };

  float col = 0.0f;
  if (steps > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int st = 0; st < steps; ++st) {
    const int buf = st & 1;
    if (st % nqb == 0) load_k(h0 + st / nqb);
    if (st + 1 < steps) load(st + 1);
    const unsigned char* qt = qs[buf];
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int ch = 2 * ks + g;
      const bf16x8_t qf = as_bf16x8(*reinterpret_cast<const uint4*>(qt + l32 * DH * 2 + ((ch ^ (l32 & (CPR - 1))) << 4)));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, kf[ks], acc, 0, 0, 0);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float4 l4 = *reinterpret_cast<const float4*>(&ls[buf][8 * a + 4 * g]);
      col += __builtin_amdgcn_exp2f(fmaf(acc[4 * a + 0], scale_log2, -l4.x));
      col += __builtin_amdgcn_exp2f(fmaf(acc[4 * a + 1], scale_log2, -l4.y));
      col += __builtin_amdgcn_exp2f(fmaf(acc[4 * a + 2], scale_log2, -l4.z));
      col += __builtin_amdgcn_exp2f(fmaf(acc[4 * a + 3], scale_log2, -l4.w));
    }
    if (st + 1 < steps) store(buf ^ 1);
    __syncthreads();
  }
  col += __shfl_xor(col, 32, 64);
  if (g == 0 && key < N) part[((int64_t)b * gridDim.y + grp) * N + key] = col;
}

// out[b, n] = bf16(fl(sum_group part[b][group][n]) * factor), groups added in order.
__global__ void pattn_lse_reduce_kernel(const float* __restrict__ part, int B, int N, int groups, float factor,
                                        uint16_t* __restrict__ out, int64_t osb) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)B * N) return;
  const int b = (int)(i / N), n = (int)(i - (int64_t)b * N);
  const float* p = part + (int64_t)b * groups * N + n;
  float t = 0.0f;
  for (int gi = 0; gi < groups; ++gi) t += p[(int64_t)gi * N];
  out[(int64_t)b * osb + n] = (uint16_t)f32_to_bf16(t * factor);
}

// Heads per group of the one-pass LSE kernel: enough groups that the grid holds about 512 workgroups.
static int lse_heads_per_group(int B, int N, int H) {
  const int kblocks = (N + kLseKeys - 1) / kLseKeys;
  const int want = (int)std::min<int64_t>(H, std::max<int64_t>(1, cdiv(512, (int64_t)kblocks * B)));
  return (H + want - 1) / want;
}

// The one-pass key-side score from lse [B, H, N] (natural log) into out, through part (B * H * N fp32
// at most: B * groups * N used).
template <int DH>
void launch_colsum_lse(const uint16_t* q, int64_t qrs, const uint16_t* kv, int64_t kvb, int64_t kvn, int64_t kvh,
                       int B, int N, int H, float scale, const float* lse, float* part, uint16_t* out, int64_t osb,
                       hipStream_t st) {
  const int hpg = lse_heads_per_group(B, N, H);
  const int groups = (H + hpg - 1) / hpg;
  const dim3 g1((unsigned)cdiv(N, kLseKeys), (unsigned)groups, (unsigned)B);
  pattn_colsum_lse_kernel<DH><<<g1, kLseWaves * 64, 0, st>>>(q, qrs, kv, kvb, kvn, kvh, N, H, hpg, scale * kLog2e,
                                                              lse, part);
  const int64_t n = (int64_t)B * N;
  pattn_lse_reduce_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(part, B, N, groups,
                                                                  1.0f / (float)((int64_t)H * N), out, osb);
}

// FORM kLse, kDense or kDenseP2 (the dense mode with a power-of-two scale of at most 1/2, e.g. 64^-0.5 = 1/8).
template <int DH, int FORM>
void launch_pattn(const uint16_t* q, int64_t qrs, const uint16_t* kv, int64_t kvb, int64_t kvn, int64_t kvh, int B,
                  int N, int H, float scale, float* ws, uint16_t* out, int64_t osb, hipStream_t st) {
  float* ref = ws;                      // the rows' references, or log-sum-exp mode's row log-sum-exp
  float* w = ws + (int64_t)B * H * N;   // the rows' weights, or log-sum-exp mode's partial column sums
  const unsigned g1 = (unsigned)(cdiv(N, 32 * kStWaves) * H * B);
  pattn_stats_kernel<DH, FORM><<<g1, kStWaves * 64, 0, st>>>(q, qrs, kv, kvb, kvn, kvh, N, H, scale, ref, w);
  if constexpr (FORM == kLse) {
    launch_colsum_lse<DH>(q, qrs, kv, kvb, kvn, kvh, B, N, H, scale, ref, w, out, osb, st);
  } else {
    // Partial column sums per 128-query block after the statistics.
    float* part = ws + 2 * (int64_t)B * H * N;
    const int nqb = (int)cdiv(N, kDnTile);
    const unsigned g2 = (unsigned)(nqb * nqb * B);
    // 32-bit offsets within a tile are unsigned: rows that run backwards (kvn < 0) take 64-bit ones.
    if (qrs >= 0 && kvn >= 0 && std::max(qrs, kvn) < ((int64_t)1 << 24))
      pattn_colsum_kernel<DH, FORM, uint32_t>
          <<<g2, 512, 0, st>>>(q, qrs, kv, kvb, kvn, kvh, N, H, scale, ref, w, part);
    else
      pattn_colsum_kernel<DH, FORM, int64_t><<<g2, 512, 0, st>>>(q, qrs, kv, kvb, kvn, kvh, N, H, scale, ref, w, part);
    const int64_t n = (int64_t)B * N;
    pattn_dense_reduce_kernel<<<(unsigned)cdiv(n, 256), 256, 0, st>>>(part, B, N, nqb, out, osb);
  }
}

template <int DH>
void launch_pattn_mode(const uint16_t* q, int64_t qrs, const uint16_t* kv, int64_t kvb, int64_t kvn, int64_t kvh, int B,
                       int N, int H, float scale, int mode, float* ws, uint16_t* out, int64_t osb, hipStream_t st) {
  int e = 0;
  const bool pow2 = scale > 0.0f && std::frexp(scale, &e) == 0.5f && e <= 0 && e > -64;
  if (mode == kLse) launch_pattn<DH, kLse>(q, qrs, kv, kvb, kvn, kvh, B, N, H, scale, ws, out, osb, st);
  else if (pow2) launch_pattn<DH, kDenseP2>(q, qrs, kv, kvb, kvn, kvh, B, N, H, scale, ws, out, osb, st);
  else launch_pattn<DH, kDense>(q, qrs, kv, kvb, kvn, kvh, B, N, H, scale, ws, out, osb, st);
}

}  // namespace oudjat

using namespace oudjat;

extern "C" int64_t oudjat_patch_attention_prob_workspace_elems(int64_t B, int64_t N, int64_t H, int mode) {
  if (B <= 0 || N <= 0 || H <= 0) return 0;
  // two arrays of row statistics (dense: references and weights; log-sum-exp mode: the row log-sum-exp, and its
  // per-head-group column sums in the second), then the dense mode's per-query-block column sums
  return 2 * B * H * N + (mode == kDense ? B * cdiv(N, kDnTile) * N : 0);
}

extern "C" int oudjat_patch_attention_prob(const uint16_t* q, int64_t q_row_stride, int64_t B, int64_t N, int64_t H,
                                           int64_t Dh, const uint16_t* kv, int64_t kv_stride_b, int64_t kv_stride_n,
                                           int64_t kv_stride_h, float scale, int mode, float* workspace,
                                           uint16_t* out, int64_t out_stride_b, oudjat_stream_t stream) {
  OUDJAT_REQUIRE(B >= 0 && N >= 0 && H > 0, OUDJAT_ERR_INVALID_ARGUMENT, "patch_attention_prob: bad size");
  OUDJAT_REQUIRE(mode == kDense || mode == kLse, OUDJAT_ERR_INVALID_ARGUMENT, "patch_attention_prob: mode %d", mode);
  OUDJAT_REQUIRE(Dh == 64 || Dh == 128, OUDJAT_ERR_UNSUPPORTED_SHAPE, "patch_attention_prob: Dh=%lld (64 or 128)",
                 (long long)Dh);
  if (B == 0 || N == 0) return OUDJAT_OK;
  OUDJAT_REQUIRE(q && kv && workspace && out, OUDJAT_ERR_INVALID_ARGUMENT, "patch_attention_prob: null pointer");
  OUDJAT_REQUIRE(q_row_stride >= H * Dh && kv_stride_h >= Dh && out_stride_b >= N, OUDJAT_ERR_UNSUPPORTED_LAYOUT,
                 "patch_attention_prob: strides");
  OUDJAT_REQUIRE(aligned(q, 16) && aligned(kv, 16) && q_row_stride % 8 == 0 && kv_stride_b % 8 == 0 &&
                     kv_stride_n % 8 == 0 && kv_stride_h % 8 == 0,
                 OUDJAT_ERR_UNSUPPORTED_LAYOUT, "patch_attention_prob: 16-byte aligned rows required");
  OUDJAT_REQUIRE(N < (1 << 24) && H < 65536 && B < 65536 && B * H * cdiv(N, 32 * kStWaves) < ((int64_t)1 << 31) &&
                     (mode == kLse || B * cdiv(N, kDnTile) * cdiv(N, kDnTile) < ((int64_t)1 << 31)),
                 OUDJAT_ERR_TOO_LARGE, "patch_attention_prob: too large");
  const hipStream_t st = as_stream(stream);
  const int b = (int)B, n = (int)N, h = (int)H;
  if (Dh == 64)
    launch_pattn_mode<64>(q, q_row_stride, kv, kv_stride_b, kv_stride_n, kv_stride_h, b, n, h, scale, mode, workspace,
                          out, out_stride_b, st);
  else
    launch_pattn_mode<128>(q, q_row_stride, kv, kv_stride_b, kv_stride_n, kv_stride_h, b, n, h, scale, mode, workspace,
                           out, out_stride_b, st);
  return check_launch("patch_attention_prob");
}

extern "C" int oudjat_patch_attention_prob_lse(const uint16_t* q, int64_t q_row_stride, int64_t B, int64_t N,
                                               int64_t H, int64_t Dh, const uint16_t* kv, int64_t kv_stride_b,
                                               int64_t kv_stride_n, int64_t kv_stride_h, float scale, const float* lse,
                                               float* workspace, uint16_t* out, int64_t out_stride_b,
                                               oudjat_stream_t stream) {
  OUDJAT_REQUIRE(B >= 0 && N >= 0 && H > 0, OUDJAT_ERR_INVALID_ARGUMENT, "patch_attention_prob_lse: bad size");
  OUDJAT_REQUIRE(Dh == 64 || Dh == 128, OUDJAT_ERR_UNSUPPORTED_SHAPE, "patch_attention_prob_lse: Dh=%lld (64 or 128)",
                 (long long)Dh);
  if (B == 0 || N == 0) return OUDJAT_OK;
  OUDJAT_REQUIRE(q && kv && lse && workspace && out, OUDJAT_ERR_INVALID_ARGUMENT,
                 "patch_attention_prob_lse: null pointer");
  OUDJAT_REQUIRE(q_row_stride >= H * Dh && kv_stride_h >= Dh && out_stride_b >= N, OUDJAT_ERR_UNSUPPORTED_LAYOUT,
                 "patch_attention_prob_lse: strides");
  OUDJAT_REQUIRE(aligned(q, 16) && aligned(kv, 16) && aligned(lse, 4) && aligned(workspace, 4) &&
                     q_row_stride % 8 == 0 && kv_stride_b % 8 == 0 && kv_stride_n % 8 == 0 && kv_stride_h % 8 == 0,
                 OUDJAT_ERR_UNSUPPORTED_LAYOUT, "patch_attention_prob_lse: 16-byte aligned rows required");
  OUDJAT_REQUIRE(N < (1 << 24) && H < 65536 && B < 65536, OUDJAT_ERR_TOO_LARGE, "patch_attention_prob_lse: too large");
  const hipStream_t st = as_stream(stream);
  const int b = (int)B, n = (int)N, h = (int)H;
  if (Dh == 64)
    launch_colsum_lse<64>(q, q_row_stride, kv, kv_stride_b, kv_stride_n, kv_stride_h, b, n, h, scale, lse, workspace,
                          out, out_stride_b, st);
  else
    launch_colsum_lse<128>(q, q_row_stride, kv, kv_stride_b, kv_stride_n, kv_stride_h, b, n, h, scale, lse, workspace,
                           out, out_stride_b, st);
  return check_launch("patch_attention_prob_lse");
}
