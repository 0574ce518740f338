// Causal GQA attention with the reference's arithmetic (src/model/forward.js:115-140; the gated form of
// src/model/forward-qwen35.js:71-105 when a.gate is set), in two launches per layer:
//   k_attn_scores  s_t = f32(sum_i q_i K_t,i (f64, exact products) * 1/sqrt(hd)) for every position t <= pos, one
//                  block per (64-position chunk, KV head, token): all of K streams in parallel.
//   k_attn_av      softmax over the scores (e = exp(s - max) in f64, stored f32; p = f32(e * (1/sum e))), then
//                  out_i = sum_t p_t V_t,i accumulated in f32 in position order, one block per (32-dim slice, query
//                  head, token, chunk of 2048 positions); the head output is also quantised for the output projection.
// Scores live in a [token][head][ctx] f32 buffer between the two. The weighted sum of a chunk keeps the reference's f32
// rounding after every position, so rows of up to 2048 positions are the reference's bits (a random-weight network turns a
// 1e-7 change there into a visible logit difference); the chunks of longer rows are joined in f64.
#include "zl_kernels.h"
#include "zl_exp.h"
#include <algorithm>
#include <climits>

namespace zl {

// Query heads handled by one score block: the largest divisor of the GQA group that is at most 8.
inline int attn_heads_per_block(int group) {
  for (int c = 8; c > 1; c--)
    if (group % c == 0) return c;
  return 1;
}

// Score dots: every position's dot is split over HD / ATTN_VPL lanes of ATTN_VPL values each (an f64 fma chain per
// lane in value order, then an xor butterfly over the position's lanes); both attention forms use this order.
constexpr int ATTN_VPL = 32;
// Positions per score block chunk: 64, or one load round of 256 threads where that is more (HD = 64).
constexpr int attn_score_chunk(int hd) { return 256 / (hd / ATTN_VPL) > 64 ? 256 / (hd / ATTN_VPL) : 64; }

// Per-head RMSNorm (weights nw, when set) and RoPE at position pos of one head vector v[0..HD) in LDS, by one wave,
// with the arithmetic of src/model/forward.js:203-211 and src/compute/ref-kernels.js:305-310, 344-363 (64-lane strided
// f64 sum of squares and butterfly; f64 rotation of each (i, i + half) or (2i, 2i + 1) pair, stored f32).
template <int HD>
struct RopeVals {
  static constexpr int PR = (HD / 2 + 63) / 64;  // rotation pairs per lane at most
  static constexpr int NW = (HD + 63) / 64;      // norm weights per lane
  float cv[PR], sv[PR], wv[NW];
};

// The lane's norm weights (a read of the table when there is no norm: no branch around the loads) ...
template <int HD>
__device__ inline void rope_load_w(RopeVals<HD> &r, const float *nw, const float *cosT, int lane) {
  const float *nwp = nw ? nw : cosT;
  #pragma unroll
  for (int k = 0; k < RopeVals<HD>::NW; k++) r.wv[k] = nwp[lane + 64 * k < HD ? lane + 64 * k : 0];
}
// ... and its rotation table values at position pos.
template <int HD>
__device__ inline void rope_load_cs(RopeVals<HD> &r, int nRot, const float *cosT, const float *sinT, int pos, int lane) {
  const int half = nRot / 2;
  #pragma unroll
  for (int k = 0; k < RopeVals<HD>::PR; k++) {
    const int i = lane + 64 * k, ic = i < half ? i : 0;
    r.cv[k] = cosT[(long)pos * half + ic];
    r.sv[k] = sinT[(long)pos * half + ic];
  }
}

// Per-head RMSNorm (weights nw, when set) and RoPE of one head vector v[0..HD) in LDS, by one wave, with the
// arithmetic of src/model/forward.js:203-211 and src/compute/ref-kernels.js:305-310, 344-363 (64-lane strided f64 sum
// of squares and butterfly; f64 rotation of each (i, i + half) or (2i, 2i + 1) pair, stored f32), from values loaded by
// rope_load_w / rope_load_cs.
template <int HD>
__device__ inline void norm_rope_apply(float *v, const RopeVals<HD> &r, const float *nw, double eps, int nRot, int neox,
                                       int lane) {
  const int half = nRot / 2;
  if (nw) {
    double ss = 0;
    for (int i = lane; i < HD; i += 64) { const double x = (double)v[i]; ss += x * x; }
    ss = wave_sum_xor(ss, 64);
    const double sc = 1.0 / sqrt(ss / (double)HD + eps);
    #pragma unroll
    for (int k = 0; k < RopeVals<HD>::NW; k++) {
      const int i = lane + 64 * k;
      if (i < HD) v[i] = (float)((double)v[i] * sc * (double)r.wv[k]);
    }
  }
  #pragma unroll
  for (int k = 0; k < RopeVals<HD>::PR; k++) {
    const int i = lane + 64 * k;
    if (i >= half) break;
    const int i0 = neox ? i : 2 * i, i1 = neox ? i + half : 2 * i + 1;
    const double c = (double)r.cv[k], sn = (double)r.sv[k];
    const double x0 = (double)v[i0], x1 = (double)v[i1];
    v[i0] = (float)(x0 * c - x1 * sn);  // pairs are disjoint across lanes
    v[i1] = (float)(x0 * sn + x1 * c);
  }
}

// Both at position pos; the table values and norm weights are requested before the sum of squares, which does not need
// them.
template <int HD>
__device__ inline void norm_rope(float *v, const float *nw, double eps, int nRot, int neox, const float *cosT,
                                 const float *sinT, int pos, int lane) {
  RopeVals<HD> r;
  rope_load_cs<HD>(r, nRot, cosT, sinT, pos, lane);
  rope_load_w<HD>(r, nw, cosT, lane);
  norm_rope_apply<HD>(v, r, nw, eps, nRot, neox, lane);
}

// Contexts from which the long-context launch forms are used (KV cache capacity in positions).
constexpr int AV_BIG_CTX = 4096;

// Scores of one 64-position chunk of one token for hg query heads sharing a KV head. Keys of positions before the
// pass (pos0) come from the cache; the pass's own keys (positions pos0 .. pos0 + b) are normed and rotated here from the
// projection output, rounded as the cache stores them, and the block of token b appends its own key and value to the
// cache (K position-major, V dimension-major), which is where the reference's pass writes them before attending
// (src/model/forward.js:203-214). The query heads are normed and rotated here too.
template <int HD, bool F16KV>
__global__ __launch_bounds__(256) void k_attn_scores(const AttnArgs a) {
  constexpr int VB = F16KV ? 2 : 4;      // bytes per cached value
  constexpr int EPW = 16 / VB;           // K values per 16-byte load
  constexpr int LP = HD / ATTN_VPL;      // lanes per position (ATTN_VPL values each)
  constexpr int NLD = ATTN_VPL / EPW;    // 16-byte loads per lane and position
  constexpr int PPI = 256 / LP;          // positions per load round
  constexpr int P = attn_score_chunk(HD);  // positions per chunk
  constexpr int R = P / PPI;             // load rounds per chunk
  static_assert(R >= 1 && P % PPI == 0, "chunk geometry");
  __shared__ float qs[8 * HD];
  __shared__ float kf[8 * HD];           // rotated keys of the pass, a batch of up to 8 positions at a time (f32)
  extern __shared__ __align__(16) uint8_t kn[];  // the chunk's new keys in cache format, from position n0: [min(P, B)][HD]
  // Workgroups go to the 8 XCDs round robin (linear id mod 8). At long contexts, where a layer's keys outgrow the
  // L2s, the blocks of the pass's tokens that read the same key chunks are given consecutive linear ids of one XCD, so
  // their K reads meet in that XCD's L2 instead of each token streaming the keys from memory again (measured: 16K
  // context, 9 tokens, 0.24 ms less per verify pass; at ~700 positions the keys stay in L2 and the order costs 0.02 ms).
  const int stB = a.step->B, stPos0 = a.step->pos0;  // the pass's step record (scalar loads, read before the pins)
  const int X = gridDim.x, XY = X * gridDim.y, Z = gridDim.z;
  pin_args(Z, a.q, a.ldq, a.qhs, a.k, a.ldkv, a.kcache, a.hpb, a.layer, a.nHead, a.nHeadKv);
  const int L = blockIdx.x + X * (blockIdx.y + gridDim.y * blockIdx.z);
  int xy, b;
  if (a.ctx >= AV_BIG_CTX && XY % 8 == 0) {
    const int q = L >> 3;
    b = q % Z;
    xy = (L & 7) + 8 * (q / Z);
  } else {
    b = L / XY;
    xy = L - b * XY;
  }
  const int bx = xy % X, by = xy / X;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int group = a.nHead / a.nHeadKv, hg = a.hpb;
  const int h0 = by * hg;        // first query head of this block
  const int kvh = h0 / group;
  const bool writer = h0 % group == 0;   // the first head group of a KV head appends the pass's K and V
  const long kvoff = ((long)a.layer * a.nHeadKv + kvh) * a.ctx * HD;
  const uint8_t *kbase = (const uint8_t *)a.kcache + kvoff * VB;
  float *srow = a.scores + ((long)b * a.nHead + h0) * a.sld;
  const int part = tid % LP, sub = tid / LP;
  uint4 u[R][NLD];
  // cached keys (positions of the pass are filled in from kn); the first chunk's keys and the query heads are requested
  // before the pass's step record arrives, so the positions past the cache's valid ones are read too (and unused)
  auto fetch = [&](int c0, int lim) {
    #pragma unroll
    for (int r = 0; r < R; r++) {
      const int t = c0 + r * PPI + sub;
      #pragma unroll
      for (int k = 0; k < NLD; k++)
        u[r][k] = t < lim ? *(const uint4 *)(kbase + ((long)t * HD + part * ATTN_VPL) * VB + 16 * k) : make_uint4(0, 0, 0, 0);
    }
  };
  // the query heads and the pass's keys, then the first chunk of cached keys: loads complete in order, so the query
  // rotation below waits for the query values alone while the keys are on their way
  constexpr int QV = 8 * HD / 256;  // query values per thread (at most 8 heads of HD values per block)
  float qv[QV];
  #pragma unroll
  for (int k = 0; k < QV; k++) {
    const int i = tid + 256 * k;
    qv[k] = i < hg * HD ? a.q[(long)b * a.ldq + (long)(h0 + i / HD) * a.qhs + i % HD] : 0.f;
  }
  // the pass's first 8 key rows of this KV head (row-major [row][HD], element tid + 256 k), for the blocks that norm
  // and rotate the pass's keys; unconditional loads (rows past B read row 0, unused)
  constexpr int KPT = 8 * HD / 256;
  const int nB = Z;
  float kr[KPT];
  #pragma unroll
  for (int k = 0; k < KPT; k++) {
    const int e = tid + 256 * k, row = e / HD < nB ? e / HD : 0;
    kr[k] = a.k[(long)row * a.ldkv + (long)kvh * HD + e % HD];
  }
  __builtin_amdgcn_sched_barrier(0);
  fetch(bx * P, a.ctx);
  __builtin_amdgcn_sched_barrier(0);
  if (b >= stB) return;
  const int pos0 = stPos0, npos = pos0 + b + 1;
  if (bx * P >= npos) return;
  #pragma unroll
  for (int k = 0; k < QV; k++)
    if (tid + 256 * k < hg * HD) qs[tid + 256 * k] = qv[k];
  __syncthreads();
  for (int h = wave; h < hg; h += 4) norm_rope<HD>(qs + h * HD, a.qNorm, a.eps, a.nRot, a.neox, a.cosT, a.sinT, npos - 1, lane);
  __syncthreads();
  for (int c0 = bx * P; c0 < npos; c0 += X * P) {
    if (c0 != bx * P) fetch(c0, pos0);
    // the pass's keys in this chunk: positions [n0, n1), tokens [n0 - pos0, n1 - pos0)
    const int n0 = max(c0, pos0), n1 = min(c0 + P, npos);
    for (int g0 = n0; g0 < n1; g0 += 8) {
      const int g1 = min(n1, g0 + 8);
      if (g0 == pos0) {  // rows 0 .. g1 - g0 - 1: the prefetched ones
        #pragma unroll
        for (int k = 0; k < KPT; k++)
          if (tid + 256 * k < (g1 - g0) * HD) kf[tid + 256 * k] = kr[k];
      } else {
        for (int i = tid; i < (g1 - g0) * HD; i += 256)
          kf[i] = a.k[(long)(g0 - pos0 + i / HD) * a.ldkv + (long)kvh * HD + i % HD];
      }
      __syncthreads();
      for (int p = g0 + wave; p < g1; p += 4)
        norm_rope<HD>(kf + (p - g0) * HD, a.kNorm, a.eps, a.nRot, a.neox, a.cosT, a.sinT, p, lane);
      __syncthreads();
      for (int i = tid; i < (g1 - g0) * HD; i += 256) {
        const int p = g0 + i / HD, d = i % HD;
        const float kv = kf[i];
        const long off = kvoff + (long)p * HD + d;
        if (F16KV) {
          const uint16_t hbits = f2h(kv);
          ((uint16_t *)kn)[(p - n0) * HD + d] = hbits;
          if (writer && p == npos - 1) {
            ((uint16_t *)a.kcache)[off] = hbits;
            ((uint16_t *)a.vcache)[(((long)a.layer * a.nHeadKv + kvh) * HD + d) * a.vstride + p] =
                f2h(a.v[(long)b * a.ldkv + (long)kvh * HD + d]);
          }
        } else {
          ((float *)kn)[(p - n0) * HD + d] = kv;
          if (writer && p == npos - 1) {
            ((float *)a.kcache)[off] = kv;
            ((float *)a.vcache)[(((long)a.layer * a.nHeadKv + kvh) * HD + d) * a.vstride + p] = a.v[(long)b * a.ldkv + (long)kvh * HD + d];
          }
        }
      }
      __syncthreads();
    }
    #pragma unroll
    for (int r = 0; r < R; r++) {
      const int t = c0 + r * PPI + sub;
      if (t >= pos0 && t < npos) {
        #pragma unroll
        for (int k = 0; k < NLD; k++) u[r][k] = *(const uint4 *)(kn + ((t - n0) * HD + part * ATTN_VPL) * VB + 16 * k);
      }
      double kv[ATTN_VPL];
      #pragma unroll
      for (int k = 0; k < NLD; k++) {
        const uint32_t w4[4] = {u[r][k].x, u[r][k].y, u[r][k].z, u[r][k].w};
        #pragma unroll
        for (int e = 0; e < EPW; e++)
          kv[k * EPW + e] = F16KV ? (double)h2f((uint16_t)((w4[e >> 1] >> (16 * (e & 1))) & 0xffff)) : (double)__uint_as_float(w4[e]);
      }
      for (int h = 0; h < hg; h++) {
        const float *qh = qs + h * HD + part * ATTN_VPL;
        double s = 0.0;
        #pragma unroll
        for (int e = 0; e < ATTN_VPL; e++) s = fma((double)qh[e], kv[e], s);
        s = wave_sum_xor(s, LP);
        if (part == (h % LP) && t < npos) srow[(long)h * a.sld + t] = (float)(s * a.scale);
      }
    }
    __syncthreads();  // kn is refilled by the next chunk
  }
}

// ---- scores of passes of several tokens on the matrix cores. v_mfma_f64_16x16x4_f64 adds its four products to the
// accumulator as four fused multiply-adds in k order (measured on gfx950, every element of random wide-range operands),
// so eight of them over dimensions 32 j .. 32 j + 31 in order are exactly the per-lane f64 fma chain of k_attn_scores
// (part j of a position's dot), and the parts are joined in the same butterfly order: the same bits. The pass's query
// rows and keys are normed and rotated first (k_attn_prep, which also appends the pass's K and V to the cache, as
// k_attn_scores' writer blocks do), so the score blocks only read.

// One wave per (token, head): query heads are normed, rotated and stored f32 to qr [B][nHead][HD]; KV heads (blockIdx.y
// >= nHead) have their key normed, rotated and appended to the cache in its format, and their value appended.
template <int HD, bool F16KV>
__global__ __launch_bounds__(64) void k_attn_prep(const AttnArgs a) {
  __shared__ float v[HD];
  const int b = blockIdx.x, hy = blockIdx.y, lane = threadIdx.x;
  const Step *st = a.step;
  if (b >= st->B) return;
  const int pos = st->pos0 + b;
  const bool isq = hy < a.nHead;
  const int h = isq ? hy : hy - a.nHead;
  const float *src = isq ? a.q + (long)b * a.ldq + (long)h * a.qhs : a.k + (long)b * a.ldkv + (long)h * HD;
  for (int i = lane; i < HD; i += 64) v[i] = src[i];
  __syncthreads();
  norm_rope<HD>(v, isq ? a.qNorm : a.kNorm, a.eps, a.nRot, a.neox, a.cosT, a.sinT, pos, lane);
  __syncthreads();
  if (isq) {
    for (int i = lane; i < HD; i += 64) a.qr[((long)b * a.nHead + h) * HD + i] = v[i];
    return;
  }
  const long kvoff = ((long)a.layer * a.nHeadKv + h) * a.ctx * HD + (long)pos * HD;
  const long voff = ((long)a.layer * a.nHeadKv + h) * HD;
  for (int d = lane; d < HD; d += 64) {
    const float vv = a.v[(long)b * a.ldkv + (long)h * HD + d];
    if (F16KV) {
      ((uint16_t *)a.kcache)[kvoff + d] = f2h(v[d]);
      ((uint16_t *)a.vcache)[(voff + d) * a.vstride + pos] = f2h(vv);
    } else {
      ((float *)a.kcache)[kvoff + d] = v[d];
      ((float *)a.vcache)[(voff + d) * a.vstride + pos] = vv;
    }
  }
}

// Block (every X-th 64-position tile of the pass, KV head, group of NWV row tiles); wave w computes row tile NWV z + w: 16
// rows r = b G + g (token b, query head kvh G + g) against every position of its tiles, 16 positions at a time. Lane l
// supplies A = the row l mod 16's dimension 32 j + 4 m + l / 16 (its query values, f64, held for the whole block) and B = key value
// [position l mod 16][dimension 32 j + 4 m + l / 16] from LDS, where the block has staged 64 positions' keys as f64;
// the accumulator of lane l element v is (row 4 v + l / 16, position l mod 16).
constexpr int MM_PT = 64;    // positions staged in LDS at a time
// NWV waves per block, one row tile each: 8 for passes of 128 rows or more per KV head (prefill chunks: every staged key
// tile serves 8 row tiles), else 4
template <int HD, bool F16KV, int NWV>
__global__ __launch_bounds__(NWV * 64) void k_attn_scores_mm(const AttnArgs a, int nrows) {
  constexpr int NP = HD / ATTN_VPL;    // parts (32 dimensions each)
  constexpr int VB = F16KV ? 2 : 4;
  constexpr int NT = NWV * 64;
  constexpr int RAW = MM_PT * HD * VB / 16 / NT;  // 16-byte K pieces per thread per staged tile
  static_assert(RAW >= 1 && RAW * NT * 16 == MM_PT * HD * VB, "staging geometry");
  typedef double d4 __attribute__((ext_vector_type(4)));
  extern __shared__ __align__(16) uint8_t lds[];
  // [MM_PT][HD + 2] keys as f64: with rows 2 doubles (4 banks) apart, the 32 lanes of a half-wave's B read (16
  // positions x 2 k-groups, one double each) fall on 64 distinct banks
  double *kd = (double *)lds;
  constexpr int KP = HD + 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n16 = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.y, tile = blockIdx.z * NWV + wave;
  const int G = a.nHead / a.nHeadKv;
  const Step *st = a.step;
  const int Bd = st->B, pos0 = st->pos0, nmax = pos0 + Bd;
  // the block's MM_PT-position tiles: bx, bx + X, ... of the pass's positions (the grid holds as many blocks per KV
  // head and row group as stay resident at once, so the tiles of a pass of any length spread evenly over them)
  const int X = gridDim.x, bx = blockIdx.x, ntile = (nmax + MM_PT - 1) / MM_PT;
  if (bx >= ntile) return;
  const long kvoff = ((long)a.layer * a.nHeadKv + kvh) * a.ctx * HD;
  const uint8_t *kbase = (const uint8_t *)a.kcache + kvoff * VB;
  // A operands: row n16 of the tile, dimensions 32 j + 4 m + g
  const int ra = tile * 16 + n16, ba = ra / G, ha = kvh * G + ra % G;
  const bool rowok = ra < nrows && ba < Bd;
  double A[NP][8];
  #pragma unroll
  for (int j = 0; j < NP; j++)
    #pragma unroll
    for (int m = 0; m < 8; m++)
      A[j][m] = rowok ? (double)a.qr[((long)ba * a.nHead + ha) * HD + 32 * j + 4 * m + g] : 0.0;
  // the rows whose accumulator elements this lane holds: 4 v + g, v = 0..3
  int rb[4], rh[4], rn[4];
  #pragma unroll
  for (int v = 0; v < 4; v++) {
    const int r = tile * 16 + 4 * v + g, bb = r / G;
    rb[v] = bb; rh[v] = kvh * G + r % G;
    rn[v] = (r < nrows && bb < Bd) ? pos0 + bb + 1 : 0;  // positions of the row (0: no row)
  }
  const bool waveok = tile * 16 < nrows;
  uint4 raw[RAW];
  auto fetch = [&](int t0) {
    #pragma unroll
    for (int k = 0; k < RAW; k++) {
      const int e = (k * NT + tid) * (16 / VB), p = e / HD, d = e % HD, t = t0 + p;
      raw[k] = t < nmax ? *(const uint4 *)(kbase + ((long)t * HD + d) * VB) : make_uint4(0, 0, 0, 0);
    }
  };
  // A thread's 16 fetched bytes become PPL 16-byte pieces of f64 keys, one run of PPL * 16 bytes per lane: the runs of
  // LPW neighbouring lanes fill a 256-byte bank window. Step s writes piece (s + rot) mod PPL, rot = (tid / LPW) mod PPL,
  // so the lanes that share bank offsets write different pieces and each 16-lane group of a write covers 64 banks.
  constexpr int PPL = 8 / VB, LPW = 256 / (PPL * 16);
  const int rot = (tid / LPW) % PPL;
  auto store = [&]() {
    #pragma unroll
    for (int k = 0; k < RAW; k++) {
      const int e = (k * NT + tid) * (16 / VB), p = e / HD, d = e % HD;
      const uint32_t w0 = raw[k].x, w1 = raw[k].y, w2 = raw[k].z, w3 = raw[k].w;
      #pragma unroll
      for (int s = 0; s < PPL; s++) {
        const int pc = (s + rot) % PPL;
        double lo, hi;
        if (F16KV) {  // piece pc = the two f16 keys of word pc
          const uint32_t wd = pc == 0 ? w0 : pc == 1 ? w1 : pc == 2 ? w2 : w3;
          lo = (double)h2f((uint16_t)(wd & 0xffff));
          hi = (double)h2f((uint16_t)(wd >> 16));
        } else {      // piece pc = the f32 keys of words 2 pc, 2 pc + 1
          lo = (double)__uint_as_float(pc == 0 ? w0 : w2);
          hi = (double)__uint_as_float(pc == 0 ? w1 : w3);
        }
        *(double2 *)(kd + p * KP + d + 2 * pc) = make_double2(lo, hi);
      }
    }
  };
  fetch(bx * MM_PT);
  for (int ti = bx; ti < ntile; ti += X) {
    const int t0 = ti * MM_PT, c1 = min(t0 + MM_PT, nmax);
    __syncthreads();  // the previous tile's reads are done
    store();
    __syncthreads();
    if (ti + X < ntile) fetch((ti + X) * MM_PT);
    if (waveok) {
      #pragma unroll 1
      for (int pt = 0; pt < MM_PT && t0 + pt < c1; pt += 16) {
        d4 acc[NP];
        #pragma unroll
        for (int j = 0; j < NP; j++) {
          acc[j] = d4{0.0, 0.0, 0.0, 0.0};
          #pragma unroll
          for (int m = 0; m < 8; m++)
            acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[j][m], kd[(pt + n16) * KP + 32 * j + 4 * m + g], acc[j], 0, 0, 0);
        }
        const int t = t0 + pt + n16;
        #pragma unroll
        for (int v = 0; v < 4; v++) {
          double sv[NP];
          #pragma unroll
          for (int j = 0; j < NP; j++) sv[j] = acc[j][v];
          // the butterfly of k_attn_scores over the position's NP lanes: pairs, then pairs of pairs
          #pragma unroll
          for (int w = 1; w < NP; w *= 2)
            #pragma unroll
            for (int j = 0; j < NP; j += 2 * w) sv[j] = sv[j] + sv[j + w];
          if (t < rn[v]) a.scores[((long)rb[v] * a.nHead + rh[v]) * a.sld + t] = (float)(sv[0] * a.scale);
        }
      }
    }
  }
}

size_t attention_mm_lds(int hd) { return (size_t)MM_PT * (hd + 2) * 8; }


// ---- chunks of a row. A row of positions 0 .. pos is cut into chunks of ATTN_CHUNK positions. Each chunk is a softmax
// and a weighted sum of its own, with the reference's arithmetic (src/compute/ref-kernels.js:313-320,
// src/model/forward.js:131-134): m_c = the chunk's largest score, e_t = exp(s_t - m_c) (f64), l_c = their sum,
// p_t = f32(f32(e_t) * (1 / l_c)), o_c = the f32 chain of p_t V_t over the chunk's positions in order. A row of one
// chunk is the reference's row bit for bit. A longer row's chunks are joined in f64 in chunk order,
//   out = f32(sum_c w_c o_c / sum_c w_c),  w_c = exp(m_c - max m) l_c,
// so its chains run side by side instead of one dependent step per position over the whole row: a 16K-position head
// took 16,384 steps of ~4 ns on one wave. Chunks start at multiples of ATTN_CHUNK, so the order is a function of the
// position alone and a token gets the same bits in a pass of any size. Against float64 the joined chunks are closer than
// the single f32 chain, whose rounding errors grow with its length.
//
// Infinities and NaN come out as in a softmax over the whole row. A chunk of a longer row without a score above -inf is
// taken against 0 in place of its maximum (chunk_max), so l_c and the probabilities are 0 where every score is -inf
// (which counts for nothing beside a finite score elsewhere, except that 0 times a V of inf or NaN is NaN) and NaN where
// one is NaN. No chunk is left out for a weight of 0.
//
// A chunk of a longer row leaves a record [m_c, l_c (lane chains), o_c of 32 dimensions] in a.rec ([token][head][32-dimension slice]
// [chunk]); the block that arrives last at the counter of its (token, head, slice) or row block joins them. The hand-off
// is that of the GEMV's K parts: device-coherent stores, complete (vmcnt(0)) before the relaxed arrival, device-coherent
// loads by the last.
constexpr int REC_D = ATTN_REC_DOUBLES;
// Chunks of a row that have blocks of their own. The blocks of caches of more chunks walk several (WALK: chunks z, z + 16,
// ...), so a launch stops growing with the cache's capacity: with a block per chunk a token at position 700 of a cache of
// 262,144 cost 4 layers of the 0.6B shapes 299 us where one of 1024 costs 176. The kernels below that have no loop over
// chunks, whose registers (constants kept across the chunks) would cost occupancy: k_attn_av 143 -> 175.
constexpr int ATTN_ZMAX = 16;
// The thread's index, in a walk as a value of its own in every chunk, so that what follows from it is formed there and not
// kept in registers across the chunks.
template <bool WALK>
__device__ __forceinline__ int thread_index() {
  int t = threadIdx.x;
  if constexpr (WALK) __asm__ volatile("" : "+v"(t));
  return t;
}
__device__ __forceinline__ double *chunk_rec(const AttnArgs &a, int b, int h, int slice, int c) {
  return a.rec + ((((long)b * a.nHead + h) * (a.hd >> 5) + slice) * a.nchunk + c) * REC_D;
}
// o of dimension `lane` on 32 consecutive lanes, m and l the same on all of them
__device__ __forceinline__ void chunk_store(double *r, int lane, double m, double l, float o) {
  __hip_atomic_store((float *)(r + 2) + lane, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (lane < 2) __hip_atomic_store(r + lane, lane == 0 ? m : l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// what a chunk's exponentials are taken against, and 1 / sum of them
__device__ __forceinline__ double chunk_max(double m, int nrow) { return nrow > ATTN_CHUNK && m == -INFINITY ? 0.0 : m; }
__device__ __forceinline__ double chunk_inv(double l) { return l == 0.0 ? 0.0 : 1.0 / l; }
// The joined outputs of dimension `lane` (32 consecutive lanes) of NS neighbouring slices of n chunks' records at r
// (slices lds apart); ml(c) gives chunk c's (m, l).
template <int NS, typename ML>
__device__ __forceinline__ void chunk_join(const double *r, long lds, int n, int lane, const ML &ml, float (&out)[NS]) {
  constexpr int NJ = NS > 1 ? 4 : 8;  // chunks whose loads are issued together
  float M = -INFINITY;
  for (int c = lane; c < n; c += 32) M = fmaxf(M, (float)ml(c).x);
  M = group_fmax(M, 32);
  double L = 0.0, O[NS];
  #pragma unroll
  for (int i = 0; i < NS; i++) O[i] = 0.0;
  for (int c0 = 0; c0 < n; c0 += 32) {
    const int nc = min(32, n - c0);
    const double2 v = ml(min(c0 + lane, n - 1));
    const double w = v.x == -INFINITY && M != -INFINITY ? v.y : exp(v.x - (double)M) * v.y;  // (l = 0 or NaN there)
    for (int j0 = 0; j0 < nc; j0 += NJ) {
      float o[NS][NJ];
      #pragma unroll
      for (int i = 0; i < NS; i++)
        #pragma unroll
        for (int j = 0; j < NJ; j++)
          o[i][j] = __hip_atomic_load((const float *)(r + i * lds + (long)(c0 + min(j0 + j, nc - 1)) * REC_D + 2) + lane,
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      #pragma unroll
      for (int j = 0; j < NJ; j++) {
        const double wj = __shfl(w, min(j0 + j, nc - 1), 32);
        if (j0 + j < nc) {
          L += wj;
          #pragma unroll
          for (int i = 0; i < NS; i++) O[i] = fma(wj, (double)o[i][j], O[i]);
        }
      }
    }
  }
  #pragma unroll
  for (int i = 0; i < NS; i++) out[i] = (float)(O[i] / L);
}

// The head output of 32 dimensions on 32 consecutive lanes: the output gate when there is one
// (src/model/forward-qwen35.js:103: o * sigmoid(gate), f64, stored f32), the f32 row, its quantisation.
__device__ __forceinline__ void attn_emit(const AttnArgs &a, int b, int h, int dim, float o) {
  const int col = h * a.hd + dim;
  if (a.gate) {
    const double g = (double)a.gate[(long)b * a.ldq + (long)h * a.qhs + dim];
    o = (float)((double)o * (1.0 / (1.0 + exp(-g))));
  }
  if (a.out) a.out[(long)b * a.ldo + col] = o;
  if (a.act.q) quant_block32(o, col, a.act, b);  // (unset: the output GEMV quantises the f32 rows itself)
}

// One block per (32-dim slice, query head, token, chunk). The slice's V rows (dimension-major in the cache) are staged
// through LDS in pieces of AV_ROW bytes per dimension, double buffered, the first one during the softmax. The chain runs
// on lanes 0-31 of wave 0, one output dimension each, reading 16 bytes of consecutive positions at a time. Bound by the
// dependent fma of the chain (~4 ns per position, at most ATTN_CHUNK of them); three blocks fit a CU's LDS.
constexpr int AV_DIMS = 32;       // output dimensions per block
constexpr int AV_ROW = 512;       // bytes of one dimension's positions per staged piece
constexpr int AV_PITCH = AV_ROW + 16;   // LDS row pitch (the pad spreads the chain's rows over the banks)
constexpr int AV_STAGE = AV_DIMS * AV_PITCH;
constexpr int AV_UNIT = 32;       // positions per unrolled step of the weighted sum

// NSC: scores per thread (256 NSC >= the positions of a chunk), held in registers from the load to the probabilities
template <bool F16KV, int NSC, bool WALK>
__device__ __forceinline__ void av_chunk(const AttnArgs &a, int chunk, int b, int stB, int stPos0, uint8_t *lds) {
  constexpr int VB = F16KV ? 2 : 4;
  constexpr int CT = AV_ROW / VB;        // positions per staged piece
  constexpr int EPP = 16 / VB;           // positions per 16-byte load
  constexpr int PPR = AV_ROW / 16;       // loads per row
  constexpr int LPT = AV_DIMS * PPR / 256;   // 16-byte loads per thread per staged piece
  constexpr int NP = 256 * NSC;          // positions per block at most
  const int h = blockIdx.y, tid = thread_index<WALK>(), wave = tid >> 6, lane = tid & 63;
  const int hd = a.hd, kvh = h / (a.nHead / a.nHeadKv), NS = hd / AV_DIMS;
  const int slice = blockIdx.x;
  const int t00 = chunk * ATTN_CHUNK, ctxc = a.ctx - t00;  // the chunk's first position, cache positions from there on
  float *p = (float *)lds;               // [NP] probabilities
  uint8_t *vbuf = lds + NP * 4;          // [2][AV_DIMS][AV_PITCH] staged V rows
  __shared__ double redd[4];
  __shared__ float redf[4];
  const uint8_t *vbase =
      (const uint8_t *)a.vcache + ((((long)a.layer * a.nHeadKv + kvh) * hd + (long)slice * AV_DIMS) * a.vstride + t00) * VB;
  uint4 pre[LPT];
  // V of piece c below `lim` positions (inside the cache row); the first piece and the scores are requested before the
  // pass's step record arrives, and what lies at or past the last position is zeroed after it
  auto fetch = [&](int c, int lim) {
    #pragma unroll
    for (int k = 0; k < LPT; k++) {
      const int idx = k * 256 + tid, dim = idx / PPR, t = c * CT + (idx % PPR) * EPP;
      pre[k] = t < lim ? *(const uint4 *)(vbase + ((long)dim * a.vstride + t) * VB) : make_uint4(0, 0, 0, 0);
    }
  };
  auto store = [&](int buf) {
    #pragma unroll
    for (int k = 0; k < LPT; k++) {
      const int idx = k * 256 + tid;
      *(uint4 *)(vbuf + buf * AV_STAGE + (idx / PPR) * AV_PITCH + (idx % PPR) * 16) = pre[k];
    }
  };
  // the scores, then the first V piece: loads complete in order, so the softmax below waits for the scores alone while V
  // is on its way
  const float *srow = a.scores + ((long)b * a.nHead + h) * a.sld + t00;
  float v[NSC];
  #pragma unroll
  for (int k = 0; k < NSC; k++) { const int t = k * 256 + tid; v[k] = srow[t < ctxc ? t : 0]; }  // (t >= npos: unused)
  __builtin_amdgcn_sched_barrier(0);
  #pragma unroll
  for (int k = 0; k < LPT; k++) {  // unconditional loads (what lies past the cache's positions reads position 0, zeroed
                                   // below with all at or past the last position): a load under a branch would make
                                   // the first use of the scores wait for it too
    const int idx = k * 256 + tid, dim = idx / PPR, t = (idx % PPR) * EPP;
    pre[k] = *(const uint4 *)(vbase + ((long)dim * a.vstride + (t < ctxc ? t : 0)) * VB);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (b >= stB) return;
  const int nrow = stPos0 + b + 1, npos = min(nrow - t00, ATTN_CHUNK);  // the row's positions, the chunk's
  if (npos <= 0) return;
  const int nch = (npos + CT - 1) / CT;
  // ---- softmax (src/compute/ref-kernels.js:313-320): thread tid holds t = tid + 256 k, its exponentials added in k order
  float mx = -INFINITY;
  #pragma unroll
  for (int k = 0; k < NSC; k++) { v[k] = k * 256 + tid < npos ? v[k] : -INFINITY; mx = fmaxf(mx, v[k]); }
  mx = group_fmax(mx, 64);
  if (lane == 0) redf[wave] = mx;
  __syncthreads();
  const double m = (double)fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3])), mz = chunk_max(m, nrow);
  double sum = 0.0;
  #pragma unroll
  for (int k0 = 0; k0 < NSC; k0 += 4) {
    if (k0 * 256 < npos) {  // (uniform)
      double e[4];  // four independent chains
      #pragma unroll
      for (int k = 0; k < 4; k++) e[k] = exp_neg((double)v[k0 + k] - mz);
      #pragma unroll
      for (int k = 0; k < 4; k++) {
        const bool on = (k0 + k) * 256 + tid < npos;
        if (on) sum += e[k];
        v[k0 + k] = on ? (float)e[k] : 0.f;
      }
    }
  }
  sum = wave_sum_xor(sum, 64);
  if (lane == 0) redd[wave] = sum;
  __syncthreads();
  const double l = (redd[0] + redd[1]) + (redd[2] + redd[3]), inv = chunk_inv(l);
  #pragma unroll
  for (int k = 0; k < NSC; k++) {  // (zeros from the last position to the end of its unit, at least)
    const int t = k * 256 + tid;
    if (k * 256 < npos) p[t] = t < npos ? (float)((double)v[k] * inv) : 0.f;
  }
  // the last piece from the last position on: zeros (the cache may hold anything there, inf and NaN of a discarded token
  // included, and a probability of 0 does not take those out of the sum); a thread's loads are of the same positions of
  // different dimensions
  auto trim = [&](int c) {
    static_assert(256 % PPR == 0, "one set of positions per thread");
    const int r = npos - c * CT - (tid % PPR) * EPP;  // how many of them lie below the last position
    uint32_t w[4];
    #pragma unroll
    for (int e = 0; e < 4; e++) w[e] = !F16KV ? (r > e ? ~0u : 0u) : r > 2 * e + 1 ? ~0u : r > 2 * e ? 0xffffu : 0u;
    #pragma unroll
    for (int k = 0; k < LPT; k++) pre[k] = make_uint4(pre[k].x & w[0], pre[k].y & w[1], pre[k].z & w[2], pre[k].w & w[3]);
  };
  if (nch == 1) trim(0);
  store(0);
  __syncthreads();
  // ---- weighted sum of V: f32 fma chain in position order, one output dimension per lane (lanes 0-31 of wave 0)
  const bool chainLane = wave == 0 && lane < AV_DIMS;
  float o = 0.f;
  for (int c = 0; c < nch; c++) {
    if (c + 1 < nch) fetch(c + 1, npos);
    if (chainLane) {
      // units of UNIT positions, software pipelined: the LDS reads of unit u + 1 are issued before the fma steps of
      // unit u, so the chain (one dependent fma per position, ~4 ns each) does not wait out an LDS latency per unit.
      // p and V are zero past the last position, so a unit may run past `cnt`: fmaf(0, 0, o) == o. The read-ahead index
      // is clamped to the chunk's last unit (a re-read, never past it).
      const int t0 = c * CT, cnt = min(CT, npos - t0), nu = (cnt + AV_UNIT - 1) / AV_UNIT;
      const uint8_t *row = vbuf + (c & 1) * AV_STAGE + lane * AV_PITCH;
      const float *pc = p + t0;
      float4 pa[AV_UNIT / 4], pb[AV_UNIT / 4];
      uint4 va[AV_UNIT * VB / 16], vb[AV_UNIT * VB / 16];
      auto read = [&](int u, float4 (&pv)[AV_UNIT / 4], uint4 (&vv)[AV_UNIT * VB / 16]) {
        #pragma unroll
        for (int k = 0; k < AV_UNIT / 4; k++) pv[k] = *(const float4 *)(pc + u * AV_UNIT + 4 * k);
        #pragma unroll
        for (int k = 0; k < AV_UNIT * VB / 16; k++) vv[k] = *(const uint4 *)(row + (u * AV_UNIT + k * EPP) * VB);
      };
      auto steps = [&](const float4 (&pv)[AV_UNIT / 4], const uint4 (&vv)[AV_UNIT * VB / 16]) {
        #pragma unroll
        for (int k = 0; k < AV_UNIT / 4; k++) {
          float v0, v1, v2, v3;
          if (F16KV) {
            const uint4 &w = vv[k >> 1];
            const uint32_t lo = (k & 1) ? w.z : w.x, hi = (k & 1) ? w.w : w.y;
            v0 = h2f((uint16_t)(lo & 0xffff)); v1 = h2f((uint16_t)(lo >> 16));
            v2 = h2f((uint16_t)(hi & 0xffff)); v3 = h2f((uint16_t)(hi >> 16));
          } else {
            const uint4 &w = vv[k];
            v0 = __uint_as_float(w.x); v1 = __uint_as_float(w.y); v2 = __uint_as_float(w.z); v3 = __uint_as_float(w.w);
          }
          o = fmaf(pv[k].x, v0, o); o = fmaf(pv[k].y, v1, o); o = fmaf(pv[k].z, v2, o); o = fmaf(pv[k].w, v3, o);
        }
      };
      // two units per iteration and no branch between a unit's reads and its steps (a branch there lets the compiler
      // sink the reads to their use); an odd last unit is already in (pa, va) after the loop
      read(0, pa, va);
      int u = 0;
      for (; u + 2 <= nu; u += 2) {
        read(u + 1, pb, vb);
        __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the steps (the scheduler moves them to their use)
        steps(pa, va);
        read(min(u + 2, nu - 1), pa, va);
        __builtin_amdgcn_sched_barrier(0);
        steps(pb, vb);
      }
      if (u < nu) steps(pa, va);
    }
    __syncthreads();
    if (c + 1 < nch) {
      if (c + 2 == nch) trim(c + 1);
      store((c + 1) & 1);
    }
    __syncthreads();
  }
  if (!chainLane) return;
  if (nrow <= ATTN_CHUNK) {
    attn_emit(a, b, h, slice * AV_DIMS + lane, o);
    return;
  }
  chunk_store(chunk_rec(a, b, h, slice, chunk), lane, m, l, o);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores are complete
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  const int n = (nrow + ATTN_CHUNK - 1) / ATTN_CHUNK;
  uint32_t *cnt = a.rcnt + ((long)b * a.nHead + h) * NS + slice;
  uint32_t at = 0;
  if (lane == 0) at = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane(at) != (uint32_t)(n - 1)) return;
  if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const double *r = chunk_rec(a, b, h, slice, 0);
  auto ml = [&](int c) {
    return make_double2(__hip_atomic_load(r + (long)c * REC_D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                        __hip_atomic_load(r + (long)c * REC_D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  float out[1];
  chunk_join<1>(r, 0, n, lane, ml, out);
  attn_emit(a, b, h, slice * AV_DIMS + lane, out[0]);
}

// Grid (slices, heads, nz x tokens), chunks slowest (a row's short last chunk would otherwise take a place on a CU ahead of
// a whole chunk of another row). Chunk 0's first loads go out before the pass's step record arrives; a block of a later
// chunk waits for the record, as in a cache longer than the row it has nothing to load.
template <bool F16KV, int NSC, bool WALK>
__global__ __launch_bounds__(256) void k_attn_av(const AttnArgs a, int nB, int nz) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int z = blockIdx.z / nB, b = blockIdx.z - z * nB;
  const int stB = a.step->B, stPos0 = a.step->pos0;  // the pass's step record (scalar loads, read before the pins)
  pin_args(a.hd, a.nHead, a.nHeadKv, a.layer, a.vstride, a.vcache, a.scores, a.sld, a.ctx);
  for (int chunk = z;; chunk += nz) {
    if (chunk > 0) {
      __asm__ volatile("");  // (keeps the test of the record a branch of its own: chunk 0 does not wait for it)
      if (b >= stB || chunk * ATTN_CHUNK > stPos0 + b) return;
    }
    av_chunk<F16KV, NSC, WALK>(a, chunk, b, stB, stPos0, lds);
    if (!WALK) return;
  }
}

// The probabilities of every (chunk, query head, token) part of a pass of several tokens, in place of its scores, and its
// (m_c, l_c). One wave per part: lane i takes k_attn_av's threads i, i + 64, i + 128 and i + 192 (their positions in their
// order, then the same four 64-lane sums and (w0 + w1) + (w2 + w3)), so a part has one maximum and no barrier. Bound by
// the f64 exponentials (~30 VALU instructions a position); with four waves per part their reductions cost as much again.
// Grid (heads, tokens, chunks): with the chunks fastest the 8 or 16 of a large cache, most of them past the row, put every
// row's live ones on the same few of the 8 XCDs (workgroup i runs on XCD i mod 8): 64 tokens of 16 heads after 7000
// positions took 19 us in a cache of 8K and 43 in one of 32K.
template <bool WALK>
__global__ __launch_bounds__(64) void k_attn_softmax_rows(const AttnArgs a) {
  constexpr int NK = ATTN_CHUNK / 64;
  const int h = blockIdx.x, b = blockIdx.y;
  const Step *st = a.step;
  const int nrow = st->pos0 + b + 1;
  if (b >= st->B) return;
  for (int chunk = blockIdx.z; chunk * ATTN_CHUNK < nrow; chunk += gridDim.z) {
    const int lane = thread_index<WALK>();
    const int t00 = chunk * ATTN_CHUNK, npos = min(nrow - t00, ATTN_CHUNK);
    float *srow = a.scores + ((long)b * a.nHead + h) * a.sld + t00;
    float v[NK], mx = -INFINITY;
    #pragma unroll
    for (int k = 0; k < NK; k += 8)
      if (k * 64 < npos) {  // (uniform; a position past the last repeats the first)
        #pragma unroll
        for (int j = k; j < k + 8; j++) { const int t = j * 64 + lane; v[j] = srow[t < npos ? t : 0]; }
      }
    #pragma unroll
    for (int k = 0; k < NK; k += 8)
      if (k * 64 < npos) {
        #pragma unroll
        for (int j = k; j < k + 8; j++) mx = fmaxf(mx, v[j]);
      }
    mx = group_fmax(mx, 64);
    const double m = (double)mx, mz = chunk_max(m, nrow);
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    #pragma unroll
    for (int k = 0; k < NK; k += 4)
      if (k * 64 < npos) {  // positions 256 (k / 4) + 64 w + lane of the four waves w
        double e[4];
        #pragma unroll
        for (int w = 0; w < 4; w++) e[w] = exp_neg((double)v[k + w] - mz);
        #pragma unroll
        for (int w = 0; w < 4; w++) {
          if ((k + w) * 64 + lane < npos) sum[w] += e[w];
          v[k + w] = (float)e[w];
        }
      }
    #pragma unroll
    for (int w = 0; w < 4; w++) sum[w] = wave_sum_xor(sum[w], 64);
    const double l = (sum[0] + sum[1]) + (sum[2] + sum[3]), inv = chunk_inv(l);
    #pragma unroll
    for (int k = 0; k < NK; k += 4)
      if (k * 64 < npos) {
        #pragma unroll
        for (int j = k; j < k + 4; j++) {
          const int t = j * 64 + lane;
          if (t < npos) srow[t] = (float)((double)v[j] * inv);
        }
      }
    if (lane == 0) a.cml[((long)b * a.nHead + h) * a.nchunk + chunk] = make_double2(m, l);
    if (!WALK) return;
  }
}

// ---- weighted sum of passes of several tokens on the matrix cores. v_mfma_f32_16x16x4_f32 adds its four products to
// the accumulator as four fused multiply-adds in k order (measured on gfx950, every element of random wide-range
// operands), so a chain of them over positions t, t + 1, ... in order is the reference's f32 chain out += p_t v_t
// (one rounding per position, src/model/forward.js:131-134) for 16 rows x 16 dimensions at once: the bits of k_attn_av.
// Block: one chunk of 16 rows r = b G + g (token b, query head kvh G + g) and 32 NDG dimensions of a KV head. A chain wave runs
// 16 CPW dimensions: one chain, or two that share the A operand (lane l supplies A = p[row l mod 16][position 4 m + l / 16],
// B = V[dimension l mod 16 (+ 16)][4 m + l / 16] and holds (row 4 (l / 16) + v, dimension l mod 16)); the producer waves stage
// piece c + 1 meanwhile: V as f32 (zero past the pass's last position) and the probabilities (already normalised by
// k_attn_softmax_rows, zero past a row's last position), with up to four pieces more on their way in registers (a piece takes
// ~0.5 us, a load from memory 2-3); one barrier per piece. Operands lie in LDS by position mod 4 (section k holds positions
// 4 m + k), so a 16-byte read gives four MFMAs' operands and the chain waves issue nothing but MFMAs and reads.
// Bound by the MFMAs (32 cycles each) and, per piece, the barrier and the first reads behind it, with the producers'
// instructions close behind (a wave alone on a SIMD issues one every ~7 cycles, two one every ~5). A wave of two chains reads
// 384 bytes of LDS per MFMA, of one chain 512, but two chains on one SIMD take twice the time of one: they are for launches
// that fill the chip anyway. Pieces of 64 positions, so two blocks of 128 dimensions fit a CU, or four of 32 (with pieces of 128
// or four producer waves fewer: 9 tokens of 32 heads after 16384 positions, 864 blocks, 451 us a pass of two layers, 453 and 474).
template <bool B> struct Whole { static constexpr bool value = B; };  // a piece below every row's last position
constexpr int MMV_RB = 16;                  // rows per block
constexpr int MMV_CT = 64;                  // positions per staged piece
constexpr int MMV_SF = MMV_CT / 4;          // floats of one position section
constexpr int MMV_RS = 4 * MMV_SF + 4;      // floats of one dimension or row (4 x an odd number: conflict-free chain reads)
// NDG x CPW: 4 x 2 (128 dimensions, two chains per wave) or 1 x 1 (32, one chain per wave)
constexpr int mmv_producers(int cpw) { return cpw == 2 ? 8 : 2; }
constexpr int mmv_waves(int ndg, int cpw) { return 2 * ndg / cpw + mmv_producers(cpw); }
template <bool F16KV, int NDG, int CPW, bool WALK>
__device__ __forceinline__ void av_mm_chunk(const AttnArgs &a, int nrows, int chunk, int L, uint8_t *lds) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int VB = F16KV ? 2 : 4, DB = 32 * NDG, RB = MMV_RB;
  constexpr int CT = MMV_CT, SF = MMV_SF, RS = MMV_RS, NPT = mmv_producers(CPW) * 64;
  constexpr int EPP = 16 / VB;                      // positions per 16-byte V load
  constexpr int UL = 16 / EPP;                      // V loads per unit of 16 positions (2 f16, 4 f32)
  constexpr int UPR = CT / 16;                      // units per dimension of a piece
  constexpr int D = F16KV ? 4 : 2;                  // pieces in flight (as many as the registers hold)
  constexpr int VU = DB * UPR / NPT;                // V units per producer thread per piece
  constexpr int PN = RB * CT / NPT;                 // probabilities per producer thread per piece
  constexpr int NCW = 2 * NDG / CPW;                // chain waves
  static_assert(VU * NPT == DB * UPR && (PN == 2 || PN == 8) && (CPW == 1 || CPW == 2), "producer units");
  float *vk = (float *)lds;                         // [2][DB][RS]: V of position 4 m + k, dimension j at j RS + k SF + m
  float *pk = vk + 2 * DB * RS;                     // [2][RB][RS]: p of row i, position 4 m + k at i RS + k SF + m
  __shared__ long roff[RB];
  __shared__ int rnp[RB], rfull[RB];                // the row's positions in the chunk, and in all
  __shared__ uint32_t arrived;
  const int tid = thread_index<WALK>(), lane = tid & 63, n16 = lane & 15, g = lane >> 4;
  // wave w of a block runs on SIMD w mod 4: every other four-wave block takes its last two for the chains, so that two blocks
  // on a CU use the matrix pipes of all four (1 % of a pass)
  const int wave = CPW == 1 ? (tid >> 6) ^ (L & 1) * 2 : tid >> 6;
  const int ND = a.hd / DB, NZ = (nrows + RB - 1) / RB;
  const int kvh = L / (ND * NZ), rbk = (L / ND) % NZ, d0 = (L % ND) * DB;
  const int G = a.nHead / a.nHeadKv;
  const Step *st = a.step;
  // positions below are relative to the chunk's first one, t00
  const int t00 = chunk * ATTN_CHUNK;
  const int Bd = st->B, pos0 = st->pos0, nmax = pos0 + Bd - t00;
  // the block's rows: scores row offsets, positions (0: no row; such a row reads the block's first one)
  const long r0h = ((long)(rbk * RB / G) * a.nHead + kvh * G) * a.sld, r00 = r0h + t00;
  if (tid < RB) {
    const int r = rbk * RB + tid, b = r / G, h = kvh * G + r % G;
    const bool live = r < nrows && b < Bd;
    roff[tid] = (live ? ((long)b * a.nHead + h) * a.sld : r0h) + t00;
    rfull[tid] = live ? pos0 + b + 1 : 0;
    rnp[tid] = max(0, min(rfull[tid] - t00, ATTN_CHUNK));
  }
  __syncthreads();
  // a piece that ends at or before every live row's last position (all pieces but the last one or two) needs no load
  // clamped and no value zeroed: fetch and stage take it in a form without those checks (rows without a live query read
  // the block's first one there; their outputs are never stored, and row i of an MFMA result depends on row i of A only)
  int nrmax = 0, nrfull = 0, nrmin = INT_MAX;
  #pragma unroll
  for (int i = 0; i < RB; i++) {
    nrmax = max(nrmax, rnp[i]);
    nrfull = max(nrfull, rfull[i]);
    nrmin = rnp[i] > 0 ? min(nrmin, rnp[i]) : nrmin;
  }
  if (nrmax == 0) return;  // (uniform)
  const int nch = (nrmax + CT - 1) / CT;
  const int nend = (nrmax + AV_UNIT - 1) / AV_UNIT * AV_UNIT;  // positions the chains run
  const uint8_t *vbase = (const uint8_t *)a.vcache + ((((long)a.layer * a.nHeadKv + kvh) * a.hd + d0) * a.vstride + t00) * VB;
  const bool producer = wave >= NCW;
  f4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  // the producers and the chain waves run loops of their own with one barrier per piece each (the same count), so the
  // chains' accumulators stay in their registers from piece to piece
  if (producer) {
    const int pt = (wave - NCW) * 64 + lane;                  // producer thread 0 .. NPT - 1
    const int pr = pt * PN / CT, pq = pt * PN % CT; // its row and first position of its PN probabilities in a piece
    const int np = rnp[pr];
    // both by buffer loads and no branch around a load, so that the waits count exactly the piece they are for. Up to D
    // pieces past the block's last one are requested (and never staged), so a load's whole offset, the piece's part
    // included, is its vector offset: that is what the range check compares with the resource's size (the end of the V
    // rows and of the pass's scores), and past it a load returns zeros without an access. A scalar offset may be left
    // out of that comparison, or be larger than the resource.
    const uint32_t vrow = (uint32_t)a.vstride * VB;
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc((void *)vbase, (short)0, (int)(DB * vrow - t00 * VB), 0x00020000);
    const long pend = (long)Bd * a.nHead * a.sld - r00;  // floats from the block's first row on
    const __amdgpu_buffer_rsrc_t pr_ =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.scores + r00), (short)0, (int)(uint32_t)min(pend * 4, 0xfffffff0l), 0x00020000);
    const uint32_t poff = (uint32_t)(roff[pr] - r00 + pq) * 4;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    struct Pre {
      u4 v[VU][UL];
      float p[PN];
    };
    // piece c's V and scores (what lies past a row's or the pass's last position is zeroed when the piece is staged)
    auto fetch = [&](int c, Pre &s) {
      const uint32_t t0 = (uint32_t)c * CT;
      #pragma unroll
      for (int k = 0; k < VU; k++) {
        const int u = k * NPT + pt, dim = u / UPR;
        const uint32_t vo = dim * vrow + (t0 + (u % UPR) * 16) * VB;
        #pragma unroll
        for (int l = 0; l < UL; l++) s.v[k][l] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(vr, vo + l * 16, 0, 0));
      }
      #pragma unroll
      for (int j = 0; j < PN; j++) s.p[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(pr_, poff + t0 * 4 + 4 * j, 0, 0));
    };
    auto stage_f = [&](auto whole, int c, const Pre &s) {
      constexpr bool W = decltype(whole)::value;
      float *vs = vk + (c & 1) * DB * RS;
      #pragma unroll
      for (int k = 0; k < VU; k++) {
        const int u = k * NPT + pt, dim = u / UPR, uu = u % UPR, t0 = c * CT + uu * 16;
        float f[16];
        #pragma unroll
        for (int e = 0; e < 16; e++) {
          const int w = e % EPP;
          const uint32_t wd = s.v[k][e / EPP][F16KV ? w >> 1 : w];
          const float x = F16KV ? h2f((uint16_t)((w & 1) ? (wd >> 16) : (wd & 0xffff))) : __uint_as_float(wd);
          f[e] = W || t0 + e < nmax ? x : 0.f;
        }
        float *drow = vs + dim * RS + uu * 4;
        #pragma unroll
        for (int q = 0; q < 4; q++) *(f4 *)(drow + q * SF) = (f4){f[q], f[q + 4], f[q + 8], f[q + 12]};
      }
      float *prow = pk + (c & 1) * RB * RS + pr * RS + (pq >> 2);
      #pragma unroll
      for (int j = 0; j < PN; j++) prow[((pq + j) & 3) * SF + (PN > 4 ? j >> 2 : 0)] = W || c * CT + pq + j < np ? s.p[j] : 0.f;
    };
    auto stage = [&](int c, const Pre &s) {
      if ((c + 1) * CT <= nrmin) stage_f(Whole<true>{}, c, s);
      else stage_f(Whole<false>{}, c, s);
    };
    // piece c lies in register set c mod D, which requests piece c + D as soon as it is staged
    Pre s[D];
    #pragma unroll
    for (int d = 0; d < D; d++) fetch(d, s[d]);
    stage(0, s[0]);
    fetch(D, s[0]);
    __syncthreads();
    for (int c0 = 0; c0 < nch; c0 += D) {  // piece c + 1 is staged while the chains run piece c
      #pragma unroll
      for (int d = 0; d < D; d++) {
        const int c = c0 + d;
        if (c >= nch) break;
        if (c + 1 < nch) stage(c + 1, s[(d + 1) % D]);
        fetch(c + 1 + D, s[(d + 1) % D]);
        __syncthreads();
      }
    }
  } else {
    __syncthreads();
    constexpr int Y = CPW == 2 ? 16 * RS : 0;       // the second chain's dimensions (none: the same reads)
    auto ld = [&](const float *q) { return *(const f4 *)q; };
    const float *vr0 = vk + (wave * 16 * CPW + n16) * RS + g * SF, *pr0 = pk + n16 * RS + g * SF;
    for (int c = 0; c < nch; c++) {
      // 16 positions per step (4 MFMAs per chain; lane group g: positions 4 m + g, m = 4 u .. 4 u + 3), the next step's
      // reads ahead of the current one's MFMAs; two steps per unit of 32 positions
      const float *vr = vr0 + (c & 1) * DB * RS, *pr = pr0 + (c & 1) * RB * RS;
      auto step = [&](const f4 &p, const f4 &v0, const f4 &v1) {
        #pragma unroll
        for (int i = 0; i < 4; i++) {
          acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i], v0[i], acc0, 0, 0, 0);
          if constexpr (CPW == 2) acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(p[i], v1[i], acc1, 0, 0, 0);
        }
      };
      const int nu = min(CT, nend - c * CT) / 16;  // an even number of steps
      f4 p0 = ld(pr), x0 = ld(vr), y0 = ld(vr + Y);
      f4 p1 = ld(pr + 4), x1 = ld(vr + 4), y1 = ld(vr + Y + 4);
      __builtin_amdgcn_sched_barrier(0);
      step(p0, x0, y0);
      #pragma unroll
      for (int u = 2; u < CT / 16; u += 2)
        if (nu > u) {
          p0 = ld(pr + 4 * u); x0 = ld(vr + 4 * u); y0 = ld(vr + Y + 4 * u);
          __builtin_amdgcn_sched_barrier(0);
          step(p1, x1, y1);
          p1 = ld(pr + 4 * u + 4); x1 = ld(vr + 4 * u + 4); y1 = ld(vr + Y + 4 * u + 4);
          __builtin_amdgcn_sched_barrier(0);
          step(p0, x0, y0);
        }
      step(p1, x1, y1);
      __syncthreads();
    }
  }
  // ---- epilogue: the outputs through LDS (the staged pieces are no longer read), a row's 32 dimensions on 32
  // consecutive lanes (one quantizeAct block)
  constexpr int OP = DB + 1;
  float *ot = (float *)lds;
  if (!producer) {
    #pragma unroll
    for (int v = 0; v < 4; v++) {
      ot[(4 * g + v) * OP + 16 * CPW * wave + n16] = acc0[v];
      if constexpr (CPW == 2) ot[(4 * g + v) * OP + 32 * wave + 16 + n16] = acc1[v];
    }
  }
  __syncthreads();
  constexpr int NH = 2 * mmv_waves(NDG, CPW);       // half-waves
  const int hw = tid >> 5, l32 = tid & 31;
  for (int e = hw; e < RB * NDG; e += NH) {
    const int i = e / NDG, sl = e % NDG;
    if (rnp[i] == 0) continue;
    const int r = rbk * RB + i, b = r / G, h = kvh * G + r % G;
    const float o = ot[i * OP + 32 * sl + l32];
    if (rfull[i] <= ATTN_CHUNK) attn_emit(a, b, h, d0 + 32 * sl + l32, o);
    else __hip_atomic_store((float *)(chunk_rec(a, b, h, d0 / 32 + sl, chunk) + 2) + l32, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (nrfull <= ATTN_CHUNK) return;  // (uniform)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores are complete
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  uint32_t *cnt = a.rcnt + L;
  if (tid == 0) arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrived != (uint32_t)((nrfull + ATTN_CHUNK - 1) / ATTN_CHUNK - 1)) return;  // (the chunks this block's rows have)
  if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int i = hw; i < RB; i += NH) {  // a row's slices together
    if (rfull[i] <= ATTN_CHUNK) continue;
    const int r = rbk * RB + i, b = r / G, h = kvh * G + r % G;
    const double2 *mlr = a.cml + ((long)b * a.nHead + h) * a.nchunk;
    float out[NDG];
    chunk_join<NDG>(chunk_rec(a, b, h, d0 / 32, 0), (long)a.nchunk * REC_D, (rfull[i] + ATTN_CHUNK - 1) / ATTN_CHUNK, l32,
                    [&](int c) { return mlr[c]; }, out);
    #pragma unroll
    for (int sl = 0; sl < NDG; sl++) attn_emit(a, b, h, d0 + 32 * sl + l32, out[sl]);
  }
}

// Grid (blocks of a chunk, nz chunks).
// XCD-aware block order: workgroup i of a chunk's blocks (a multiple of 8) goes to XCD i mod 8, and logical block
// L = (i mod 8) (blocks / 8) + i / 8 gives each XCD a contiguous run of L, ordered dimension block fastest, then row block,
// then KV head, so the blocks that read the same V share one L2
template <bool F16KV, int NDG, int CPW, bool WALK>
__global__ __launch_bounds__(mmv_waves(NDG, CPW) * 64, CPW == 1 ? 4 : NDG * 6 / 4) void k_attn_av_mm(const AttnArgs a, int nrows) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (L >= a.hd / (32 * NDG) * ((nrows + MMV_RB - 1) / MMV_RB) * a.nHeadKv) return;
  const int nmax = a.step->pos0 + a.step->B;
  for (int chunk = blockIdx.y; chunk * ATTN_CHUNK < nmax; chunk += gridDim.y) {
    av_mm_chunk<F16KV, NDG, CPW, WALK>(a, nrows, chunk, L, lds);
    if (!WALK) return;
    __syncthreads();  // the chunk's LDS has been read
  }
}

static size_t attention_av_mm_lds(int ndg) { return (size_t)2 * (32 * ndg + MMV_RB) * MMV_RS * 4; }

// ---- position-split weighted sum (only where it is asked for). Here one block per (256-position chunk, query head, token) takes
// the chunk's scores, its max m_c, e_t = exp(s_t - m_c) and l_c = sum e_t in f64, and o_c[i] = sum e_t V_t,i in f64
// (V staged through LDS with coalesced loads); k_attn_merge then forms out_i = f32(sum_c w_c o_c[i] / sum_c w_c l_c),
// w_c = exp(m_c - max_c m_c), adding the chunks in chunk order. Every order is a function of the position count only,
// so batched and single-token passes agree bit for bit. The result is the softmax-weighted sum in f64, rounded once:
// it differs from the reference's f32 chain (src/model/forward.js:134-139) by that chain's own rounding error, and from the
// joined chunks above by the rounding errors of their chains.
template <bool F16KV>
__global__ __launch_bounds__(256) void k_attn_av_split(const AttnArgs a) {
  extern __shared__ __align__(16) uint8_t lds[];
  constexpr int VB = F16KV ? 2 : 4, C = ATTN_SPLIT_C, EPP = 16 / VB;
  __shared__ double e[C];
  __shared__ double redd[4];
  __shared__ float redf[4];
  const int c = blockIdx.x, h = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hd = a.hd, kvh = h / (a.nHead / a.nHeadKv), t0 = c * C;
  const Step *st = a.step;
  if (b >= st->B) return;
  const int npos = st->pos0 + b + 1;
  if (t0 >= npos) return;
  const int cnt = min(C, npos - t0);
  // V rows of the chunk [hd][C] (dimension-major cache rows), 16 bytes per load, consecutive threads along a row
  const uint8_t *vbase = (const uint8_t *)a.vcache + ((long)a.layer * a.nHeadKv + kvh) * hd * a.vstride * VB;
  // LDS row pitch of C * VB + 4 bytes (an odd number of words): the lanes of a wave, one dimension each, read the same
  // position of consecutive rows from distinct banks
  const int ppr = C / EPP, pitch = C * VB + 4;  // 16-byte pieces per row
  for (int idx = tid; idx < hd * ppr; idx += 256) {
    const int dim = idx / ppr, t = t0 + (idx % ppr) * EPP;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (t < npos) v = *(const uint4 *)(vbase + ((long)dim * a.vstride + t) * VB);
    uint32_t *d = (uint32_t *)(lds + (long)dim * pitch + (idx % ppr) * 16);
    d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
  }
  const float *srow = a.scores + ((long)b * a.nHead + h) * a.sld + t0;
  const float s = tid < cnt ? srow[tid] : -INFINITY;
  float mx = group_fmax(s, 64);
  if (lane == 0) redf[wave] = mx;
  __syncthreads();
  const float m = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
  const double ev = tid < cnt ? exp((double)s - (double)m) : 0.0;
  e[tid] = ev;
  double l = wave_sum_xor(ev, 64);
  if (lane == 0) redd[wave] = l;
  __syncthreads();
  l = (redd[0] + redd[1]) + (redd[2] + redd[3]);
  // o_c[i]: thread (i = tid mod hd, q = tid / hd) adds positions q, q + R, ... (R = 256 / hd), then the R partial sums
  // meet in LDS in q order
  const int R = 256 / hd, i = tid % hd, q = tid / hd;
  double o = 0.0;
  const uint8_t *row = lds + (long)i * pitch;
  for (int t = q; t < cnt; t += R) {
    const float v = F16KV ? h2f(((const uint16_t *)row)[t]) : ((const float *)row)[t];
    o = fma(e[t], (double)v, o);
  }
  __syncthreads();  // the staged V is no longer read: its LDS holds the partial sums
  double *po = (double *)lds;
  po[tid] = o;
  __syncthreads();
  if (tid < hd) {
    double tot = po[tid];
    for (int k = 1; k < R; k++) tot += po[k * hd + tid];
    double *dst = a.part + (((long)b * a.nHead + h) * a.nch + c) * (hd + 2);
    dst[2 + tid] = tot;
    if (tid == 0) { dst[0] = (double)m; dst[1] = l; }
  }
}

__global__ __launch_bounds__(256) void k_attn_merge(const AttnArgs a) {
  const int h = blockIdx.x, b = blockIdx.y, i = threadIdx.x, hd = a.hd;
  const Step *st = a.step;
  if (b >= st->B || i >= hd) return;
  const int npos = st->pos0 + b + 1, nch = (npos + ATTN_SPLIT_C - 1) / ATTN_SPLIT_C;
  const double *pr = a.part + ((long)b * a.nHead + h) * a.nch * (hd + 2);
  double M = -INFINITY;
  for (int c = 0; c < nch; c++) M = fmax(M, pr[(long)c * (hd + 2)]);
  double L = 0.0, O = 0.0;
  for (int c = 0; c < nch; c++) {
    const double *pc = pr + (long)c * (hd + 2);
    const double w = exp(pc[0] - M);
    L += w * pc[1];
    O += w * pc[2 + i];
  }
  float o = (float)(O / L);
  const int col = h * hd + i;
  if (a.gate) {  // gated attention output (src/model/forward-qwen35.js:103): o * sigmoid(gate), f64, stored f32
    const double g = (double)a.gate[(long)b * a.ldq + (long)h * a.qhs + i];
    o = (float)((double)o * (1.0 / (1.0 + exp(-g))));
  }
  if (a.out) a.out[(long)b * a.ldo + col] = o;
  if (a.act.q) quant_block32(o, col, a.act, b);  // (unset: the output GEMV quantises the f32 rows itself)
}

size_t attention_split_lds(int hd, int kvF16) { return (size_t)hd * (ATTN_SPLIT_C * (kvF16 ? 2 : 4) + 4); }

// Dynamic LDS of one k_attn_av block: the probabilities of its positions and two staged pieces of V.
static size_t attention_lds(int nsc) { return (size_t)256 * nsc * 4 + 2 * (size_t)AV_STAGE; }

constexpr int LONG_CTX = 8192;  // contexts from which passes of 2 tokens or more take the matrix-core forms

AttnForm attention_form(int ctx) {
  AttnForm f;
  // matrix-core score dots for passes of 16 tokens or more (prefill chunks), and of 2 or more where the context is long
  // (verify passes at long contexts); ZEROLLM_ATTN_MM_B overrides the token count (tests)
  const char *em = getenv("ZEROLLM_ATTN_MM_B");
  f.mmMinB = em ? atoi(em) : ctx >= LONG_CTX ? 2 : 16;
  // their weighted sums on the matrix cores likewise: from 16 tokens on, and from 2 where the context is long
  const char *ea = getenv("ZEROLLM_ATTN_MMAV_B");
  f.mmAvMinB = ea ? atoi(ea) : em ? f.mmMinB : ctx >= LONG_CTX ? 2 : 16;
  return f;
}

template <bool F16KV, int NDG, int CPW, bool WALK>
static void launch_av_mm_w(const AttnArgs &a, int nrows, hipStream_t st) {
  static bool attr = false;  // dynamic LDS above 64 KB must be requested per kernel
  const size_t lds = attention_av_mm_lds(NDG);
  if (!attr) {
    ZL_HIP(hipFuncSetAttribute((const void *)k_attn_av_mm<F16KV, NDG, CPW, WALK>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = true;
  }
  const int nb = a.hd / (32 * NDG) * a.nHeadKv * ((nrows + MMV_RB - 1) / MMV_RB);  // (dimensions, KV head, rows) blocks
  const dim3 grid((nb + 7) / 8 * 8, std::min(a.nchunk, ATTN_ZMAX));
  hipLaunchKernelGGL((k_attn_av_mm<F16KV, NDG, CPW, WALK>), grid, dim3(mmv_waves(NDG, CPW) * 64), lds, st, a, nrows);
}
template <bool F16KV, int NDG, int CPW>
static void launch_av_mm_k(const AttnArgs &a, int nrows, hipStream_t st) {
  if (a.nchunk > ATTN_ZMAX) launch_av_mm_w<F16KV, NDG, CPW, true>(a, nrows, st);
  else launch_av_mm_w<F16KV, NDG, CPW, false>(a, nrows, st);
}
// One chain per wave and 32 dimensions per block, where each chain wave then has a SIMD's matrix pipe to itself or nearly so
// (a CU holds four blocks), two chains per wave and 128 dimensions, which read V and p less often per MFMA, where the launch
// fills the chip several times over. Only the cache's capacity is known here, so the line is drawn between rows of a quarter
// and of all of it. Whole passes in 32- against 128-dimension blocks: verify 8B, 9 tokens (96 blocks a chunk, 16 chunks) after
// 3000 positions 305 and 346 us, after 15000 403 and 418, after 28000 521 and 526; 5 tokens (64) after 5000 of 8K 292 and 308,
// after 28000 of 32K 456 and 444; prompt 8B in 16 tokens (128) after 7000 1478 and 1519, after 28000 2243 and 2146; in 64 tokens
// (512) after 700 537 and 545, after 7000 841 and 815.
constexpr long MMV_ONE_CHAIN_BLOCKS = 1536;
template <bool F16KV>
static void launch_av_mm(const AttnArgs &a, int nrows, hipStream_t st) {
  const long blocks = (long)a.hd / 32 * a.nHeadKv * ((nrows + MMV_RB - 1) / MMV_RB) * std::min(a.nchunk, ATTN_ZMAX);
  if (a.hd == 64 || blocks <= MMV_ONE_CHAIN_BLOCKS) launch_av_mm_k<F16KV, 1, 1>(a, nrows, st);
  else launch_av_mm_k<F16KV, 4, 2>(a, nrows, st);
}

template <int HD, bool F16KV>
static void launch_scores_mm(const AttnArgs &a, dim3 gp, int nrows, hipStream_t st) {
  constexpr bool canWide = HD <= 128;  // (256-dimension rows in 8-wave blocks would spill)
  static bool attr = false;  // dynamic LDS above 64 KB must be requested per kernel
  if (!attr) {
    ZL_HIP(hipFuncSetAttribute((const void *)k_attn_scores_mm<HD, F16KV, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, 140 * 1024));
    if constexpr (canWide)
      ZL_HIP(hipFuncSetAttribute((const void *)k_attn_scores_mm<HD, F16KV, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, 140 * 1024));
    attr = true;
  }
  hipLaunchKernelGGL((k_attn_prep<HD, F16KV>), gp, dim3(64), 0, st, a);
  // as many position blocks per (KV head, row group) as stay resident together (LDS bounds the blocks per CU, and the
  // registers of 8-wave blocks one per CU), at most one per tile of the cache: a pass's tiles then spread over them in
  // one round
  const bool wide = canWide && nrows >= 128;
  const int nwv = wide ? 8 : 4, zg = (nrows + 16 * nwv - 1) / (16 * nwv), ntc = (a.ctx + MM_PT - 1) / MM_PT;
  const size_t lds = attention_mm_lds(HD);
  const int slots = 256 * (wide ? 1 : std::max(1, (int)(160 * 1024 / lds)));
  const dim3 gm((unsigned)std::max(1, std::min(ntc, slots / (a.nHeadKv * zg))), a.nHeadKv, zg);
  if constexpr (canWide) {
    if (wide) {
      hipLaunchKernelGGL((k_attn_scores_mm<HD, F16KV, 8>), gm, dim3(512), lds, st, a, nrows);
      return;
    }
  }
  hipLaunchKernelGGL((k_attn_scores_mm<HD, F16KV, 4>), gm, dim3(256), lds, st, a, nrows);
}

template <int HD, bool F16KV>
static void launch_scores_k(const AttnArgs &a, dim3 grid, int B, hipStream_t st) {
  const size_t kn = (size_t)std::min(64, B) * HD * (F16KV ? 2 : 4);
  hipLaunchKernelGGL((k_attn_scores<HD, F16KV>), grid, dim3(256), kn, st, a);
}

template <bool F16KV>
static void launch_av_k(const AttnArgs &a, int B, hipStream_t st) {
  const int nz = std::min(a.nchunk, ATTN_ZMAX);
  const dim3 grid(a.hd / AV_DIMS, a.nHead, nz * B);
  if (a.ctx <= 1024) hipLaunchKernelGGL((k_attn_av<F16KV, 4, false>), grid, dim3(256), attention_lds(4), st, a, B, nz);
  else if (a.nchunk <= ATTN_ZMAX) hipLaunchKernelGGL((k_attn_av<F16KV, 8, false>), grid, dim3(256), attention_lds(8), st, a, B, nz);
  else hipLaunchKernelGGL((k_attn_av<F16KV, 8, true>), grid, dim3(256), attention_lds(8), st, a, B, nz);
}

template <bool F16KV>
static void launch_av_split_k(const AttnArgs &a, dim3 grid, size_t lds, hipStream_t st) {
  static size_t attr = 64 * 1024;
  if (lds > attr) {
    ZL_HIP(hipFuncSetAttribute((const void *)k_attn_av_split<F16KV>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr = lds;
  }
  hipLaunchKernelGGL((k_attn_av_split<F16KV>), grid, dim3(256), lds, st, a);
}

void launch_attention(const AttnArgs &a0, int B, hipStream_t st) {
  AttnArgs a = a0;
  // the weighted-sum form: split, the matrix cores, or the lane chains
  const bool avmm = !a.part && a.qr && a.mmAvMinB > 0 && B >= a.mmAvMinB;
  ZL_REQUIRE(a.nchunk == (a.ctx + ATTN_CHUNK - 1) / ATTN_CHUNK && a.cml && (a.nchunk == 1 || (a.rec && a.rcnt)), ZL_ERR_ARG,
             "attention: chunk records missing");
  ZL_REQUIRE(!a.part || a.nch * ATTN_SPLIT_C >= a.ctx, ZL_ERR_ARG, "attention: split partials below the context");
  ZL_REQUIRE(a.hd == 64 || a.hd == 128 || a.hd == 256, ZL_ERR_UNSUPPORTED, "attention: head_dim must be 64, 128 or 256");
  ZL_REQUIRE(a.sld >= a.ctx, ZL_ERR_ARG, "attention: score stride below the context");
  ZL_REQUIRE(a.qhs >= a.hd && a.ldq >= a.nHead * a.qhs, ZL_ERR_ARG, "attention: query head stride below the head size");
  const int group = a.nHead / a.nHeadKv;
  a.hpb = attn_heads_per_block(group);
  const int chunks = (a.ctx + attn_score_chunk(a.hd) - 1) / attn_score_chunk(a.hd);
  if (a.qr && a.mmMinB > 0 && B >= a.mmMinB) {
    const dim3 gp(B, a.nHead + a.nHeadKv);
    const int nrows = B * group;
    switch (a.hd * 2 + a.kvF16) {
      case 128: launch_scores_mm<64, false>(a, gp, nrows, st); break;
      case 129: launch_scores_mm<64, true>(a, gp, nrows, st); break;
      case 256: launch_scores_mm<128, false>(a, gp, nrows, st); break;
      case 257: launch_scores_mm<128, true>(a, gp, nrows, st); break;
      case 512: launch_scores_mm<256, false>(a, gp, nrows, st); break;
      case 513: launch_scores_mm<256, true>(a, gp, nrows, st); break;
    }
  } else {
    dim3 gs(chunks < 64 ? chunks : 64, a.nHead / a.hpb, B);
    switch (a.hd * 2 + a.kvF16) {
      case 128: launch_scores_k<64, false>(a, gs, B, st); break;
      case 129: launch_scores_k<64, true>(a, gs, B, st); break;
      case 256: launch_scores_k<128, false>(a, gs, B, st); break;
      case 257: launch_scores_k<128, true>(a, gs, B, st); break;
      case 512: launch_scores_k<256, false>(a, gs, B, st); break;
      case 513: launch_scores_k<256, true>(a, gs, B, st); break;
    }
  }
  ZL_HIP(hipGetLastError());
  if (a.part) {
    const dim3 gv(a.nch, a.nHead, B);
    const size_t lds = attention_split_lds(a.hd, a.kvF16);
    if (a.kvF16) launch_av_split_k<true>(a, gv, lds, st);
    else launch_av_split_k<false>(a, gv, lds, st);
    ZL_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_attn_merge, dim3(a.nHead, B), dim3(std::max(64, a.hd)), 0, st, a);
    ZL_HIP(hipGetLastError());
    return;
  }
  if (avmm) {
    // the probabilities of every row part, then the weighted sums on the matrix cores
    const bool walk = a.nchunk > ATTN_ZMAX;
    const dim3 gr(a.nHead, B, std::min(a.nchunk, ATTN_ZMAX));
    if (walk) hipLaunchKernelGGL(k_attn_softmax_rows<true>, gr, dim3(64), 0, st, a);
    else hipLaunchKernelGGL(k_attn_softmax_rows<false>, gr, dim3(64), 0, st, a);
    const int nrows = group * B;
    if (a.kvF16) launch_av_mm<true>(a, nrows, st);
    else launch_av_mm<false>(a, nrows, st);
    ZL_HIP(hipGetLastError());
    return;
  }
  if (a.kvF16) launch_av_k<true>(a, B, st);
  else launch_av_k<false>(a, B, st);
  ZL_HIP(hipGetLastError());
}

}  // namespace zl
