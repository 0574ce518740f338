// GEMV dispatch: K-part choice, token chunks, per-format tile kernels (zl_gemv.h, instantiated in zl_gemv_*.hip) and
// the float-weight kernel.
#include <type_traits>

#include "zl_kernels.h"

namespace zl {

// Float weights (F32/F16/BF16) use the f32 activation (src/compute/ref-kernels.js:278-299): a wave takes R rows and MT
// tokens; lane l adds the products of columns l, l + 64, ... in order in f64 (each product is exact), a butterfly joins
// the lanes, so a sum's bits depend on neither R nor MT.
//
// Bound by HBM where M is small (the matrix is read once per MT tokens) and by the f64 multiply-adds beyond. UN columns
// of every row and token are requested together: one element at a time each step waited out a memory latency, and a
// pass per token read the matrix M times. F16: 151936 x 4096 at 1 token 1120 -> 201 us (6.2 TB/s), 4096 x 12288 at 16
// tokens 1779 -> 69, 512 x 1024 at 1 and 5 tokens 12.0 -> 7.9 and 37.2 -> 8.0.
template <int TY>
__device__ __forceinline__ float float_weight(const uint8_t *row, int c) {
  if constexpr (TY == T_F32) return ((const float *)row)[c];
  else if constexpr (TY == T_F16) return h2f(((const uint16_t *)row)[c]);
  else return __uint_as_float((uint32_t)((const uint16_t *)row)[c] << 16);
}

template <int TY, int EPI, int MT, int R>
__global__ __launch_bounds__(256) void k_gemv_float(const GemvArgs a, int rows_total, const float *__restrict__ xf, int ldx) {
  constexpr int NR = EPI == EPI_SWIGLU ? 2 : 1;  // matrices per output row: gate and up
  constexpr int NW = NR * R;                     // weight rows of the wave
  constexpr int UN = NW + MT <= 5 ? 8 : NW + MT <= 8 ? 4 : 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = (blockIdx.x * 4 + wave) * R, t0 = blockIdx.y * MT;
  if (row0 >= rows_total) return;
  const uint8_t *wr[NW];
  int seg[R], lr[R];  // (rows past the last one repeat it; not stored)
  #pragma unroll
  for (int i = 0; i < R; i++) {
    const int row = min(row0 + i, rows_total - 1);
    int si = 0, base = 0;
    if constexpr (EPI == EPI_STORE) {
      if (a.nseg > 1 && row >= a.seg[0].rows) { si = 1; base = a.seg[0].rows; }
      if (a.nseg > 2 && row >= a.seg[0].rows + a.seg[1].rows) { si = 2; base = a.seg[0].rows + a.seg[1].rows; }
    }
    seg[i] = si;
    lr[i] = row - base;
  }
#define ZL_SEG(i, f) (seg[i] == 0 ? a.seg[0].f : seg[i] == 1 ? a.seg[1].f : a.seg[2].f)
  const int cols = a.seg[0].m.cols;
  const long rb = (long)cols * (TY == T_F32 ? 4 : 2);
  #pragma unroll
  for (int i = 0; i < R; i++) {
    wr[i] = ZL_SEG(i, m.qs) + lr[i] * rb;
    if constexpr (NR == 2) wr[R + i] = a.seg[1].m.qs + lr[i] * rb;
  }
  const float *xr[MT];  // (tokens past M repeat the last one; not stored)
  #pragma unroll
  for (int t = 0; t < MT; t++) xr[t] = xf + (long)min(t0 + t, a.M - 1) * ldx;
  double acc[NW][MT];
  #pragma unroll
  for (int i = 0; i < NW; i++)
    #pragma unroll
    for (int t = 0; t < MT; t++) acc[i][t] = 0.0;
  int c = lane;
  for (; c + 64 * (UN - 1) < cols; c += 64 * UN) {
    float w[UN][NW], x[UN][MT];
    #pragma unroll
    for (int k = 0; k < UN; k++) {
      #pragma unroll
      for (int i = 0; i < NW; i++) w[k][i] = float_weight<TY>(wr[i], c + 64 * k);
      #pragma unroll
      for (int t = 0; t < MT; t++) x[k][t] = xr[t][c + 64 * k];
    }
    #pragma unroll
    for (int k = 0; k < UN; k++)
      #pragma unroll
      for (int i = 0; i < NW; i++)
        #pragma unroll
        for (int t = 0; t < MT; t++) acc[i][t] = fma((double)w[k][i], (double)x[k][t], acc[i][t]);
  }
  for (; c < cols; c += 64)
    #pragma unroll
    for (int i = 0; i < NW; i++) {
      const double w = (double)float_weight<TY>(wr[i], c);
      #pragma unroll
      for (int t = 0; t < MT; t++) acc[i][t] = fma(w, (double)xr[t][c], acc[i][t]);
    }
  #pragma unroll
  for (int i = 0; i < NW; i++)
    #pragma unroll
    for (int t = 0; t < MT; t++) acc[i][t] = wave_sum_xor(acc[i][t], 64);
  #pragma unroll
  for (int i = 0; i < R; i++)
    #pragma unroll
    for (int t = 0; t < MT; t++) {
      const int tt = t0 + t;
      if (lane != i * MT + t || row0 + i >= rows_total || tt >= a.M) continue;  // lane i MT + t stores sum (i, t)
      if constexpr (EPI == EPI_SWIGLU) {
        const double g = (double)(float)acc[i][t], u = (double)(float)acc[R + i][t];
        a.hb[(long)tt * a.ldh + lr[i]] = (float)(g / (1.0 + exp(-g)) * u);
      } else if constexpr (EPI == EPI_RESID) {
        float *xp = a.resid + (long)tt * a.ldr + lr[i];
        *xp = (float)((double)*xp + (double)(float)acc[i][t]);
      } else {
        float y = (float)acc[i][t];
        const float *bias = ZL_SEG(i, bias);
        if (bias) y = (float)((double)y + (double)bias[lr[i]]);
        ZL_SEG(i, out)[(long)tt * ZL_SEG(i, ldo) + lr[i]] = y;
      }
    }
#undef ZL_SEG
}

// Four rows per wave share its activation loads where that still leaves four waves per CU, one row otherwise; the
// tokens in the fewest groups of at most 8, spread evenly.
template <int TY, int EPI>
static void launch_gemv_float(const GemvArgs &a, int rows, const float *xf, int ldx, hipStream_t st) {
  const int groups = (a.M + 7) / 8, per = (a.M + groups - 1) / groups;
  auto go = [&](auto mt, auto r) {
    constexpr int MT = mt.value, R = r.value;
    hipLaunchKernelGGL((k_gemv_float<TY, EPI, MT, R>), dim3((rows + 4 * R - 1) / (4 * R), (a.M + MT - 1) / MT), dim3(256), 0, st, a, rows, xf, ldx);
  };
  auto tokens = [&](auto r) {
    if (per <= 1) go(std::integral_constant<int, 1>{}, r);
    else if (per <= 2) go(std::integral_constant<int, 2>{}, r);
    else if (per <= 4) go(std::integral_constant<int, 4>{}, r);
    else if (per <= 6) go(std::integral_constant<int, 6>{}, r);
    else go(std::integral_constant<int, 8>{}, r);
  };
  if (rows >= 4096) tokens(std::integral_constant<int, 4>{});
  else tokens(std::integral_constant<int, 1>{});
}
template <int TY>
static void launch_gemv_float_epi(const GemvArgs &a, int epi, int rows, const float *xf, int ldx, hipStream_t st) {
  if (epi == EPI_STORE) launch_gemv_float<TY, EPI_STORE>(a, rows, xf, ldx, st);
  else if (epi == EPI_RESID) launch_gemv_float<TY, EPI_RESID>(a, rows, xf, ldx, st);
  else launch_gemv_float<TY, EPI_SWIGLU>(a, rows, xf, ldx, st);
}

// Launch shape, a function of the matrix shape only (so every summation order is independent of the token count):
// - waves per matrix: 4 when there are enough tiles to fill the GPU with workgroups, else 8 (4 for gate/up pairs, whose
//   workgroup runs the gate and the up rows on two halves). Against 16 (8 per gate/up half) each wave holds more slabs,
//   so more of its compute overlaps the loads, and fewer waves meet in the reduction: 5-25 % faster at M = 1, 5, 9 for
//   every 8B and 0.6B projection shape;
// - K parts: 1 (no cross-workgroup sum) unless a part would exceed the staged-activation limit (GT_KR_MAX slabs) or
//   give a wave more than GT_NMAX slabs; for large single-output matrices of fewer tiles than CUs, more parts where that
//   lowers the slabs the busiest CU streams while every wave keeps at least two slabs (attn_output 4096 x 4096: 4 parts,
//   256 workgroups; attn_v 1024 x 4096: 4 parts, so that its launch mixed with attn_q/attn_k's 160 workgroups stays
//   within one round of 256). Not for gate/up pairs: their workgroups hold too many registers to overlap, so rounds of
//   K parts cost more than they save.
void gemv_shape(int ntiles, int nslab, bool swiglu, int *ks, int *nw) {
  const int w = ntiles >= 256 || swiglu ? 4 : 8;  // waves per matrix
  int k = 1;
  while ((nslab + k - 1) / k > 96 || ((nslab + k - 1) / k + w - 1) / w > 16) k *= 2;
  // large matrices of fewer tiles than CUs: more K parts while that lowers the most slabs one CU streams (workgroups
  // run in rounds of 256), keeping at least two slabs per wave
  if (!swiglu && ntiles < 256 && (long)ntiles * nslab >= 1024) {
    auto load = [&](int kk) { return (long)((ntiles * kk + 255) / 256) * ((nslab + kk - 1) / kk); };
    for (int kk = k * 2; kk <= 8 && (nslab + kk - 1) / kk >= 2 * w; kk *= 2)
      if (load(kk) < load(k)) k = kk;
  }
  *ks = k;
  *nw = swiglu ? 2 * w : w;  // a gate/up pair: w waves per matrix
}

// Tokens per GEMM launch (ZEROLLM_GEMM_MAXM, read when a launch is enqueued, so a captured graph keeps the value of its
// capture; below GEMM_MIN_M every launch stays on the GEMV kernels in chunks of at most GEMV_MAX_MT tokens: the same
// bits, more weight passes). Default 64, one launch per prefill chunk: measured against two launches of 32 (whose
// sums fit a wave's registers, where 64 tokens spill a few), 16K-token prefill 6.47 -> 6.21 s (target), 2.69 -> 2.32 s
// (draft).
static int gemm_max_m() {
  const char *e = getenv("ZEROLLM_GEMM_MAXM");
  const int m = e ? atoi(e) : 64;
  return m < GEMM_MIN_M ? 0 : std::min(m, 64);
}

// Launches of at least GEMM_MIN_M tokens (ZEROLLM_GEMM_MINM moves it, for measurements) of the formats the GEMM takes,
// without a fused prologue.
static int gemm_min_m() {
  const char *e = getenv("ZEROLLM_GEMM_MINM");
  return e ? std::max(1, atoi(e)) : GEMM_MIN_M;
}
bool gemm_takes(const GemvArgs &a) {
  const int t = a.seg[0].m.type;
  return gemm_max_m() > 0 && a.M >= gemm_min_m() && !a.xf && (t == T_Q8_0 || t == T_Q4_K || t == T_Q5_K || t == T_Q6_K);
}

long gemv_part_need(const GemvArgs &a) {
  if (a.ks == 1) return 0;
  if (gemm_takes(a)) {  // the split of the chunks' sizes that takes the most (chunks differ by one token at most)
    const int cap = gemm_max_m(), nch = (a.M + cap - 1) / cap;
    long need = 0;
    for (int k = 0; k < 2; k++) {
      GemvArgs c = a;
      c.M = k ? (a.M + nch - 1) / nch : std::max(1, a.M / nch);
      for (const bool swiglu : {false, true}) {
        const GemmPlan p = gemm_plan(c, swiglu);
        need = std::max(need, (long)p.blocks * a.ks * 2 * 16 * p.U * p.G * 16 * p.RG);
      }
    }
    return need;
  }
  return (long)a.ntiles * a.ks * 2 * GEMV_MAX_MT * 64;
}

void launch_gemv(const GemvArgs &a0, int epi, const float *xf, int ldx, hipStream_t st) {
  const int fmt = a0.seg[0].m.type;
  for (int i = 1; i < a0.nseg; i++)
    ZL_REQUIRE(a0.seg[i].m.type == fmt && a0.seg[i].m.nslab == a0.nslab, ZL_ERR_ARG, "gemv: segments differ in type or width");
  if (!is_quant(fmt)) {
    int rows_total = 0;
    for (int i = 0; i < a0.nseg; i++) rows_total += (epi == EPI_SWIGLU && i > 0) ? 0 : a0.seg[i].rows;
    if (fmt == T_F32) launch_gemv_float_epi<T_F32>(a0, epi, rows_total, xf, ldx, st);
    else if (fmt == T_F16) launch_gemv_float_epi<T_F16>(a0, epi, rows_total, xf, ldx, st);
    else if (fmt == T_BF16) launch_gemv_float_epi<T_BF16>(a0, epi, rows_total, xf, ldx, st);
    else throw Error(ZL_ERR_UNSUPPORTED, "gemv: unsupported weight type");
    ZL_HIP(hipGetLastError());
    return;
  }
  ZL_REQUIRE(a0.ks >= 1 && a0.ntiles >= 1, ZL_ERR_ARG, "gemv: bad launch shape");
  ZL_REQUIRE(a0.ks == 1 || (a0.part && a0.cnt && a0.ntiles <= GEMV_CNT_TILES && gemv_part_need(a0) <= GEMV_PART_DOUBLES),
             ZL_ERR_ARG, "gemv: split-K work space missing or too small");
  ZL_REQUIRE(a0.act.q && a0.act.ra && a0.act.rb && a0.act.rc && a0.act.ld % 64 == 0 && a0.act.ld >= a0.nslab * 64,
             ZL_ERR_ARG, "gemv: activation records missing");
  // as few weight passes as chunks of at most 64 (GEMM) or GEMV_MAX_MT tokens allow, with the tokens spread evenly
  // over them; every input and output row is addressed from offset pointers, and the results do not depend on the
  // chunking
  const bool gemm = gemm_takes(a0);
  const int cap = gemm ? gemm_max_m() : GEMV_MAX_MT;
  const int nch = (a0.M + cap - 1) / cap;
  for (int c = 0, t0 = 0; c < nch; c++) {
    GemvArgs b = a0;
    b.M = (a0.M - t0) / (nch - c);  // the remaining tokens over the remaining chunks, the larger chunks last
    ZL_REQUIRE(b.M >= 1 && b.M <= cap, ZL_ERR_ARG, "gemv: bad token chunk");
    if (t0) {
      b.act = act_rows(a0.act, t0);
      for (int i = 0; i < b.nseg; i++) if (b.seg[i].out) b.seg[i].out += (long)t0 * b.seg[i].ldo;
      if (b.resid) b.resid += (long)t0 * b.ldr;
      if (b.hb) b.hb += (long)t0 * b.ldh;
      if (b.qout.q) b.qout = act_rows(a0.qout, t0);
      b.xrow0 += t0;  // fused prologue: the chunk's own input rows
    }
    t0 += b.M;
    if (gemm) {  // every weight read once for all the chunk's tokens, on the matrix cores; same results
      switch (fmt) {
        case T_Q8_0: launch_gemm_fmt<T_Q8_0>(b, epi, st); break;
        case T_Q4_K: launch_gemm_fmt<T_Q4_K>(b, epi, st); break;
        case T_Q5_K: launch_gemm_fmt<T_Q5_K>(b, epi, st); break;
        default: launch_gemm_fmt<T_Q6_K>(b, epi, st); break;
      }
      ZL_HIP(hipGetLastError());
      continue;
    }
    if (gemv_mfma_ok(b, epi)) {  // Q4_K and Q8_0 at 2..8 tokens: the int8 dots on the matrix cores, same results
      launch_gemv_mfma(b, epi, st);
      ZL_HIP(hipGetLastError());
      continue;
    }
    switch (fmt) {
      case T_Q8_0: launch_gemv_fmt<T_Q8_0>(b, epi, st); break;
      case T_Q4_0: launch_gemv_fmt<T_Q4_0>(b, epi, st); break;
      case T_Q5_0: launch_gemv_fmt<T_Q5_0>(b, epi, st); break;
      case T_Q4_K: launch_gemv_fmt<T_Q4_K>(b, epi, st); break;
      case T_Q5_K: launch_gemv_fmt<T_Q5_K>(b, epi, st); break;
      case T_Q6_K: launch_gemv_fmt<T_Q6_K>(b, epi, st); break;
      default: throw Error(ZL_ERR_UNSUPPORTED, "gemv: unsupported weight type");
    }
    ZL_HIP(hipGetLastError());
  }
}

}  // namespace zl
