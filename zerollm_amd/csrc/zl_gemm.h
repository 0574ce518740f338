// Quantised GEMM for 10..64 tokens (prefill chunks, wide verify passes), included by the per-format zl_gemm_*.hip
// files. Every weight byte is read once per launch for all the launch's tokens, as the reference's batched kernels read
// each weight tile once for every token of a chunk (src/compute/wasm/kernels.js:127-240,
// src/compute/wasm/kquant-kernels.js:337-504); the int8 block dots run on the matrix cores and the f64 block terms are
// the reference's (src/compute/ref-kernels.js:132-277), per (row, token) in exactly the order of k_gemv_tiles
// (zl_gemv.h): the same slabs per wave, slab by slab, block 0 then block 1 (Q6_K: both blocks in one term), the same
// halving tree over the waves and the same K parts. A token therefore gets the same bits whatever the size of
// the pass it is in (1..9 tokens through the GEMV kernels, 10..64 here).
//
// Mapping (64-row tiles; blocks of 96 and 32 rows are six and two row groups of 16 in place of four). The workgroup is the
// GEMV's (K part, 64-row tile) with its W waves (gate/up pairs: W / 2 per matrix); wave wl of a matrix walks
// slabs s0 + wl + WH i as in k_gemv_tiles, but for every token of the launch at once. One
// v_mfma_i32_16x16x64_i8 multiplies A (16 tokens: lane l supplies token l mod 16's values of the slab's value quarter
// g = l / 16) by B (16 rows of the tile: lane l supplies row l mod 16's values of quarter g) into D[token][row]; lane l
// receives tokens 4 g + v (v = 0..3) of row l mod 16. To keep one 32-value block (Q6_K: one 16-value group) per dot, A
// holds the token's values only in the quarters of that block and zeros elsewhere: two MFMAs per (16 tokens, 16 rows)
// and slab (Q6_K: four). The B operands are built from the row-layout planes (lane l reads row 16 j + l mod 16's
// 16-byte part of quarter g and the scale words), so no second copy of the weights is needed.
//
// Accumulators. Lane l holds acc[j][u][v] = the running f64 sum of row 16 j + l mod 16 (j = 0..3 row groups of the
// tile) and token 16 u + 4 g + v (u = 0..U-1 token groups): 16 U doubles. Its f64 factors (Q4_K/Q5_K d*sc and dmin*mn
// of the two blocks, Q6_K d, Q8_0 the two block scales) are formed per slab for its four rows.
//
// Activations. Per round i (slabs s0 + WH i + wl of every wave wl of a matrix) the workgroup stages the int8 values and
// block records of those WH slabs for all tokens in LDS ([wl][token][64 B], then [wl][token][32 B]), double-buffered:
// the next round's bytes are loaded into registers while the current round computes and stored to LDS after it, and
// one barrier per round hands the buffer over. (Direct global-to-LDS loads would make the compiler wait for every
// load in flight, the weights' included, before each LDS read.)
#pragma once
#include "zl_gemv.h"

namespace zl {

constexpr int GEMM_MAX_M = 64;   // tokens per launch at most (four groups of 16)
// token groups of a launch whose sums lie in LDS together (96-row blocks: 96 KB each)
constexpr int gemm_ub(int U, int RG) { return U < 2 || RG == 6 ? 1 : 2; }

typedef int gm_i32x4 __attribute__((ext_vector_type(4)));

// One slab of one lane as loaded: for each of J row groups j (lane mod 16 = row of the group) the 16 bytes of value
// quarter g's plane part, the extra-bit word(s), the scale-code word and the super-block / block scale word.
template <int FMT, int J>
struct GmRaw {
  static constexpr int HW = FMT == T_Q6_K ? 4 : FMT == T_Q5_K ? 1 : 0;
  uint32_t q[J][4];
  uint32_t h[J][HW > 0 ? HW : 1];
  uint32_t sc[J];
  uint32_t dw[J];
};

// Slab s of the row groups RG lb + j0 .. + J - 1 (16 rows each) of a matrix of nq row groups; groups past the last one
// read it again (their sums are not stored). RG = 4: row groups j0 .. of tile lb.
template <int FMT, int J, int RG>
__device__ __forceinline__ void gm_load(const Rsrc &R, int lb, int j0, int nq, int s, int nslab, int n16, int g, bool valid, GmRaw<FMT, J> &o) {
  const int oob = valid ? 0 : 0x40000000;
  s = valid ? s : 0;
  #pragma unroll
  for (int j = 0; j < J; j++) {
    const int q = RG == 4 ? 4 * lb : min(RG * lb + j0 + j, nq - 1);
    const int ts = (q >> 2) * nslab + s, sbi = (q >> 2) * (nslab >> 2) + (s >> 2);
    const int r = (RG == 4 ? 16 * (j0 + j) : 0) + n16;  // row of the tile, in the lane's offset
    const int rs = RG == 4 ? 0 : 16 * (q & 3);           // and what the wave's offset adds to it
    u32x4 v;
    if constexpr (FMT == T_Q8_0) {
      // part g (values 16 g .. 16 g + 15) of row r is 16-byte unit 64 g + r of the tile-slab
      v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(R.qs, oob + (g * 64 + r) * 16, ts * 4096 + rs * 16, 0));
    } else {
      // 4-bit planes: part (g & 1) holds the low nibbles of values 16 (g & 1) .. + 15 and the high nibbles 32 later
      v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(R.qs, oob + ((g & 1) * 64 + r) * 16, ts * 2048 + rs * 16, 0));
    }
    o.q[j][0] = v.x; o.q[j][1] = v.y; o.q[j][2] = v.z; o.q[j][3] = v.w;
    if constexpr (FMT == T_Q6_K) {
      const u32x4 x = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(R.qx, oob + r * 16, ts * 1024 + rs * 16, 0));
      o.h[j][0] = x.x; o.h[j][1] = x.y; o.h[j][2] = x.z; o.h[j][3] = x.w;
    } else if constexpr (FMT == T_Q5_K) {
      o.h[j][0] = __builtin_amdgcn_raw_buffer_load_b32(R.qx, oob + r * 8 + 4 * (g >> 1), ts * 512 + rs * 8, 0);
    }
    if constexpr (FMT == T_Q4_K || FMT == T_Q5_K || FMT == T_Q6_K) o.sc[j] = __builtin_amdgcn_raw_buffer_load_b32(R.sc, oob + r * 4, ts * 256 + rs * 4, 0);
    if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) o.dw[j] = __builtin_amdgcn_raw_buffer_load_b32(R.dd, oob + r * 4, sbi * 256 + rs * 4, 0);
    else if constexpr (FMT == T_Q6_K) o.dw[j] = __builtin_amdgcn_raw_buffer_load_b16(R.dd, oob + r * 2, sbi * 128 + rs * 2, 0);
    else o.dw[j] = __builtin_amdgcn_raw_buffer_load_b32(R.dd, oob + r * 4, ts * 256 + rs * 4, 0);
  }
}

// B operands (the 16 values of quarter g of the lane's J rows, as int8) and the exact f64 factors of the rows:
//   Q8_0 f = {d0, d1};  Q4_K/Q5_K f = {d*sc0, d*sc1, dmin*mn0, dmin*mn1};  Q6_K f = {d} and the four group scales, a byte each, in gs.
// The products are those k_gemv_tiles forms (zl_gemv.h unpack), so every term below is bit for bit its term.
template <int FMT>
constexpr int gm_nf = FMT == T_Q6_K ? 1 : FMT == T_Q8_0 ? 2 : 4;
template <int FMT, int J>
__device__ __forceinline__ void gm_unpack(const GmRaw<FMT, J> &o, int g, gm_i32x4 B[J], double f[J][gm_nf<FMT>], uint32_t gs[J]) {
  #pragma unroll
  for (int j = 0; j < J; j++) {
    #pragma unroll
    for (int k = 0; k < 4; k++) {
      uint32_t w = o.q[j][k];
      if constexpr (FMT != T_Q8_0) w = (w >> (4 * (g >> 1))) & 0x0F0F0F0Fu;
      if constexpr (FMT == T_Q5_K) {
        // bit 16 (g & 1) + 4 k + i of the word is the fifth bit of byte i of this dword
        w |= ((((o.h[j][0] >> (16 * (g & 1) + 4 * k)) & 15u) * 0x00204081u) & 0x01010101u) << 4;
      }
      // top two bits of value 16 g + byte; the codes 0..63 become the signed values -32..31 (no carry between the bytes)
      if constexpr (FMT == T_Q6_K) w = ((w | (((o.h[j][k] >> (2 * g)) & 0x03030303u) << 4)) + 0x60606060u) ^ 0x80808080u;
      B[j][k] = (int)w;
    }
    const double d0 = (double)h2f((uint16_t)(o.dw[j] & 0xffff)), d1 = (double)h2f((uint16_t)(o.dw[j] >> 16));
    if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) {
      f[j][0] = d0 * (double)(o.sc[j] & 0xff);
      f[j][1] = d0 * (double)((o.sc[j] >> 8) & 0xff);
      f[j][2] = d1 * (double)((o.sc[j] >> 16) & 0xff);
      f[j][3] = d1 * (double)((o.sc[j] >> 24) & 0xff);
    } else if constexpr (FMT == T_Q6_K) {
      f[j][0] = d0;
      gs[j] = o.sc[j];
    } else {
      f[j][0] = d0; f[j][1] = d1;
    }
  }
}

// RG: 16-row groups per workgroup. 4: a tile. 6: 96 rows, taken three groups at a time against the same staged tokens,
// for launches whose workgroups of 64 rows would fill the last of their rounds of 256 (one per CU) badly; 2: half a tile,
// for launches of few tiles (two of 8 waves fit a CU): see gemm_plan.
template <int FMT, int EPI, int W, int U, int RG>
__global__ __launch_bounds__(W * 64, RG == 2 ? 4 : 1) void k_gemm(const GemvArgs a) {
  extern __shared__ __align__(16) uint8_t xl[];
  constexpr int NR = EPI == EPI_SWIGLU ? 2 : 1;
  constexpr int WH = NR == 2 ? W / 2 : W;                 // waves per matrix
  constexpr int NH = RG == 6 || (U > 2 && FMT != T_Q6_K) ? 2 : 1, JH = RG / NH;  // row groups JH at a time (fewer operand registers)
  constexpr int DEPTH = U <= 2 && FMT != T_Q6_K && NH == 1 ? 2 : 1;  // slabs of weights in flight beyond the one computed
  constexpr int BR = RG * 16;                              // rows per workgroup
  constexpr int MP = 16 * U;                               // staged tokens (the last group padded with the last token)
  constexpr int RB = WH * MP * 96;                         // LDS bytes of one round: values, then records
  constexpr int CH = RB / 1024;                            // 1 KB staging chunks per round
  constexpr int SPW = (CH + W - 1) / W;                    // staging loads per wave and round,
  constexpr int SPH = (SPW + NH - 1) / NH;                 // and with each of its NH parts
  static_assert(RB % 1024 == 0, "whole staging chunks");
  const int kp = blockIdx.x, blk = blockIdx.y;
  // token group z of the launch's G (blockIdx.z): tokens tb .. tb + Ml - 1, staged as rows 0 .. MP - 1. A (row, token)
  // sum does not depend on which workgroup holds the token, so the groups only spread a small matrix over more CUs.
  const int zg = blockIdx.z, G = gridDim.z, tb = zg * MP, Ml = min(MP, a.M - tb);
  const int lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = NR == 2 ? __builtin_amdgcn_readfirstlane(wave / WH) : 0;
  const int wl = wave - grp * WH;
  const int ks = a.ks, M = Ml;  // this group's tokens
  // first row blocks of the second and third segment
  const int blk1 = RG == 6 ? gemm_blocks6(a.seg[0].rows) : a.seg[1].tile0 * 4 / RG;
  const int blk2 = RG == 6 ? blk1 + gemm_blocks6(a.seg[1].rows) : a.seg[2].tile0 * 4 / RG;
  const int si = __builtin_amdgcn_readfirstlane(EPI == EPI_SWIGLU ? 0 : (a.nseg > 2 && blk >= blk2) ? 2 : (a.nseg > 1 && blk >= blk1) ? 1 : 0);
#define ZL_SEG(f) (si == 0 ? a.seg[0].f : si == 1 ? a.seg[1].f : a.seg[2].f)
  const int lb = blk - (si == 0 ? 0 : si == 1 ? blk1 : blk2), rows = ZL_SEG(rows), nq = (rows + 15) >> 4;
  const int nslab = a.nslab;
  const Rsrc R0 = {make_rsrc(ZL_SEG(m.qs), ZL_SEG(nqs)), make_rsrc(ZL_SEG(m.qx), ZL_SEG(nqx)), make_rsrc(ZL_SEG(m.sc), ZL_SEG(nsc)),
                   make_rsrc(ZL_SEG(m.dd), ZL_SEG(ndd))};
  const Rsrc R1 = NR == 2 ? Rsrc{make_rsrc(a.seg[1].m.qs, a.seg[1].nqs), make_rsrc(a.seg[1].m.qx, a.seg[1].nqx),
                                 make_rsrc(a.seg[1].m.sc, a.seg[1].nsc), make_rsrc(a.seg[1].m.dd, a.seg[1].ndd)}
                          : R0;
  const Rsrc R = grp == 0 ? R0 : R1;
  const int kr = a.kr, s0 = kp * kr, s1 = min(nslab, s0 + kr), nsl = s1 - s0;
  const int n = nsl > wl ? (nsl - wl + WH - 1) / WH : 0;  // this wave's slabs: s0 + wl + WH i, i < n
  const int nr = (nsl + WH - 1) / WH;                      // rounds (the most slabs a wave of the workgroup has)
  const uint8_t *xq = (const uint8_t *)a.act.q;
  const uint8_t *xr = (const uint8_t *)(FMT == T_Q6_K ? (const void *)a.act.rb : (const void *)a.act.ra);
  const long ldq = a.act.ld, ldr = (long)(a.act.ld >> 5) * 16;

  // ---- staging of round r into buffer r & 1 (chunk c of the round is LDS bytes [1024 c, 1024 c + 1024) of the
  // buffer), through registers: the loads are issued at the start of the previous round and the LDS stores follow its
  // compute, so the compiler's load counters track them exactly and the weight loads in flight are never waited for
  auto stage_load = [&](int r, int k0, u32x4 *sg) {  // loads k0 .. of the wave's SPW
    #pragma unroll
    for (int k = k0; k < k0 + SPH; k++) {
      const int c = min(wave + W * k, CH - 1);  // surplus loads repeat the last chunk (the same bytes)
      const bool isv = c < WH * U;
      const int o = (isv ? c : c - WH * U) * 1024 + lane * 16;
      const int per = isv ? MP * 64 : MP * 32, rb = isv ? 64 : 32;
      const int w_ = o / per, rem = o - w_ * per, t = min(rem / rb, M - 1), e = rem % rb;
      const int s = min(s0 + w_ + WH * r, nslab - 1);  // rounds past the last one read a slab in range (unused)
      sg[k - k0] = *(const u32x4 *)(isv ? xq + (long)(tb + t) * ldq + (long)s * 64 + e : xr + (long)(tb + t) * ldr + (long)s * 32 + e);
    }
  };
  auto stage_store = [&](int r, int k0, const u32x4 *sg) {
    uint8_t *buf = xl + (r & 1) * RB;
    #pragma unroll
    for (int k = k0; k < k0 + SPH; k++) {
      const int c = min(wave + W * k, CH - 1);
      *(u32x4 *)(buf + c * 1024 + lane * 16) = sg[k - k0];
    }
  };

  double acc[RG][U][4];
  #pragma unroll
  for (int j = 0; j < RG; j++)
    #pragma unroll
    for (int u = 0; u < U; u++)
      #pragma unroll
      for (int v = 0; v < 4; v++) acc[j][u][v] = 0.0;

  auto load = [&](int i, int h, GmRaw<FMT, JH> &b) {
    gm_load<FMT, JH, RG>(R, lb, h * JH, nq, s0 + wl + WH * i, nslab, n16, g, i < n, b);
  };
  GmRaw<FMT, JH> ring[DEPTH * NH];
  {
    u32x4 sg[NH * SPH];
    #pragma unroll
    for (int h = 0; h < NH; h++) stage_load(0, h * SPH, sg + h * SPH);
    #pragma unroll
    for (int d = 0; d < DEPTH; d++)
      #pragma unroll
      for (int h = 0; h < NH; h++) load(d, h, ring[d * NH + h]);
    #pragma unroll
    for (int h = 0; h < NH; h++) stage_store(0, h * SPH, sg + h * SPH);
    __syncthreads();
  }

  // one round: the wave's slab r (weights in `slots`, activations in buffer r & 1), the next round's activations staged
  auto round = [&](int r, GmRaw<FMT, JH> *slots) {
    #pragma unroll
    for (int h = 0; h < NH; h++) {
      u32x4 sg[SPH];
      gm_i32x4 B[JH];
      double f[JH][gm_nf<FMT>];
      uint32_t gs[JH];
      gm_unpack<FMT, JH>(slots[h], g, B, f, gs);
      // the operands are formed here, before the slot is reloaded (not sunk to their uses below), so the reload can
      // land in the slot's own registers
      #pragma unroll
      for (int j = 0; j < JH; j++) {
        asm volatile("" : "+v"(B[j]));
        #pragma unroll
        for (int k = 0; k < gm_nf<FMT>; k++) asm volatile("" : "+v"(f[j][k]));
        if constexpr (FMT == T_Q6_K) asm volatile("" : "+v"(gs[j]));
      }
      __builtin_amdgcn_sched_barrier(0);  // issue order: the staging loads, then the weights (the stores below wait for
      stage_load(r + 1, h * SPH, sg);     // the former only)
      __builtin_amdgcn_sched_barrier(0);
      load(r + DEPTH, h, slots[h]);  // past the wave's last slab: no memory access
      __builtin_amdgcn_sched_barrier(0);
      if (r < n) {
        const uint8_t *buf = xl + (r & 1) * RB;
        const uint8_t *vals = buf + wl * MP * 64, *recs = buf + WH * MP * 64 + wl * MP * 32;
        #pragma unroll
        for (int u = 0; u < U; u++) {
          const uint4 av = *(const uint4 *)(vals + (16 * u + n16) * 64 + 16 * g);
          if constexpr (FMT == T_Q6_K) {
            // the two groups of a block join in integers, the slab's two blocks in one product with d: 9 VALU instructions
            // per (row, token) and slab where a term per group took 16 (4096 x 12288 at 64 tokens 73.8 -> 48.9 us, bound by
            // their issue). One slab ahead in flight: two (40 registers each) spilled. Row group j's sums are formed while
            // the matrix cores run j + 1's dots (the barriers keep the scheduler from holding all four row groups' dots in
            // registers at once)
            gm_i32x4 A[4], D[2][4];
            double xd[2][4];
            #pragma unroll
            for (int b = 0; b < 4; b++) A[b] = g == b ? gm_i32x4{(int)av.x, (int)av.y, (int)av.z, (int)av.w} : gm_i32x4{0, 0, 0, 0};
            #pragma unroll
            for (int v = 0; v < 4; v++)
              #pragma unroll
              for (int blk = 0; blk < 2; blk++) xd[blk][v] = *(const double *)(recs + (16 * u + 4 * g + v) * 32 + blk * 16);
            auto dots = [&](int j) {
              #pragma unroll
              for (int b = 0; b < 4; b++) D[j & 1][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[b], B[j], gm_i32x4{0, 0, 0, 0}, 0, 0, 0);
            };
            dots(0);
            #pragma unroll
            for (int j = 0; j < JH; j++) {
              __builtin_amdgcn_sched_barrier(0);
              if (j < JH - 1) dots(j + 1);
              const gm_i32x4 (&d)[4] = D[j & 1];
              int sc[4];
              #pragma unroll
              for (int k = 0; k < 4; k++) sc[k] = (int)(int8_t)(gs[j] >> (8 * k));
              #pragma unroll
              for (int v = 0; v < 4; v++) {
                const int e0 = __mul24(d[0][v], sc[0]) + __mul24(d[1][v], sc[1]);
                const int e1 = __mul24(d[2][v], sc[2]) + __mul24(d[3][v], sc[3]);
                double &s = acc[h * JH + j][u][v];
                s = fma(f[j][0], fma(xd[1][v], (double)e1, xd[0][v] * (double)e0), s);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          } else {
            #pragma unroll
            for (int b = 0; b < 2; b++) {
              const bool on = (g >> 1) == b;  // this lane's quarter lies in block b
              const gm_i32x4 A = on ? gm_i32x4{(int)av.x, (int)av.y, (int)av.z, (int)av.w} : gm_i32x4{0, 0, 0, 0};
              gm_i32x4 D[JH];
              #pragma unroll
              for (int j = 0; j < JH; j++) D[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, B[j], gm_i32x4{0, 0, 0, 0}, 0, 0, 0);
              #pragma unroll
              for (int v = 0; v < 4; v++) {
                const uint4 rc = *(const uint4 *)(recs + (16 * u + 4 * g + v) * 32 + b * 16);
                const double xd = dbl(rc.x, rc.y);
                #pragma unroll
                for (int j = 0; j < JH; j++) {
                  double &s = acc[h * JH + j][u][v];
                  if constexpr (FMT == T_Q8_0) {
                    s = fma((double)D[j][v] * f[j][b], xd, s);
                  } else {
                    s = fma(xd, fma(f[j][b], (double)D[j][v], -(f[j][2 + b] * dbl(rc.z, rc.w))), s);
                  }
                }
              }
            }
          }
        }
      }
      stage_store(r + 1, h * SPH, sg);  // buffer (r + 1) & 1 was last read in round r - 1, before the previous barrier
    }
    __syncthreads();
  };
  // whole groups of DEPTH rounds (a round past the last only stages and loads unused bytes), so each slot of the ring
  // keeps its registers from one iteration to the next
  for (int r = 0; r < nr; r += DEPTH) {
    round(r, ring);
    if constexpr (DEPTH == 2) round(r + 1, ring + NH);
  }

  // ---- every wave parks its sums, then each wave adds its share of the (row, token) sums over the waves of each matrix
  // in the order of a halving tree (as k_gemv_tiles) and runs the epilogue (or stores a K part). Its NU units of 64 sums
  // go through each step together, so their loads and chains overlap: one by one the hand-off's loads alone were NU
  // round trips. Unit k: 64-row tiles, token wave + W k and row `lane`; 96- and 32-row blocks, 32 rows (a whole block of the
  // quantised output) of two tokens.
  constexpr int UPG = RG / (W / 4), RU = RG / 2;  // units per wave and token group; 32-row units per block
  constexpr int NU = U * UPG;
  auto unit_t = [&](int k) {
    return RG == 4 ? wave + W * k : 16 * (k / UPG) + 2 * (wave + W * ((k % UPG) / RU)) + (lane >> 5);
  };
  auto unit_r = [&](int k) { return RG == 4 ? lane : 32 * ((k % UPG) % RU) + (lane & 31); };
  double *red = (double *)xl;  // [token group of a batch][W][RG j][4 v][64 lanes]
  const int PW = NR * MP * BR;  // doubles per K part
  double *pp = a.part + (((long)blk * G + zg) * ks + kp) * PW;
  const int row0 = lb * BR;
  float rres[NU];  // the residual values, requested ahead of the reduction
  if constexpr (EPI == EPI_RESID) {
    #pragma unroll
    for (int k = 0; k < NU; k++) rres[k] = a.resid[(long)(tb + min(unit_t(k), M - 1)) * a.ldr + min(row0 + unit_r(k), rows - 1)];
  }
  auto epilogue = [&](int k, int t, int row, double g0, double u0) {
    const bool live = row < rows;
    if constexpr (EPI == EPI_SWIGLU) {
      const double gv = (double)(float)g0, uu = (double)(float)u0;
      const float hv = live ? (float)(gv / (1.0 + exp(-gv)) * uu) : 0.f;  // src/compute/ref-kernels.js:322
      if (live) a.hb[(long)t * a.ldh + row] = hv;
      if (a.qout.q && (RG == 4 || row < ((rows + 63) & ~63))) quant_block32(hv, row, a.qout, t);
    } else if constexpr (EPI == EPI_RESID) {
      const double y = (double)(float)g0;
      if (live) a.resid[(long)t * a.ldr + row] = (float)((double)rres[k] + y);
    } else {
      const float y = (float)g0;
      if (live) {
        const float *bias = ZL_SEG(bias);
        ZL_SEG(out)[(long)t * ZL_SEG(ldo) + row] = bias ? (float)((double)y + (double)bias[row]) : y;
      }
    }
  };
  double sums[NU][NR];
  constexpr int UB = gemm_ub(U, RG);  // token groups parked at a time
  #pragma unroll
  for (int u0 = 0; u0 < U; u0 += UB) {
    if (u0 > 0) __syncthreads();  // the previous groups' sums have been read
    #pragma unroll
    for (int u = u0; u < u0 + UB && u < U; u++)
      #pragma unroll
      for (int j = 0; j < RG; j++)
        #pragma unroll
        for (int v = 0; v < 4; v++) red[((((u - u0) * W + wave) * RG + j) * 4 + v) * 64 + lane] = acc[j][u][v];
    __syncthreads();
    #pragma unroll
    for (int k = u0 * UPG; k < NU && k < (u0 + UB) * UPG; k++) {
      const int t = unit_t(k), tt = t & 15, rr = unit_r(k);  // (tokens past M: sums of padding, not stored)
      // (row rr, token t): row group rr / 16 in lane 16 (tt / 4) + rr mod 16, slot v = tt mod 4
      const int src = 16 * (tt >> 2) + n16, jv = (rr >> 4) * 4 + (tt & 3);
      #pragma unroll
      for (int r = 0; r < NR; r++) {
        double vv[WH];
        #pragma unroll
        for (int w = 0; w < WH; w++) vv[w] = red[((((k / UPG - u0) * W + r * WH + w) * RG * 4) + jv) * 64 + src];
        #pragma unroll
        for (int half = WH / 2; half >= 1; half >>= 1)
          #pragma unroll
          for (int w = 0; w < half; w++) vv[w] = vv[w] + vv[w + half];
        sums[k][r] = vv[0];
      }
    }
  }
  if (ks > 1) {
    // ---- K parts: the last part of the row block to arrive adds all parts' sums in part order (as k_gemv_tiles)
    __shared__ uint32_t last;
    #pragma unroll
    for (int k = 0; k < NU; k++)
      if (unit_t(k) < M) {
        #pragma unroll
        for (int r = 0; r < NR; r++)
          __hip_atomic_store(pp + (r * MP + unit_t(k)) * BR + unit_r(k), sums[k][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's stores are complete
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    uint32_t *cnt = a.cnt + (long)blk * G + zg;
    if (threadIdx.x == 0) last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(ks - 1);
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double *p0 = a.part + ((long)blk * G + zg) * ks * PW;
    for (int q0 = 0; q0 < ks; q0 += 4) {  // four parts' loads of all the wave's sums are issued together
      double pv[NU][NR][4];
      #pragma unroll
      for (int k = 0; k < NU; k++)
        #pragma unroll
        for (int r = 0; r < NR; r++)
          #pragma unroll
          for (int q = 0; q < 4; q++)
            pv[k][r][q] = __hip_atomic_load(p0 + (long)min(q0 + q, ks - 1) * PW + (r * MP + min(unit_t(k), M - 1)) * BR + unit_r(k),
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      #pragma unroll
      for (int k = 0; k < NU; k++)
        #pragma unroll
        for (int r = 0; r < NR; r++)
          #pragma unroll
          for (int q = 0; q < 4; q++) {
            if (q0 + q == 0) sums[k][r] = pv[k][r][0];
            else if (q0 + q < ks) sums[k][r] += pv[k][r][q];
          }
    }
  }
  #pragma unroll
  for (int k = 0; k < NU; k++)
    if (unit_t(k) < M) epilogue(k, tb + unit_t(k), row0 + unit_r(k), sums[k][0], sums[k][NR - 1]);
#undef ZL_SEG
}

// LDS bytes of a launch: two staging rounds, or the waves' sums.
template <int W, int U, int RG>
constexpr size_t gemm_lds(bool swiglu) {
  return std::max((size_t)2 * (swiglu ? W / 2 : W) * 16 * U * 96, (size_t)gemm_ub(U, RG) * W * RG * 4 * 64 * 8);
}

template <int FMT, int EPI, int W, int U, int RG = 4>
inline void launch_gemm_k(const GemvArgs &a, const GemmPlan &p, hipStream_t st) {
  const size_t lds = gemm_lds<W, U, RG>(EPI == EPI_SWIGLU);
  static bool done = false;
  if (!done) {
    ZL_HIP(hipFuncSetAttribute((const void *)k_gemm<FMT, EPI, W, U, RG>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    done = true;
  }
  hipLaunchKernelGGL((k_gemm<FMT, EPI, W, U, RG>), dim3((unsigned)a.ks, (unsigned)p.blocks, (unsigned)p.G), dim3(W * 64), lds, st, a);
}

template <int FMT, int EPI, int W>
inline void launch_gemm_w(const GemvArgs &a, hipStream_t st) {
  const GemmPlan p = gemm_plan(a, EPI == EPI_SWIGLU);
  ZL_REQUIRE(a.ks == 1 || (long)p.blocks * p.G <= GEMV_CNT_TILES, ZL_ERR_ARG, "gemm: too many split-K counters");
  if constexpr (gemm_has6(FMT)) {
    if (p.RG == 6) return launch_gemm_k<FMT, EPI, W, 2, 6>(a, p, st);
  }
  if (p.RG == 2) return launch_gemm_k<FMT, EPI, W, 1, 2>(a, p, st);
  switch (p.U) {
    case 1: launch_gemm_k<FMT, EPI, W, 1>(a, p, st); break;
    case 2: launch_gemm_k<FMT, EPI, W, 2>(a, p, st); break;
    case 3: launch_gemm_k<FMT, EPI, W, 3>(a, p, st); break;
    default: launch_gemm_k<FMT, EPI, W, 4>(a, p, st); break;
  }
}

template <int FMT>
void launch_gemm_fmt(const GemvArgs &a, int epi, hipStream_t st) {
  ZL_REQUIRE(a.M >= 1 && a.M <= GEMM_MAX_M && (a.nwave == 4 || a.nwave == 8) && (epi != EPI_SWIGLU || a.nwave == 8) &&
                 a.ks >= 1 && a.ks <= 8 && !a.xf && a.kr >= 1,
             ZL_ERR_ARG, "gemm: launch shape out of range");
  if (epi == EPI_SWIGLU) {
    launch_gemm_w<FMT, EPI_SWIGLU, 8>(a, st);
  } else if (epi == EPI_RESID) {
    if (a.nwave == 4) launch_gemm_w<FMT, EPI_RESID, 4>(a, st);
    else launch_gemm_w<FMT, EPI_RESID, 8>(a, st);
  } else {
    if (a.nwave == 4) launch_gemm_w<FMT, EPI_STORE, 4>(a, st);
    else launch_gemm_w<FMT, EPI_STORE, 8>(a, st);
  }
}

}  // namespace zl
