// The 64-column steps of the blocked Cholesky factorisation (FP64).
//
// A step's 64x64 diagonal block is one serial chain of 64 pivots, and it is the
// critical path of a panel: the design keeps that chain in the registers of one
// wavefront and moves everything else beside it.
//
// Blocks of 16x16 travel in the "operand layout": value e (0..3) of lane l is
// element (l % 16, 4 e + l / 16).  It is what v_mfma_f64_16x16x4 takes as either
// operand at k = 4 e.., and the transposed product of two such blocks comes out of
// the accumulators in it again (their element e of lane l is (4 e + l / 16, l % 16)
// of the product), so that a chain of block products needs no LDS in between.
#pragma once

#include "nka_common.hpp"

namespace nka {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int CH_NB = 64;

// An entry of a triangular solve's output that has not been solved yet: a
// signalling NaN, which arithmetic never returns; a value with its bit pattern is
// published as the default NaN.
constexpr uint64_t kUnsolved = 0x7FF4D15EA5E0F00DULL;
constexpr uint64_t kDefaultNaN = 0x7FF8000000000000ULL;

// 1/sqrt(a) from the hardware estimate (about 2^-23 relative error) refined by
// two Newton-Raphson steps y <- y + y (1/2 - (a/2) y^2), each of which squares
// the relative error.
__device__ inline double rsqrt_refined(double a) {
  const double h = 0.5 * a;
  double y = __builtin_amdgcn_rsq(a);
  y = fma(y, fma(-(h * y), y, 0.5), y);
  y = fma(y, fma(-(h * y), y, 0.5), y);
  return y;
}

// Bounded wait of a wavefront for an LDS flag of its own workgroup set by
// another wavefront (workgroup-scope acquire).  The setter always runs to its
// publication, so the wait ends; past the bound the factorisation is reported as
// failed at this step (*info = k0 + 1) and the wavefront goes on.  A factorisation
// already reported as failed (*info set, possibly by another workgroup of the
// launch, after which a wavefront that read it at its start has left) ends the wait
// too: its result is discarded.
constexpr int64_t kLdsSpinLimit = 1LL << 24;
__device__ inline void lds_wait(const int* flag, int32_t* info, int64_t k0) {
  int64_t spins = 0;
  while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(const_cast<int*>(flag), __ATOMIC_ACQUIRE,
                                                          __HIP_MEMORY_SCOPE_WORKGROUP)) == 0) {
    ++spins;
    // (a normal wait ends within a few thousand polls, before *info is read)
    if (spins > 16384 && (spins & 255) == 0 &&
        __builtin_amdgcn_readfirstlane(__hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0)
      break;
    if (spins > kLdsSpinLimit) {
      if ((threadIdx.x & 63) == 0) atomicCAS(info, 0, (int32_t)(k0 + 1));
      break;
    }
  }
}

// Publish an LDS flag of the workgroup (every lane stores it; the release orders
// each lane's earlier LDS accesses before it).
__device__ inline void lds_publish(int* flag) {
  __hip_atomic_store(flag, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Lane J of the lane's row of 16, for two values.
template <int J>
__device__ __forceinline__ void row_bcast2(double& a, double& b, double x, double y) {
  // two wait states between a VALU write and its DPP read
  asm("s_nop 1\n\t"
      "v_mov_b64_dpp %0, %2 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b64_dpp %1, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf"
      : "=&v"(a), "=&v"(b)
      : "v"(x), "v"(y), "n"(J));
}

// a += (a of lane J of the row) s, and so for b, c and d.
template <int J>
__device__ __forceinline__ void row_fmac4(double s, double& a, double& b, double& c, double& d) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d)
      : "v"(s), "n"(J));
}

// Pivot J of a symmetric 16x16 block, lane i = row i % 16 (all four rows of lanes
// hold the same): row i -= (x_iJ / x_JJ) row J for i > J, on the columns right of J
// and on the first J + 1 columns of the unit matrix carried along in E.  `ajj` is
// the pivot in every lane and r its reciprocal (estimate and one Newton step; the
// second opens the block), and both are left for the next pivot.
//
// One asm block, since a DPP operand must not be read within two wait states of its
// write by a vector instruction and only the order of the instructions keeps that
// without idle slots: the three opening instructions keep any register copy that
// the compiler places before the block away, and x_J+1 is read as the next pivot
// two instructions after its update.  (FP64 FMAs issue every 4 cycles and depend
// at no extra cost, the reciprocal estimate takes 16, an `s_nop 1` 8.)
template <int J>
__device__ __forceinline__ void pivot16(double (&x)[16], double (&E)[16], double& ajj, double& r, int i) {
  // column J + 1 + n of x while there is one, then the columns of E
  auto at = [&](int n) __attribute__((always_inline)) -> double& {
    return J + 1 + n < 16 ? x[(J + 1 + n) & 15] : E[(J + 1 + n) & 15];
  };
  const double xm = i > J ? x[J] : 0.0;
  double s, f;
#define NKA_ROW_FMAC(n) "v_fmac_f64_dpp %" #n ", %" #n ", %18 row_newbcast:%21 row_mask:0xf bank_mask:0xf\n\t"
  asm("v_fma_f64 %19, -%16, %17, 1.0\n\t"
      "v_fma_f64 %17, %17, %19, %17\n\t"
      "v_mul_f64 %18, %20, -%17\n\t"
      NKA_ROW_FMAC(0) NKA_ROW_FMAC(1) NKA_ROW_FMAC(2)
      "v_mov_b64_dpp %16, %0 row_newbcast:%22 row_mask:0xf bank_mask:0xf\n\t"
      NKA_ROW_FMAC(3)
      "v_rcp_f64 %17, %16\n\t"
      NKA_ROW_FMAC(4) NKA_ROW_FMAC(5) NKA_ROW_FMAC(6)
      "v_fma_f64 %19, -%16, %17, 1.0\n\t"
      "v_fma_f64 %17, %17, %19, %17\n\t"
      NKA_ROW_FMAC(7) NKA_ROW_FMAC(8) NKA_ROW_FMAC(9) NKA_ROW_FMAC(10) NKA_ROW_FMAC(11)
      NKA_ROW_FMAC(12) NKA_ROW_FMAC(13) NKA_ROW_FMAC(14) NKA_ROW_FMAC(15)
      : "+v"(at(0)), "+v"(at(1)), "+v"(at(2)), "+v"(at(3)), "+v"(at(4)), "+v"(at(5)), "+v"(at(6)), "+v"(at(7)),
        "+v"(at(8)), "+v"(at(9)), "+v"(at(10)), "+v"(at(11)), "+v"(at(12)), "+v"(at(13)), "+v"(at(14)), "+v"(at(15)),
        "+v"(ajj), "+v"(r), "=&v"(s), "=&v"(f)
      : "v"(xm), "n"(J), "n"((J + 1) & 15));
#undef NKA_ROW_FMAC
}

// All pivots (the last one has no row below it).
template <int J>
__device__ __forceinline__ void pivots16(double (&x)[16], double (&E)[16], double& ajj, double& r, int i) {
  pivot16<J>(x, E, ajj, r, i);
  if constexpr (J < 14) pivots16<J + 1>(x, E, ajj, r, i);
}

// Value e of the operand layout from a whole row per lane.
__device__ __forceinline__ void row_to_operand(const double (&r)[16], double (&o)[4], int lane) {
  const bool g1 = (lane & 16) != 0, g2 = (lane & 32) != 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double a = g1 ? r[4 * e + 1] : r[4 * e], b = g1 ? r[4 * e + 3] : r[4 * e + 2];
    o[e] = g2 ? b : a;
  }
}

// A whole row per lane from the operand layout.
__device__ __forceinline__ void operand_to_row(const double (&o)[4], double (&r)[16]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    double a = o[e], b = o[e];
    swap_rows16(a, b);  // rows of lanes 0 0 2 2 and 1 1 3 3
    double a2 = a, b2 = b;
    swap_halves(a, a2);
    swap_halves(b, b2);
    r[4 * e] = a;
    r[4 * e + 1] = b;
    r[4 * e + 2] = a2;
    r[4 * e + 3] = b2;
  }
}

// b a^T of two blocks in operand layout (`a` from LDS, [4][64]), in operand layout;
// with b as stored in the accumulators instead (element (4 e + l / 16, l % 16)), a b
// in that layout.
__device__ __forceinline__ doublex4 block_product(const double (&a)[4], const double (&b)[4]) {
  doublex4 s = (doublex4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], s, 0, 0, 0);
  return s;
}
__device__ __forceinline__ doublex4 block_product(const double* a, const double (&b)[4], int lane) {
  const double r[4] = {a[lane], a[64 + lane], a[128 + lane], a[192 + lane]};
  return block_product(r, b);
}

struct PanelLds {
  double P[4][16][64];     // 64 rows of the previous step's columns, operand layout
  double Mi[4][4][64];     // inverses of L's diagonal blocks
  double Lo[6][4][64];     // L's blocks (1,0) (2,0) (2,1) (3,0) (3,1) (3,2)
  double R[3][2][4][64];   // strip i = 1..3: block (i, i-1), diagonal block, up to date
  double Lx[4][4][64];     // L's diagonal blocks before the columns' scaling,
  double Ly[4][16];        // and that scaling
  int flags[16];           // [0..3] Mi, [4..9] Lo, [10..12] R, [13..15] P read by wavefront 1..3
};
__device__ constexpr int lo_index(int i, int k) { return i * (i - 1) / 2 + k; }

// The K = 64 products with the previous step's columns take them in an order of
// their own, 8 (q / 2) + 2 (l / 16) + q % 2 for product q, so that a lane reads 16
// bytes at a time and four lanes 64 bytes of a row.
typedef double pair_t __attribute__((ext_vector_type(2), aligned(8)));
template <int N>
__device__ __forceinline__ void load_k_pairs(const double* row, int q0, int lane, double (&v)[N]) {
#pragma unroll
  for (int q = 0; q < N; q += 2) {
    const pair_t d = *(const pair_t*)(row + 4 * (q0 + q) + 2 * (lane >> 4));
    v[q] = d.x;
    v[q + 1] = d.y;
  }
}

// Rows 16 s.. of the 64 rows at P (row r: P + r * lda; rows from `rows` on re-read
// the last) for products q0..q0 + 7.
__device__ __forceinline__ void load_strip_half(const double* P, int64_t lda, int64_t rows, int s, int q0, int lane,
                                                double (&v)[8]) {
  const int64_t r = 16 * s + (lane & 15);
  load_k_pairs(P + min<int64_t>(r, rows - 1) * lda, q0, lane, v);
}

// U[k] -= (strip of 16 rows, pb) (rows 16 k.. of P)^T, K = 64, k < NBLK.
template <int NBLK>
__device__ __forceinline__ void strip_update(const double (*P)[16][64], const double (&pb)[16], double (&U)[NBLK][4],
                                             int lane) {
  // two blocks at a time: enough to cover a product's latency, and within 128 registers
#pragma unroll
  for (int k0 = 0; k0 < NBLK; k0 += 2) {
    doublex4 acc[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) acc[k] = (doublex4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 16; ++q)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (k0 + k < NBLK) acc[k] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[k0 + k][q][lane], pb[q], acc[k], 0, 0, 0);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k0 + k < NBLK) U[k0 + k][e] -= acc[k][e];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Blocks (I, 0..I) of the symmetric diagonal block at C (lower triangle valid;
// identity from row and column nb on).
template <int I>
__device__ __forceinline__ void load_diag_strip(const double* C, int64_t lda, int nb, int lane, double (&u)[I + 1][4]) {
  const int r = 16 * I + (lane & 15), g = lane >> 4;
  if (nb == CH_NB) {
    const double* row = C + r * lda + g;
    const double* block = C + 16 * I * lda + 16 * I;
#pragma unroll
    for (int k = 0; k < I; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) u[k][e] = row[16 * k + 4 * e];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int a = lane & 15, c = 4 * e + g;
      u[I][e] = block[max(a, c) * lda + min(a, c)];
    }
  } else {
#pragma unroll
    for (int k = 0; k <= I; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = 16 * k + 4 * e + g;
        const int hi = max(r, c), lo = min(r, c);
        const double v = C[(int64_t)min(hi, nb - 1) * lda + min(lo, nb - 1)];
        u[k][e] = hi < nb ? v : (r == c ? 1.0 : 0.0);
      }
  }
}

// Rows 16 I.. of the diagonal block, one wavefront (I = 1..3): the previous step's
// update, then the blocks left of the diagonal as the inverses come in; block
// (I, I-1) and the diagonal block are handed to wavefront 0 as soon as they need
// nothing but L's columns up to I - 2.
template <int I, bool UPDATE>
__device__ __forceinline__ void diag_strip(PanelLds& s, double (&U)[I + 1][4], int lane, int32_t* info, int64_t k0) {
  if constexpr (UPDATE) {
    double pb[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) pb[q] = s.P[I][q][lane];
    strip_update<I + 1>(s.P, pb, U, lane);
  }
  lds_publish(&s.flags[12 + I]);
#pragma unroll
  for (int p = 0; p + 1 < I; ++p) {
    lds_wait(&s.flags[p], info, k0);
    const doublex4 x = block_product(&s.Mi[p][0][0], U[p], lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      U[p][e] = x[e];
      s.Lo[lo_index(I, p)][e][lane] = x[e];
    }
    lds_publish(&s.flags[4 + lo_index(I, p)]);
#pragma unroll
    for (int k = p + 1; k <= I; ++k) {
      doublex4 y;
      if (k < I) {
        lds_wait(&s.flags[4 + lo_index(k, p)], info, k0);
        y = block_product(&s.Lo[lo_index(k, p)][0][0], U[p], lane);
      } else {
        y = block_product(U[p], U[p]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) U[k][e] -= y[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s.R[I - 1][0][e][lane] = U[I - 1][e];
    s.R[I - 1][1][e][lane] = U[I][e];
  }
  lds_publish(&s.flags[9 + I]);
}

// The diagonal blocks, one wavefront: c is block (0, 0), up to date.  Returns the
// first failing column + 1 + k0 (a pivot that is not positive and finite), or 0.
__device__ __forceinline__ int diag_chain(PanelLds& s, double (&c)[4], int lane, int32_t* info, int64_t k0) {
  const int i = lane & 15;
  int bad = 0;
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    double x[16], E[16];
    operand_to_row(c, x);
#pragma unroll
    for (int q = 0; q < 16; ++q) E[q] = q == i ? 1.0 : 0.0;
    double ajj, dummy;
    row_bcast2<0>(ajj, dummy, x[0], x[0]);
    double r = __builtin_amdgcn_rcp(ajj);
    r = fma(r, fma(-ajj, r, 1.0), r);
    pivots16<0>(x, E, ajj, r, i);
    // the pivots d are x's diagonal; L = x / sqrt(d) by columns, its inverse
    // E / sqrt(d) by rows
    double lx[4], lin[4];
    double d = x[0];
#pragma unroll
    for (int q = 1; q < 16; ++q) d = q == i ? x[q] : d;
    const double y = rsqrt_refined(d);
    row_to_operand(E, lin, lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lin[e] *= y;
      s.Mi[p][e][lane] = lin[e];
    }
    lds_publish(&s.flags[p]);
    if (p < 3) {
      lds_wait(&s.flags[10 + p], info, k0);
      double b[4], dp[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = s.R[p][0][e][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) dp[e] = s.R[p][1][e][lane];
      doublex4 xl = block_product(lin, b);
      // in the products' shadow
      row_to_operand(x, lx, lane);
      const int lo = (p + 1) * p / 2 + p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        b[e] = xl[e];
        s.Lo[lo][e][lane] = xl[e];
      }
      xl = block_product(b, b);
      lds_publish(&s.flags[4 + lo]);
#pragma unroll
      for (int e = 0; e < 4; ++e) c[e] = dp[e] - xl[e];
    } else {
      row_to_operand(x, lx, lane);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s.Lx[p][e][lane] = lx[e];
    if (lane < 16) s.Ly[p][i] = y;
    const uint32_t fail = (uint32_t)__ballot(!(d > 0.0 && isfinite(d))) & 0xffffu;
    if (fail && !bad) bad = (int)(k0 + 16 * p + __builtin_ctz(fail) + 1);
  }
  return bad;
}

// Rows r0.. (16) below the diagonal block and, with UPDATE, their part of the
// previous step's columns.  Rows from n on re-read the last.
template <bool UPDATE>
__device__ __forceinline__ void load_factor_strip(const double* A, int64_t lda, int64_t n, int64_t k0, int64_t r0,
                                                  int lane, double (&U)[4][4], double (&pb)[16]) {
  const double* row = A + min<int64_t>(r0 + (lane & 15), n - 1) * lda + k0;
  if constexpr (UPDATE) load_k_pairs(row - CH_NB, 0, lane, pb);
  row += lane >> 4;
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) U[k][e] = row[16 * k + 4 * e];
}

// The strip's update and solve, column block by column block as the factor comes
// in.  The solved blocks are formed once more with the operands exchanged, which
// puts them into the accumulators by rows, for stores of whole lines.
template <bool UPDATE>
__device__ __forceinline__ void factor_strip(PanelLds& s, double* A, int64_t lda, int64_t n, int64_t k0, int64_t r0,
                                             int lane, int32_t* info, double (&U)[4][4], double (&pb)[16]) {
  if constexpr (UPDATE) strip_update<4>(s.P, pb, U, lane);
  double* out = A + (r0 + (lane >> 4)) * lda + k0 + (lane & 15);
  const int64_t left = n - r0 - (lane >> 4);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
#pragma unroll
    for (int k = 0; k < p; ++k) {
      lds_wait(&s.flags[4 + lo_index(p, k)], info, k0);
      const doublex4 y = block_product(&s.Lo[lo_index(p, k)][0][0], U[k], lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) U[p][e] -= y[e];
    }
    lds_wait(&s.flags[p], info, k0);
    const double m[4] = {s.Mi[p][0][lane], s.Mi[p][1][lane], s.Mi[p][2][lane], s.Mi[p][3][lane]};
    const doublex4 o = block_product(U[p], m);
    if (p < 3) {
      const doublex4 x = block_product(m, U[p]);
#pragma unroll
      for (int e = 0; e < 4; ++e) U[p][e] = x[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * e < left) out[4 * e * lda + 16 * p] = o[e];
  }
}
// One 64-column step k0 of a panel, in one launch of eight wavefronts per
// workgroup with two roles.  `nb` columns (64 but for the matrix's last block).
//
// Workgroups [0, n_factor): the step's columns.  With UPDATE the previous step's
// rank-64 update of them is applied first.  Every workgroup factors the diagonal
// block itself (wavefronts 0-3), so that the solve of the rows below,
// L21 = A21 L11^{-T} (`strips` times 16 of them, wavefronts 5-7 and 1), needs no
// second launch; wavefront 4 idles, since FP64 matrix products on a SIMD hold up
// the vector FP64 of the other wavefront on it.  Three strips while the workgroups
// fit on the chip (the fourth ends 1.3 us after the chain), else four.
// Workgroup 0 writes L11 to `slot` (64x64 row-major, identity from nb on, zeros
// above the diagonal) and reports a failed pivot in *info; L11 reaches A's diagonal
// block in the inversion kernel at the end, since a workgroup that starts late
// still reads the unfactored block from A.
//
// The other workgroups apply the previous step's update to the panel's columns
// right of this step, 128 rows x 64 columns each, by the same strips.  The roles
// write disjoint columns and read only what earlier launches wrote.
//
// Bound by the chain of 64 pivots and the block products between them in wavefront
// 0: of 11.4 us in the kernel at n = 1680 the loads take 3.4, the chain 7.6 (a
// 16x16 block 1.3, the products to the next one 0.5) and the stores 0.5; 14.4 us
// from launch to launch.  With the pivots' columns broadcast through LDS and the
// rest of the block updated between the sub-panels by the same wavefront the step
// took 20.1 us (23 at 8384).
template <bool UPDATE>
__global__ void __launch_bounds__(512, 4) panel_step_kernel(double* __restrict__ A, int64_t lda, int64_t n,
                                                            int64_t k0, int nb, int strips, int n_factor, int64_t cols_b,
                                                            int tiles_n_b, double* __restrict__ slot,
                                                            int32_t* __restrict__ info) {
  extern __shared__ __align__(16) unsigned char smem[];
  PanelLds& s = *(PanelLds*)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int32_t failed = __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // (read first, looked at with the rows)
  if (tid < 16) s.flags[tid] = 0;  // ordered by the barrier below
  const bool factor = (int)blockIdx.x < n_factor;
  // the previous step's columns; rows k0.. as the factored columns, or the rows of
  // this workgroup's 64 columns right of the step
  const uint32_t tile = blockIdx.x - (uint32_t)n_factor, ti = factor ? 0 : tile / (uint32_t)tiles_n_b;
  const int64_t c0 = factor ? k0 : k0 + CH_NB + (int64_t)(tile - ti * (uint32_t)tiles_n_b) * CH_NB;
  // this wavefront's strip: of the factored columns for wavefronts 5-7 and, with
  // four strips, after its part of the diagonal block, wavefront 1; of the columns
  // right for all
  const int64_t r0 = factor ? k0 + CH_NB + (int64_t)blockIdx.x * 16 * strips + (w == 1 ? 48 : 16 * (w - 5))
                            : k0 + CH_NB + (int64_t)ti * 128 + 16 * w;
  const int cols = factor ? nb : (int)min<int64_t>(CH_NB, k0 + CH_NB + cols_b - c0);
  if (!factor && k0 + CH_NB + (int64_t)ti * 128 + 127 < c0) return;  // above the diagonal
  const double* Pc = A + c0 * lda + k0 - CH_NB;
  double v[8];
  if constexpr (UPDATE) load_strip_half(Pc, lda, cols, w >> 1, 8 * (w & 1), lane, v);
  // (every wavefront meets the one barrier below in its own branch)
  auto stage = [&]() __attribute__((always_inline)) {
    if constexpr (UPDATE) {
#pragma unroll
      for (int q = 0; q < 8; ++q) s.P[w >> 1][8 * (w & 1) + q][lane] = 16 * (w >> 1) + (lane & 15) < cols ? v[q] : 0.0;
    }
    __syncthreads();
  };
  const double* D = A + k0 * lda + k0;
  if (factor && w == 0) {
    __builtin_amdgcn_s_setprio(3);  // the chain goes first where wavefronts share a SIMD
    double u[1][4];
    load_diag_strip<0>(D, lda, nb, lane, u);
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
    if constexpr (UPDATE) {
      doublex4 a[2] = {(doublex4){0.0, 0.0, 0.0, 0.0}, (doublex4){0.0, 0.0, 0.0, 0.0}};
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const double p = s.P[0][q][lane];
        a[q & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(p, p, a[q & 1], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) u[0][e] -= a[0][e] + a[1][e];
    }
    const int bad = diag_chain(s, u[0], lane, info, k0);
    if (blockIdx.x == 0 && lane == 0 && bad) atomicCAS(info, 0, bad);
  } else if (factor && (w == 1 || w > 4)) {
    // (rows below the block imply that it has 64 columns)
    double U[4][4], pb[16], u[2][4];
    const bool rows = r0 < n && (w != 1 || strips == 4);
    if (w == 1) load_diag_strip<1>(D, lda, nb, lane, u);
    if (rows) load_factor_strip<UPDATE>(A, lda, n, k0, r0, lane, U, pb);
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
    if (w == 1) {
      __builtin_amdgcn_s_setprio(2);
      diag_strip<1, UPDATE>(s, u, lane, info, k0);
      __builtin_amdgcn_s_setprio(0);
    } else if (UPDATE && rows) {
      // the matrix cores serve the diagonal block first
      lds_wait(&s.flags[w == 6 ? 11 : 8 + w], info, k0);
    }
    if (rows) factor_strip<UPDATE>(s, A, lda, n, k0, r0, lane, info, U, pb);
  } else if (factor && w == 2) {
    __builtin_amdgcn_s_setprio(1);
    double u[3][4];
    load_diag_strip<2>(D, lda, nb, lane, u);
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
    diag_strip<2, UPDATE>(s, u, lane, info, k0);
  } else if (factor && w == 3) {
    __builtin_amdgcn_s_setprio(1);
    double u[4][4];
    load_diag_strip<3>(D, lda, nb, lane, u);
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
    diag_strip<3, UPDATE>(s, u, lane, info, k0);
  } else if (factor) {
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
  } else {
    // 16 rows of the columns right of the step, by rows (a lane holds one column)
    double U[4][4], pb[16];
    const int64_t row = min<int64_t>(r0 + (lane & 15), n - 1);
    load_k_pairs(A + row * lda + k0 - CH_NB, 0, lane, pb);
    double* C = A + r0 * lda + c0 + (lane & 15);
    const int64_t left = n - r0 - (lane >> 4);  // rows from this lane's first
    // rows and columns past the last re-read it; they are not stored
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double* rowc = A + min<int64_t>(r0 + (lane >> 4) + 4 * e, n - 1) * lda + c0;
#pragma unroll
      for (int k = 0; k < 4; ++k) U[k][e] = rowc[min(16 * k + (lane & 15), cols - 1)];
    }
    if (__builtin_amdgcn_readfirstlane(failed) != 0) return;
    stage();
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
      doublex4 acc[2] = {(doublex4){0.0, 0.0, 0.0, 0.0}, (doublex4){0.0, 0.0, 0.0, 0.0}};
#pragma unroll
      for (int q = 0; q < 16; ++q)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(pb[q], s.P[k + t][q][lane], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * e < left && 16 * (k + t) + (lane & 15) < cols)
            C[((lane >> 4) + 4 * e) * lda + 16 * (k + t)] = U[k + t][e] - acc[t][e];
    }
  }
  if (blockIdx.x != 0) return;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < CH_NB * CH_NB / 512; ++t) {
    const int idx = tid + 512 * t, r = idx >> 6, c = idx & 63;
    const int bi = r >> 4, bj = c >> 4;
    double x = 0.0;
    const int op = ((c & 15) >> 2) * 64 + (c & 3) * 16 + (r & 15);
    if (bi == bj) x = c <= r ? (&s.Lx[bi][0][0])[op] * s.Ly[bi][c & 15] : 0.0;
    else if (bj < bi) x = (&s.Lo[lo_index(bi, bj)][0][0])[op];
    slot[idx] = x;
  }
}

// Pivot J of the substitution: row i of E -= (l_iJ / l_JJ) row J for i > J, columns
// 0..J (in fours); y = 1 / l_ii in lane i.
template <int J>
__device__ __forceinline__ void substitute16(const double (&l)[16], double (&E)[16], double y, int i) {
  double yj, dummy;
  row_bcast2<J>(yj, dummy, y, y);
  const double s = i > J ? -(l[J] * yj) : 0.0;
  row_fmac4<J>(s, E[0], E[1], E[2], E[3]);
  if constexpr (J >= 4) row_fmac4<J>(s, E[4], E[5], E[6], E[7]);
  if constexpr (J >= 8) row_fmac4<J>(s, E[8], E[9], E[10], E[11]);
  if constexpr (J >= 12) row_fmac4<J>(s, E[12], E[13], E[14], E[15]);
  if constexpr (J < 14) substitute16<J + 1>(l, E, y, i);
}

// inv_b = L_bb^{-1} for every 64x64 diagonal block b of the factor, one workgroup
// per block.  The factored block is read from its slot in `inv` (row-major,
// identity padding, zeros above the diagonal), copied into A's diagonal block, and
// replaced by its inverse (row-major): wavefront p inverts diagonal block p by
// substitution, then forms block column p of the inverse,
// X_pp = M_p, X_rp = -M_r sum_{p <= k < r} L_rk X_kp, in registers.
// Bound by latencies: 8 us at 27 blocks, 39 us with a lane per column of the 64x64
// block.
__global__ void __launch_bounds__(256) trtri_blocks_kernel(double* __restrict__ A, int64_t lda, int64_t n,
                                                           double* __restrict__ inv, double* __restrict__ y,
                                                           const int32_t* __restrict__ info) {
  if (*info != 0) return;
  __shared__ double Lo[6][4][64], Mi[4][4][64];
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t k0 = (int64_t)blockIdx.x * CH_NB;
  const int nb = (int)min<int64_t>(CH_NB, n - k0);
  double* blk = inv + (int64_t)blockIdx.x * CH_NB * CH_NB;
  // what the solves start from
  if (tid < nb) ((uint64_t*)y)[k0 + tid] = kUnsolved;
  double v[16], l[16], E[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) l[q] = blk[(16 * w + i) * CH_NB + 16 * w + q];
#pragma unroll
  for (int t = 0; t < 16; ++t) v[t] = blk[tid + 256 * t];
  double rd = 1.0;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    E[q] = q == i ? 1.0 : 0.0;
    rd = q == i ? l[q] : rd;
  }
  rd = 1.0 / rd;
  substitute16<0>(l, E, rd, i);
  double o[4];
  row_to_operand(E, o, lane);
#pragma unroll
  for (int e = 0; e < 4; ++e) Mi[w][e][lane] = o[e] * rd;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int idx = tid + 256 * t, r = idx >> 6, c = idx & 63;
    if ((c >> 4) < (r >> 4)) Lo[lo_index(r >> 4, c >> 4)][(c & 15) >> 2][(c & 3) * 16 + (r & 15)] = v[t];
    if (r < nb && c <= r) A[(k0 + r) * lda + k0 + c] = v[t];
  }
  __syncthreads();  // every read of the slot is done
  double X[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (r < w) {
#pragma unroll
      for (int e = 0; e < 4; ++e) X[r][e] = 0.0;
    } else if (r == w) {
      // element (4 e + l / 16, l % 16)
#pragma unroll
      for (int e = 0; e < 4; ++e) X[r][e] = Mi[w][i >> 2][(i & 3) * 16 + 4 * e + (lane >> 4)];
    } else {
      double T[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < r; ++k) {
        if (k < w) continue;
        const doublex4 t = block_product(&Lo[lo_index(r, k)][0][0], X[k], lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) T[e] += t[e];
      }
      const doublex4 t = block_product(&Mi[r][0][0], T, lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) X[r][e] = -t[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) blk[(16 * r + 4 * e + (lane >> 4)) * CH_NB + 16 * w + i] = X[r][e];
  }
}

}  // namespace nka
