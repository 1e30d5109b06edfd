// Dense linear algebra of the SR / minSR solve on gfx950 matrix cores.
//
// nka_gram_bf16x3  S = O_L^T O_L or T = O_L O_L^T (+ shift I + offset 11^T)
//                  (netket/optimizer/qgt/qgt_jacobian_dense.py:136-161,
//                   netket/_src/ngd/sr.py:58-63, netket/_src/ngd/srt.py:55-66)
//                  from a bf16 hi/lo split with three v_mfma_f32_32x32x16_bf16
//                  products per tile (hi.hi + hi.lo + lo.hi), FP32 accumulate.
// nka_gemm_nt_f64 / nka_syrk_f64
//                  FP64 v_mfma_f64_16x16x4 products, used by the Cholesky
//                  trailing update, its panel solve and FP64 Gram matrices.
// nka_potrf_f64 / nka_potrs_f64
//                  blocked right-looking Cholesky and the two triangular
//                  solves (jax.scipy.linalg.cho_factor / cho_solve as called by
//                  netket/optimizer/solver/solvers.py:241-270).
// nka_gemv_f64, nka_check_finite, nka_sgd_update, nka_centre_scale, nka_stats_moments
//                  vector helpers of the step.
#include "nka_common.hpp"
#include "nka_panel.hpp"
#include "netket_amd.h"
#include <mutex>

namespace nka {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Map a linear block id onto the lower-triangular tile pair (ti >= tj).
__device__ inline void tri_tile(int64_t b, int& ti, int& tj) {
  int64_t i = (int64_t)((sqrt(8.0 * (double)b + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= b) ++i;
  while (i * (i + 1) / 2 > b) --i;
  ti = (int)i;
  tj = (int)(b - i * (i + 1) / 2);
}

// Spread consecutive block ids over the 8 XCDs in contiguous chunks: the
// hardware dispatches block b to XCD b % 8, so block b is given the work item
// (b % 8) * ceil(G/8) + b / 8; neighbouring tiles (which share operand rows)
// then run on the same XCD and share its L2.
// The grid is launched with a multiple of 8 blocks (G = 8 * per), which makes
// the map a bijection of [0, G); ids past the real work count exit early.
__device__ inline int64_t xcd_remap(int64_t b, int64_t G) {
  const int64_t per = G / 8;
  return (b % 8) * per + b / 8;
}
inline unsigned grid_mult8(int64_t tiles) { return (unsigned)(((tiles + 7) / 8) * 8); }

// ---------------------------------------------------------------------------
// bf16x3 Gram: 128x128 output tile per workgroup, 4 waves of 64x64, K step 64.
// ---------------------------------------------------------------------------
constexpr int GB_K = 64;    // K step (bf16 elements): one 128-byte line per row and plane
constexpr int GB_LD = 72;   // LDS row stride in bf16 (64 + 8 pad: 144 bytes)
constexpr int GB_CPR = GB_K / 8;              // 16-byte chunks per row and plane

// Epilogue of the RBM neural tangent kernel, T = O_c O_c^T scaled, from
// Theta = t t^T (the bf16x3 product) and S = sigma sigma^T:
//   T_ij = scale ((hb + S_ij) Theta_ij + ha S_ij - v_i - v_j + c) + offset
// (+ shift on the diagonal), with S_ij = N - 2 popcount(bits_i ^ bits_j)
// exact from the packed spins.
struct GramRbmEpi {
  const uint32_t* bits;   // (n, nw): bit b of word w is (sigma_{32w+b} > 0)
  int nw, nwp, N;         // words per row, LDS row stride (multiple of 4), sites
  const double* v;
  const double* c;
  double hb, ha, scale;
  // two-layer network (NP = 3): the passes 1 and 2 take these planes, and
  //   T_ij = scale ((hb2 + H_ij) G_ij + (hb + X_ij) D_ij - v_i - v_j + c) + offset
  // with H = h1 h1^T (pass 0), G = g2 g2^T (pass 1), D = d1 d1^T (pass 2),
  // X = x x^T from the packed spins
  const uint16_t* xh1;
  const uint16_t* xl1;
  const uint16_t* xh2;
  const uint16_t* xl2;
  int64_t K1, K2, ld1, ld2;
  double hb2;
};

// WT: wave tile edge (64 or 96); the workgroup tile is 2 WT x 2 WT (four
// waves), so each wave holds (WT/32)^2 accumulators of 32x32.  A 192-wide
// tile reads 12 operand fragments from LDS per 27 products (128-wide: 8 per
// 12) and re-reads each operand row panel from L2 a third fewer times; it
// needs 110 KB of LDS, so one workgroup runs per CU.
// NP: products per tile, 1 (the Gram, or the RBM tangent kernel when RBM) or
// 3 (the two-layer network's tangent kernel, RBM set), each K loop in turn.
template <bool RBM, int WT, int NP = 1>
__global__ void __launch_bounds__(256, 1) gram_bf16x3_kernel(const uint16_t* __restrict__ xh,
                                                          const uint16_t* __restrict__ xl, int64_t n,
                                                          int64_t K, int64_t ldx, double shift,
                                                          double offset, double* __restrict__ out,
                                                          int64_t ldo, int64_t n_tiles_total,
                                                          GramRbmEpi ep) {
  constexpr int TT = 2 * WT;                 // workgroup tile edge
  constexpr int MI = WT / 32;                // 32x32 tiles per wave edge
  constexpr int NIT = TT * GB_CPR / 256;     // 16-byte chunks per thread and plane
  __shared__ __attribute__((aligned(16))) uint16_t sA[2][TT * GB_LD];  // [plane][row*LD + k]
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][TT * GB_LD];
  const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if (bid >= n_tiles_total) return;
  int ti, tj;
  tri_supertile(bid, (n + TT - 1) / TT, ti, tj);
  const int64_t i0 = (int64_t)ti * TT, j0 = (int64_t)tj * TT;
  const int tid = threadIdx.x, wid = tid / 64, lane = lane_id();
  const int wm = (wid >> 1) * WT, wn = (wid & 1) * WT;  // wave tile origin in block tile
  const bool diag_tile = (ti == tj);

  floatx16 accs[NP][MI][MI];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
      for (int b = 0; b < MI; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) accs[p][a][b][e] = 0.0f;

#pragma unroll
  for (int pass = 0; pass < NP; ++pass) {
    const uint16_t* xh_p = pass == 0 ? xh : pass == 1 ? ep.xh1 : ep.xh2;
    const uint16_t* xl_p = pass == 0 ? xl : pass == 1 ? ep.xl1 : ep.xl2;
    const int64_t K_p = pass == 0 ? K : pass == 1 ? ep.K1 : ep.K2;
    const int64_t ld_p = pass == 0 ? ldx : pass == 1 ? ep.ld1 : ep.ld2;
    if (pass > 0) __syncthreads();  // the previous pass's last slab has been read
    // Each operand slab is TT rows x GB_K k = TT GB_CPR chunks of 8 bf16;
    // thread tid moves chunks tid + 256 it (it < NIT) of each of the (up to)
    // four planes.  The next slab is fetched into registers while the current
    // one is used.
    uint4 pf[NIT][4];
    // chunks it0 <= it < it1 of the slab at k0
    auto fetch_part = [&](int64_t k0, int it0, int it1) {
  #pragma unroll
      for (int it = 0; it < NIT; ++it) {
        if (it < it0 || it >= it1) continue;
        const int chunk = tid + it * 256;
        const int r = chunk / GB_CPR, kc = (chunk % GB_CPR) * 8;
        const int64_t kk = k0 + kc;
        uint4 z = {0, 0, 0, 0};
        pf[it][0] = z;
        pf[it][1] = z;
        pf[it][2] = z;
        pf[it][3] = z;
        if (i0 + r < n && kk < K_p) {
          pf[it][0] = *(const uint4*)(xh_p + (i0 + r) * ld_p + kk);
          pf[it][1] = *(const uint4*)(xl_p + (i0 + r) * ld_p + kk);
        }
        if (!diag_tile && j0 + r < n && kk < K_p) {
          pf[it][2] = *(const uint4*)(xh_p + (j0 + r) * ld_p + kk);
          pf[it][3] = *(const uint4*)(xl_p + (j0 + r) * ld_p + kk);
        }
      }
    };
    fetch_part(0, 0, NIT);
    for (int64_t k0 = 0; k0 < K_p; k0 += GB_K) {
      __syncthreads();
  #pragma unroll
      for (int it = 0; it < NIT; ++it) {
        const int chunk = tid + it * 256;
        const int r = chunk / GB_CPR, kc = (chunk % GB_CPR) * 8;
        *(uint4*)(&sA[0][r * GB_LD + kc]) = pf[it][0];
        *(uint4*)(&sA[1][r * GB_LD + kc]) = pf[it][1];
        if (!diag_tile) {
          *(uint4*)(&sB[0][r * GB_LD + kc]) = pf[it][2];
          *(uint4*)(&sB[1][r * GB_LD + kc]) = pf[it][3];
        }
      }
      __syncthreads();
      const uint16_t* Bh = diag_tile ? sA[0] : sB[0];
      const uint16_t* Bl = diag_tile ? sA[1] : sB[1];
      const bool more = k0 + GB_K < K_p;
  #pragma unroll
      for (int ks = 0; ks < GB_K; ks += 16) {
        // the next slab's loads are spread over the first K sub-steps, so the
        // memory pipeline works through them while the products run
        if (more) {
          constexpr int per = (NIT + GB_K / 16 - 2) / (GB_K / 16 - 1);
          const int q = ks / 16;
          if (q < GB_K / 16 - 1) fetch_part(k0 + GB_K, q * per, (q + 1) * per < NIT ? (q + 1) * per : NIT);
        }
        __builtin_amdgcn_sched_barrier(0);
        const int kq = ks + (lane >> 5) * 8;
        bf16x8 ah[MI], al[MI], bh[MI], bl[MI];
  #pragma unroll
        for (int a = 0; a < MI; ++a) {
          const int row = wm + a * 32 + (lane & 31);
          ah[a] = *(const bf16x8*)(&sA[0][row * GB_LD + kq]);
          al[a] = *(const bf16x8*)(&sA[1][row * GB_LD + kq]);
        }
  #pragma unroll
        for (int b = 0; b < MI; ++b) {
          const int row = wn + b * 32 + (lane & 31);
          bh[b] = *(const bf16x8*)(&Bh[row * GB_LD + kq]);
          bl[b] = *(const bf16x8*)(&Bl[row * GB_LD + kq]);
        }
        // small products first, four independent accumulators between
        // consecutive updates of the same accumulator
  #pragma unroll
        for (int a = 0; a < MI; ++a)
  #pragma unroll
          for (int b = 0; b < MI; ++b)
            accs[pass][a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[a], bh[b], accs[pass][a][b], 0, 0, 0);
  #pragma unroll
        for (int a = 0; a < MI; ++a)
  #pragma unroll
          for (int b = 0; b < MI; ++b)
            accs[pass][a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bl[b], accs[pass][a][b], 0, 0, 0);
  #pragma unroll
        for (int a = 0; a < MI; ++a)
  #pragma unroll
          for (int b = 0; b < MI; ++b)
            accs[pass][a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bh[b], accs[pass][a][b], 0, 0, 0);
      }
    }
  }
  // store: element e of lane l in a 32x32 tile is (row (e/4)*8 + (l/32)*4 + e%4, col l%32)
  if constexpr (!RBM) {
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
      for (int b = 0; b < MI; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t gi = i0 + wm + a * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
          const int64_t gj = j0 + wn + b * 32 + (lane & 31);
          if (gi < n && gj <= gi) {
            double v = (double)accs[0][a][b][e] + offset;
            if (gi == gj) v += shift;
            out[gi * ldo + gj] = v;
          }
        }
  } else {
    // spins of the tile's 128 rows and 128 columns into the operand LDS
    __syncthreads();
    uint32_t* rb = (uint32_t*)&sA[0][0];
    uint32_t* cb = (uint32_t*)&sB[0][0];
    const int nwp = ep.nwp;
    for (int idx = tid; idx < TT * nwp; idx += 256) {
      const int r = idx / nwp, w = idx % nwp;
      uint32_t x = 0, y = 0;
      if (w < ep.nw) {
        if (i0 + r < n) x = ep.bits[(i0 + r) * ep.nw + w];
        if (j0 + r < n) y = ep.bits[(j0 + r) * ep.nw + w];
      }
      rb[idx] = x;
      cb[idx] = y;
    }
    __syncthreads();
    int cnt[MI][MI][16];
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
      for (int b = 0; b < MI; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) cnt[a][b][e] = 0;
    for (int w = 0; w < nwp; w += 4) {
      uint4 cq[MI];
#pragma unroll
      for (int b = 0; b < MI; ++b) cq[b] = *(const uint4*)&cb[(wn + b * 32 + (lane & 31)) * nwp + w];
#pragma unroll
      for (int a = 0; a < MI; ++a)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int rl = wm + a * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
          const uint4 rq = *(const uint4*)&rb[rl * nwp + w];
#pragma unroll
          for (int b = 0; b < MI; ++b)
            cnt[a][b][e] += __builtin_popcount(rq.x ^ cq[b].x) + __builtin_popcount(rq.y ^ cq[b].y) +
                            __builtin_popcount(rq.z ^ cq[b].z) + __builtin_popcount(rq.w ^ cq[b].w);
        }
    }
    const double cc = *ep.c;
#pragma unroll
    for (int a = 0; a < MI; ++a)
#pragma unroll
      for (int b = 0; b < MI; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t gi = i0 + wm + a * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
          const int64_t gj = j0 + wn + b * 32 + (lane & 31);
          if (gi < n && gj <= gi) {
            const double S = (double)(ep.N - 2 * cnt[a][b][e]);
            double v;
            if constexpr (NP == 1) {
              const double Th = (double)accs[0][a][b][e];
              v = ep.scale * ((ep.hb + S) * Th + ep.ha * S - ep.v[gi] - ep.v[gj] + cc) + offset;
            } else {
              const double Hh = (double)accs[0][a][b][e];
              const double Gg = (double)accs[NP - 2][a][b][e];
              const double Dd = (double)accs[NP - 1][a][b][e];
              v = ep.scale * ((ep.hb2 + Hh) * Gg + (ep.hb + S) * Dd - ep.v[gi] - ep.v[gj] + cc) + offset;
            }
            if (gi == gj) v += shift;
            out[gi * ldo + gj] = v;
          }
        }
  }
}

// Largest LDS row stride (words) of the packed spins in the RBM epilogue: the
// tile's rows must fit in one operand buffer (2 planes x rows x GB_LD bf16).
constexpr int kGramRbmMaxNwp = (int)(2 * GB_LD * sizeof(uint16_t) / sizeof(uint32_t)) / 4 * 4;
// wave tile edges of the Gram and of the RBM tangent kernel
constexpr int kGramWT = 96;
constexpr int kGramRbmWT = 64;

// ---------------------------------------------------------------------------
// C = A (Bh + Bl)^T in FP32 (ma x nb), K contiguous in both operands (row
// stride ldk, a multiple of 64; K too, zero beyond the true K).  A is one bf16
// plane whose entries bf16 holds exactly (products of +-1 spins, 0 and 1); B
// is split into two bf16 planes.  Each fragment pair therefore takes two
// products (v_mfma_f32_32x32x16_bf16) instead of the Gram's three, and A's LDS
// slab is a single plane.  Tiles are numbered down the columns (the ma side
// fastest), so the workgroups that share a B column panel (the larger operand)
// sit on one XCD and read it through one L2.
// The FP32 accumulation inside the MFMA rounds with a bias (the error of a
// plain sum over 16384 samples grows like the number of accumulations times
// 2^-24, not like its square root), so the products are accumulated on the
// matrix cores for 64 kExactAChunk samples (128 accumulations) at a time and
// each chunk is added into a separate FP32 total with round-to-nearest vector
// adds.  Both kernels take the products of an entry in the same order.
// ---------------------------------------------------------------------------
constexpr int kExactAChunk = 16;
constexpr int kExactAMIA = 3, kExactAMIB = 2;  // 32 x 32 blocks per wavefront
constexpr int kExactAK = 32;                   // samples per K step
constexpr int kExactABuf = 4;                  // K steps held in LDS

// 192 x 128 tiles, four wavefronts of 96 x 64, one workgroup per CU: the
// accumulators and totals take 192 registers, and a sub-step of 16 samples
// reads 7 fragments from LDS for 12 products.  Operands go from global memory
// straight into LDS, three K steps ahead; one request (an LDS read of the other
// sub-step's fragments, or a load of a later step) stands behind each product.
// A row's four 16-byte chunks of a K step are stored in the order
// chunk ^ (row / 4 % 4): fragment reads (32 consecutive rows, one chunk) are
// free of bank conflicts over the 64 banks.  Bound by the matrix cores.
// 2081 x 8385 x 16384: 1.24 ms (0.92 PFLOP/s executed, a library bf16 product
// reaches 1.09), 1.42 with the slab prefetched into registers and one buffer.
// Whole dense S there 1.80 -> 1.57 ms; the whole SR step, whose FP64 products
// then run at a lower clock, 8.25 -> 8.18 ms.
// ldk < 2^26, so that 16 rows lie within a buffer descriptor's offsets.
__global__ void __launch_bounds__(256, 1) gemm_exact_a_kernel(const uint16_t* __restrict__ a, int64_t ma,
                                                           const uint16_t* __restrict__ bh,
                                                           const uint16_t* __restrict__ bl, int64_t nb, int64_t K,
                                                           int64_t ldk, float* __restrict__ c, int64_t ldc,
                                                           int64_t tiles_m, int64_t n_tiles_total) {
  constexpr int MIA = kExactAMIA, MIB = kExactAMIB, TA = 64 * MIA, TB = 64 * MIB;
  constexpr int ROWB = 2 * kExactAK, BYTES = (TA + 2 * TB) * ROWB;  // a row's and a K step's bytes
  constexpr int LOADS = BYTES / 1024 / 4;                           // 16-row loads per wavefront and K step
  constexpr int AHEAD = kExactABuf - 1;                             // K steps in flight ahead of the products
  static_assert(ROWB == 64 && BYTES % 4096 == 0, "whole loads per wavefront");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kExactABuf][BYTES];
  const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if (bid >= n_tiles_total) return;
  const int64_t i0 = (bid % tiles_m) * TA, j0 = (bid / tiles_m) * TB;
  const int tid = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = (wid >> 1) * 32 * MIA, wn = (wid & 1) * 32 * MIB;
  const int64_t steps = K / kExactAK;

  // Each of the wavefront's loads covers 16 rows of A or of one plane of B: a
  // buffer descriptor of those rows (rows past the operand's end read as zero),
  // and for this lane row lane / 4 and the chunk that belongs in slot lane % 4.
  __amdgpu_buffer_rsrc_t src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (wid * LOADS + i) * 16;  // first row in the stacked tile (A, B hi, B lo)
    const int b = row - TA;
    const int64_t first = row < TA ? i0 + row : j0 + b % TB, rows = row < TA ? ma : nb;
    const uint16_t* base = row < TA ? a : b < TB ? bh : bl;
    const int64_t left = min<int64_t>(max<int64_t>(rows - first, 0), 16);
    const uint64_t addr = (uint64_t)(base + (left > 0 ? first : 0) * ldk);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)addr);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(addr >> 32));
    src[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0,
                                               __builtin_amdgcn_readfirstlane((int)(2 * left * ldk)), 0x00020000);
  }
  // (row / 4) % 4 of the stacked row is that of the row among the 16
  const int voff = (lane >> 2) * 2 * (int)ldk + (((lane & 3) ^ ((lane >> 4) & 3)) * 16);
  auto issue = [&](int buf, int64_t t, int i) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        src[i], (__attribute__((address_space(3))) void*)&smem[buf][(wid * LOADS + i) * 1024], 16, voff,
        (int)(t * ROWB), 0, 0);
  };
  floatx16 acc[MIA][MIB], tot[MIA][MIB];
#pragma unroll
  for (int x = 0; x < MIA; ++x)
#pragma unroll
    for (int y = 0; y < MIB; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[x][y][e] = tot[x][y][e] = 0.0f;

  // fragment f (A blocks, B lo, B hi) of sub-step ks of the step in `buf`
  const int fr = lane & 31, sw = (fr >> 2) & 3;
  const int foff[2] = {fr * ROWB + ((lane >> 5) ^ sw) * 16, fr * ROWB + ((2 + (lane >> 5)) ^ sw) * 16};
  auto frag = [&](int buf, int ks, int f) __attribute__((always_inline)) {
    const int y = f - MIA;
    const int row = f < MIA ? wm + f * 32 : TA + (y < MIB ? TB + y * 32 : (y - MIB) * 32) + wn;
    return *(const bf16x8*)(smem[buf] + row * ROWB + foff[ks]);
  };
  // Two phases of 12 products per K step: a phase multiplies one sub-step's
  // fragments while it reads the other's (the next step's first ones in phase 1)
  // and issues its share of the loads of the step AHEAD.  (The last steps are
  // requested again past the end: the count of loads in flight is the same at
  // every step.)
  constexpr int NF = MIA + 2 * MIB, NP = 2 * MIA * MIB, SPLIT = NP - NF;
  static_assert(SPLIT >= 0 && LOADS >= SPLIT && LOADS - SPLIT <= NP, "requests fit behind the products");
  bf16x8 fg[2][NF];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
#pragma unroll
    for (int k = 0; k < LOADS; ++k) issue(i, min<int64_t>(i, steps - 1), k);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((AHEAD - 1) * LOADS) : "memory");
#pragma unroll
  for (int f = 0; f < NF; ++f) fg[0][f] = frag(0, 0, f);
  int buf = 0;
  for (int64_t t = 0; t < steps; ++t) {
    if (t != 0 && t % (64 / kExactAK * kExactAChunk) == 0) {
#pragma unroll
      for (int x = 0; x < MIA; ++x)
#pragma unroll
        for (int y = 0; y < MIB; ++y)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            tot[x][y][e] += acc[x][y][e];
            acc[x][y][e] = 0.0f;
          }
    }
    const int next = (buf + 1) % kExactABuf, into = (buf + AHEAD) % kExactABuf;
    const int64_t tl = min<int64_t>(t + AHEAD, steps - 1);
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
      if (ph == 1)
        // this wavefront's loads of step t + 1 have landed and its reads of step t
        // are done; after the barrier that holds for all four
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((AHEAD - 2) * LOADS + SPLIT) : "memory");
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        // small products first
        const int x = q / MIB % MIA, y = q % MIB, pl = q / (MIA * MIB);
        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg[ph][x], fg[ph][MIA + pl * MIB + y], acc[x][y], 0, 0, 0);
        if (q < NF) fg[ph ^ 1][q] = ph == 0 ? frag(buf, 1, q) : frag(next, 0, q);
        if (ph == 0 && q >= NF) issue(into, tl, q - NF);
        if (ph == 1 && q >= NP - (LOADS - SPLIT)) issue(into, tl, SPLIT + q - (NP - (LOADS - SPLIT)));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    buf = next;
  }
  // no load may be in flight into LDS when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // element e of lane l in a 32x32 block is (row (e/4)*8 + (l/32)*4 + e%4, col l%32)
#pragma unroll
  for (int x = 0; x < MIA; ++x)
#pragma unroll
    for (int y = 0; y < MIB; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t gi = i0 + wm + x * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
        const int64_t gj = j0 + wn + y * 32 + (lane & 31);
        if (gi < ma && gj < nb) c[gi * ldc + gj] = tot[x][y][e] + acc[x][y][e];
      }
}

// 64 x 64 tiles (a 32 x 32 block per wavefront, four workgroups per CU) for
// products whose large tiles would leave CUs idle.  K step, slab prefetch and
// fragment layout are the Gram kernel's.
__global__ void __launch_bounds__(256, 4) gemm_exact_a_small_kernel(const uint16_t* __restrict__ a, int64_t ma,
                                                                 const uint16_t* __restrict__ bh,
                                                                 const uint16_t* __restrict__ bl, int64_t nb,
                                                                 int64_t K, int64_t ldk, float* __restrict__ c,
                                                                 int64_t ldc, int64_t tiles_m,
                                                                 int64_t n_tiles_total) {
  constexpr int MIA = 1, MIB = 1, TA = 64 * MIA, TB = 64 * MIB;
  constexpr int NITA = TA * GB_CPR / 256, NITB = TB * GB_CPR / 256;
  constexpr int NIT = NITA > NITB ? NITA : NITB;
  __shared__ __attribute__((aligned(16))) uint16_t sA[TA * GB_LD];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][TB * GB_LD];
  const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if (bid >= n_tiles_total) return;
  const int64_t i0 = (bid % tiles_m) * TA, j0 = (bid / tiles_m) * TB;
  const int tid = threadIdx.x, wid = tid / 64, lane = lane_id();
  const int wm = (wid >> 1) * 32 * MIA, wn = (wid & 1) * 32 * MIB;

  floatx16 acc[MIA][MIB];
  float tot[MIA][MIB][16];
#pragma unroll
  for (int x = 0; x < MIA; ++x)
#pragma unroll
    for (int y = 0; y < MIB; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[x][y][e] = 0.0f;
        tot[x][y][e] = 0.0f;
      }

  // chunks it0 <= it < it1 of the slab at k0: A, B hi, B lo
  uint4 pa[NITA], pb[NITB][2];
  auto fetch_part = [&](int64_t k0, int it0, int it1) {
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      if (it < it0 || it >= it1) continue;
      const int chunk = tid + it * 256;
      const int r = chunk / GB_CPR, kc = (chunk % GB_CPR) * 8;
      const int64_t kk = k0 + kc;
      const uint4 z = {0, 0, 0, 0};
      if (it < NITA) {
        pa[it] = z;
        if (i0 + r < ma && kk < K) pa[it] = *(const uint4*)(a + (i0 + r) * ldk + kk);
      }
      if (it < NITB) {
        pb[it][0] = z;
        pb[it][1] = z;
        if (j0 + r < nb && kk < K) {
          pb[it][0] = *(const uint4*)(bh + (j0 + r) * ldk + kk);
          pb[it][1] = *(const uint4*)(bl + (j0 + r) * ldk + kk);
        }
      }
    }
  };
  fetch_part(0, 0, NIT);
  for (int64_t k0 = 0; k0 < K; k0 += GB_K) {
    if (k0 != 0 && k0 % (GB_K * kExactAChunk) == 0) {
#pragma unroll
      for (int x = 0; x < MIA; ++x)
#pragma unroll
        for (int y = 0; y < MIB; ++y)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            tot[x][y][e] += acc[x][y][e];
            acc[x][y][e] = 0.0f;
          }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int chunk = tid + it * 256;
      const int r = chunk / GB_CPR, kc = (chunk % GB_CPR) * 8;
      if (it < NITA) *(uint4*)(&sA[r * GB_LD + kc]) = pa[it];
      if (it < NITB) {
        *(uint4*)(&sB[0][r * GB_LD + kc]) = pb[it][0];
        *(uint4*)(&sB[1][r * GB_LD + kc]) = pb[it][1];
      }
    }
    __syncthreads();
    const bool more = k0 + GB_K < K;
#pragma unroll
    for (int ks = 0; ks < GB_K; ks += 16) {
      // the next slab's loads spread over the first K sub-steps
      if (more) {
        constexpr int per = (NIT + GB_K / 16 - 2) / (GB_K / 16 - 1);
        const int q = ks / 16;
        if (q < GB_K / 16 - 1) fetch_part(k0 + GB_K, q * per, (q + 1) * per < NIT ? (q + 1) * per : NIT);
      }
      __builtin_amdgcn_sched_barrier(0);
      const int kq = ks + (lane >> 5) * 8;
      bf16x8 af[MIA], bhf[MIB], blf[MIB];
#pragma unroll
      for (int x = 0; x < MIA; ++x) af[x] = *(const bf16x8*)(&sA[(wm + x * 32 + (lane & 31)) * GB_LD + kq]);
#pragma unroll
      for (int y = 0; y < MIB; ++y) {
        const int row = wn + y * 32 + (lane & 31);
        bhf[y] = *(const bf16x8*)(&sB[0][row * GB_LD + kq]);
        blf[y] = *(const bf16x8*)(&sB[1][row * GB_LD + kq]);
      }
      // small products first
#pragma unroll
      for (int x = 0; x < MIA; ++x)
#pragma unroll
        for (int y = 0; y < MIB; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[x], blf[y], acc[x][y], 0, 0, 0);
#pragma unroll
      for (int x = 0; x < MIA; ++x)
#pragma unroll
        for (int y = 0; y < MIB; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[x], bhf[y], acc[x][y], 0, 0, 0);
    }
  }
  // element e of lane l in a 32x32 tile is (row (e/4)*8 + (l/32)*4 + e%4, col l%32)
#pragma unroll
  for (int x = 0; x < MIA; ++x)
#pragma unroll
    for (int y = 0; y < MIB; ++y)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t gi = i0 + wm + x * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
        const int64_t gj = j0 + wn + y * 32 + (lane & 31);
        if (gi < ma && gj < nb) c[gi * ldc + gj] = tot[x][y][e] + acc[x][y][e];
      }
}

// ---------------------------------------------------------------------------
// FP64 NT GEMM: C = beta C + alpha A B^T (+ shift on the diagonal),
// 64x64 tile per workgroup, 4 waves of 32x32, K step 16, for K that is no multiple
// of the K step (the kernel below takes the others).  lower_only skips tiles above
// the diagonal and elements with j > i.
// ---------------------------------------------------------------------------
constexpr int GD_T = 64;
constexpr int GD_K = 16;
constexpr int GD_LD = 17;  // padded LDS stride (doubles)

__global__ void __launch_bounds__(256) gemm_nt_f64_kernel(const double* a, int64_t lda, const double* b,
                                                          int64_t ldb, double* c, int64_t ldc, int64_t m,
                                                          int64_t n, int64_t K, double alpha, double beta,
                                                          double shift, int lower_only, int64_t tiles_n,
                                                          int64_t n_tiles_total, const int32_t* info) {
  if (info && *info != 0) return;
  __shared__ double sA[GD_T * GD_LD];
  __shared__ double sB[GD_T * GD_LD];
  const int64_t bid = xcd_remap(blockIdx.x, gridDim.x);
  if (bid >= n_tiles_total) return;
  int ti, tj;
  if (lower_only) {
    tri_tile(bid, ti, tj);
  } else {
    ti = (int)(bid / tiles_n);
    tj = (int)(bid % tiles_n);
  }
  const int64_t i0 = (int64_t)ti * GD_T, j0 = (int64_t)tj * GD_T;
  const int tid = threadIdx.x, wid = tid / 64, lane = lane_id();
  const int wm = (wid >> 1) * 32, wn = (wid & 1) * 32;
  doublex4 acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = (doublex4){0.0, 0.0, 0.0, 0.0};

  for (int64_t k0 = 0; k0 < K; k0 += GD_K) {
    __syncthreads();
    // 64 rows x 16 k per operand = 1024 doubles; 256 threads x 4
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int idx = tid + it * 256;
      const int r = idx >> 4, kc = idx & 15;
      const int64_t kk = k0 + kc;
      sA[r * GD_LD + kc] = (i0 + r < m && kk < K) ? a[(i0 + r) * lda + kk] : 0.0;
      sB[r * GD_LD + kc] = (j0 + r < n && kk < K) ? b[(j0 + r) * ldb + kk] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < GD_K; ks += 4) {
      const int kq = ks + (lane >> 4);
      double av[2], bv[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) av[x] = sA[(wm + x * 16 + (lane & 15)) * GD_LD + kq];
#pragma unroll
      for (int y = 0; y < 2; ++y) bv[y] = sB[(wn + y * 16 + (lane & 15)) * GD_LD + kq];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[x], bv[y], acc[x][y], 0, 0, 0);
    }
  }
  __syncthreads();
  // element e of lane l in a 16x16 tile is (row l/16 + 4e, col l%16); C is
  // read before any of it is written, so the loads' latencies overlap
  double cv[2][2][4];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t gi = i0 + wm + x * 16 + (lane >> 4) + 4 * e;
        const int64_t gj = j0 + wn + y * 16 + (lane & 15);
        cv[x][y][e] = (beta != 0.0 && gi < m && gj < n && (!lower_only || gj <= gi)) ? c[gi * ldc + gj] : 0.0;
      }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t gi = i0 + wm + x * 16 + (lane >> 4) + 4 * e;
        const int64_t gj = j0 + wn + y * 16 + (lane & 15);
        if (gi < m && gj < n && (!lower_only || gj <= gi)) {
          double v = alpha * acc[x][y][e];
          if (beta != 0.0) v += beta * cv[x][y][e];
          if (gi == gj) v += shift;
          c[gi * ldc + gj] = v;
        }
      }
}

// ---------------------------------------------------------------------------
// FP64 NT GEMM for K a multiple of 16: C = beta C + alpha A B^T (+ shift on the
// diagonal) on a T x T tile per workgroup, T = 128 (4 waves of 64x64, 4x4
// v_mfma_f64_16x16x4 blocks, two workgroups per CU) or 64, K step 16, LDS tiles in
// two buffers.  The tile after the next is loaded into registers and the
// next one stored to the other buffer while the current one is multiplied; the
// tiles are k-major so a fragment read is 16 consecutive rows.  lower_only
// skips tiles above the diagonal and elements with j > i.  A, B and C must
// not overlap.  Bound by the matrix cores: 73.9 TFLOP/s at 16384^2 x 4096 and 69.4
// at 8192^2 x 768 (68.7 and 58.9 with one buffer, two barriers per K step and the
// requests in front of the products; the peak is 78.6).
// ---------------------------------------------------------------------------
constexpr int G2_T = 128;
constexpr int G2_K = 16;
// LDS tile of T rows, k-major: row k starts at (T + 16) k (+ 16 from k = 8 on)
// doubles, so that the two k rows that half a wavefront reads fall into different
// banks, and so do the two (k, k + 8) that it writes.
template <int T>
__device__ constexpr int g2_row(int k) { return k * (T + 16) + (k >= 8 ? 16 : 0); }
constexpr int g2_tile(int T) { return G2_K * (T + 16) + 16; }

template <int T, bool VEC, bool SPLIT>
__device__ __forceinline__ void gemm_big_tile(const double* __restrict__ a, int64_t lda, const double* __restrict__ b,
                                     int64_t ldb, double* __restrict__ c, int64_t ldc, int64_t m, int64_t n,
                                     int64_t K, double alpha, double beta, double shift, int lower_only, int64_t tiles_n,
                                     int64_t bid, double* sA, double* sB, double* __restrict__ wout) {
  int ti, tj;
  if (lower_only) {
    tri_supertile(bid, tiles_n, ti, tj);
  } else {
    ti = (int)(bid / tiles_n);
    tj = (int)(bid % tiles_n);
  }
  constexpr int NB = T / 32;            // 16x16 blocks per wavefront and direction
  constexpr int PER = 2 * NB;           // values per thread, operand and K tile
  const int64_t i0 = (int64_t)ti * T, j0 = (int64_t)tj * T;
  const int tid = threadIdx.x, wid = tid / 64, lane = lane_id();
  const int wm = (wid >> 1) * (T / 2), wn = (wid & 1) * (T / 2);
  // global -> register mapping: 16 / PER threads per row, PER values of k each.
  // Rows past the edge re-read the last row (K is a multiple of 16, so every load
  // is in bounds); their products are never stored.
  const int lr = tid / (16 / PER), lk = (tid % (16 / PER)) * PER;
  const double* pa = a + min<int64_t>(i0 + lr, m - 1) * lda + lk;
  const double* pb = b + min<int64_t>(j0 + lr, n - 1) * ldb + lk;
  double ra[PER], rb[PER];
  // request q (< 2 PER) of a tile: 16 bytes (VEC; q < PER) or 8
  auto load_one = [&](int64_t k0, int q) __attribute__((always_inline)) {
    if (VEC) {
      if (q >= PER) return;
      const int h = q % (PER / 2);
      const double2 v = *reinterpret_cast<const double2*>((q < PER / 2 ? pa : pb) + k0 + 2 * h);
      if (q < PER / 2) {
        ra[2 * h] = v.x;
        ra[2 * h + 1] = v.y;
      } else {
        rb[2 * h] = v.x;
        rb[2 * h + 1] = v.y;
      }
    } else if (q < PER) {
      ra[q % PER] = pa[k0 + q % PER];
    } else {
      rb[q % PER] = pb[k0 + q % PER];
    }
  };
  auto load = [&](int64_t k0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2 * PER; ++q) load_one(k0, q);
  };
  doublex4 acc[NB][NB];
#pragma unroll
  for (int x = 0; x < NB; ++x)
#pragma unroll
    for (int y = 0; y < NB; ++y) acc[x][y] = (doublex4){0.0, 0.0, 0.0, 0.0};
  constexpr int TILE = g2_tile(T);
  double* wa = sA + g2_row<T>(lk) + lr;
  double* wb = sB + g2_row<T>(lk) + lr;
  auto store = [&](int q, int buf) __attribute__((always_inline)) {  // q < PER: A, else B (lk + PER <= 8 or >= 8)
    if (q < PER) wa[buf * TILE + (q % PER) * (T + 16)] = ra[q % PER];
    else wb[buf * TILE + (q % PER) * (T + 16)] = rb[q % PER];
  };
  load(0);
#pragma unroll
  for (int q = 0; q < 2 * PER; ++q) store(q, 0);
  load(min<int64_t>(G2_K, K - G2_K));
  const double* fa = sA + (lane >> 4) * (T + 16) + wm + (lane & 15);
  const double* fb = sB + (lane >> 4) * (T + 16) + wn + (lane & 15);
  double fr[2][2 * NB];  // the fragments of a product group and the next
  auto frag = [&](int ks, int q, int buf) __attribute__((always_inline)) {
    fr[ks & 1][q] = q < NB ? fa[buf * TILE + g2_row<T>(4 * ks) + 16 * q] : fb[buf * TILE + g2_row<T>(4 * ks) + 16 * (q - NB)];
  };
  int buf = 0;
  for (int64_t k0 = 0; k0 < K; k0 += G2_K) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2 * NB; ++q) frag(0, q, buf);
    // one memory request (T = 64: two) behind each product: the next group's
    // fragments, then the next tile's stores to the other buffer and the loads of the
    // one after it (past the last tile it is loaded and stored again, and not read)
    const int64_t kn = min<int64_t>(k0 + 2 * G2_K, K - G2_K);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int t = 0; t < NB * NB; ++t) {
        const int x = t / NB, y = t % NB;
        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[ks & 1][x], fr[ks & 1][NB + y], acc[x][y], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4 / NB; ++u) {
          const int q = t * (4 / NB) + u;  // < 4 NB
          if (q < 2 * NB) {
            if (ks < 3) frag(ks + 1, q, buf);
          } else if (ks < 2) {
            store(2 * NB * ks + q - 2 * NB, buf ^ 1);
          } else {
            load_one(kn, 2 * NB * (ks - 2) + q - 2 * NB);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    buf ^= 1;
  }
  // element e of lane l in a 16x16 block is (row l/16 + 4e, col l%16)
  if constexpr (SPLIT) {
    // partial product of a K slice: the raw tile, row-major
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int y = 0; y < NB; ++y)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          wout[(wm + x * 16 + (lane >> 4) + 4 * e) * T + wn + y * 16 + (lane & 15)] = acc[x][y][e];
    return;
  }
  // C is read in batches of one 16-row block (16 values per lane) before
  // any of the batch is written, and the batch's results are all formed
  // before its stores: the compiler cannot prove the addresses distinct for a
  // runtime ldc, so element-wise read-modify-write waited for each store.
  // Interior tiles (inside C and, for lower_only, below the diagonal) take
  // unpredicated loads and stores, which keep each store's data in its own
  // registers; edge tiles check every element.
  const bool interior = i0 + T <= m && j0 + T <= n && (!lower_only || j0 + T <= i0);
#pragma unroll
  for (int xb = 0; xb < NB; ++xb) {
    double cv[1][NB][4];
#pragma unroll
    for (int x = 0; x < 1; ++x)
#pragma unroll
      for (int y = 0; y < NB; ++y)
#pragma unroll
        for (int e = 0; e < 4; ++e) cv[x][y][e] = 0.0;
    if (beta != 0.0) {
#pragma unroll
      for (int x = 0; x < 1; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int64_t gi = i0 + wm + (xb + x) * 16 + (lane >> 4) + 4 * e;
            const int64_t gj = j0 + wn + y * 16 + (lane & 15);
            if (interior || (gi < m && gj < n && (!lower_only || gj <= gi))) cv[x][y][e] = c[gi * ldc + gj];
          }
    }
#pragma unroll
    for (int x = 0; x < 1; ++x)
#pragma unroll
      for (int y = 0; y < NB; ++y)
#pragma unroll
        for (int e = 0; e < 4; ++e) cv[x][y][e] = alpha * acc[xb + x][y][e] + beta * cv[x][y][e];
    if (interior) {
#pragma unroll
      for (int x = 0; x < 1; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            c[(i0 + wm + (xb + x) * 16 + (lane >> 4) + 4 * e) * ldc + j0 + wn + y * 16 + (lane & 15)] = cv[x][y][e];
    } else {
#pragma unroll
      for (int x = 0; x < 1; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int64_t gi = i0 + wm + (xb + x) * 16 + (lane >> 4) + 4 * e;
            const int64_t gj = j0 + wn + y * 16 + (lane & 15);
            if (gi < m && gj < n && (!lower_only || gj <= gi))
              c[gi * ldc + gj] = gi == gj ? cv[x][y][e] + shift : cv[x][y][e];
          }
    }
  }
}


// One tile per workgroup (a grid smaller than the tile count makes each
// workgroup walk tiles bid, bid + G, ..., consecutive in the super-block order).
// SPLIT = false: one tile per unit u < n_units (tile ids from 0), whole K,
// C updated.  SPLIT = true: unit u is slice u % S (kc columns of K) of tile
// n_main + u / S, whose raw product goes to work + u * 128 * 128 for
// gemm_big_reduce_kernel.
template <int T, bool VEC, bool SPLIT>
__global__ void __launch_bounds__(256, T == 128 ? 2 : 3) gemm_nt_f64_big_kernel(const double* __restrict__ a, int64_t lda,
                                                              const double* __restrict__ b, int64_t ldb,
                                                              double* __restrict__ c, int64_t ldc, int64_t m,
                                                              int64_t n, int64_t K, double alpha, double beta,
                                                              double shift, int lower_only, int64_t tiles_n,
                                                              int64_t n_units, int64_t n_main, int S,
                                                              int64_t kc, double* __restrict__ work,
                                                              const int32_t* info) {
  if (info && *info != 0) return;
  extern __shared__ __align__(16) unsigned char smem[];
  double* sA = (double*)smem;  // two tiles of each operand
  double* sB = sA + 2 * g2_tile(T);
  const int64_t G = gridDim.x;
  for (int64_t u = xcd_remap(blockIdx.x, G); u < n_units; u += G) {
    if (!SPLIT) {
      gemm_big_tile<T, VEC, false>(a, lda, b, ldb, c, ldc, m, n, K, alpha, beta, shift, lower_only, tiles_n, u, sA, sB,
                                nullptr);
    } else {
      const int64_t tile = n_main + u / S;
      const int64_t kb = (u % S) * kc, kl = min<int64_t>(kc, K - kb);
      gemm_big_tile<T, VEC, true>(a + kb, lda, b + kb, ldb, c, ldc, m, n, kl, alpha, beta, 0.0, lower_only, tiles_n, tile,
                               sA, sB, work + u * (int64_t)(G2_T * G2_T));
    }
    __syncthreads();
  }
}

// C = beta C + alpha sum_part W[part] for the split tail tiles, parts summed
// in a fixed order.  One workgroup per (tail tile, 32-row band).
__global__ void __launch_bounds__(256) gemm_big_reduce_kernel(const double* __restrict__ work, double* __restrict__ c,
                                                              int64_t ldc, int64_t m, int64_t n, double alpha,
                                                              double beta, int lower_only, int64_t tiles_n,
                                                              int64_t n_main, int S, const int32_t* info) {
  if (info && *info != 0) return;
  const int64_t r = blockIdx.x / 4;  // tail tile index
  const int band = blockIdx.x % 4;
  const int64_t tile = n_main + r;
  int ti, tj;
  if (lower_only) {
    tri_supertile(tile, tiles_n, ti, tj);
  } else {
    ti = (int)(tile / tiles_n);
    tj = (int)(tile % tiles_n);
  }
  const double* w = work + r * S * (int64_t)(G2_T * G2_T);
  // 16 elements per thread, the loads of a slice (and of C) all in flight;
  // each element sums its slices in slice order
  constexpr int PER = 32 * G2_T / 256;
  double acc[PER], cv[PER];
  bool keep[PER];
  int64_t off[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int idx = threadIdx.x + e * 256;
    const int li = band * 32 + idx / G2_T, lj = idx % G2_T;
    const int64_t gi = (int64_t)ti * G2_T + li, gj = (int64_t)tj * G2_T + lj;
    keep[e] = gi < m && gj < n && (!lower_only || gj <= gi);
    off[e] = keep[e] ? gi * ldc + gj : 0;
    acc[e] = 0.0;
    cv[e] = (beta != 0.0 && keep[e]) ? c[off[e]] : 0.0;
  }
  for (int p = 0; p < S; ++p) {
    const double* wp = w + (int64_t)p * G2_T * G2_T + band * 32 * G2_T;
#pragma unroll
    for (int e = 0; e < PER; ++e) acc[e] += wp[threadIdx.x + e * 256];
  }
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    if (keep[e]) {
      double v = alpha * acc[e];
      if (beta != 0.0) v += beta * cv[e];
      c[off[e]] = v;
    }
  }
}

// Zero n 32-bit words (a fill kernel rather than a memset node, so that a
// captured graph replays it correctly).
__global__ void zero_u32_kernel(uint32_t* __restrict__ p, int64_t n) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    p[k] = 0u;
}

// ---------------------------------------------------------------------------
// Triangular solves with the blocked factor, one launch each.  Workgroup k
// owns the 64-row block k; it waits (bounded spin in global memory) for every
// block it depends on, and only ever on blocks with a smaller workgroup id,
// which the hardware dispatched earlier, so the wait always ends.
//
// The solved entries are their own flags: the output vector holds kUnsolved
// before the launch, each entry is written once, as a 64-bit atomic store, and a
// reader polls the entries it needs with 64-bit atomic loads until none holds
// kUnsolved.  One memory round trip per dependency, and no ordering between
// different entries is needed.
//
// A wait that exceeds its bound takes the entry for NaN, which then reaches every
// entry that depends on it: after a forward solve that ran out, the whole solution.
// In the backward solve the entries above it are not reached, so a wait that runs out
// there sets *err (zeroed by the forward launch) before its rows are published, and
// two parties turn the rest into NaN: the workgroup of the last block to be solved,
// which depends on all others and so has waited for them or run out itself, fills the
// vector if it sees *err; and a wavefront that publishes later than that sees *err
// after its rows are out and takes them back.
// ---------------------------------------------------------------------------
constexpr int64_t kSpinLimit = 1LL << 26;

// The entry *p (lanes with active), polled with relaxed agent-scope loads
// (they read the L2 copy); inactive lanes get 0.  Wave-uniform loop; `late` is set when
// `limit` polls were not enough.
__device__ inline double poll_entry(const double* p, bool active, int64_t limit, bool& late) {
  uint64_t u = 0;
  int64_t spins = 0;
  while (true) {
    if (active) u = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!__any(active && u == kUnsolved)) break;
    __builtin_amdgcn_s_sleep(1);
    if (++spins > limit) {
      late = true;
      break;
    }
  }
  if (u == kUnsolved) u = kDefaultNaN;
  return active ? __longlong_as_double((long long)u) : 0.0;
}

__device__ inline void publish_entry(double* p, double v) {
  uint64_t u = (uint64_t)__double_as_longlong(v);
  if (u == kUnsolved) u = kDefaultNaN;
  __hip_atomic_store((uint64_t*)p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a b += y_c L[c], c = 0..15, y_c that of lane c of the lane's row of 16 (two sums).
__device__ __forceinline__ void row_dot16(double& a, double& b, double y, const double (&L)[16]) {
#define NKA_ROW_FMAC(acc, n, c) "v_fmac_f64_dpp %" #acc ", %2, %" #n " row_newbcast:" #c " row_mask:0xf bank_mask:0xf\n\t"
  // (two wait states between the write of y and its DPP reads)
  asm("s_nop 1\n\t"
      NKA_ROW_FMAC(0, 3, 0) NKA_ROW_FMAC(1, 4, 1) NKA_ROW_FMAC(0, 5, 2) NKA_ROW_FMAC(1, 6, 3)
      NKA_ROW_FMAC(0, 7, 4) NKA_ROW_FMAC(1, 8, 5) NKA_ROW_FMAC(0, 9, 6) NKA_ROW_FMAC(1, 10, 7)
      NKA_ROW_FMAC(0, 11, 8) NKA_ROW_FMAC(1, 12, 9) NKA_ROW_FMAC(0, 13, 10) NKA_ROW_FMAC(1, 14, 11)
      NKA_ROW_FMAC(0, 15, 12) NKA_ROW_FMAC(1, 16, 13) NKA_ROW_FMAC(0, 17, 14) NKA_ROW_FMAC(1, 18, 15)
      : "+v"(a), "+v"(b)
      : "v"(y), "v"(L[0]), "v"(L[1]), "v"(L[2]), "v"(L[3]), "v"(L[4]), "v"(L[5]), "v"(L[6]), "v"(L[7]), "v"(L[8]),
        "v"(L[9]), "v"(L[10]), "v"(L[11]), "v"(L[12]), "v"(L[13]), "v"(L[14]), "v"(L[15]));
#undef NKA_ROW_FMAC
}
// Sum over the four rows of lanes, in every one.
__device__ __forceinline__ double sum_rows(double v) {
  double w = v;
  swap_rows16(v, w);
  v += w;
  w = v;
  swap_halves(v, w);
  return v + w;
}

// Both solves.  Workgroup k (block kb) of four wavefronts, 16 rows of the block
// each; lane l has row l % 16 and a quarter of the columns, and the entries of the
// solution reach it from the lanes of its row of 16, so that neither LDS nor a
// barrier lies between an entry's arrival and the next block's.
//
//   x_k = inv_kk (b_k - sum_j L_kj x_j) = s_k - (inv_kk L_k,prev) x_prev
//
// The product W = inv_kk L_k,prev is formed ahead of time on the matrix cores, and
// s_k, which takes all blocks but the last to come, while that one is being solved:
// what is left in the chain per block is one memory round trip and 16 FMAs.
// Bound by that chain: 29 + 28 us at 27 blocks and 147 + 141 at 131 (1.1 us a
// block), against 40 + 46 and 203 + 237 with the block's sums and its inverse's
// product taken through LDS after the last entry's arrival.
//
// forward (BWD false): L y = b from block 0 up; b's entries become unsolved ones
// (the next launch fills them with x).  Backward: L^T x = y from the last block
// down; y's entries become unsolved again, for another solve with the factor.
template <bool BWD>
__global__ void __launch_bounds__(256, 2) trsv_lookback(const double* __restrict__ A, int64_t lda, int64_t n,
                                                        const double* __restrict__ inv, double* rhs, double* out,
                                                        const int32_t* __restrict__ info, int32_t* err,
                                                        int64_t limit) {
  __shared__ double ts[CH_NB];
  bool late = false;
  const int nblk = gridDim.x;
  const int kb = BWD ? nblk - 1 - (int)blockIdx.x : (int)blockIdx.x;
  const int64_t k0 = (int64_t)kb * CH_NB;
  const int nb = (int)min<int64_t>(CH_NB, n - k0);
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int r = 16 * w + i;             // row of the block
  const int rc = min(r, nb - 1);        // rows past nb re-read the last; their sums are never used
  if (*info != 0) {
    // a failed factorisation leaves NaN in the solution, as LAPACK-based cho_solve
    // does on a matrix that is not positive definite
    if (BWD && tid < nb) out[k0 + tid] = __longlong_as_double((long long)kDefaultNaN);
    return;
  }
  if (!BWD && kb == 0 && tid == 0) *err = 0;
  const double* invk = inv + (int64_t)kb * CH_NB * CH_NB;
  const int m = BWD ? nblk - 1 - kb : kb;      // blocks before this one
  // the t-th of them, in the order in which they are solved
  auto first = [&](int t) { return (int64_t)(BWD ? nblk - 1 - t : t) * CH_NB; };
  // a lane's columns (BWD: rows) of a tile: pairs, so that four lanes read 64 bytes
  auto col = [&](int c) { return 8 * (c >> 1) + 2 * g + (c & 1); };
  double iv[16], W[16], rk = 0.0;
  if constexpr (BWD) {
#pragma unroll
    for (int c = 0; c < 16; ++c) iv[c] = invk[col(c) * CH_NB + r];
  } else {
    load_k_pairs(invk + r * CH_NB, 0, lane, iv);
  }
  if (r < nb) rk = rhs[k0 + r];
  if (m > 0) {
    const int64_t j0 = first(m - 1);
    const int mb = (int)min<int64_t>(CH_NB, n - j0);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      double a[16];
      if constexpr (BWD) {
        load_k_pairs(A + (j0 + min(16 * cb + i, mb - 1)) * lda + k0, 0, lane, a);
      } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) a[q] = A[(k0 + min(col(q), nb - 1)) * lda + j0 + 16 * cb + i];
      }
      doublex4 acc = (doublex4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 16; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], iv[q], acc, 0, 0, 0);
      // element e is W[r][16 cb + 4 e + g]
#pragma unroll
      for (int e = 0; e < 4; ++e) W[4 * cb + e] = acc[e];
    }
  }
  auto load = [&](int t, double (&L)[16]) __attribute__((always_inline)) {
    const int64_t j0 = first(t);
    if constexpr (BWD) {
      // rows past the matrix re-read the last one and meet a zero entry of x
      const int mb = (int)min<int64_t>(CH_NB, n - j0);
#pragma unroll
      for (int c = 0; c < 16; ++c) L[c] = A[(j0 + min(col(c), mb - 1)) * lda + k0 + rc];
    } else {
      load_k_pairs(A + (k0 + rc) * lda + j0, 0, lane, L);
    }
  };
  // the tiles of four blocks in flight; the last block is left for W
  double L[4][16];
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (u + 1 < m) load(u, L[u]);
  const int cl = 8 * (i >> 1) + 2 * g + (i & 1);  // the entry that lane l holds for a tile
  double s0 = 0.0, s1 = 0.0;
  for (int t0 = 0; t0 + 1 < m; t0 += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (t0 + u + 1 >= m) break;
      const int64_t j = first(t0 + u) + cl;
      const double x = poll_entry(out + j, j < n, limit, late);
      row_dot16(s0, s1, x, L[u]);
      if (t0 + u + 5 < m) load(t0 + u + 4, L[u]);
    }
  }
  const double tr = r < nb ? rk - sum_rows(s0 + s1) : 0.0;
  if (g == 0) ts[r] = tr;
  __syncthreads();
  s0 = s1 = 0.0;
  row_dot16(s0, s1, ts[cl], iv);
  double v = sum_rows(s0 + s1);
  if (g == 0 && r < nb) ((uint64_t*)rhs)[k0 + r] = kUnsolved;
  if (m > 0) {
    const int64_t j = first(m - 1) + 4 * i + g;   // W's order of columns
    const double x = poll_entry(out + j, j < n, limit, late);
    s0 = s1 = 0.0;
    row_dot16(s0, s1, x, W);
    v -= sum_rows(s0 + s1);
  }
  if (BWD && late) {
    if (lane == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence();  // *err before the rows that it belongs to
  }
  if (g == 0 && r < nb) publish_entry(out + k0 + r, v);
  if constexpr (BWD) {
    if (kb == 0) __syncthreads();
    __threadfence();  // the rows (and, in the last block, the entries it waited for) before the look at *err
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
      if (kb == 0) {
        for (int64_t q = tid; q < n; q += 256) publish_entry(out + q, __longlong_as_double((long long)kDefaultNaN));
      } else if (g == 0 && r < nb) {
        publish_entry(out + k0 + r, __longlong_as_double((long long)kDefaultNaN));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Vector helpers
// ---------------------------------------------------------------------------
// y = alpha op(A) x + beta y.  trans 0: row dot products (one wave per row);
// trans 1: column sums (thread per column); trans 2: symmetric from lower.
__global__ void __launch_bounds__(256) gemv_n_kernel(const double* __restrict__ A, int64_t lda, int64_t m,
                                                     int64_t n, const double* __restrict__ x, double alpha,
                                                     double beta, double* __restrict__ y, int sym_lower) {
  const int wid = threadIdx.x / 64, lane = lane_id();
  for (int64_t r = (int64_t)blockIdx.x * 4 + wid; r < m; r += (int64_t)gridDim.x * 4) {
    double s = 0.0;
    if (!sym_lower) {
      for (int64_t c = lane; c < n; c += 64) s += A[r * lda + c] * x[c];
    } else {
      for (int64_t c = lane; c <= r; c += 64) s += A[r * lda + c] * x[c];
      for (int64_t c = r + 1 + lane; c < n; c += 64) s += A[c * lda + r] * x[c];
    }
    s = wave_sum(s);
    if (lane == 0) y[r] = alpha * s + (beta != 0.0 ? beta * y[r] : 0.0);
  }
}

__global__ void __launch_bounds__(256) gemv_t_partial(const double* __restrict__ A, int64_t lda, int64_t m,
                                                      int64_t n, const double* __restrict__ x,
                                                      double* __restrict__ part, int64_t rows_per) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * rows_per;
  const int64_t r1 = min(m, r0 + rows_per);
  if (c >= n) return;
  double s = 0.0;
  for (int64_t r = r0; r < r1; ++r) s += A[r * lda + c] * x[r];
  part[(int64_t)blockIdx.y * n + c] = s;
}

__global__ void gemv_t_reduce(const double* __restrict__ part, int nparts, int64_t n, double alpha,
                              double beta, double* __restrict__ y) {
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int p = 0; p < nparts; ++p) s += part[(int64_t)p * n + c];
    y[c] = alpha * s + (beta != 0.0 ? beta * y[c] : 0.0);
  }
}

__global__ void check_finite_kernel(const double* __restrict__ x, int64_t n, int32_t* __restrict__ flag) {
  int bad = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    bad |= !isfinite(x[i]);
  if (__any(bad) && lane_id() == 0) atomicOr(flag, 1);
}

template <class T>
__global__ void sgd_kernel(T* __restrict__ p, const double* __restrict__ dp, int64_t n, T lr) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const T g = (T)dp[i];
    const T u = -lr * g;
    p[i] = p[i] + u;
  }
}

__global__ void axpy_kernel(int64_t n, double alpha, const double* __restrict__ x, double* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] += alpha * x[i];
}

__global__ void centre_scale_kernel(const double* __restrict__ e, int64_t n, const double* __restrict__ mean,
                                    double scale, double* __restrict__ out) {
  const double mu = *mean;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (e[i] - mu) * scale;
}

// Moments of data (C, L) for the blocking statistics: one workgroup.
__device__ inline double block_sum(double v, double* red) {
  v = wave_sum(v);
  const int wid = threadIdx.x / 64;
  __syncthreads();
  if (lane_id() == 0) red[wid] = v;
  __syncthreads();
  double t = 0.0;
  const int nw = blockDim.x / 64;
  for (int w = 0; w < nw; ++w) t += red[w];
  return t;
}

// Mean of the group means and variance around it (two passes); group g of
// size gs starts at element start(g) of data (C, L).
struct GroupSpec {
  int kind;  // 0: chains (size L); 1: blocks of lb within each chain; 2: half chains
  int C, L, lb, nbc, h;
};
__device__ inline int64_t group_count(const GroupSpec& g) {
  return g.kind == 0 ? g.C : (g.kind == 1 ? (int64_t)g.C * g.nbc : 2 * (int64_t)g.C);
}
__device__ inline double group_mean(const double* d, const GroupSpec& g, int64_t q) {
  int64_t start;
  int sz;
  if (g.kind == 0) {
    start = q * g.L;
    sz = g.L;
  } else if (g.kind == 1) {
    start = (q / g.nbc) * g.L + (q % g.nbc) * g.lb;
    sz = g.lb;
  } else {
    start = (q / 2) * g.L + (q % 2) * g.h;
    sz = g.h;
  }
  double a = 0.0;
#pragma unroll 16
  for (int l = 0; l < sz; ++l) a += d[start + l];
  return sz > 0 ? a / (double)sz : 0.0;
}
__device__ inline double group_var(const double* d, const GroupSpec& g, double* red) {
  const int64_t cnt = group_count(g);
  double s = 0.0, first = 0.0;  // (a thread's first group, for the second pass)
  for (int64_t q = threadIdx.x; q < cnt; q += blockDim.x) {
    const double x = group_mean(d, g, q);
    if (q == threadIdx.x) first = x;
    s += x;
  }
  const double mu = block_sum(s, red) / (double)cnt;
  double v = 0.0;
  for (int64_t q = threadIdx.x; q < cnt; q += blockDim.x) {
    const double x = (q == threadIdx.x ? first : group_mean(d, g, q)) - mu;
    v += x * x;
  }
  return block_sum(v, red) / (double)cnt;
}

// One workgroup; bound by the latency of its passes over data that fits the caches,
// so a thread's loads are in flight together, and the mean of a thread's first group is
// kept for the second pass (all of them up to 1024 groups; 16 chains of 63 and of 1000:
// 22.8 -> 11.5 us, 242 -> 33 us).
__global__ void __launch_bounds__(1024) stats_kernel(const double* __restrict__ d, int C, int L,
                                                     double* __restrict__ out) {
  __shared__ double red[16];
  const int64_t n = (int64_t)C * L;
  double s = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) s += d[i];
  const double mean = block_sum(s, red) / (double)n;
  double v = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double x = d[i] - mean;
    v += x * x;
  }
  const double var = block_sum(v, red) / (double)n;
  // block size l_block = max(1, L / 32) and floor(L / l_block) blocks per chain;
  // split R-hat halves drop the last element when L is odd
  GroupSpec g;
  g.C = C;
  g.L = L;
  g.lb = max(1, L / 32);
  g.nbc = L / g.lb;
  g.h = L / 2;
  g.kind = 0;
  const double cvar = group_var(d, g, red);
  g.kind = 1;
  const double bvar = group_var(d, g, red);
  g.kind = 2;
  const double hvar = g.h > 0 ? group_var(d, g, red) : 0.0;
  if (threadIdx.x == 0) {
    out[0] = mean;
    out[1] = var;
    out[2] = cvar;
    out[3] = (double)((int64_t)C * g.nbc);
    out[4] = bvar;
    out[5] = hvar;
    out[6] = (double)g.lb;
    out[7] = (double)n;
  }
}

// Copy the lower triangle onto the upper one (row-major, FP64): one 64x64 tile
// of the lower triangle per workgroup, transposed through LDS, so that both
// the reads and the writes run along rows (an element-wise copy reads the lower
// triangle down its columns: 0.41 ms at n = 8384).
constexpr int SY_T = 64;
__global__ void __launch_bounds__(256) symmetrize_kernel(double* __restrict__ a, int64_t n, int64_t lda) {
  __shared__ double tile[SY_T][SY_T + 1];
  int ti, tj;
  tri_tile(blockIdx.x, ti, tj);
  const int64_t i0 = (int64_t)ti * SY_T, j0 = (int64_t)tj * SY_T;
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
#pragma unroll
  for (int r = r0; r < SY_T; r += 4)
    if (i0 + r < n && j0 + c < n) tile[r][c] = a[(i0 + r) * lda + j0 + c];
  __syncthreads();
#pragma unroll
  for (int r = r0; r < SY_T; r += 4)
    if (j0 + r < n && i0 + c < n && j0 + r < i0 + c) a[(j0 + r) * lda + i0 + c] = tile[c][r];
}

// RBM neural tangent kernel on the bf16x3 Gram tiles (called from the NTK
// entry point): Theta from the split tanh values xh + xl (n x K, ldx), S from
// the packed spins.  Returns false when the spins do not fit the epilogue.
bool launch_gram_rbm(const uint16_t* xh, const uint16_t* xl, int64_t n, int64_t K, int64_t ldx,
                     const uint32_t* bits, int nw, int N, const double* v, const double* c, double hb,
                     double ha, double scale, double shift, double offset, double* out, int64_t ldo,
                     hipStream_t s) {
  const int nwp = (nw + 3) / 4 * 4;
  if (nwp > kGramRbmMaxNwp) return false;
  const int64_t T = (n + 2 * kGramRbmWT - 1) / (2 * kGramRbmWT);
  const int64_t tiles = T * (T + 1) / 2;
  GramRbmEpi ep{bits, nw, nwp, N, v, c, hb, ha, scale};
  hipLaunchKernelGGL((gram_bf16x3_kernel<true, kGramRbmWT>), dim3(grid_mult8(tiles)), dim3(256), 0, s, xh, xl,
                     n, K, ldx, shift, offset, out, ldo, tiles, ep);
  return true;
}

// Workgroups of the 128-tile kernel resident at once (two per CU), from the
// device's CU count (queried once per process for the current device).
static int64_t big_gemm_slots() {
  static int64_t slots = 0;
  if (slots == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
      slots = 2 * (int64_t)cus;
    else
      slots = 512;
  }
  return slots;
}

// C = A (Bh + Bl)^T (FP32) for an exact single-plane A; K and ldk multiples
// of 64, operands 16-byte aligned (checked by the caller).
void launch_gemm_exact_a(const uint16_t* a, int64_t ma, const uint16_t* bh, const uint16_t* bl, int64_t nb,
                         int64_t K, int64_t ldk, float* c, int64_t ldc, hipStream_t s) {
  if (ma == 0 || nb == 0) return;
  constexpr int TA = 64 * kExactAMIA, TB = 64 * kExactAMIB;
  const int64_t tm = (ma + TA - 1) / TA, tn = (nb + TB - 1) / TB;
  // A round of 192x128 tiles over the chip takes 1.05 us per K slab of 64, 64x64 tiles
  // 0.2 + 0.35 per tile and CU (0.65 at least): the small ones where they are
  // fewer.  Same sums.  Whole dense S at 36 sites x 36 units, 6912 samples (121
  // tiles of 64x64): 136 us against 165; 36 x 72, 4096 (462): 140 against 152;
  // 48 x 96, 4096 (1387, two rounds): 300 against 300; 64 x 64, 4096 (1089): 228 against 190.
  const int64_t sm = (ma + 63) / 64, sn = (nb + 63) / 64, cus = big_gemm_slots() / 2;
  if (sm * sn + 146 < 768 * ((tm * tn + cus - 1) / cus) || ldk >= 1 << 26)
    hipLaunchKernelGGL(gemm_exact_a_small_kernel, dim3(grid_mult8(sm * sn)), dim3(256), 0, s, a, ma, bh, bl, nb, K,
                       ldk, c, ldc, sm, sm * sn);
  else
    hipLaunchKernelGGL(gemm_exact_a_kernel, dim3(grid_mult8(tm * tn)), dim3(256), 0, s, a,
                       ma, bh, bl, nb, K, ldk, c, ldc, tm, tm * tn);
}

// The two-layer network's tangent kernel on the bf16x3 Gram tiles (called from
// the network's NTK entry point): H, G and D from the split h1, g2 and d1
// (hi + lo planes, n rows each), X from the packed spins.  Returns false when
// the spins do not fit the epilogue.
bool launch_gram_ffnn(const uint16_t* h1h, const uint16_t* h1l, int64_t K0, int64_t ld0, const uint16_t* g2h,
                      const uint16_t* g2l, int64_t K1, int64_t ld1, const uint16_t* d1h, const uint16_t* d1l,
                      int64_t K2, int64_t ld2, int64_t n, const uint32_t* bits, int nw, int N, const double* v,
                      const double* c, double hb1, double hb2, double scale, double shift, double offset,
                      double* out, int64_t ldo, hipStream_t s) {
  const int nwp = (nw + 3) / 4 * 4;
  if (nwp > kGramRbmMaxNwp) return false;
  const int64_t T = (n + 2 * kGramRbmWT - 1) / (2 * kGramRbmWT);
  const int64_t tiles = T * (T + 1) / 2;
  GramRbmEpi ep{bits, nw, nwp, N, v, c, hb1, 0.0, scale, g2h, g2l, d1h, d1l, K1, K2, ld1, ld2, hb2};
  hipLaunchKernelGGL((gram_bf16x3_kernel<true, kGramRbmWT, 3>), dim3(grid_mult8(tiles)), dim3(256), 0, s, h1h,
                     h1l, n, K0, ld0, shift, offset, out, ldo, tiles, ep);
  return true;
}

}  // namespace nka

using namespace nka;

extern "C" {

int nka_gram_bf16x3(const uint16_t* x_hi, const uint16_t* x_lo, int64_t n, int64_t k, int64_t ldx,
                    double shift, double offset, double* out, int64_t ldo, void* stream) {
  NKA_CHECK_ARG(n >= 0 && k >= 0 && ldx >= k && ldo >= n, "nka_gram_bf16x3: bad sizes");
  NKA_CHECK_ARG(ldx % 8 == 0 && k % 8 == 0,
                "nka_gram_bf16x3: k and ldx must be multiples of 8 (pad with zeros)");
  NKA_CHECK_ARG(((uintptr_t)x_hi % 16) == 0 && ((uintptr_t)x_lo % 16) == 0,
                "nka_gram_bf16x3: operands must be 16-byte aligned");
  if (n == 0) return NKA_OK;
  const int64_t T = (n + 2 * kGramWT - 1) / (2 * kGramWT);
  const int64_t tiles = T * (T + 1) / 2;
  NKA_CHECK_ARG(tiles < (1LL << 31), "nka_gram_bf16x3: matrix too large");
  hipLaunchKernelGGL((gram_bf16x3_kernel<false, kGramWT>), dim3(grid_mult8(tiles)), dim3(256), 0,
                     (hipStream_t)stream, x_hi, x_lo, n, k, ldx, shift, offset, out, ldo, tiles, GramRbmEpi{});
  NKA_CHECK_LAUNCH("nka_gram_bf16x3");
  return NKA_OK;
}

static int gemm_launch(const double* a, int64_t lda, const double* b, int64_t ldb, double* c,
                       int64_t ldc, int64_t m, int64_t n, int64_t k, double alpha, double beta,
                       double shift, int lower, const int32_t* info, hipStream_t s) {
  const int64_t tm = (m + GD_T - 1) / GD_T, tn = (n + GD_T - 1) / GD_T;
  const int64_t tiles = lower ? tm * (tm + 1) / 2 : tm * tn;
  if (tiles == 0) return NKA_OK;
  hipLaunchKernelGGL(gemm_nt_f64_kernel, dim3(grid_mult8(tiles)), dim3(256), 0, s, a, lda, b, ldb, c,
                     ldc, m, n, k, alpha, beta, shift, lower, tn, tiles, info);
  return NKA_OK;
}


// Tail-split workspace of the 128-tile GEMM: at most kMaxSplitUnits raw tiles.
constexpr int64_t kMaxSplitUnits = 1024;

// The 128-tile kernel needs K to be a multiple of its K step; other shapes
// take the 64-tile kernel.  With a workspace, the tiles of the last, partial
// round of the grid are split along K so that the round is filled, and their
// slices are summed into C by a second launch.
static void gemm_big_launch(const double* a, int64_t lda, const double* b, int64_t ldb, double* c,
                            int64_t ldc, int64_t m, int64_t n, int64_t k, double alpha, double beta,
                            int lower, const int32_t* info, hipStream_t s, double* work = nullptr,
                            int64_t work_units = 0, double shift = 0.0) {
  if (m <= 0 || n <= 0) return;
  if (k % G2_K != 0 || k == 0) {
    gemm_launch(a, lda, b, ldb, c, ldc, m, n, k, alpha, beta, shift, lower, info, s);
    return;
  }
  int64_t tm = (m + G2_T - 1) / G2_T, tn = (n + G2_T - 1) / G2_T;
  int64_t tiles = lower ? tm * (tm + 1) / 2 : tm * tn;
  const int64_t slots = big_gemm_slots();
  const int64_t n_main = (tiles / slots) * slots;
  const int64_t tail = tiles - n_main;
  // slices per tail tile: fill the round, keep >= 4 K steps per slice
  int S = 1;
  if (work && tail > 0) {
    const int64_t max_s = std::max<int64_t>(1, k / (4 * G2_K));
    S = (int)std::min<int64_t>(std::min<int64_t>(slots / tail, max_s), work_units / tail);
    if (S < 2) S = 1;
  }
  const int64_t kc = S > 1 ? ((k + S - 1) / S + G2_K - 1) / G2_K * G2_K : k;
  if (S > 1) S = (int)((k + kc - 1) / kc);  // slices actually needed with kc columns each
  int64_t main_tiles = S > 1 ? n_main : tiles;
  // 64x64 tiles where their rounds over the chip are cheaper: a round of 128x128
  // tiles takes 1.88 us per K step, one of 64x64 tiles 0.56 (0.74 if it is the only
  // one).  X X^T of 1008 x 8384, 2560 x 8384, 4096 x 8384: 376, 1191, 2626 us with
  // 64x64 tiles, 980, 1042, 2981 with 128x128.  In place of slices and their sum
  // only for one round and K up to 1024 (solves at n = 5500 and 6500: 2.63 and 3.64
  // ms against 2.69 and 3.70): a longer single sum doubles the solve's error.
  const int64_t t64 = lower ? ((m + 63) / 64) * ((m + 63) / 64 + 1) / 2 : ((m + 63) / 64) * ((n + 63) / 64);
  const int64_t r64 = (t64 + slots / 2 - 1) / (slots / 2), r128 = (tiles + slots / 2 - 1) / (slots / 2);
  const bool small = 3 * r64 < 10 * r128 && (S == 1 || (r64 == 1 && k <= 1024));
  if (small) {
    tm = (m + 63) / 64;
    tn = (n + 63) / 64;
    main_tiles = t64;
    S = 1;
  }
  const bool vec = ((uintptr_t)a % 16 == 0) && ((uintptr_t)b % 16 == 0) && lda % 2 == 0 && ldb % 2 == 0;
  const int lds = 4 * g2_tile(small ? 64 : 128) * (int)sizeof(double);
  auto launch = [&](auto kernel, int64_t units, int64_t first, int slices, int64_t width) {
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(kernel, dim3(grid_mult8(units)), dim3(256), lds, s, a, lda, b, ldb, c, ldc, m, n, k, alpha, beta,
                       shift, lower, tn, units, first, slices, width, work, info);
  };
  if (main_tiles > 0) {
    if (small && vec) launch(gemm_nt_f64_big_kernel<64, true, false>, main_tiles, 0, 1, k);
    else if (small) launch(gemm_nt_f64_big_kernel<64, false, false>, main_tiles, 0, 1, k);
    else if (vec) launch(gemm_nt_f64_big_kernel<128, true, false>, main_tiles, 0, 1, k);
    else launch(gemm_nt_f64_big_kernel<128, false, false>, main_tiles, 0, 1, k);
  }
  if (S > 1) {
    if (vec) launch(gemm_nt_f64_big_kernel<128, true, true>, tail * S, main_tiles, S, kc);
    else launch(gemm_nt_f64_big_kernel<128, false, true>, tail * S, main_tiles, S, kc);
  }
  if (S > 1)
    hipLaunchKernelGGL(gemm_big_reduce_kernel, dim3((unsigned)(tail * 4)), dim3(256), 0, s, work, c, ldc, m, n,
                       alpha, beta, lower, tn, main_tiles, S, info);
}

int nka_syrk_f64(const double* x, int64_t n, int64_t k, int64_t ldx, double alpha, double beta,
                 double shift, double* c, int64_t ldc, void* stream) {
  NKA_CHECK_ARG(n >= 0 && k >= 0 && ldx >= k && ldc >= n, "nka_syrk_f64: bad sizes");
  gemm_big_launch(x, ldx, x, ldx, c, ldc, n, n, k, alpha, beta, 1, nullptr, (hipStream_t)stream, nullptr, 0, shift);
  NKA_CHECK_LAUNCH("nka_syrk_f64");
  return NKA_OK;
}

int nka_gemm_nt_f64(const double* a, int64_t lda, const double* b, int64_t ldb, double* c,
                    int64_t ldc, int64_t m, int64_t n, int64_t k, double alpha, double beta,
                    void* stream) {
  NKA_CHECK_ARG(m >= 0 && n >= 0 && k >= 0 && lda >= k && ldb >= k && ldc >= n,
                "nka_gemm_nt_f64: bad sizes");
  if (k == 0) {
    gemm_launch(a, lda, b, ldb, c, ldc, m, n, k, alpha, beta, 0.0, 0, nullptr, (hipStream_t)stream);
  } else {
    // 128x128 tiles when K is a multiple of their K step, else 64x64 tiles
    gemm_big_launch(a, lda, b, ldb, c, ldc, m, n, k, alpha, beta, 0, nullptr, (hipStream_t)stream);
  }
  NKA_CHECK_LAUNCH("nka_gemm_nt_f64");
  return NKA_OK;
}

// Workspace: 64x64 inverses of the diagonal blocks, the intermediate vector and the
// error word of the solves, and the K-slices of the trailing products' split tail tiles
// (up to kMaxSplitUnits raw 128x128 tiles, fewer for small n).
static int64_t split_units(int64_t n) {
  const int64_t t = (n + G2_T - 1) / G2_T;
  return std::min<int64_t>(kMaxSplitUnits, 2 * t * (t + 1) / 2);
}
static constexpr int64_t ws_head(int64_t n, int64_t nblk) {
  return (nblk * CH_NB * CH_NB * (int64_t)sizeof(double) + (n + 64) * (int64_t)sizeof(double) + 256 + 255) / 256 * 256;
}

int64_t nka_potrf_workspace(int64_t n) {
  if (n <= 0) return 0;
  return ws_head(n, (n + CH_NB - 1) / CH_NB) + split_units(n) * G2_T * G2_T * (int64_t)sizeof(double);
}

static inline double* ws_inv(void* ws) { return (double*)ws; }
static inline double* ws_vec(void* ws, int64_t nblk) {
  return (double*)ws + nblk * CH_NB * CH_NB;
}
static inline int32_t* ws_err(void* ws, int64_t n, int64_t nblk) {
  return (int32_t*)(ws_vec(ws, nblk) + n + 64);
}
static inline double* ws_split(void* ws, int64_t n, int64_t nblk) {
  return (double*)((char*)ws + ws_head(n, nblk));
}

// Right-looking Cholesky with up to three levels of blocking.  An outer
// panel of NB0 columns is factored as panels of NB1 columns, each by 64-column
// steps (diagonal block and panel solve in one launch, then the update of the
// NB1-panel's remaining columns); after each NB1-panel the rest of the outer
// panel receives a rank-NB1 update, and after the outer panel the trailing
// matrix one rank-NB0 update.  A long K keeps the MFMA GEMM near its peak and
// reads and writes the trailing matrix fewer times; the widths trade that
// against the tile-count quantisation of the narrower updates.  The inverses
// of the diagonal blocks, used by the triangular solves, are formed at the
// end.
// The launches of the factorisation.  split / n_split are the K-slices of
// the trailing products' split tail tiles (nullptr / 0: no split).
static void potrf_run(double* a, int64_t n, int64_t lda, void* workspace, double* split, int64_t n_split,
                      int32_t* info, hipStream_t s) {
  static_assert(sizeof(PanelLds) <= 80 * 1024, "two workgroups per CU");
  (void)hipFuncSetAttribute((const void*)panel_step_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)sizeof(PanelLds));
  (void)hipFuncSetAttribute((const void*)panel_step_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)sizeof(PanelLds));
  double* inv = ws_inv(workspace);
  const int64_t nblk = (n + CH_NB - 1) / CH_NB;
  // Panel widths.  Up to n = 5000 as few panels as can be of at most 2048 columns:
  // the steps' own updates (K = 64) are cheaper there than a product and the sum of
  // its slices (whole solves at n = 960, 1680, 2600, 4096: 276, 510, 863, 1707 us,
  // against 345, 595, 971, 1800 us with panels of 768).  Then 768 (6000, 8384,
  // 12288: 3.37, 6.55, 15.8 ms, against 3.43, 6.70, 16.2 with 512 and 3.38, 6.65,
  // 15.9 with 1024), and (4096, 512) from 16384 (32.4 ms there against 33.0 with 768).
  const bool large = n >= 16384;
  const int64_t few = (n + 2047) / 2048, one = ((n + few - 1) / few + CH_NB - 1) / CH_NB * CH_NB;
  const int64_t NB0 = large ? 4096 : n <= 5000 ? one : 768, NB1 = large ? 512 : NB0;
  for (int64_t K0 = 0; K0 < n; K0 += NB0) {
    const int64_t n0 = std::min<int64_t>(NB0, n - K0);
    for (int64_t K1 = K0; K1 < K0 + n0; K1 += NB1) {
      const int64_t n1 = std::min<int64_t>(NB1, K0 + n0 - K1);
      // 64-column steps, one launch each.  The first step of the panel factors
      // its columns as the trailing updates left them; a later one applies the
      // previous step's update to its columns itself, and to the columns further
      // right beside it.
      for (int64_t k0 = K1; k0 < K1 + n1; k0 += CH_NB) {
        const int nb = (int)std::min<int64_t>(CH_NB, n - k0);
        const int64_t rest = std::max<int64_t>(n - k0 - CH_NB, 0);
        double* slot = inv + (k0 / CH_NB) * CH_NB * CH_NB;
        const int strips = rest <= 256 * 48 ? 3 : 4;
        const int64_t nf = std::max<int64_t>((rest + 16 * strips - 1) / (16 * strips), 1);
        if (k0 == K1) {
          hipLaunchKernelGGL(panel_step_kernel<false>, dim3((unsigned)nf), dim3(512), sizeof(PanelLds), s, a, lda, n,
                             k0, nb, strips, (int)nf, (int64_t)0, 1, slot, info);
        } else {
          const int64_t cols_b = std::max<int64_t>(K1 + n1 - (k0 + CH_NB), 0);
          const int64_t tn = std::max<int64_t>((cols_b + 63) / 64, 1);
          const int64_t tiles_b = cols_b > 0 ? (rest + 127) / 128 * tn : 0;
          hipLaunchKernelGGL(panel_step_kernel<true>, dim3((unsigned)(nf + tiles_b)), dim3(512), sizeof(PanelLds), s,
                             a, lda, n, k0, nb, strips, (int)nf, cols_b, (int)tn, slot, info);
        }
      }
      // update of the outer panel's columns right of this NB1-column panel
      // (K = NB1): the lower triangle of its square top, then the rows below it
      const int64_t cols1 = K0 + n0 - (K1 + n1);
      if (cols1 > 0) {
        const int64_t rows1 = n - (K1 + n1);
        const double* l = a + (K1 + n1) * lda + K1;
        double* c = a + (K1 + n1) * lda + (K1 + n1);
        gemm_big_launch(l, lda, l, lda, c, lda, cols1, cols1, n1, -1.0, 1.0, 1, info, s, split, n_split);
        if (rows1 > cols1)
          gemm_big_launch(l + cols1 * lda, lda, l, lda, c + cols1 * lda, lda, rows1 - cols1, cols1, n1, -1.0,
                          1.0, 0, info, s, split, n_split);
      }
    }
    // trailing update (K = NB0)
    const int64_t rest2 = n - K0 - n0;
    if (rest2 > 0) {
      const double* l21 = a + (K0 + n0) * lda + K0;
      double* a22 = a + (K0 + n0) * lda + (K0 + n0);
      gemm_big_launch(l21, lda, l21, lda, a22, lda, rest2, rest2, n0, -1.0, 1.0, 1, info, s, split, n_split);
    }
  }
  hipLaunchKernelGGL(trtri_blocks_kernel, dim3((unsigned)nblk), dim3(256), 0, s, a, lda, n, inv, ws_vec(workspace, nblk),
                     info);
}

int nka_potrf_f64(double* a, int64_t n, int64_t lda, void* workspace, int32_t* info,
                  void* stream) {
  NKA_CHECK_ARG(n >= 0 && lda >= n && a && workspace && info, "nka_potrf_f64: bad arguments");
  if (n == 0) return NKA_OK;
  const int64_t nblk = (n + CH_NB - 1) / CH_NB;
  NKA_CHECK_ARG(nblk < (1LL << 31), "nka_potrf_f64: too large");
  potrf_run(a, n, lda, workspace, ws_split(workspace, n, nblk), split_units(n), info, (hipStream_t)stream);
  NKA_CHECK_LAUNCH("nka_potrf_f64");
  return NKA_OK;
}

// The launches of the two triangular solves, whose waits end after `limit` polls.
static void potrs_run(const double* a, int64_t n, int64_t lda, void* ws, double* b, const int32_t* info,
                      hipStream_t s, int64_t limit) {
  const int64_t nblk = (n + CH_NB - 1) / CH_NB;
  const double* inv = ws_inv(ws);
  double* y = ws_vec(ws, nblk);
  int32_t* err = ws_err(ws, n, nblk);
  // (y is as the factorisation or the last solve left it: unsolved)
  hipLaunchKernelGGL(trsv_lookback<false>, dim3((unsigned)nblk), dim3(256), 0, s, a, lda, n, inv, b, y, info, err,
                     limit);
  hipLaunchKernelGGL(trsv_lookback<true>, dim3((unsigned)nblk), dim3(256), 0, s, a, lda, n, inv, y, b, info, err,
                     limit);
}

int nka_potrs_f64_bounded(const double* a, int64_t n, int64_t lda, const void* workspace, double* b,
                          const int32_t* info, int64_t polls, void* stream) {
  NKA_CHECK_ARG(n >= 0 && lda >= n && a && workspace && b && info && polls >= 0, "nka_potrs_f64: bad arguments");
  if (n == 0) return NKA_OK;
  NKA_CHECK_ARG((n + CH_NB - 1) / CH_NB < (1LL << 31), "nka_potrs_f64: too large");
  potrs_run(a, n, lda, (void*)workspace, b, info, (hipStream_t)stream, polls);
  NKA_CHECK_LAUNCH("nka_potrs_f64");
  return NKA_OK;
}

int nka_potrs_f64(const double* a, int64_t n, int64_t lda, const void* workspace, double* b,
                  const int32_t* info, void* stream) {
  return nka_potrs_f64_bounded(a, n, lda, workspace, b, info, kSpinLimit, stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Factor and solve with no allocation and no caller workspace.  The scratch
// (inverses of the diagonal blocks, the intermediate vector and the error word
// of the solves) is a static device array of a fixed size;
// host code reaches it only through the address hipGetSymbolAddress returns
// for the current device.  Trailing products run unsplit here (the split of
// tail tiles would need up to 128 MiB more), so the last bits can differ from
// nka_potrf_f64 + nka_potrs_f64 by the order of the K sums of those tiles.
// ---------------------------------------------------------------------------
constexpr int64_t kNoAllocMaxN = 32768;
constexpr int64_t kNoAllocNblk = (kNoAllocMaxN + CH_NB - 1) / CH_NB;
constexpr int64_t kNoAllocBytes = ws_head(kNoAllocMaxN, kNoAllocNblk);

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64];

// The device address of `scratch` on the current device, looked up once per device.
static void* scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    set_error("nka_cholesky_solve_f64_noalloc: no current HIP device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("nka_cholesky_solve_f64_noalloc: hipGetSymbolAddress: %s", hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

// Scale-invariant regularisation of the QGT (netket/optimizer/qgt/qgt_jacobian_common.py:21-60):
// d_k = sqrt(S_kk + offset) from the diagonal of the unregularised S.
__global__ void qgt_diag_scale_kernel(const double* __restrict__ a, int64_t n, int64_t lda, double offset,
                                      double* __restrict__ d) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    d[k] = sqrt(a[k * lda + k] + offset);
}
// mode 0: lower triangle S_ij / (d_i d_j) + shift delta_ij (the rescaled system);
// mode 1: S_kk + shift d_k^2 on the diagonal only (to_dense of the scaled QGT).
__global__ void qgt_rescale_kernel(double* __restrict__ a, int64_t n, int64_t lda, const double* __restrict__ d,
                                   double shift, int mode) {
  if (mode == 1) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
      a[k * lda + k] += shift * d[k] * d[k];
    return;
  }
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    const double di = d[i];
    for (int64_t j = threadIdx.x; j <= i; j += blockDim.x) {
      double v = a[i * lda + j] / (di * d[j]);
      if (j == i) v += shift;
      a[i * lda + j] = v;
    }
  }
}
__global__ void mul_div_kernel(const double* __restrict__ x, const double* __restrict__ d, int64_t n, int divide,
                               double* __restrict__ out) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    out[k] = divide ? x[k] / d[k] : x[k] * d[k];
}

__global__ void select_on_flag_kernel(const int32_t* __restrict__ flag, const double* __restrict__ src,
                                      double* __restrict__ x, int64_t n) {
  if (*flag == 0) return;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    x[k] = src ? src[k] : 0.0;
}

extern "C" {

int64_t nka_cholesky_solve_noalloc_max_n(void) { return kNoAllocMaxN; }

int nka_cholesky_solve_f64_noalloc(double* a, int64_t n, int64_t lda, double* b, int32_t* info,
                                   void* stream) {
  NKA_CHECK_ARG(n >= 0 && lda >= n && info && (n == 0 || (a && b)),
                "nka_cholesky_solve_f64_noalloc: bad arguments");
  NKA_CHECK_ARG(n <= kNoAllocMaxN, "nka_cholesky_solve_f64_noalloc: n = %lld exceeds the maximum %lld of the "
                "static scratch; use nka_potrf_f64 / nka_potrs_f64 with a workspace",
                (long long)n, (long long)kNoAllocMaxN);
  void* ws = scratch_on_current_device();
  if (!ws) return NKA_ERR_HIP;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, (uint32_t*)info, (int64_t)1);
  if (n == 0) {
    NKA_CHECK_LAUNCH("nka_cholesky_solve_f64_noalloc");
    return NKA_OK;
  }
  potrf_run(a, n, lda, ws, nullptr, 0, info, s);
  potrs_run(a, n, lda, ws, b, info, s, kSpinLimit);
  NKA_CHECK_LAUNCH("nka_cholesky_solve_f64_noalloc");
  return NKA_OK;
}

int nka_qgt_rescale_f64(double* a, int64_t n, int64_t lda, double offset, double shift, int mode,
                        double* scale, void* stream) {
  NKA_CHECK_ARG(n >= 0 && lda >= n && (mode == 0 || mode == 1) && (n == 0 || (a && scale)),
                "nka_qgt_rescale_f64: bad arguments");
  if (n == 0) return NKA_OK;
  hipStream_t s = (hipStream_t)stream;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(qgt_diag_scale_kernel, dim3(g), dim3(256), 0, s, a, n, lda, offset, scale);
  const unsigned g2 = mode == 1 ? g : (unsigned)std::min<int64_t>(n, 8192);
  hipLaunchKernelGGL(qgt_rescale_kernel, dim3(g2), dim3(256), 0, s, a, n, lda, scale, shift, mode);
  NKA_CHECK_LAUNCH("nka_qgt_rescale_f64");
  return NKA_OK;
}

int nka_mul_div_f64(const double* x, const double* d, int64_t n, int divide, double* out, void* stream) {
  NKA_CHECK_ARG(n >= 0 && (n == 0 || (x && d && out)), "nka_mul_div_f64: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(mul_div_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, x, d, n, divide, out);
  NKA_CHECK_LAUNCH("nka_mul_div_f64");
  return NKA_OK;
}

int nka_select_on_flag_f64(const int32_t* flag, const double* src, double* x, int64_t n, void* stream) {
  NKA_CHECK_ARG(n >= 0 && flag && (n == 0 || x), "nka_select_on_flag_f64: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(select_on_flag_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, flag, src, x, n);
  NKA_CHECK_LAUNCH("nka_select_on_flag_f64");
  return NKA_OK;
}

int nka_gemv_f64(const double* a, int64_t lda, int64_t m, int64_t n, int trans, const double* x,
                 double alpha, double beta, double* y, void* workspace, void* stream) {
  NKA_CHECK_ARG(m >= 0 && n >= 0 && a && x && y, "nka_gemv_f64: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  if (trans == 0 || trans == 2) {
    const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>((m + 3) / 4, 4096));
    hipLaunchKernelGGL(gemv_n_kernel, dim3(g), dim3(256), 0, s, a, lda, m, n, x, alpha, beta, y,
                       trans == 2 ? 1 : 0);
  } else if (trans == 1) {
    NKA_CHECK_ARG(workspace != nullptr, "nka_gemv_f64: transposed product needs a workspace");
    const int64_t rows_per = 256;
    const int64_t parts = (m + rows_per - 1) / rows_per;
    NKA_CHECK_ARG(parts <= 65535, "nka_gemv_f64: too many rows");
    dim3 grid((unsigned)((n + 255) / 256), (unsigned)std::max<int64_t>(parts, 1));
    hipLaunchKernelGGL(gemv_t_partial, grid, dim3(256), 0, s, a, lda, m, n, x, (double*)workspace,
                       rows_per);
    const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 4096));
    hipLaunchKernelGGL(gemv_t_reduce, dim3(g), dim3(256), 0, s, (const double*)workspace,
                       (int)std::max<int64_t>(parts, 1), n, alpha, beta, y);
  } else {
    set_error("nka_gemv_f64: bad trans %d", trans);
    return NKA_ERR_ARG;
  }
  NKA_CHECK_LAUNCH("nka_gemv_f64");
  return NKA_OK;
}

int nka_check_finite(const double* x, int64_t n, int32_t* flag, void* stream) {
  NKA_CHECK_ARG(n >= 0 && flag && (n == 0 || x), "nka_check_finite: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 1024);
  hipLaunchKernelGGL(check_finite_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, x, n, flag);
  NKA_CHECK_LAUNCH("nka_check_finite");
  return NKA_OK;
}

int nka_sgd_update(void* params, int dtype, const double* dp, int64_t n, double lr, void* stream) {
  NKA_CHECK_ARG(n >= 0 && (n == 0 || (params && dp)), "nka_sgd_update: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
  if (dtype == NKA_F32)
    hipLaunchKernelGGL(sgd_kernel<float>, dim3(g), dim3(256), 0, (hipStream_t)stream,
                       (float*)params, dp, n, (float)lr);
  else if (dtype == NKA_F64)
    hipLaunchKernelGGL(sgd_kernel<double>, dim3(g), dim3(256), 0, (hipStream_t)stream,
                       (double*)params, dp, n, lr);
  else {
    set_error("nka_sgd_update: bad dtype");
    return NKA_ERR_ARG;
  }
  NKA_CHECK_LAUNCH("nka_sgd_update");
  return NKA_OK;
}

int nka_axpy_f64(int64_t n, double alpha, const double* x, double* y, void* stream) {
  NKA_CHECK_ARG(n >= 0 && (n == 0 || (x && y)), "nka_axpy_f64: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(axpy_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, n, alpha, x, y);
  NKA_CHECK_LAUNCH("nka_axpy_f64");
  return NKA_OK;
}

int nka_centre_scale(const double* e, int64_t n, const double* mean, double scale, double* out,
                     void* stream) {
  NKA_CHECK_ARG(n >= 0 && (n == 0 || (e && mean && out)), "nka_centre_scale: bad arguments");
  if (n == 0) return NKA_OK;
  const unsigned g = (unsigned)std::min<int64_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(centre_scale_kernel, dim3(g), dim3(256), 0, (hipStream_t)stream, e, n, mean,
                     scale, out);
  NKA_CHECK_LAUNCH("nka_centre_scale");
  return NKA_OK;
}

int nka_symmetrize_f64(double* a, int64_t n, int64_t lda, void* stream) {
  NKA_CHECK_ARG(n >= 0 && lda >= n && (n == 0 || a), "nka_symmetrize_f64: bad arguments");
  if (n == 0) return NKA_OK;
  const int64_t T = (n + SY_T - 1) / SY_T;
  NKA_CHECK_ARG(T * (T + 1) / 2 < (1LL << 31), "nka_symmetrize_f64: too large");
  hipLaunchKernelGGL(symmetrize_kernel, dim3((unsigned)(T * (T + 1) / 2)), dim3(256), 0, (hipStream_t)stream, a, n,
                     lda);
  NKA_CHECK_LAUNCH("nka_symmetrize_f64");
  return NKA_OK;
}

int nka_stats_moments(const double* data, int n_chains, int chain_length, double* out8,
                      void* stream) {
  NKA_CHECK_ARG(n_chains > 0 && chain_length > 0 && data && out8, "nka_stats_moments: bad arguments");
  hipLaunchKernelGGL(stats_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, data, n_chains,
                     chain_length, out8);
  NKA_CHECK_LAUNCH("nka_stats_moments");
  return NKA_OK;
}

}  // extern "C"
