// Dense S of an FP64 RBM from its structure, on the int8 matrix cores
// (matrix = O_L^T O_L + diag_shift I of netket/_src/ngd/sr.py:43-55 and
// QGTJacobianDenseT.to_dense, netket/optimizer/qgt/qgt_jacobian_dense.py:136-161).
//
// As for FP32 models (nka_ntk.hip) every entry of O^T O is one entry of
// C = P Q^T over the samples, P the distinct spin-pair products (+-1) and Q
// the distinct pair products of the centred activations.  Here Q is held as
// 55-bit fixed point with one power-of-two scale per row, in seven planes of
// balanced base-256 digits (int8), so that P Q_d^T is an exact int32 product
// on v_mfma_i32_32x32x32_i8 for each digit plane d and C comes out with a
// single rounding per entry and slice or chunk of the samples (usually one of
// each), where an FP64 product of the Jacobian rounds at every accumulation.
//
// Seven int8 products of Na Nb Ns (Na Nb about Np^2 / 4) replace Ns Np^2
// FP64 operations; the int8 rate is 64 times the FP64 one.  64 sites, 128
// hidden units, 16384 samples (S 8384^2, mirrored): 47.7 ms as the FP64
// product of the Jacobian, 3.0 ms here, and the error of S against extended
// precision fell from 3.5e-15 to 1.0e-15 (relative norms).
#include "nka_common.hpp"
#include "nka_qgt.hpp"

namespace nka {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int Q8_D = 7;        // digit planes of Q
constexpr int Q8_BITS = 54;    // |q| 2^(54 - e) <= 2^54 for a row with |q| < 2^e
constexpr int Q8_K = 64;       // samples (bytes) per K step
constexpr int Q8_BUF = 4;      // K steps held in LDS
constexpr int Q8_MI = 2;       // 32-row blocks of P per wavefront
constexpr int Q8_TA = 64 * Q8_MI, Q8_TB = 64;
constexpr int Q8_SMALLEST = -400;   // least row exponent (keeps every scale finite)

// c_j = mean over the samples of tT[j][:] and e_j with |t_j - c_j| < 2^e_j for
// every sample, one workgroup per hidden unit.  ex[j] = e_j as a double, NaN
// when an activation is (the sums of its pairs then are NaN as well).
__global__ void __launch_bounds__(256) qgt64_means_kernel(const double* __restrict__ tT, int64_t ns, int M,
                                                          double* __restrict__ c, double* __restrict__ ex) {
  __shared__ double red[4];
  const int wid = threadIdx.x >> 6;
  for (int j = blockIdx.x; j < M; j += gridDim.x) {
    const double* t = tT + (int64_t)j * ns;
    double acc = 0.0;
    for (int64_t s = threadIdx.x; s < ns; s += 256) acc += t[s];
    acc = wave_sum(acc);
    __syncthreads();
    if (lane_id() == 0) red[wid] = acc;
    __syncthreads();
    const double mean = (red[0] + red[1] + red[2] + red[3]) / (double)ns;
    double mx = 0.0;
    for (int64_t s = threadIdx.x; s < ns; s += 256) mx = fmax(mx, fabs(t[s] - mean));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, NKA_WAVE));
    __syncthreads();
    if (lane_id() == 0) red[wid] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
      mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
      const int e = mx > 0.0 ? ilogb(mx) + 1 : Q8_SMALLEST;
      c[j] = mean;
      ex[j] = mean == mean ? (double)max(e, Q8_SMALLEST) : mean;   // a NaN activation makes the mean NaN
    }
  }
}

// The two hidden units (j <= l; -1: none) of row r of Q.
__device__ inline void qgt_hidden_pair(int64_t r, int M, int64_t& j, int64_t& l) {
  j = l = -1;
  if (r >= 1 && r <= M) {
    j = r - 1;
  } else if (r > M) {
    const int64_t b = r - 1 - M;
    l = tri_root(b);
    j = b - l * (l + 1) / 2;
  }
}

// P (rows x ldk int8, +-1) from the transposed spins sT (+-1, 0 past ns): the
// bytes of a product of two signs are (a ^ b) | 1.  Past ns P may hold
// anything, since Q is zero there.  One workgroup per row, 16 samples per
// thread and step.
__global__ void __launch_bounds__(256) qgt64_spin_pairs_kernel(const int8_t* __restrict__ sT, int N, int64_t ldk,
                                                               int64_t rows, int8_t* __restrict__ P) {
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    int64_t i = -1, k = -1;
    if (r >= 1 && r <= N) {
      i = r - 1;
    } else if (r > N) {
      const int64_t b = r - 1 - N;
      k = tri_root(b) + 1;
      i = b - k * (k - 1) / 2;
    }
    for (int64_t s0 = (int64_t)threadIdx.x * 16; s0 < ldk; s0 += 256 * 16) {
      uint4 v = {0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};
      if (i >= 0) v = *(const uint4*)(sT + i * ldk + s0);
      if (k >= 0) {
        const uint4 b = *(const uint4*)(sT + k * ldk + s0);
        v.x = (v.x ^ b.x) | 0x01010101u;
        v.y = (v.y ^ b.y) | 0x01010101u;
        v.z = (v.z ^ b.z) | 0x01010101u;
        v.w = (v.w ^ b.w) | 0x01010101u;
      }
      *(uint4*)(P + r * ldk + s0) = v;
    }
  }
}

// Bytes k of four words, packed into one word each (4x4 byte transpose).
__device__ inline void bytes4x4(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t (&o)[4]) {
  const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u);  // a0 b0 a1 b1
  const uint32_t ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);  // a2 b2 a3 b3
  const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u);
  const uint32_t cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
  o[0] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
  o[1] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
  o[2] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
  o[3] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
}

// Q: row r of the pair products q (1, t'_j, t'_j t'_l with t' = t - c) as the
// integer I = rint(q 2^(54 - e)), e = e_j + e_l, in seven planes of balanced
// base-256 digits: I + 0x80..80 has the bytes d + 128, and a byte's digit is
// its value with the top bit flipped.  |I| <= 2^54 fits the seven digits.
// (A product below 2^-55 of 2^e is lost, 2^-53 of the product of its units' largest.)
// rscale[r] = 2^(e - 54).  Plane d, row r, sample s is Q[(d rows + r) ldk + s];
// zero past ns.  One workgroup per row, 4 samples per thread and step: the
// loads of a wavefront then cover whole lines, and its stores 256 bytes per
// plane.  Bound by the 7 bytes written per entry.  (t of unit j: tT + j ldt.)
__global__ void __launch_bounds__(256) qgt64_hidden_digits_kernel(const double* __restrict__ tT, int64_t ldt,
                                                                  int64_t ns, int M,
                                                                  const double* __restrict__ cmean,
                                                                  const double* __restrict__ ex, int64_t ldk,
                                                                  int64_t rows, uint8_t* __restrict__ Q,
                                                                  double* __restrict__ rscale) {
  const bool vec = (ldt % 2) == 0 && (((uintptr_t)tT) % 16) == 0;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    int64_t j, l;
    qgt_hidden_pair(r, M, j, l);
    const double ej = j >= 0 ? ex[j] : 1.0, el = l >= 0 ? ex[l] : 0.0;
    const double e = ej + el;
    const bool nan = e != e;
    const double up = nan ? 0.0 : ldexp(1.0, Q8_BITS - (int)e);
    if (threadIdx.x == 0) rscale[r] = nan ? e : ldexp(1.0, (int)e - Q8_BITS);
    const double cj = j >= 0 ? cmean[j] : 0.0, cl = l >= 0 ? cmean[l] : 0.0;
    for (int64_t s0 = (int64_t)threadIdx.x * 4; s0 < ldk; s0 += 256 * 4) {
      double f[4];
      auto load4 = [&](const double* t, double (&v)[4]) {
        if (vec && s0 + 4 <= ns) {
          const double2 a = *(const double2*)(t + s0), b = *(const double2*)(t + s0 + 2);
          v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = s0 + q < ns ? t[s0 + q] : 0.0;
        }
      };
      if (j < 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) f[q] = 1.0;
      } else {
        load4(tT + j * ldt, f);
#pragma unroll
        for (int q = 0; q < 4; ++q) f[q] -= cj;
        if (l >= 0) {
          double h[4];
          load4(tT + l * ldt, h);
#pragma unroll
          for (int q = 0; q < 4; ++q) f[q] *= h[q] - cl;
        }
      }
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // v is a whole number, so its low word is in [0, 2^32)
        const double v = s0 + q < ns ? rint(f[q] * up) : 0.0;
        const double vh = floor(v * 0x1p-32);
        const uint32_t vl = (uint32_t)fma(vh, -0x1p32, v);
        const uint64_t I = ((uint64_t)(uint32_t)(int32_t)vh << 32) + vl + 0x0080808080808080ull;
        lo[q] = (uint32_t)I ^ 0x80808080u;
        hi[q] = (uint32_t)(I >> 32) ^ 0x00808080u;
      }
      uint32_t o[2][4];
      bytes4x4(lo[0], lo[1], lo[2], lo[3], o[0]);
      bytes4x4(hi[0], hi[1], hi[2], hi[3], o[1]);
#pragma unroll
      for (int d = 0; d < Q8_D; ++d) *(uint32_t*)(Q + ((int64_t)d * rows + r) * ldk + s0) = o[d / 4][d % 4];
    }
  }
}

// C = P Q^T (FP64), one 128 x 64 tile per workgroup: four wavefronts of 64 x 32
// with one int32 accumulator per digit plane and 32 x 32 block (2 x 7), so a
// K sub-step of 32 samples reads 2 + 7 operand fragments from LDS for 14
// products.  Operands go from global memory straight into LDS (16 bytes per lane),
// three K steps ahead of the one that is multiplied, which leaves the registers to
// the 224 accumulators.  A row's four 16-byte chunks of a K step are stored in the
// order chunk ^ (row / 4 % 4), which makes the fragment reads (32 consecutive
// rows, one chunk) free of bank conflicts over the 64 banks.
// Tiles are numbered down the columns, so the workgroups that share a panel of
// Q (the larger operand) run on one XCD and read it through one L2.
// Bound by the matrix cores (48% busy at the clock the card holds here): 2.36 to
// 2.56 ms over cards at 2081 x 8385 x 16384 (1.6e15 int8 operations/s).  Where it took
// 2.40 ms, it took 3.07 (34% busy) with the loads and LDS reads issued ahead of a
// step's products instead of between them, and 3.15 with two buffers instead of four.
// blockIdx.y: slice of K (whole K steps); slice y writes C + y * slab, or with `add`
// (a further chunk of the samples) adds to it.
__global__ void __launch_bounds__(256, 1) qgt64_gemm_kernel(const int8_t* __restrict__ P, int64_t ma,
                                                         const uint8_t* __restrict__ Q, int64_t nb,
                                                         const double* __restrict__ rscale, int64_t ldk,
                                                         double* __restrict__ C, int64_t ldc, int64_t slab,
                                                         int64_t tiles_m, int64_t n_tiles, int64_t steps_per_slice,
                                                         int add) {
  constexpr int A_BYTES = Q8_TA * Q8_K, B_BYTES = Q8_D * Q8_TB * Q8_K;
  constexpr int LOADS = (A_BYTES + B_BYTES) / 1024 / 4;   // 16-row wavefront loads per wavefront and K step
  static_assert((A_BYTES + B_BYTES) % 4096 == 0, "whole loads per wavefront");
  constexpr int AHEAD = Q8_BUF - 1;                       // K steps in flight ahead of the products
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Q8_BUF][A_BYTES + B_BYTES];
  const int64_t G = gridDim.x;
  const int64_t bid = (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  if (bid >= n_tiles) return;
  const int64_t i0 = (bid % tiles_m) * Q8_TA, j0 = (bid / tiles_m) * Q8_TB;
  const int tid = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = (wid >> 1) * 32 * Q8_MI, wn = (wid & 1) * 32;
  const int64_t steps = ldk / Q8_K;
  const int64_t t0 = (int64_t)blockIdx.y * steps_per_slice;
  const int64_t t1 = min<int64_t>(steps, t0 + steps_per_slice);

  // Each of the wavefront's loads covers 16 rows of P or of one plane: a buffer
  // descriptor of those rows (rows past the operand's end read as zero), and
  // for this lane row lane / 4 and the chunk that belongs in slot lane % 4.
  __amdgpu_buffer_rsrc_t src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (wid * LOADS + i) * 16;            // first row in the stacked tile (P rows, then the planes')
    const int b = row - Q8_TA;
    const int64_t first = row < Q8_TA ? i0 + row : j0 + b % Q8_TB, rows = row < Q8_TA ? ma : nb;
    const uint8_t* base = row < Q8_TA ? (const uint8_t*)P : Q + (int64_t)(b / Q8_TB) * nb * ldk;
    const int64_t left = min<int64_t>(max<int64_t>(rows - first, 0), 16);
    const uint64_t addr = (uint64_t)(base + (left > 0 ? first : 0) * ldk);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)addr);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(addr >> 32));
    src[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0,
                                               __builtin_amdgcn_readfirstlane((int)(left * ldk)), 0x00020000);
  }
  // (row / 4) % 4 of the stacked row is that of the row among the 16
  const int voff = (lane >> 2) * (int)ldk + (((lane & 3) ^ ((lane >> 4) & 3)) * 16);
  auto issue = [&](int buf, int64_t t, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        src[i], (__attribute__((address_space(3))) void*)&smem[buf][(wid * LOADS + i) * 1024], 16, voff,
        (int)(t * Q8_K), 0, 0);
  };
  i32x16 acc[Q8_D][Q8_MI];
#pragma unroll
  for (int d = 0; d < Q8_D; ++d)
#pragma unroll
    for (int x = 0; x < Q8_MI; ++x)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[d][x][e] = 0;

  // fragment f (P blocks, then planes) of sub-step ks of the step in `buf`
  const int fr = lane & 31, sw = (fr >> 2) & 3;
  const int foff[2] = {fr * Q8_K + ((lane >> 5) ^ sw) * 16, fr * Q8_K + ((2 + (lane >> 5)) ^ sw) * 16};
  auto frag = [&](int buf, int ks, int f) {
    const int row = f < Q8_MI ? wm + f * 32 : Q8_TA + (f - Q8_MI) * Q8_TB + wn;
    return *(const i32x4*)(smem[buf] + row * Q8_K + foff[ks]);
  };
  // Each K step is two phases of 14 products.  A phase multiplies one
  // sub-step's fragments while it reads the other's (the next step's first
  // ones in phase 1) and issues its share of the loads of the step AHEAD,
  // one request behind each product, so neither the LDS reads nor the issue of
  // the loads stands between two products.  (The last steps are requested
  // again past the end: the count of loads in flight is the same at every step.)
  constexpr int NF = Q8_MI + Q8_D, NP = Q8_MI * Q8_D, SPLIT = NP - NF;
  static_assert(SPLIT >= 0 && LOADS >= SPLIT && LOADS - SPLIT <= NP, "requests fit behind the products");
  i32x4 fg[2][NF];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
#pragma unroll
    for (int k = 0; k < LOADS; ++k) issue(i, min<int64_t>(t0 + i, t1 - 1), k);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((AHEAD - 1) * LOADS) : "memory");
#pragma unroll
  for (int f = 0; f < NF; ++f) fg[0][f] = frag(0, 0, f);
  int buf = 0;
  for (int64_t t = t0; t < t1; ++t) {
    const int next = (buf + 1) % Q8_BUF, into = (buf + AHEAD) % Q8_BUF;
    const int64_t tl = min<int64_t>(t + AHEAD, t1 - 1);
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
      if (ph == 1)
        // this wavefront's loads of step t + 1 have landed and its reads of step t
        // are done; after the barrier that holds for all four
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((AHEAD - 2) * LOADS + SPLIT) : "memory");
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        const int d = q / Q8_MI, x = q % Q8_MI;
        acc[d][x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fg[ph][x], fg[ph][Q8_MI + d], acc[d][x], 0, 0, 0);
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
  const int64_t gj = j0 + wn + (lane & 31);
  if (gj < nb) {
    const double rs = rscale[gj];
    double* out = C + (int64_t)blockIdx.y * slab;
#pragma unroll
    for (int x = 0; x < Q8_MI; ++x)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t gi = i0 + wm + x * 32 + (e / 4) * 8 + (lane >> 5) * 4 + (e & 3);
        if (gi < ma) {
          // both halves are exact integers below 2^53; one rounding in the sum
          const int64_t lo = (int64_t)acc[0][x][e] + ((int64_t)acc[1][x][e] << 8) + ((int64_t)acc[2][x][e] << 16) +
                             ((int64_t)acc[3][x][e] << 24);
          const int64_t hi = (int64_t)acc[4][x][e] + ((int64_t)acc[5][x][e] << 8) + ((int64_t)acc[6][x][e] << 16);
          const double v = fma((double)hi, 0x1p32, (double)lo) * rs;
          out[gi * ldc + gj] = add ? out[gi * ldc + gj] + v : v;
        }
      }
  }
}

// C += the slices' partial sums, in slice order.
__global__ void __launch_bounds__(256) qgt64_reduce_kernel(double* __restrict__ C, int64_t total, int64_t slab,
                                                           int slices) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    double v = C[i];
    for (int y = 1; y < slices; ++y) v += C[i + y * slab];
    C[i] = v;
  }
}

// S from C, one workgroup per augmented spin pair (u_hi >= u_lo in [-1, N)):
// the entries S[p][q] with p = (u_hi, w), q = (u_lo, x) for w, x in [-1, M),
// each written once into the lower triangle.  With K(w, x) the covariance sum
// of s_uhi t'_w and s_ulo t'_x (t'_-1 = 1, c_-1 = 0),
//   S_pq = scale (K(w,x) + c_w K(-1,x) + c_x K(w,-1) + c_w c_x K(-1,-1)) (+ shift if p == q),
//   K(w, x) = C[r, (w,x)] - C[r_hi, (w,-1)] C[r_lo, (x,-1)] / ns:
// every term is centred by itself, so no large sums cancel between them.
// The pair's row of C and the two spins' sums are staged in LDS when they fit.
template <bool LDS_ROW>
__global__ void __launch_bounds__(512) qgt64_unpack_kernel(nka_rbm m, const double* __restrict__ c, int64_t ldc,
                                                           int64_t nb, const double* __restrict__ cmean, double ns,
                                                           double scale, double shift, double* __restrict__ out,
                                                           int64_t ldo) {
  extern __shared__ double crow64[];
  const int N = m.n_visible, M = m.n_hidden;
  const int64_t n_pairs = (int64_t)(N + 1) * (N + 2) / 2;
  const int W = M + 1;
  const double rns = 1.0 / ns;
  const int wid = threadIdx.x >> 6, lane = lane_id();
  for (int64_t b = blockIdx.x; b < n_pairs; b += gridDim.x) {
    const int64_t ah = tri_root(b);
    const int uh = (int)ah - 1, ul = (int)(b - ah * (ah + 1) / 2) - 1;
    const double* row = c + qgt_spin_row(uh, ul, N) * ldc;
    const double* rowh = c + qgt_spin_row(uh, -1, N) * ldc;  // entries 0..M: sums of (u_hi, w)
    const double* rowl = c + qgt_spin_row(ul, -1, N) * ldc;
    if (LDS_ROW) {
      __syncthreads();
      for (int64_t e = threadIdx.x; e < nb; e += blockDim.x) crow64[e] = row[e];
      for (int e = threadIdx.x; e < W; e += blockDim.x) {
        crow64[nb + e] = rowh[e];
        crow64[nb + W + e] = rowl[e];
      }
      __syncthreads();
      row = crow64;
      rowh = crow64 + nb;
      rowl = crow64 + nb + W;
    }
    auto cov = [&](int w, int x) {
      return row[qgt_hidden_row(w, x, M)] - rowh[w + 1] * (rowl[x + 1] * rns);
    };
    // (sums of signs: whole numbers below 2^22, so one rounding)
    const double k00 = (row[0] * ns - rowh[0] * rowl[0]) * rns;
    auto entry = [&](int w, int64_t p, double cw, double kw, int x) {
      const int64_t q = qgt_param(ul, x, m);
      if (q < 0 || (uh == ul && p < q)) return;  // the symmetric diagonal pair: each entry once
      double v = w < 0 && x < 0 ? k00 : cov(w, x);
      if (x >= 0) {
        const double cx = cmean[x];
        if (w >= 0) v += cw * cov(-1, x) + cx * kw + cw * cx * k00;
        else v += cx * kw;
      } else if (w >= 0) {
        v += cw * k00;
      }
      v *= scale;
      if (p == q) v += shift;
      if (p >= q)
        out[p * ldo + q] = v;
      else
        out[q * ldo + p] = v;
    };
    // rows w of the block, one wavefront each; lanes along x >= 0, whose
    // positions q are consecutive in S
    for (int w = wid - 1; w < M; w += 8) {
      const int64_t p = qgt_param(uh, w, m);
      if (p < 0) continue;
      const double cw = w >= 0 ? cmean[w] : 0.0;
      const double kw = cov(w, -1);
      for (int x = lane; x < M; x += 64) entry(w, p, cw, kw, x);
    }
    // the column x = -1 (the visible bias of u_lo), one row per thread
    for (int w = (int)threadIdx.x - 1; w < M; w += blockDim.x) {
      const int64_t p = qgt_param(uh, w, m);
      if (p < 0) continue;
      entry(w, p, w >= 0 ? cmean[w] : 0.0, 0.0, -1);
    }
  }
}

constexpr int64_t kQ8Spare = 256 << 20;
static int64_t q8_ldc(const nka_rbm& m) { return (qgt_rows_q(m) + 31) / 32 * 32; }
static int64_t q8_np(const nka_rbm& m) {
  return (m.bias_off >= 0 ? m.n_hidden : 0) + (int64_t)m.n_visible * m.n_hidden +
         (m.visible_off >= 0 ? m.n_visible : 0);
}
// The samples go through in chunks (all of them at once where that fits) whose planes,
// with C, take no more than the FP64 Jacobian that they stand for and 256 MB: 7 bytes
// per activation pair and sample are 0.44 alpha Jacobians, and C is a quarter of S.  A
// chunk holds 512 samples at least.
// Slices of K: enough workgroups for the chip when the tiles alone are few,
// with at least 8 K steps each.
struct Q8Plan {
  int64_t chunk;        // samples of a chunk, padded
  int64_t tiles_m, tiles, slices, steps_per_slice;
  int64_t fixed;        // bytes of C, the scales and the means
};
static Q8Plan q8_plan(const nka_rbm& m, int64_t ns) {
  Q8Plan p;
  const int64_t rp = qgt_rows_p(m), rq = qgt_rows_q(m);
  const int64_t ldk = qgt_ldk(ns);
  p.tiles_m = (rp + Q8_TA - 1) / Q8_TA;
  p.tiles = p.tiles_m * ((rq + Q8_TB - 1) / Q8_TB);
  const int64_t wanted = std::min<int64_t>(256 / p.tiles, 16);
  p.fixed = qgt_round(std::max<int64_t>(wanted, 1) * rp * q8_ldc(m) * 8) + qgt_round(rq * 8) +
            2 * qgt_round((int64_t)m.n_hidden * 8);
  const int64_t per_sample = m.n_visible + rp + Q8_D * rq, room = 8 * q8_np(m) * ldk + kQ8Spare - p.fixed - 1024;
  const int64_t fits = std::max<int64_t>(room > 0 ? room / per_sample : 0, 512);
  const int64_t chunks = (ldk + fits - 1) / fits;
  p.chunk = std::min<int64_t>(ldk, ((ldk + chunks - 1) / chunks + Q8_K - 1) / Q8_K * Q8_K);
  if (p.chunk > fits) p.chunk = fits / Q8_K * Q8_K;
  const int64_t steps = p.chunk / Q8_K;
  const int64_t sl = std::max<int64_t>(std::min<int64_t>(wanted, steps / 8), 1);
  p.steps_per_slice = (steps + sl - 1) / sl;
  p.slices = (steps + p.steps_per_slice - 1) / p.steps_per_slice;
  return p;
}
// 128 ns per digit sum has to stay below 2^31
constexpr int64_t kQ8MaxSamples = 1 << 22;

}  // namespace nka

using namespace nka;

extern "C" {

int64_t nka_rbm_qgt_f64_workspace(const nka_rbm* m, int64_t ns) {
  if (!m || ns <= 0 || ns > kQ8MaxSamples || m->n_visible < 1 || m->n_hidden < 1) return 0;
  const Q8Plan p = q8_plan(*m, ns);
  return qgt_round((int64_t)m->n_visible * p.chunk) + qgt_round(qgt_rows_p(*m) * p.chunk) +
         qgt_round(Q8_D * qgt_rows_q(*m) * p.chunk) + p.fixed;
}

int nka_rbm_qgt_f64(const nka_rbm* m, const int8_t* sigma, const double* tT, int64_t ns, double scale, double shift,
                    double* out, int64_t ldo, void* workspace, void* stream) {
  NKA_CHECK_ARG(m && m->params && sigma && tT && out && workspace && ns > 0, "nka_rbm_qgt_f64: bad arguments");
  NKA_CHECK_ARG(m->dtype == NKA_F64, "nka_rbm_qgt_f64: FP64 models only");
  NKA_CHECK_ARG(ns <= kQ8MaxSamples, "nka_rbm_qgt_f64: too many samples");
  NKA_CHECK_ARG(m->n_visible >= 1 && m->n_hidden >= 1, "nka_rbm_qgt_f64: empty model");
  const int N = m->n_visible, M = m->n_hidden;
  NKA_CHECK_ARG(ldo >= q8_np(*m), "nka_rbm_qgt_f64: ldo < n_params");
  const Q8Plan pl = q8_plan(*m, ns);
  NKA_CHECK_ARG((int64_t)(N + 1) * (N + 2) / 2 < (1LL << 31) && pl.tiles < (1LL << 31),
                "nka_rbm_qgt_f64: too many units");
  hipStream_t s = (hipStream_t)stream;
  const int64_t rp = qgt_rows_p(*m), rq = qgt_rows_q(*m), ldc = q8_ldc(*m);
  unsigned char* w = (unsigned char*)workspace;
  int8_t* sT = (int8_t*)w;
  w += qgt_round((int64_t)N * pl.chunk);
  int8_t* P = (int8_t*)w;
  w += qgt_round(rp * pl.chunk);
  uint8_t* Q = (uint8_t*)w;
  w += qgt_round(Q8_D * rq * pl.chunk);
  double* C = (double*)w;
  w += qgt_round(pl.slices * rp * ldc * 8);
  double* rscale = (double*)w;
  w += qgt_round(rq * 8);
  double* cmean = (double*)w;
  w += qgt_round((int64_t)M * 8);
  double* ex = (double*)w;
  hipLaunchKernelGGL(qgt64_means_kernel, dim3((unsigned)std::min<int64_t>(M, 65536)), dim3(256), 0, s, tT, ns, M,
                     cmean, ex);
  const unsigned grid = (unsigned)((pl.tiles + 7) / 8 * 8);
  const int64_t slab = rp * ldc;
  for (int64_t s0 = 0; s0 < ns; s0 += pl.chunk) {
    // (each slice has the first steps_per_slice K steps of the chunk, so all of them
    // are written: a last chunk keeps the length, zero past its samples)
    const int64_t nc = std::min<int64_t>(pl.chunk, ns - s0), ldk = pl.chunk;
    launch_qgt_spins_t(sigma + s0 * N, nc, N, ldk, sT, s);
    hipLaunchKernelGGL(qgt64_spin_pairs_kernel, dim3((unsigned)std::min<int64_t>(rp, 65536)), dim3(256), 0, s,
                       (const int8_t*)sT, N, ldk, rp, P);
    hipLaunchKernelGGL(qgt64_hidden_digits_kernel, dim3((unsigned)std::min<int64_t>(rq, 65536)), dim3(256), 0, s,
                       tT + s0, ns, nc, M, (const double*)cmean, (const double*)ex, ldk, rq, Q, rscale);
    hipLaunchKernelGGL(qgt64_gemm_kernel, dim3(grid, (unsigned)pl.slices), dim3(256), 0, s, (const int8_t*)P, rp,
                       (const uint8_t*)Q, rq, (const double*)rscale, ldk, C, ldc, slab, pl.tiles_m, pl.tiles,
                       pl.steps_per_slice, s0 > 0 ? 1 : 0);
  }
  if (pl.slices > 1)
    hipLaunchKernelGGL(qgt64_reduce_kernel, dim3((unsigned)std::min<int64_t>((slab + 255) / 256, 4096)), dim3(256), 0,
                       s, C, slab, slab, (int)pl.slices);
  const unsigned gu = (unsigned)std::min<int64_t>((int64_t)(N + 1) * (N + 2) / 2, 65536);
  const size_t row_bytes = (size_t)(rq + 2 * (M + 1)) * sizeof(double);
  constexpr size_t kMaxRow = 128 * 1024;  // of the 160 KB of a CU
  if (row_bytes <= kMaxRow) {
    if (row_bytes > 64 * 1024)
      NKA_CHECK_HIP(hipFuncSetAttribute((const void*)qgt64_unpack_kernel<true>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxRow),
                    "nka_rbm_qgt_f64");
    hipLaunchKernelGGL(qgt64_unpack_kernel<true>, dim3(gu), dim3(512), row_bytes, s, *m, (const double*)C, ldc, rq,
                       (const double*)cmean, (double)ns, scale, shift, out, ldo);
  } else {
    hipLaunchKernelGGL(qgt64_unpack_kernel<false>, dim3(gu), dim3(512), 0, s, *m, (const double*)C, ldc, rq,
                       (const double*)cmean, (double)ns, scale, shift, out, ldo);
  }
  NKA_CHECK_LAUNCH("nka_rbm_qgt_f64");
  return NKA_OK;
}

}  // extern "C"
