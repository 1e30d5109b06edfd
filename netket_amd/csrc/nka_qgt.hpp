// Index maps of the RBM's structured S, shared by its FP32 (bf16 planes) and
// FP64 (int8 digit planes) forms.
#pragma once

#include "nka_common.hpp"
#include "netket_amd.h"

namespace nka {

// Augmented spin index u in [-1, N) (-1: the constant 1).  Row of P holding
// s~_u s~_u'.
__device__ __host__ inline int64_t qgt_spin_row(int u, int v, int N) {
  if (u == v) return 0;
  if (u < 0) return 1 + v;
  if (v < 0) return 1 + u;
  const int64_t i = u < v ? u : v, k = u < v ? v : u;
  return 1 + N + k * (k - 1) / 2 + i;
}
// Augmented hidden index w in [-1, M).  Row of Q holding t~_w t~_w'.
__device__ __host__ inline int64_t qgt_hidden_row(int w, int x, int M) {
  if (w < 0 && x < 0) return 0;
  if (w < 0) return 1 + x;
  if (x < 0) return 1 + w;
  const int64_t j = w < x ? w : x, l = w < x ? x : w;
  return 1 + M + l * (l + 1) / 2 + j;
}
// Largest e with e (e + 1) / 2 <= b.
__device__ inline int64_t tri_root(int64_t b) {
  int64_t e = (int64_t)((sqrt(8.0 * (double)b + 1.0) - 1.0) * 0.5);
  while ((e + 1) * (e + 2) / 2 <= b) ++e;
  while (e * (e + 1) / 2 > b) --e;
  return e;
}
// Position of parameter (u, w) in the flat vector, or -1 when it is not one.
__device__ inline int64_t qgt_param(int u, int w, const nka_rbm& m) {
  if (u < 0) return (w < 0 || m.bias_off < 0) ? -1 : m.bias_off + w;
  if (w < 0) return m.visible_off < 0 ? -1 : m.visible_off + u;
  return m.kernel_off + (int64_t)u * m.n_hidden + w;
}

// Rows of the sample dimension (padded), of P and of Q.
inline int64_t qgt_ldk(int64_t ns) { return (ns + 63) / 64 * 64; }
inline int64_t qgt_rows_p(const nka_rbm& m) { return 1 + (int64_t)m.n_visible + (int64_t)m.n_visible * (m.n_visible - 1) / 2; }
inline int64_t qgt_rows_q(const nka_rbm& m) { return 1 + (int64_t)m.n_hidden + (int64_t)m.n_hidden * (m.n_hidden + 1) / 2; }
inline int64_t qgt_round(int64_t b) { return (b + 255) / 256 * 256; }

// sT (N x ldk int8) = sigma^T as +-1, zero past the ns samples (nka_ntk.hip).
void launch_qgt_spins_t(const int8_t* sigma, int64_t ns, int N, int64_t ldk, int8_t* sT, hipStream_t s);

}  // namespace nka
