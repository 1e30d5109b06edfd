// Parts shared by the RBM samplers (nka_sampler.hip: FP32 and the one-chain-per-
// wavefront kernels; nka_sampler64.hip: several FP64 chains per wavefront).
#pragma once

#include "nka_rbm.hpp"

namespace nka {

constexpr int kMaxClusterSlots = 16;  // clusters per lane: n_clusters <= 1024

struct SweepArgs {
  int rule;
  const int32_t* clusters;
  int n_clusters;
  const uint32_t* weights;      // exchange: integer weight per cluster (NULL: uniform)
  int C, sweep_size, n_discard, chain_length;
  double machine_pow;
  uint32_t k0, k1;
  uint64_t counter;
  const uint64_t* counter_dev;  // when set, the counter is read from device memory
};

// Sum (product) over the LPC lanes of this lane's group (LPC = 16 or 32), in
// every lane; the partner lanes of a step add the same two operands.
template <int LPC, class T>
__device__ inline T group_sum(T v) {
  v = row_sum(v);
  if (LPC == 32) {
    T w = v;
    swap_rows16(v, w);
    v += w;
  }
  return v;
}
template <int LPC, class T>
__device__ inline T group_prod(T v) {
  v = row_prod(v);
  if (LPC == 32) {
    T w = v;
    swap_rows16(v, w);
    v *= w;
  }
  return v;
}

// One exchange proposal of this group's chain (spins xs, group g of LPC lanes;
// lane gl holds the clusters gl + LPC r in cu[r], cv[r], -1 for none; cl_s all
// clusters in LDS): the sites of the k-th differing cluster, k from the draw,
// the number of differing clusters (0: no move, returns false) and their number
// after the swap (at least 1).
template <int LPC, int RSG>
__device__ __forceinline__ bool group_exchange(const int8_t* xs, const int32_t* cl_s, int n_clusters,
                                               const int (&cu)[RSG], const int (&cv)[RSG], int g, uint32_t draw,
                                               int& s0, int& s1, int& n_diff, int& n_new) {
  constexpr uint64_t GMASK = (1ull << LPC) - 1ull;
  // the differing clusters as a bit set in cluster order: cluster cl = gl +
  // LPC * r is bit cl % 64 of word cl / 64
  constexpr int NW = (RSG * LPC + 63) / 64;
  uint64_t word[NW];
  int8_t xu[RSG], xv[RSG];
#pragma unroll
  for (int w = 0; w < NW; ++w) word[w] = 0;
#pragma unroll
  for (int r = 0; r < RSG; ++r) {
    xu[r] = cu[r] >= 0 ? xs[cu[r]] : (int8_t)0;
    xv[r] = cu[r] >= 0 ? xs[cv[r]] : (int8_t)0;
    const uint64_t gbits = (__ballot(xu[r] != xv[r]) >> (g * LPC)) & GMASK;
    word[(LPC * r) / 64] |= gbits << ((LPC * r) % 64);
  }
  n_diff = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) n_diff += __popcll(word[w]);
  const bool valid = n_diff > 0;
  int k = (int)bounded(draw, (uint32_t)max(n_diff, 1));
  int sel = 0;
  bool found = false;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int cnt = __popcll(word[w]);
    if (!found && k < cnt) {
      sel = 64 * w + kth_set_bit(word[w], k);
      found = true;
    } else if (!found) {
      k -= cnt;
    }
  }
  if (!valid || sel >= n_clusters) sel = 0;
  s0 = cl_s[2 * sel];
  s1 = cl_s[2 * sel + 1];
  // differing clusters after the swap (sigma'_u = sigma_v, sigma'_v = sigma_u)
  const int8_t y0 = xs[s0], y1 = xs[s1];
  n_new = 0;
#pragma unroll
  for (int r = 0; r < RSG; ++r) {
    const int a = cu[r], bb = cv[r];
    const int8_t xa = a == s0 ? y1 : (a == s1 ? y0 : xu[r]);
    const int8_t xb = bb == s0 ? y1 : (bb == s1 ? y0 : xv[r]);
    n_new += __popcll((__ballot(a >= 0 && xa != xb) >> (g * LPC)) & GMASK);
  }
  n_new = max(n_new, 1);
  return valid;
}

// Several FP64 chains per wavefront (nka_sampler64.hip); false when the model
// or the rule does not fit it.
bool launch_group64(const nka_rbm& m, const SweepArgs& sa, int8_t* sigma, double* lp, int8_t* smp, double* lps,
                    int64_t* nacc, const nka_sweep_job* jobs, int n_jobs, hipStream_t s);
// FP32 local-rule sweeps with W in the caches (nka_sampler_wide.hip).
void launch_wide(const nka_rbm& m, const SweepArgs& sa, int8_t* sigma, float* lp, int8_t* smp, float* lps,
                 int64_t* nacc, const nka_sweep_job* jobs, int n_jobs, hipStream_t s);
int device_cus();

}  // namespace nka
