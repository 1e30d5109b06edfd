// Metropolis sweeps of FP64 RBMs with several chains per wavefront (semantics,
// rules and random streams as in nka_sampler.hip).
//
// A wavefront holds G chains, one per group of LPC = 64 / G lanes; lane gl of a
// group owns the hidden units gl + LPC jj.  The chains are sequential, so a
// proposal's latency and its FP64 instructions are what counts.  With
//   sum_j log_cosh(theta_j) = sum_j |theta_j| + log prod_j (1 + e^{-2|theta_j|}) - M log 2
// the acceptance test needs no logarithm at all: with P the product over a
// chain's units (at most 2^256) and A the change of sum |theta|,
//   u < exp(2 log psi' / psi + log n_diff / n_new)
//     <=>  u P0^2 n_new < exp(2 (A + visible)) P^2 n_diff,
// so a proposal costs one exponential per unit (20 instructions) and one for the
// test, where log_cosh took an exponential and a log1p of the library per unit.
// The sums and products over a group stay in the VALU (DPP and row swaps).  The
// local rule's site does not depend on the state, so its W row and bias are read
// one proposal ahead.
//
// Bound by the FP64 issue rate with many chains, by the serial latency of a
// proposal (about 800 cycles) with few.  Measured, against one exponential and
// one log1p of the library per unit and a draw per proposal: 4096 chains, 64
// sites, 128 hidden units, exchange, 576 proposals: 5.22 -> 0.85 ms (W, 64 KB, now
// staged in LDS as well); 16 chains, 16 sites and units, local rule, 1264
// proposals: 0.91 -> 0.45 ms.
#include "nka_sampler.hpp"

namespace nka {

// The logarithm out of line: it is off the common path (other powers than 2,
// and once per kept sweep), and inlined its constants would take the scalar
// registers that exp_f64's live in.
__device__ __attribute__((noinline)) double log_call(double x) { return log(x); }

template <int G, int JG, int RSG, bool EXCH>
__device__ __forceinline__ void group64_body(const nka_rbm& m, const SweepArgs& sa, int8_t* __restrict__ sigma,
                                             double* __restrict__ log_prob, int8_t* __restrict__ samples,
                                             double* __restrict__ lp_samples, int64_t* __restrict__ n_accepted,
                                             int bx) {
  constexpr int LPC = NKA_WAVE / G;
  extern __shared__ unsigned char smem[];
  const RbmView<double> v = rbm_view<double>(m);
  const int N = v.N, M = v.M;
  const int wid = threadIdx.x / NKA_WAVE, waves = blockDim.x / NKA_WAVE;
  const int lane = lane_id(), g = lane / LPC, gl = lane % LPC;
  // LDS: [W] [visible bias a] [cluster pairs] [spins of each chain]
  const size_t wbytes = pad16((size_t)N * M * sizeof(double));
  const double* W = (const double*)smem;
  double* a_s = (double*)(smem + wbytes);
  int32_t* cl_s = (int32_t*)(smem + wbytes + pad16((size_t)N * sizeof(double)));
  int8_t* xs = (int8_t*)cl_s + pad16((size_t)2 * sa.n_clusters * sizeof(int32_t)) + (wid * G + g) * pad16(N);
  for (int i = threadIdx.x; i < N; i += blockDim.x) a_s[i] = v.a ? v.a[i] : 0.0;
  for (int i = threadIdx.x; i < 2 * sa.n_clusters; i += blockDim.x) cl_s[i] = sa.clusters[i];
  stage_w<double>((double*)smem, v.W, N, M);  // ends with a workgroup barrier
  if ((bx * waves + wid) * G >= sa.C) return;  // whole wavefront past the last chain
  const int c_raw = (bx * waves + wid) * G + g;
  const bool live = c_raw < sa.C;              // groups past the last chain repeat it
  const int c = live ? c_raw : sa.C - 1;

  for (int i = gl; i < N; i += LPC) xs[i] = sigma[(int64_t)c * N + i];
  wave_lds_sync();
  // register slot jj of a lane holds hidden unit gl + LPC * ((jj + g) mod JG):
  // the rotation by the group index makes the groups of a wavefront read
  // different LDS bank ranges of their W rows in the same instruction
  // (a slot past the last unit holds 1e300, which no change moves and whose
  // factor 1 + e^{-2|theta|} is 1; it reads the last unit's weights)
  double th[JG];
  int jo[JG];
  double P0 = 1.0;
#pragma unroll
  for (int jj = 0; jj < JG; ++jj) {
    const int j = gl + LPC * ((jj + g) & (JG - 1));
    th[jj] = 1e300;
    jo[jj] = min(j, M - 1);
    if (j < M) {
      double acc = v.b ? v.b[j] : 0.0;
      for (int i = 0; i < N; ++i) {
        const double w = W[(size_t)i * M + j];
        acc += (xs[i] > 0) ? w : -w;
      }
      th[jj] = acc;
      P0 = fma(P0, exp_f64(-2.0 * fabs(acc)), P0);
    }
  }
  P0 = group_prod<LPC>(P0);
  const double pw = sa.machine_pow;
  // machine_pow log psi of the current state
  auto log_prob_now = [&]() {
    double part = 0.0;
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) part += gl + LPC * ((jj + g) & (JG - 1)) < M ? fabs(th[jj]) : 0.0;
    for (int i = gl; i < N; i += LPC) part += (xs[i] > 0) ? a_s[i] : -a_s[i];
    return pw * (group_sum<LPC>(part) + log_call(P0) - 0.69314718055994530942 * (double)M);
  };

  // cluster slots of this lane: cl = gl + LPC * r, r < RSG (RSG * LPC >= n_clusters)
  int cu[RSG], cv[RSG];
#pragma unroll
  for (int r = 0; r < RSG; ++r) {
    const int cl = gl + LPC * r;
    const bool ok = EXCH && cl < sa.n_clusters;
    cu[r] = ok ? cl_s[2 * cl] : -1;
    cv[r] = ok ? cl_s[2 * cl + 1] : -1;
  }

  int64_t nacc = 0;
  uint64_t q = sa.counter;
  if (sa.counter_dev) {
    const uint64_t cd = *sa.counter_dev;
    q = ((uint64_t)uniform_value<uint32_t>((uint32_t)(cd >> 32)) << 32) |
        (uint64_t)uniform_value<uint32_t>((uint32_t)cd);
  }
  DrawBlock<LPC> draws;
  draws.refill(q, (uint32_t)c, sa.k0, sa.k1);
  u32x4 rnd_next = draws.at(q, (uint32_t)c, sa.k0, sa.k1);
  // local rule: site, W row and bias of the next proposal
  int site_next = 0;
  double w_next[JG], a_next = 0.0;
  auto fetch = [&]() {
    site_next = (int)bounded(rnd_next.x, (uint32_t)N);
    a_next = a_s[site_next];
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) w_next[jj] = W[site_next * M + jo[jj]];
  };
  if (!EXCH) fetch();
  const int n_sweeps = sa.n_discard + sa.chain_length;
  for (int sw = 0; sw < n_sweeps; ++sw) {
    for (int p = 0; p < sa.sweep_size; ++p) {
      const u32x4 rnd = rnd_next;
      ++q;
      rnd_next = draws.at(q, (uint32_t)c, sa.k0, sa.k1);
      int s0, s1 = 0, n_diff = 1, n_new = 1;
      bool valid = true;
      double d[JG], vis;
      int8_t x0, x1 = 0;
      if (!EXCH) {
        s0 = site_next;
        x0 = xs[s0];
        const double f = x0 > 0 ? -2.0 : 2.0;
        vis = f * a_next;
#pragma unroll
        for (int jj = 0; jj < JG; ++jj) d[jj] = f * w_next[jj];
        fetch();
      } else {
        valid = group_exchange<LPC, RSG>(xs, cl_s, sa.n_clusters, cu, cv, g, rnd.x, s0, s1, n_diff, n_new);
        x0 = xs[s0];
        x1 = xs[s1];
        const double f0 = x0 > 0 ? -2.0 : 2.0, f1 = x1 > 0 ? -2.0 : 2.0;
        vis = f0 * a_s[s0] + f1 * a_s[s1];
#pragma unroll
        for (int jj = 0; jj < JG; ++jj) d[jj] = f0 * W[s0 * M + jo[jj]] + f1 * W[s1 * M + jo[jj]];
      }
      double A = 0.0, P = 1.0;
      double t[JG];
#pragma unroll
      for (int jj = 0; jj < JG; ++jj) {
        t[jj] = th[jj] + d[jj];
        A += fabs(t[jj]) - fabs(th[jj]);
        P = fma(P, exp_f64(-2.0 * fabs(t[jj])), P);
      }
      A = group_sum<LPC>(A) + vis;
      P = group_prod<LPC>(P);
      const double u = uniform01<double>(rnd);
      double lhs = P0 * P0, rhs = P * P, x = 2.0 * A;
      if (pw != 2.0) {
        lhs = rhs = 1.0;
        x = pw * (A + log_call(P / P0));
      }
      const bool acc = u * lhs * (double)n_new < exp_f64(x) * rhs * (double)n_diff;
      if (valid && acc) {
#pragma unroll
        for (int jj = 0; jj < JG; ++jj) th[jj] = t[jj];
        P0 = P;
        if (gl == 0) {
          xs[s0] = (int8_t)(-x0);
          if (EXCH) xs[s1] = (int8_t)(-x1);
        }
        ++nacc;
      }
      wave_lds_sync();
    }
    if (sw >= sa.n_discard && live) {
      const int k = sw - sa.n_discard;
      int8_t* dst = samples + ((int64_t)c * sa.chain_length + k) * N;
      for (int i = gl; i < N; i += LPC) dst[i] = xs[i];
    }
    if (sw >= sa.n_discard && lp_samples) {
      const double lp = log_prob_now();
      if (live && gl == 0) lp_samples[(int64_t)c * sa.chain_length + sw - sa.n_discard] = lp;
    }
  }
  const double lp = log_prob_now();
  if (live) {
    for (int i = gl; i < N; i += LPC) sigma[(int64_t)c * N + i] = xs[i];
    if (gl == 0) {
      log_prob[c] = lp;
      n_accepted[c] += nacc;
    }
  }
}

template <int G, int JG, int RSG, bool EXCH>
__global__ void __launch_bounds__(512) rbm_metropolis_group64_kernel(nka_rbm m, SweepArgs sa,
                                                                     int8_t* __restrict__ sigma,
                                                                     double* __restrict__ log_prob,
                                                                     int8_t* __restrict__ samples,
                                                                     double* __restrict__ lp_samples,
                                                                     int64_t* __restrict__ n_accepted) {
  group64_body<G, JG, RSG, EXCH>(m, sa, sigma, log_prob, samples, lp_samples, n_accepted, blockIdx.x);
}

// The same sweeps for a batch of jobs of one shape: blockIdx.y selects the job
// (its parameters, chains, outputs and random stream).
template <int G, int JG, int RSG, bool EXCH>
__global__ void __launch_bounds__(512) rbm_metropolis_group64_kernel_batched(const nka_sweep_job* __restrict__ jobs,
                                                                             SweepArgs sa) {
  const nka_sweep_job& j = jobs[blockIdx.y];
  SweepArgs s = sa;
  s.k0 = (uint32_t)j.seed;
  s.k1 = (uint32_t)(j.seed >> 32);
  s.counter = j.counter;
  s.counter_dev = j.counter_dev;
  group64_body<G, JG, RSG, EXCH>(j.model, s, j.sigma, (double*)j.log_prob, j.samples, (double*)j.log_prob_samples,
                                 j.n_accepted, blockIdx.x);
}

struct Group64 {
  const nka_rbm& m;
  const SweepArgs& sa;
  int8_t* sigma;
  double* lp;
  int8_t* smp;
  double* lps;
  int64_t* nacc;
  const nka_sweep_job* jobs;
  int n_jobs;
  int waves;
  size_t lds;
  hipStream_t s;

  template <int G, int JG, int RSG, bool EXCH>
  void run() const {
    const unsigned g = (unsigned)((sa.C + waves * G - 1) / (waves * G));
    if (jobs) {
      allow(rbm_metropolis_group64_kernel_batched<G, JG, RSG, EXCH>);
      hipLaunchKernelGGL((rbm_metropolis_group64_kernel_batched<G, JG, RSG, EXCH>), dim3(g, n_jobs),
                         dim3(64 * waves), lds, s, jobs, sa);
    } else {
      allow(rbm_metropolis_group64_kernel<G, JG, RSG, EXCH>);
      hipLaunchKernelGGL((rbm_metropolis_group64_kernel<G, JG, RSG, EXCH>), dim3(g), dim3(64 * waves), lds, s, m, sa,
                         sigma, lp, smp, lps, nacc);
    }
  }
  // dynamic LDS above the default 64 KB needs the function attribute
  template <class K>
  void allow(K kernel) const {
    if (lds > 64 * 1024)
      (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  }
  template <int G, int JG>
  void rule() const {
    const int need = (sa.n_clusters + NKA_WAVE / G - 1) / (NKA_WAVE / G);
    if (sa.rule != NKA_RULE_EXCHANGE) run<G, JG, 1, false>();
    else if (need <= 1) run<G, JG, 1, true>();
    else if (need <= 2) run<G, JG, 2, true>();
    else if (need <= 4) run<G, JG, 4, true>();
    else if (need <= 8) run<G, JG, 8, true>();
    else run<G, JG, 16, true>();
  }
  template <int G>
  void units() const {
    const int need = (m.n_hidden + NKA_WAVE / G - 1) / (NKA_WAVE / G);
    if (need <= 1) rule<G, 1>();
    else if (need <= 2) rule<G, 2>();
    else if (need <= 4) rule<G, 4>();
    else rule<G, 8>();
  }
};

// LDS of a workgroup: W, the visible bias, the clusters, a chain's spins.
static size_t group64_lds(const nka_rbm& m, const SweepArgs& sa, int waves, int G) {
  return pad16((size_t)m.n_visible * m.n_hidden * sizeof(double)) + pad16((size_t)m.n_visible * sizeof(double)) +
         pad16((size_t)2 * sa.n_clusters * sizeof(int32_t)) + (size_t)waves * G * pad16(m.n_visible);
}

// Chains per wavefront: 4 of 16 lanes when the units then fit one register slot
// (the shortest reduction), or when M <= 128 and there are chains enough for two
// such wavefronts per SIMD; else 2 of 32 lanes when M <= 256.  W goes to LDS:
// two workgroups of four wavefronts per CU while they fit, else one of eight.
// Weighted exchange, larger models and a W beyond 156 KB take a wavefront per
// chain (nka_sampler.hip).
bool launch_group64(const nka_rbm& m, const SweepArgs& sa, int8_t* sigma, double* lp, int8_t* smp, double* lps,
                    int64_t* nacc, const nka_sweep_job* jobs, int n_jobs, hipStream_t s) {
  if (sa.weights) return false;
  const bool four = m.n_hidden <= 16 || (m.n_hidden <= 128 && (int64_t)sa.C >= (int64_t)4 * 8 * device_cus());
  for (int G : {4, 2}) {
    if (G == 4 && !four) continue;
    const int lpc = NKA_WAVE / G;
    if (m.n_hidden > 8 * lpc) continue;
    if (sa.rule == NKA_RULE_EXCHANGE && sa.n_clusters > kMaxClusterSlots * lpc) continue;
    const int waves = group64_lds(m, sa, 4, G) <= 78 * 1024 ? 4 : 8;
    const size_t lds = group64_lds(m, sa, waves, G);
    if (lds > 156 * 1024) continue;
    const Group64 k{m, sa, sigma, lp, smp, lps, nacc, jobs, n_jobs, waves, lds, s};
    if (G == 4) k.units<4>();
    else k.units<2>();
    return true;
  }
  return false;
}

}  // namespace nka
