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
// Bound by the vector units with many chains (79% busy; 333 instructions per proposal
// of two chains with four units a lane, a third of them exponentials, the rest the
// choice of the exchange, the draws and the reductions), by the serial latency of a
// proposal (about 800 cycles) with few.  Measured, against one exponential and
// one log1p of the library per unit and a draw per proposal: 4096 chains, 64
// sites, 128 hidden units, exchange, 576 proposals: 5.22 -> 0.81 ms (W, 64 KB, now
// staged in LDS as well); 16 chains, 16 sites and units, local rule, 1264
// proposals: 0.91 -> 0.36 ms (two proposals per step, see below).
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
      P0 = fma(P0, exp_m2abs(acc), P0);
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
        P = fma(P, exp_m2abs(t[jj]), P);
      }
      A = group_sum<LPC>(A) + vis;
      P = group_prod<LPC>(P);
      const double u = uniform01<double>(rnd);
      double lhs = P0 * P0, rhs = P * P, x = 2.0 * A;
      if (pw != 2.0) {
        lhs = rhs = 1.0;
        x = pw * (A + log_call(P / P0));
      }
      // (both sides carry a few roundings of the products; the exponential's is one more)
      const bool acc = u * lhs * (double)n_new < exp_f64<false>(x) * rhs * (double)n_diff;
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

// Local rule with few chains: two proposals per step.
//
// One chain per wavefront.  While proposal q is tested (lanes 0-15), q + 1 is
// tested for both outcomes of q (lanes 16-31: q rejected; 32-47: q accepted), each
// with the operations that it would see one after the other; the two decisions are
// then taken together.  The serial chain of a test (W row, exponentials, product,
// comparison) is what bounds few chains, and it is paid once per two proposals.  The
// spins are bits in a register (lane l: sites 32 l ..), so that no LDS round trip
// lies between a decision and the next test.
// 16 chains, 16 sites and units, 1264 proposals: 0.36 ms, against 0.46 one at a time.
template <int JG>
__device__ __forceinline__ void pair64_body(const nka_rbm& m, const SweepArgs& sa, int8_t* __restrict__ sigma,
                                            double* __restrict__ log_prob, int8_t* __restrict__ samples,
                                            double* __restrict__ lp_samples, int64_t* __restrict__ n_accepted, int bx) {
  constexpr int LPC = 16;
  extern __shared__ unsigned char smem[];
  const RbmView<double> v = rbm_view<double>(m);
  const int N = v.N, M = v.M;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / NKA_WAVE), waves = blockDim.x / NKA_WAVE;
  const int lane = lane_id(), e = lane >> 4, gl = lane & 15;
  const double* W = (const double*)smem;
  double* a_s = (double*)(smem + pad16((size_t)N * M * sizeof(double)));
  for (int i = threadIdx.x; i < N; i += blockDim.x) a_s[i] = v.a ? v.a[i] : 0.0;
  stage_w<double>((double*)smem, v.W, N, M);  // ends with a workgroup barrier
  const int c = bx * waves + wid;
  if (c >= sa.C) return;

  uint32_t xb = 0;
  for (int i0 = 0; i0 < N; i0 += NKA_WAVE) {
    const uint64_t up = __ballot(i0 + lane < N && sigma[(int64_t)c * N + min(i0 + lane, N - 1)] > 0);
    if (lane == i0 / 32) xb = (uint32_t)up;
    if (lane == i0 / 32 + 1) xb = (uint32_t)(up >> 32);
  }
  auto spin_up = [&](int i) { return ((uint32_t)__builtin_amdgcn_readlane((int)xb, i >> 5) >> (i & 31)) & 1u; };
  // unit gl + 16 jj (a slot past the last holds 1e300, as above)
  double th[JG], P0 = 1.0;
  int jo[JG];
#pragma unroll
  for (int jj = 0; jj < JG; ++jj) {
    const int j = gl + LPC * jj;
    th[jj] = 1e300;
    jo[jj] = min(j, M - 1);
    if (j < M) {
      double acc = v.b ? v.b[j] : 0.0;
      for (int i = 0; i < N; ++i) {
        const double w = W[(size_t)i * M + j];
        acc += spin_up(i) ? w : -w;
      }
      th[jj] = acc;
      P0 = fma(P0, exp_m2abs(acc), P0);
    }
  }
  P0 = group_prod<LPC>(P0);
  const double pw = sa.machine_pow;
  auto log_prob_now = [&]() {
    double part = 0.0;
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) part += gl + LPC * jj < M ? fabs(th[jj]) : 0.0;
    for (int i0 = 0; i0 < N; i0 += LPC) {
      const int i = i0 + gl;
      const uint32_t w = (uint32_t)__shfl((int)xb, min(i, N - 1) >> 5);
      part += i < N ? ((w >> (i & 31)) & 1u ? a_s[i] : -a_s[i]) : 0.0;
    }
    return pw * (group_sum<LPC>(part) + log_call(P0) - 0.69314718055994530942 * (double)M);
  };

  int64_t nacc = 0;
  uint64_t q = sa.counter;
  if (sa.counter_dev) {
    const uint64_t cd = *sa.counter_dev;
    q = ((uint64_t)uniform_value<uint32_t>((uint32_t)(cd >> 32)) << 32) |
        (uint64_t)uniform_value<uint32_t>((uint32_t)cd);
  }
  DrawBlock<NKA_WAVE> draws;
  draws.refill(q, (uint32_t)c, sa.k0, sa.k1);
  // the next two proposals' draws, sites, W rows and visible biases
  u32x4 r0n, r1n;
  int s0n, s1n;
  double w0n[JG], w1n[JG], a0n, a1n;
  auto fetch = [&]() __attribute__((always_inline)) {
    r0n = draws.at(q, (uint32_t)c, sa.k0, sa.k1);
    r1n = draws.at(q + 1, (uint32_t)c, sa.k0, sa.k1);
    s0n = __builtin_amdgcn_readfirstlane((int)bounded(r0n.x, (uint32_t)N));
    s1n = __builtin_amdgcn_readfirstlane((int)bounded(r1n.x, (uint32_t)N));
    a0n = a_s[s0n];
    a1n = a_s[s1n];
#pragma unroll
    for (int jj = 0; jj < JG; ++jj) {
      w0n[jj] = W[s0n * M + jo[jj]];
      w1n[jj] = W[s1n * M + jo[jj]];
    }
  };
  fetch();
  const int n_sweeps = sa.n_discard + sa.chain_length;
  for (int sw = 0; sw < n_sweeps; ++sw) {
    for (int p = 0; p < sa.sweep_size; p += 2) {
      const bool two = p + 1 < sa.sweep_size;
      const u32x4 rnd = e == 0 ? r0n : r1n;
      const int s0 = s0n, s1 = s1n;
      // x' - x of a site; the second site's after the first was accepted
      const double f0 = spin_up(s0) ? -2.0 : 2.0, f1 = spin_up(s1) ? -2.0 : 2.0;
      const double f1a = s0 == s1 ? -f1 : f1;
      const double fe = e == 2 ? f1a : f1;
      const double vis = e == 0 ? f0 * a0n : fe * a1n;
      double A = 0.0, P = 1.0, u[JG], w1[JG];
#pragma unroll
      for (int jj = 0; jj < JG; ++jj) {
        u[jj] = th[jj] + f0 * w0n[jj];
        w1[jj] = w1n[jj];
        const double from = e == 2 ? u[jj] : th[jj];
        const double t = e == 0 ? u[jj] : from + fe * w1[jj];
        A += fabs(t) - fabs(from);
        P = fma(P, exp_m2abs(t), P);
      }
      q += two ? 2 : 1;
      fetch();
      A = group_sum<LPC>(A) + vis;
      P = group_prod<LPC>(P);
      auto lane_value = [](double x, int l) {
        return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                                __builtin_amdgcn_readlane(__double2loint(x), l));
      };
      const double Pq = lane_value(P, 0);
      const double Pe = e == 2 ? Pq : P0;
      double lhs = Pe * Pe, rhs = P * P, x = 2.0 * A;
      if (pw != 2.0) {
        lhs = rhs = 1.0;
        x = pw * (A + log_call(P / Pe));
      }
      const uint64_t acc = __ballot(uniform01<double>(rnd) * lhs < exp_f64<false>(x) * rhs);
      const bool acc0 = acc & 1ull;
      const bool acc1 = two && (acc >> (acc0 ? 32 : 16) & 1ull);
      if (acc0) {
#pragma unroll
        for (int jj = 0; jj < JG; ++jj) th[jj] = u[jj];
        P0 = Pq;
        xb ^= lane == s0 >> 5 ? 1u << (s0 & 31) : 0u;
        ++nacc;
      }
      if (acc1) {
        const double f = acc0 ? f1a : f1;
#pragma unroll
        for (int jj = 0; jj < JG; ++jj) th[jj] += f * w1[jj];
        P0 = lane_value(P, acc0 ? 32 : 16);
        xb ^= lane == s1 >> 5 ? 1u << (s1 & 31) : 0u;
        ++nacc;
      }
    }
    if (sw >= sa.n_discard) {
      const int k = sw - sa.n_discard;
      int8_t* dst = samples + ((int64_t)c * sa.chain_length + k) * N;
      for (int i0 = 0; i0 < N; i0 += NKA_WAVE) {
        const int i = i0 + lane;
        const uint32_t w = (uint32_t)__shfl((int)xb, min(i, N - 1) >> 5);
        if (i < N) dst[i] = (w >> (i & 31)) & 1u ? (int8_t)1 : (int8_t)-1;
      }
      if (lp_samples) {
        const double lp = log_prob_now();
        if (lane == 0) lp_samples[(int64_t)c * sa.chain_length + k] = lp;
      }
    }
  }
  const double lp = log_prob_now();
  for (int i0 = 0; i0 < N; i0 += NKA_WAVE) {
    const int i = i0 + lane;
    const uint32_t w = (uint32_t)__shfl((int)xb, min(i, N - 1) >> 5);
    if (i < N) sigma[(int64_t)c * N + i] = (w >> (i & 31)) & 1u ? (int8_t)1 : (int8_t)-1;
  }
  if (lane == 0) {
    log_prob[c] = lp;
    n_accepted[c] += nacc;
  }
}

template <int JG>
__global__ void __launch_bounds__(256) rbm_metropolis_pair64_kernel(nka_rbm m, SweepArgs sa, int8_t* __restrict__ sigma,
                                                                    double* __restrict__ log_prob,
                                                                    int8_t* __restrict__ samples,
                                                                    double* __restrict__ lp_samples,
                                                                    int64_t* __restrict__ n_accepted) {
  pair64_body<JG>(m, sa, sigma, log_prob, samples, lp_samples, n_accepted, blockIdx.x);
}
template <int JG>
__global__ void __launch_bounds__(256) rbm_metropolis_pair64_kernel_batched(const nka_sweep_job* __restrict__ jobs,
                                                                            SweepArgs sa) {
  const nka_sweep_job& j = jobs[blockIdx.y];
  SweepArgs s = sa;
  s.k0 = (uint32_t)j.seed;
  s.k1 = (uint32_t)(j.seed >> 32);
  s.counter = j.counter;
  s.counter_dev = j.counter_dev;
  pair64_body<JG>(j.model, s, j.sigma, (double*)j.log_prob, j.samples, (double*)j.log_prob_samples, j.n_accepted,
                  blockIdx.x);
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
  template <int JG>
  void pair() const {
    const unsigned g = (unsigned)((sa.C + waves - 1) / waves);
    if (jobs) {
      allow(rbm_metropolis_pair64_kernel_batched<JG>);
      hipLaunchKernelGGL((rbm_metropolis_pair64_kernel_batched<JG>), dim3(g, n_jobs), dim3(64 * waves), lds, s, jobs,
                         sa);
    } else {
      allow(rbm_metropolis_pair64_kernel<JG>);
      hipLaunchKernelGGL((rbm_metropolis_pair64_kernel<JG>), dim3(g), dim3(64 * waves), lds, s, m, sa, sigma, lp, smp,
                         lps, nacc);
    }
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
  // two proposals per step while every chain of a job has a SIMD of its own and its
  // units fit four a lane (16 units: 1.30x at 16 chains, 1.16x at 1024, 0.97x at 2048;
  // 64 units: 1.07x, 1.01x, 0.75x).  The kernels add a chain's units in different
  // orders, so the choice looks at one job alone: a batched job's chains are those that
  // it has by itself.
  if (sa.rule == NKA_RULE_LOCAL && m.n_hidden <= 64 && m.n_visible <= 32 * NKA_WAVE && sa.C <= 4 * device_cus()) {
    const size_t lds = pad16((size_t)m.n_visible * m.n_hidden * sizeof(double)) +
                       pad16((size_t)m.n_visible * sizeof(double));
    if (lds <= 156 * 1024) {
      const Group64 k{m, sa, sigma, lp, smp, lps, nacc, jobs, n_jobs, 4, lds, s};
      if (m.n_hidden <= 16) k.pair<1>();
      else if (m.n_hidden <= 32) k.pair<2>();
      else k.pair<4>();
      return true;
    }
  }
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
