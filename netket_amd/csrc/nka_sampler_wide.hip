// Local-rule Metropolis sweeps of FP32 RBMs whose W does not fit in LDS
// (semantics and random streams as in nka_sampler.hip).
//
// One wavefront per chain, lane l owning the units j = l + 64 jj.  The site of a
// local-rule proposal does not depend on the state, so the W row of the next
// proposal is loaded one proposal ahead and its cache latency overlaps the
// current one; two row buffers take turns.  The change of log psi uses
//   sum_j [lc(t_j) - lc(theta_j)] = (1/kappa) sum_j (|t'_j| - |theta'_j|)
//                                  + ln2 log2( prod_j (1 + 2^-|t'_j|) / P0 )
// (lc(t) = |t| + log(1 + e^{-2|t|}) - log 2, t' = kappa t, kappa = 2/ln 2):
// one exp2 per unit instead of an exp and a log.  Each lane keeps theta' of
// its units and 1/P0 of its product (< 2^64 over at most 64 units); an
// accepted move replaces both by the proposal's.
//
// A row is read through a buffer descriptor of its M values: lanes past the last
// unit read zero, so no unit needs a bounds check, and the slots' offsets are
// scalar.  Units per lane come in steps of two (a slot past the last unit costs as
// much as a real one).  Bound by the vector unit (92% busy): five instructions per unit, one of
// them an exp2.  8192 chains, 400 sites, 3200 units, 3600
// proposals: 45.3 -> 22.6 to 25.1 ms over cards, against a bounds check per load, one row buffer copied to the
// other after each proposal, a draw per lane and units in steps of eight.
#include "nka_sampler.hpp"

namespace nka {

constexpr float kKappaS = 2.8853900817779268f;    // 2 / ln 2
constexpr float kLn2S = 0.69314718055994531f;

// (three wavefronts per SIMD up to 50 units per lane: 168 registers each, at the
// cost of a few spills off the loop at 50; 24.2 -> 22.6 ms there)
template <int JL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(JL <= 50 ? 3 : 2)))
rbm_metropolis_wide_kernel(nka_rbm m, SweepArgs sa, int8_t* __restrict__ sigma, float* __restrict__ log_prob,
                           int8_t* __restrict__ samples, float* __restrict__ lp_samples,
                           int64_t* __restrict__ n_accepted, const nka_sweep_job* __restrict__ jobs) {
  if (jobs) {
    // one of a batch of jobs of this shape: its parameters, chains, outputs and
    // random stream
    const nka_sweep_job& j = jobs[blockIdx.y];
    m = j.model;
    sa.k0 = (uint32_t)j.seed;
    sa.k1 = (uint32_t)(j.seed >> 32);
    sa.counter = j.counter;
    sa.counter_dev = j.counter_dev;
    sigma = j.sigma;
    log_prob = (float*)j.log_prob;
    samples = j.samples;
    lp_samples = (float*)j.log_prob_samples;
    n_accepted = j.n_accepted;
  }
  extern __shared__ unsigned char smem[];
  const RbmView<float> v = rbm_view<float>(m);
  const int N = v.N, M = v.M;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / NKA_WAVE), waves = blockDim.x / NKA_WAVE;
  const int lane = lane_id();
  int8_t* xs = (int8_t*)smem + wid * pad16(N);
  const int c = blockIdx.x * waves + wid;
  if (c >= sa.C) return;
  for (int i = lane; i < N; i += NKA_WAVE) xs[i] = sigma[(int64_t)c * N + i];
  wave_lds_sync();

  auto load_row = [&](int site, float (&w)[JL]) __attribute__((always_inline)) {
    const uint64_t addr = (uint64_t)(v.W + (size_t)site * M);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)addr);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(addr >> 32));
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0, M * 4, 0x00020000);
    // (an opaque lane offset: the slots' constant parts then stay immediate
    // offsets of the loads instead of being kept in registers over the sweep)
    int off = lane * 4;
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int jj = 0; jj < JL; ++jj)
      w[jj] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off + jj * 256, 0, 0));
  };
  // theta of this lane's units: all JL loads of a row in flight per site
  float th[JL], wa[JL], wb[JL];
#pragma unroll
  for (int jj = 0; jj < JL; ++jj) {
    const int j = lane + NKA_WAVE * jj;
    th[jj] = (j < M && v.b) ? v.b[j] : 0.0f;
  }
  for (int i = 0; i < N; ++i) {
    const bool up = xs[i] > 0;
    load_row(i, wa);
#pragma unroll
    for (int jj = 0; jj < JL; ++jj) th[jj] += up ? wa[jj] : -wa[jj];
  }
  const float pw = (float)sa.machine_pow;
  float lcs = 0.0f, P0 = 1.0f;
#pragma unroll
  for (int jj = 0; jj < JL; ++jj) {
    lcs += lane + NKA_WAVE * jj < M ? log_cosh<float>(th[jj]) : 0.0f;
    th[jj] *= kKappaS;
    P0 = fmaf(P0, __builtin_amdgcn_exp2f(-fabsf(th[jj])), P0);
  }
  float rP0 = 1.0f / P0;
  float lp = pw * (wave_sum(lcs) + visible_term<float>(xs, v.a, N));

  int64_t nacc = 0;
  uint64_t q = sa.counter;
  if (sa.counter_dev) {
    const uint64_t cd = *sa.counter_dev;
    q = ((uint64_t)uniform_value<uint32_t>((uint32_t)(cd >> 32)) << 32) |
        (uint64_t)uniform_value<uint32_t>((uint32_t)cd);
  }
  DrawBlock<NKA_WAVE> draws;
  draws.refill(q, (uint32_t)c, sa.k0, sa.k1);
  u32x4 rnd_next = draws.at(q, (uint32_t)c, sa.k0, sa.k1);
  int site_next = (int)bounded(rnd_next.x, (uint32_t)N);
  load_row(site_next, wa);
  // one proposal: its row is in w; the next one's goes to wn
  auto propose = [&](float (&w)[JL], float (&wn)[JL]) __attribute__((always_inline)) {
    const u32x4 rnd = rnd_next;
    const int site = site_next;
    ++q;
    rnd_next = draws.at(q, (uint32_t)c, sa.k0, sa.k1);
    site_next = (int)bounded(rnd_next.x, (uint32_t)N);
    load_row(site_next, wn);
    const bool up = xs[site] > 0;
    const float g = up ? -2.0f * kKappaS : 2.0f * kKappaS;
    float A = 0.0f, P = 1.0f;
#pragma unroll
    for (int jj = 0; jj < JL; ++jj) {
      const float t = fmaf(g, w[jj], th[jj]);
      A += fabsf(t) - fabsf(th[jj]);
      P = fmaf(P, __builtin_amdgcn_exp2f(-fabsf(t)), P);
    }
    float delta = wave_sum(A * (1.0f / kKappaS) + kLn2S * __builtin_amdgcn_logf(P * rP0));
    if (v.a) delta += up ? -2.0f * v.a[site] : 2.0f * v.a[site];
    delta = uniform_value<float>(delta);
    const float u = uniform_value<float>(uniform01<float>(rnd));
    if (u < exp_t<float>(pw * delta)) {
      // recompute t rather than keep it live through the reduction (an
      // opaque copy of g stops the compiler from reusing the values)
      float gr = g;
      asm volatile("" : "+v"(gr));
#pragma unroll
      for (int jj = 0; jj < JL; ++jj) th[jj] = fmaf(gr, w[jj], th[jj]);
      rP0 = 1.0f / P;
      if (lane == 0) xs[site] = (int8_t)(-xs[site]);
      lp += pw * delta;
      ++nacc;
      wave_lds_sync();
    }
  };
  const int n_sweeps = sa.n_discard + sa.chain_length;
  for (int sw = 0; sw < n_sweeps; ++sw) {
    int p = 0;
    for (; p + 1 < sa.sweep_size; p += 2) {
      propose(wa, wb);
      propose(wb, wa);
    }
    if (p < sa.sweep_size) {
      propose(wa, wb);
#pragma unroll
      for (int jj = 0; jj < JL; ++jj) wa[jj] = wb[jj];
    }
    if (sw >= sa.n_discard) {
      const int t = sw - sa.n_discard;
      int8_t* dst = samples + ((int64_t)c * sa.chain_length + t) * N;
      for (int i = lane; i < N; i += NKA_WAVE) dst[i] = xs[i];
      if (lp_samples && lane == 0) lp_samples[(int64_t)c * sa.chain_length + t] = lp;
    }
  }
  for (int i = lane; i < N; i += NKA_WAVE) sigma[(int64_t)c * N + i] = xs[i];
  if (lane == 0) {
    log_prob[c] = lp;
    n_accepted[c] += nacc;
  }
}

template <int JL>
static void launch_wide_jl(const nka_rbm& m, const SweepArgs& sa, int8_t* sigma, float* lp, int8_t* smp, float* lps,
                           int64_t* nacc, const nka_sweep_job* jobs, int n_jobs, hipStream_t s) {
  if constexpr (JL > 2) {
    if (m.n_hidden <= (JL - 2) * NKA_WAVE) {
      launch_wide_jl<JL - 2>(m, sa, sigma, lp, smp, lps, nacc, jobs, n_jobs, s);
      return;
    }
  }
  constexpr int waves = 4;
  const unsigned g = (unsigned)((sa.C + waves - 1) / waves);
  hipLaunchKernelGGL(rbm_metropolis_wide_kernel<JL>, dim3(g, jobs ? n_jobs : 1), dim3(64 * waves),
                     waves * pad16(m.n_visible), s, m, sa, sigma, lp, smp, lps, nacc, jobs);
}

void launch_wide(const nka_rbm& m, const SweepArgs& sa, int8_t* sigma, float* lp, int8_t* smp, float* lps,
                 int64_t* nacc, const nka_sweep_job* jobs, int n_jobs, hipStream_t s) {
  launch_wide_jl<kMaxJL>(m, sa, sigma, lp, smp, lps, nacc, jobs, n_jobs, s);
}

}  // namespace nka
