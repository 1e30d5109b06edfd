"""GPU parity of the Metropolis sampler: identical chains to the oracle on the
same Philox stream (FP64), and the sampled distribution vs exact |psi|^2."""

import numpy as np
import pytest
import torch

import netket_amd as nk
from oracle import operators as O
from oracle import rbm as orbm
from oracle import sampler as osamp

pytestmark = pytest.mark.gpu


def _model(N, alpha, dtype, seed, scale):
    model = nk.models.RBM(alpha=alpha, param_dtype=dtype)
    lay = model.layout(N)
    rng = np.random.default_rng(seed)
    flat_np = rng.normal(scale=scale, size=lay["n_params"]).astype(dtype)
    return model, torch.as_tensor(flat_np, device="cuda"), orbm.RBMParams(
        flat_np.astype(np.float64), N, lay["M"])


@pytest.mark.parametrize("N,n_down", [(10, None), (12, 6), (64, 32), (7, 3)])
def test_random_states_match_oracle(gpu, N, n_down):
    print(f"case random_states N={N} n_down={n_down}", flush=True)
    hi = nk.hilbert.Spin(0.5, N=N, total_sz=None if n_down is None else (N - 2 * n_down) / 2)
    sa = nk.sampler.MetropolisLocal(hi, n_chains=37)
    st = sa.init_state(None, None, seed=1234)
    ref = osamp.random_states(37, N, n_down, 1234, 0)
    np.testing.assert_array_equal(st.sigma.cpu().numpy(), ref)
    if n_down is not None:
        assert np.all((st.sigma.cpu().numpy() < 0).sum(axis=1) == n_down)


@pytest.mark.parametrize("rule,n_chains", [("local", 6), ("exchange", 6), ("local", 8192),
                                           ("exchange", 8192), ("exchange-weighted", 6),
                                           ("exchange-weighted", 8192)])
def test_chains_identical_to_oracle_fp64(gpu, rule, n_chains):
    # 8192 chains of a small model run four chains per wavefront, fewer run
    # two; weighted exchange (NN and NNN clusters, ExchangeRule probabilities
    # per distance) runs one chain per wavefront
    print(f"case chains {rule} n_chains={n_chains}", flush=True)
    N = 10
    model, flat, p = _model(N, 2, np.float64, 3, 0.4)
    g = nk.graph.Chain(N)
    weights = None
    if rule == "local":
        hi = nk.hilbert.Spin(0.5, N=N)
        sa = nk.sampler.MetropolisLocal(hi, n_chains=n_chains, sweep_size=7)
        clusters = None
    elif rule == "exchange":
        hi = nk.hilbert.Spin(0.5, N=N, total_sz=0)
        sa = nk.sampler.MetropolisExchange(hi, graph=g, n_chains=n_chains, sweep_size=7)
        clusters = sa.rule.clusters
    else:
        hi = nk.hilbert.Spin(0.5, N=N, total_sz=0)
        sa = nk.sampler.MetropolisExchange(hi, graph=g, d_max=2, probabilities=[1.0, 0.37],
                                           n_chains=n_chains, sweep_size=7)
        clusters, weights = sa.rule.clusters, sa.rule.weights
        rule = "exchange"
    st = sa.init_state(model, flat, seed=99)
    sigma0 = st.sigma.cpu().numpy().copy()
    counter0 = st.counter
    samples, st = sa.sample_fused(model, flat, st, 3, 9)
    # the oracle follows every chain of a small batch, and a spread of chains
    # (both ends, the first and last of a wavefront's group) of a large one
    ids = np.arange(n_chains) if n_chains <= 64 else np.array([0, 1, 2, 3, 4, 4095, 4096, 8190, 8191])
    ref, ref_sigma, ref_acc = osamp.metropolis(p, sigma0[ids], rule=rule, clusters=clusters, n_discard=3,
                                               chain_length=9, sweep_size=7, seed=99, counter=counter0,
                                               chain_ids=ids, weights=weights)
    np.testing.assert_array_equal(samples.cpu().numpy()[ids], ref)
    np.testing.assert_array_equal(st.sigma.cpu().numpy()[ids], ref_sigma)
    np.testing.assert_array_equal(st.n_accepted_proc.cpu().numpy()[ids], ref_acc)
    # log_prob of the chain state is 2 Re log psi of the final configurations
    np.testing.assert_allclose(st.log_prob.cpu().numpy()[ids], 2 * orbm.log_psi(p, ref_sigma), rtol=1e-12)


def _kl(counts, probs):
    q = counts / counts.sum()
    m = q > 0
    return float(np.sum(q[m] * np.log(q[m] / probs[m])))


@pytest.mark.parametrize("rule,dtype", [("local", np.float64), ("local", np.float32),
                                        ("exchange", np.float64), ("exchange", np.float32),
                                        ("exchange-weighted", np.float32)])
def test_distribution_matches_exact(gpu, rule, dtype):
    # sampled frequencies vs exact |psi|^2 (FullSumState semantics), KL divergence
    print(f"case distribution {rule} {np.dtype(dtype)}", flush=True)
    # weights small enough that |psi|^2 is not sharply multimodal, so chains
    # started from random states equilibrate within the discarded sweeps
    N = 8
    model, flat, p = _model(N, 1, dtype, 7, 0.25)
    if rule == "local":
        hi = nk.hilbert.Spin(0.5, N=N)
        sa = nk.sampler.MetropolisLocal(hi, n_chains=1024)
        states = O.states_all(N)
    elif rule == "exchange":
        hi = nk.hilbert.Spin(0.5, N=N, total_sz=0)
        sa = nk.sampler.MetropolisExchange(hi, graph=nk.graph.Chain(N), n_chains=1024)
        states = O.states_all(N, n_down=4)
    else:
        # distance-3 swaps tried 5x as often as nearest-neighbour ones
        hi = nk.hilbert.Spin(0.5, N=N, total_sz=0)
        sa = nk.sampler.MetropolisExchange(hi, graph=nk.graph.Chain(N), d_max=3, probabilities=[1.0, 2.0, 5.0],
                                           n_chains=1024)
        states = O.states_all(N, n_down=4)
    st = sa.init_state(model, flat, seed=5)
    samples, st = sa.sample_fused(model, flat, st, 100, 200)
    s = samples.cpu().numpy().reshape(-1, N)
    keys = O.state_index(s)
    order = np.argsort(O.state_index(states))
    skeys = O.state_index(states)[order]
    pos = np.searchsorted(skeys, keys)
    assert np.all(skeys[pos] == keys), "sample outside the Hilbert space"
    counts = np.bincount(pos, minlength=len(states)).astype(float)
    probs = orbm.exact_probability(p, states[order])
    kl = _kl(counts, probs)
    print(f"KL = {kl:.3e} over {len(states)} states, {s.shape[0]} samples", flush=True)
    # expected KL of an exact sampler ~ (K-1)/(2 n) = 6e-4 (local), 2e-4 (exchange)
    assert kl < 4e-3
    if rule != "local":
        assert np.all((s < 0).sum(axis=1) == N // 2)


@pytest.mark.parametrize("alpha", [300, 430, 500])
def test_distribution_matches_exact_wide_model(gpu, alpha):
    # FP32 models whose W exceeds the LDS budget take the local-rule kernel
    # that loads the next proposal's W row ahead and uses the exp2 product
    # form of the log-amplitude change (M = 2400: 40 units per lane,
    # M = 3440: 56, M = 4000: 64)
    print(f"case distribution wide local alpha={alpha}", flush=True)
    N = 8
    model, flat, p = _model(N, alpha, np.float32, 11, 0.05)
    hi = nk.hilbert.Spin(0.5, N=N)
    sa = nk.sampler.MetropolisLocal(hi, n_chains=1024)
    states = O.states_all(N)
    st = sa.init_state(model, flat, seed=6)
    samples, st = sa.sample_fused(model, flat, st, 100, 200)
    s = samples.cpu().numpy().reshape(-1, N)
    keys = O.state_index(s)
    order = np.argsort(O.state_index(states))
    skeys = O.state_index(states)[order]
    pos = np.searchsorted(skeys, keys)
    assert np.all(skeys[pos] == keys), "sample outside the Hilbert space"
    counts = np.bincount(pos, minlength=len(states)).astype(float)
    probs = orbm.exact_probability(p, states[order])
    kl = _kl(counts, probs)
    print(f"KL = {kl:.3e} over {len(states)} states, {s.shape[0]} samples", flush=True)
    assert kl < 4e-3
    # the chain's log_prob stays 2 log psi of its state (FP32 running sum)
    lp_ref = 2 * orbm.log_psi(p, st.sigma.cpu().numpy())
    np.testing.assert_allclose(st.log_prob.cpu().numpy(), lp_ref, rtol=1e-4, atol=1e-3)


def test_mcstate_sample_shapes_and_reset(gpu):
    N = 12
    hi = nk.hilbert.Spin(0.5, N=N)
    sa = nk.sampler.MetropolisLocal(hi, n_chains=16)
    vs = nk.vqs.MCState(sa, nk.models.RBM(alpha=1), n_samples=1008, n_discard_per_chain=16, seed=0)
    assert vs.chain_length == 63 and vs.n_samples == 1008
    s1 = vs.samples
    assert tuple(s1.shape) == (16, 63, N)
    assert vs.samples is s1
    vs.reset()
    s2 = vs.samples
    assert s2 is not s1
    acc = vs.sampler_state.acceptance
    assert 0.0 < acc <= 1.0


@pytest.mark.parametrize("rule,N,alpha,n_chains,power", [
    ("local", 16, 1, 5, 2.0),        # 16 units: four chains per wavefront, one unit a lane
    ("local", 17, 1, 7, 1.0),        # 17 units: two chains; another machine power
    ("exchange", 12, 5, 9, 2.0),     # 60 units, the last lanes without a second one
    ("exchange", 16, 16, 3, 3.0),    # 256 units, the most of the grouped kernel
    ("local", 100, 1, 33, 2.0),      # W of 80 KB: one workgroup of eight wavefronts per CU
    ("local", 10, 30, 4, 2.0),       # 300 units: one chain per wavefront
    ("exchange", 8, 40, 4, 1.0),
])
def test_fp64_chains_identical_to_oracle_over_sizes(gpu, rule, N, alpha, n_chains, power):
    # 12 sweeps of 9 proposals cross the runs of 16, 32 and 64 draws shared out
    # over a chain's lanes
    print(f"case fp64 chains {rule} N={N} M={alpha * N} chains={n_chains} power={power}", flush=True)
    model, flat, p = _model(N, alpha, np.float64, 11, 0.6 / np.sqrt(alpha * N))
    if rule == "local":
        sa = nk.sampler.MetropolisLocal(nk.hilbert.Spin(0.5, N=N), n_chains=n_chains, sweep_size=9,
                                        machine_pow=power)
        clusters = None
    else:
        sa = nk.sampler.MetropolisExchange(nk.hilbert.Spin(0.5, N=N, total_sz=0), graph=nk.graph.Chain(N),
                                           n_chains=n_chains, sweep_size=9, machine_pow=power)
        clusters = sa.rule.clusters
    st = sa.init_state(model, flat, seed=21)
    sigma0 = st.sigma.cpu().numpy().copy()
    counter0 = st.counter
    (samples, lps), st = sa.sample_fused(model, flat, st, 4, 8, return_log_probabilities=True)
    ref, ref_sigma, ref_acc = osamp.metropolis(p, sigma0, rule=rule, clusters=clusters, n_discard=4,
                                               chain_length=8, sweep_size=9, seed=21, counter=counter0,
                                               machine_pow=power)
    np.testing.assert_array_equal(samples.cpu().numpy(), ref)
    np.testing.assert_array_equal(st.sigma.cpu().numpy(), ref_sigma)
    np.testing.assert_array_equal(st.n_accepted_proc.cpu().numpy(), ref_acc)
    # log psi is a sum of N M + M terms rounded to 2^-53 of their size
    lp_ref = power * orbm.log_psi(p, ref.reshape(-1, N)).reshape(n_chains, 8)
    tol = 1e-12 * np.abs(lp_ref).max()
    np.testing.assert_allclose(lps.cpu().numpy(), lp_ref, rtol=0, atol=tol)
    np.testing.assert_allclose(st.log_prob.cpu().numpy(), lp_ref[:, -1], rtol=0, atol=tol)


@pytest.mark.parametrize("N,alpha,n_chains,sweep", [(130, 1, 5, 131), (150, 3, 9, 70), (200, 16, 4, 33)])
def test_wide_model_chains_carry_their_own_log_prob(gpu, N, alpha, n_chains, sweep):
    # W past LDS, unit counts that are no multiple of a wavefront (130 and 450:
    # the last slots partly or wholly past the end) or fill 50 slots exactly
    # (3200), odd sweeps (the two row buffers swap roles between sweeps): the
    # running log-probability is that of the final configuration, and a second
    # run repeats the chains
    print(f"case wide sampler N={N} M={alpha * N} chains={n_chains} sweep={sweep}", flush=True)
    model, flat, p = _model(N, alpha, np.float32, 13, 0.3 / np.sqrt(alpha * N))
    sa = nk.sampler.MetropolisLocal(nk.hilbert.Spin(0.5, N=N), n_chains=n_chains, sweep_size=sweep)
    out = []
    for _ in range(2):
        st = sa.init_state(model, flat, seed=3)
        samples, st = sa.sample_fused(model, flat, st, 2, 5)
        out.append(samples.cpu().numpy())
    np.testing.assert_array_equal(out[0], out[1])
    np.testing.assert_array_equal(st.sigma.cpu().numpy(), out[0][:, -1])
    assert st.n_accepted > 0
    ref = 2 * orbm.log_psi(p, st.sigma.cpu().numpy())
    # 7 sweeps of accumulated FP32 steps
    np.testing.assert_allclose(st.log_prob.cpu().numpy(), ref, rtol=0, atol=1e-4 * np.abs(ref).max())


@pytest.mark.parametrize("N,M,n_chains,sweep,power", [
    (16, 16, 3, 16, 2.0),        # two proposals per step
    (16, 16, 1030, 9, 2.0),      # more chains than SIMDs: one at a time
    (3, 5, 4, 7, 2.0),           # three sites: both proposals of a step often flip the same one
    (2, 64, 2, 5, 1.0),
    (33, 33, 5, 33, 2.0),        # odd sweeps end with a single proposal; spins in two words
    (70, 20, 2, 3, 2.0),
    (1100, 17, 2, 40, 2.0),      # W of 150 KB, spins over 35 lanes
])
def test_fp64_local_chains_two_proposals_per_step(gpu, N, M, n_chains, sweep, power):
    print(f"case fp64 pairs N={N} M={M} chains={n_chains} sweep={sweep} power={power}", flush=True)
    model, flat, p = _model(N, (M + 0.5) / N, np.float64, 12, 0.7 / np.sqrt(M))
    assert p.W.shape == (N, M)
    sa = nk.sampler.MetropolisLocal(nk.hilbert.Spin(0.5, N=N), n_chains=n_chains, sweep_size=sweep,
                                    machine_pow=power)
    st = sa.init_state(model, flat, seed=23)
    sigma0 = st.sigma.cpu().numpy().copy()
    counter0 = st.counter
    (samples, lps), st = sa.sample_fused(model, flat, st, 3, 4, return_log_probabilities=True)
    ref, ref_sigma, ref_acc = osamp.metropolis(p, sigma0, rule="local", clusters=None, n_discard=3,
                                               chain_length=4, sweep_size=sweep, seed=23, counter=counter0,
                                               machine_pow=power)
    np.testing.assert_array_equal(samples.cpu().numpy(), ref)
    np.testing.assert_array_equal(st.sigma.cpu().numpy(), ref_sigma)
    np.testing.assert_array_equal(st.n_accepted_proc.cpu().numpy(), ref_acc)
    lp_ref = power * orbm.log_psi(p, ref.reshape(-1, N)).reshape(n_chains, 4)
    tol = 1e-12 * np.abs(lp_ref).max()
    np.testing.assert_allclose(lps.cpu().numpy(), lp_ref, rtol=0, atol=tol)
    np.testing.assert_allclose(st.log_prob.cpu().numpy(), lp_ref[:, -1], rtol=0, atol=tol)
