"""Launches on batches that fit the chip (k_resident, up to 4096 worlds: one world on two waves up to 1024,
then two per wave) against the work-queue form (k_rollout, k_physics), which the fenced hand-over keeps at
every size: every output, the final state and the contact histogram bit for bit. The two forms share the
physics, and the policy's sums run in the same order on the vector ALUs as on v_mfma_f32_16x16x4f32, so the
tolerance is zero. Each case asserts the form that it is about."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g1():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import g1env
    return g1env


def _form(N):
    """The form of a batch at the default hand-over on the 256 CUs of an MI355X."""
    return "duo" if N <= 1024 else "pair" if N <= 4096 else "queue"


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


# the smallest batches; both sides of two waves per world and of two worlds per wave (odd counts; 4097 worlds
# take the queue with either hand-over); layers of one to eight row blocks, ragged widths, one to three hidden
# layers; a horizon of zero
@pytest.mark.parametrize("N,H,S,hidden,act,given", [
    (1, 3, 10, (256, 256), 0, False), (3, 2, 4, (17, 1), 1, True), (1023, 2, 5, (200, 72), 1, False),
    (1024, 2, 5, (256, 256), 0, True), (1025, 2, 5, (512, 512, 256), 1, True), (2047, 2, 4, (300,), 0, False),
    (4095, 2, 4, (64, 513 - 1, 130), 0, False), (4096, 3, 3, (256, 256), 0, False), (4097, 2, 3, (256, 256), 0, False),
    (4097, 2, 3, (300, 40), 1, False), (40, 0, 10, (128, 65), 1, False),
    (130, 12, 10, (256, 256), 0, False), (512, 3, 10, (256, 256), 0, True), (513, 3, 10, (256, 256), 0, True)])
def test_resident_rollout_equals_work_queue(g1, N, H, S, hidden, act, given):
    import configs
    import torch
    rng = np.random.default_rng(N + H)
    qp, qv, pa, steps = configs.reset_states(rng, N)
    qv = rng.normal(0, 0.3, qv.shape).astype(np.float32)
    pa = rng.normal(0, 0.3, pa.shape).astype(np.float32)
    steps[::5] = 998        # time-outs and auto-resets inside the horizon
    W = _dev(configs.policy_init(rng, hidden=hidden))
    mean, var = _dev(rng.normal(0, 0.1, 100).astype(np.float32)), _dev(rng.uniform(0.5, 2.0, 100).astype(np.float32))
    an, rn = (_dev(x) for x in configs.rollout_noise(rng, H, N)) if given else (None, None)
    got = []
    for fences in (0, 1):
        with g1.Env(N, substeps=S, pgs_iters=8, seed=9) as env:
            env.set_policy(hidden, act)
            env.set_handover(fences)
            assert env.launch_form() == ("queue" if fences else _form(N))
            env.set_state(qp, qv, pa, steps)
            env.ncon_hist(enable=True)
            out = []
            for _ in range(2):   # the second continues from the first's state and noise counters
                tr = g1.Trajectory(H, N)
                for t in tr.tensors():
                    t.fill_(7.0)
                tr.run(env, W, mean, var, an, rn)
                torch.cuda.synchronize()
                out += [tr.numpy()[f].view(np.uint32) for f in tr.FIELDS]
            got.append(out + [x.view(np.uint32) for x in env.get_state()] + [env.ncon_hist(enable=False)])
            assert env.check() == 0
    for i, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), i
    assert H == 0 or (got[0][5] != 0).any()   # some world finished


@pytest.mark.parametrize("hidden,act", [((256, 256), 0), ((256, 256), 1), ((512, 512, 256), 1)])
@pytest.mark.parametrize("N", [64, 1030])
@pytest.mark.parametrize("scale", ["wide", "subnormal", "huge"])
def test_policy_sums_equal_mfma_over_the_range_of_fp32(g1, scale, N, hidden, act):
    """The resident policy's fma chains against the MFMA tiles' sums where their order and rounding show most:
    weights spread over 2^-40 .. 2^40; weights whose products and sums are subnormal; weights whose sums overflow.
    Every output of one control step and the bootstrap value bit for bit (NaN against NaN)."""
    import configs
    import torch
    rng = np.random.default_rng(5)
    qp, qv, pa, steps = configs.reset_states(rng, N)
    qv = rng.normal(0, 0.3, qv.shape).astype(np.float32)
    W = configs.policy_init(rng, hidden=hidden)
    n = W.size - 29   # the log standard deviations stay
    if scale == "wide":
        W[:n] *= np.exp2(rng.integers(-40, 41, n)).astype(np.float32)
    elif scale == "subnormal":
        n = 100 * hidden[0]   # the first layer: subnormal activations through the others
        W[:n] *= np.exp2(rng.integers(-142, -127, n)).astype(np.float32)
    else:
        W[:n] *= np.exp2(rng.integers(40, 127, n)).astype(np.float32)
    W, mean, var = _dev(W), _dev(np.zeros(100, np.float32)), _dev(np.ones(100, np.float32))
    got = []
    for fences in (0, 1):
        with g1.Env(N, substeps=1, pgs_iters=8, seed=9) as env:
            env.set_policy(hidden, act)
            env.set_handover(fences)
            assert env.launch_form() == ("queue" if fences else _form(N))
            env.set_state(qp, qv, pa, steps)
            tr = g1.Trajectory(1, N)
            tr.run(env, W, mean, var)
            torch.cuda.synchronize()
            got.append(tr.numpy())
            assert env.check() == 0
    for f in g1.Trajectory.FIELDS:
        a, b = (x[f] for x in got)
        assert np.array_equal(np.where(np.isnan(a), 0, a.view(np.uint32)), np.where(np.isnan(b), 0, b.view(np.uint32))), f
        assert np.array_equal(np.isnan(a), np.isnan(b)), f
    V = got[0]["V"]
    if scale == "subnormal":
        assert (np.abs(V) < np.finfo(np.float32).tiny).all() and (V != 0).mean() > 0.5


@pytest.mark.parametrize("N,S", [(1, 10), (33, 1), (512, 10), (513, 10), (1024, 5), (1025, 4), (4095, 3), (4096, 2)])
def test_resident_control_steps_equal_work_queue(g1, N, S):
    """Host steps (observation, reward, done; a finished world restarts) and zero-action physics: the two forms'
    outputs and states bit for bit."""
    import configs
    rng = np.random.default_rng(N)
    qp, qv, pa, steps = configs.reset_states(rng, N, noise=0.1)
    qv = rng.normal(0, 0.3, qv.shape).astype(np.float32)
    steps[::3] = 998
    acts = rng.normal(0, 0.5, (3, N, 29)).astype(np.float32)
    got = []
    for fences in (0, 1):
        with g1.Env(N, substeps=S, pgs_iters=8, seed=4) as env:
            env.set_handover(fences)
            assert env.launch_form() == ("queue" if fences else _form(N))
            env.set_state(qp, qv, pa, steps)
            env.ncon_hist(enable=True)
            out = [x for a in acts for x in env.step(a)]
            env.bench_phys(2)
            got.append([x.view(np.uint32) for x in out + list(env.get_state())] + [env.ncon_hist(enable=False)])
            assert env.check() == 0
    for i, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), i
