"""Steps that whole pairs of launches of a small batch leave over, and the tuner's
choice for such batches (needs a GPU).

The left-over steps run without tile status, from a member table of their own:
it follows changes of parameters, fields and angle bounds between calls, and
calls too short for a pair take up the status afresh.  Compared with a batch in
graph mode bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


SIZES = [(100, 90), (65, 33), (130, 61), (3, 3)]


def same(a, b, what):
    for m in range(len(SIZES)):
        for name, x, y in zip(("phi", "T", "theta"), a.fields(m), b.fields(m)):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (what, m, name)


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_left_over_steps_follow_the_members(kb, prec):
    params = [kb.default_params(delta=0.04, aniso=6.0, K=1.6, noise_a=0.01, boundary=m % 2, seed=m,
                                instance=m) for m in range(len(SIZES))]
    rng = np.random.default_rng(4)
    with kb.Batch(SIZES, params, prec) as a, kb.Batch(SIZES, params, prec) as b:
        b.set_mode("graph", 2)
        for k, n in enumerate((7, 9, 2, 7, 1, 13, 5, 11, 8)):
            a.step(n)
            b.step(n)
            same(a, b, (k, n))
            m = k % len(SIZES)
            nx, ny = SIZES[m]
            if k % 3 == 0:      # other parameters, and the other boundary
                params[m] = params[m].replace(K=1.0 + 0.1 * k, boundary=1 - params[m].boundary)
                for c in (a, b):
                    c.set_params(m, params[m])
            elif k % 3 == 1:    # angles beyond the reduced sin / cos range
                f = [rng.random((ny, nx)), np.zeros((ny, nx)), np.full((ny, nx), 3.0e3 * k)]
                for c in (a, b):
                    c.set_fields(m, *f)
            else:
                for c in (a, b):
                    c.reset_disk(m, -1, -1, 4.0)


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("trial", [2, 4, 16])
def test_tuner_times_whole_launches(kb, trial, prec):
    """Several steps a launch take a third of the time of one step a launch on
    batches of this size, so launch mode wins however short the trial is."""
    sizes = [(100, 100)] * 5
    with kb.Batch(sizes, kb.default_params(noise_a=0.01), prec) as b:
        b.reset_disk(-1, -1, -1, 6.0)
        b.step(61)
        before = [b.fields(m) for m in range(5)]
        assert b.autotune(trial)[0] == "launch"
        assert b.step_count == 61
        for m in range(5):
            for x, y in zip(before[m], b.fields(m)):
                assert np.array_equal(x, y), m
