"""Stored angles that are not finite, in cells without a gradient (needs a GPU).

Such an angle is kept, and eps of it is NaN, so the step makes phi NaN around
it whatever phi is: small tiles, one step a launch and three, give NaN exactly
in the oracle's cells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("solid", [0, 1])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
# one step a launch in 32 x 8 and 32 x 16 tiles, three in 32 x 8 .. 32 x 20
@pytest.mark.parametrize("prec,nx,ny", [("f32", 100, 70), ("f64", 100, 70), ("f32", 400, 400),
                                        ("f64", 400, 400), ("f32", 1030, 771)])
def test_phi_is_nan_where_the_oracles_is(kb, O, prec, nx, ny, bad, solid, boundary):
    p = kb.default_params(delta=0.04, aniso=6.0, noise_a=0.01, boundary=boundary, seed=1)
    q = O.default_params(**{k: getattr(p, k) for k in ("delta", "aniso", "noise_a", "boundary",
                                                       "seed")})
    dt = np.float64 if prec == "f64" else np.float32
    phi, T = np.full((ny, nx), 1.0 if solid else 0.0, dt), np.zeros((ny, nx), dt)
    theta = np.zeros((ny, nx), dt)
    phi[10:14, 20:24] = 0.5                 # a nucleus elsewhere
    theta[44, 50] = theta[23, 64] = theta[0, nx - 1] = bad
    with np.errstate(all="ignore"):
        ref = O.run(O.State(phi.copy(), T.copy(), theta.copy()), q, 3)
    for n in (1, 3):
        with kb.Solver(nx, ny, prec, p) as s:
            s.set_fields(phi, T, theta)
            for _ in range(3 // n):
                s.step(n)
            for name, got, want in zip(("phi", "T"), s.fields(), (ref.phi, ref.T)):
                assert np.array_equal(np.isnan(got), np.isnan(want)), (n, name)
                assert np.isnan(want).any()


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_batches_give_nan_where_the_oracle_does(kb, O, prec):
    sizes = [(100, 70), (70, 33), (64, 64)]
    dt = np.float64 if prec == "f64" else np.float32
    p = [kb.default_params(noise_a=0.01, boundary=m % 2, seed=m) for m in range(3)]
    with kb.Batch(sizes, p, prec) as b:
        want = []
        for m, (nx, ny) in enumerate(sizes):
            phi, T, theta = (np.zeros((ny, nx), dt) for _ in range(3))
            theta[20, 40] = np.nan
            b.set_fields(m, phi, T, theta)
            q = O.default_params(noise_a=0.01, boundary=m % 2, seed=m)
            with np.errstate(all="ignore"):
                want.append(O.run(O.State(phi, T, theta), q, 6))
        b.step(6)
        for m in range(3):
            assert np.isnan(want[m].phi).any()
            assert np.array_equal(np.isnan(b.phase(m)), np.isnan(want[m].phi)), m
