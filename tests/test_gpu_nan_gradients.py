"""NaN and infinite phi and T among cells with gradients (needs a GPU): from step
to step phi, T and theta are NaN in the oracle's cells, in the small tiles, the
64 x 30 tiles, the two-pass kernel and batches.  (Where gx < -eps and gy is NaN,
theta is pi + atan(NaN).)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


def nans(fields):
    return [np.isnan(f) for f in fields]


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("bad", ["nan", "-nan", "inf", "T nan", "T -nan"])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_nan_cells_are_the_oracles(kb, O, prec, bad, boundary):
    nx, ny = 72, 50
    dt = np.float64 if prec == "f64" else np.float32
    rng = np.random.default_rng(8)
    y, x = np.mgrid[:ny, :nx]
    # phi falls from the left (gx < 0) with gradients everywhere, so that every angle is set
    phi = (0.8 - 0.5 * x / nx + 0.1 * np.sin(y) + 0.05 * rng.random((ny, nx))).astype(dt)
    T = (0.2 * rng.random((ny, nx))).astype(dt)
    theta = rng.uniform(0, 6, (ny, nx)).astype(dt)
    value = dt(np.inf) if bad == "inf" else np.copysign(dt(np.nan), dt(-1 if "-" in bad else 1))
    for cx, cy in ((30, 20), (33, 31), (70, 1)):
        (T if bad[0] == "T" else phi)[cy, cx] = value
    p = kb.default_params(delta=0.04, aniso=6.0, noise_a=0.01, boundary=boundary, seed=1)
    q = O.default_params(delta=0.04, aniso=6.0, noise_a=0.01, boundary=boundary, seed=1)
    runs = {"fused": kb.Solver(nx, ny, prec, p), "two_pass": kb.Solver(nx, ny, prec, p),
            "graph": kb.Batch([(nx, ny)], p, prec), "three": kb.Solver(nx, ny, prec, p),
            "batch": kb.Batch([(nx, ny)], p, prec)}
    runs["two_pass"].set_kernel("two_pass")
    runs["graph"].set_mode("graph", 2)
    for s in runs.values():
        s.set_fields(*(() if isinstance(s, kb.Solver) else (0,)), phi, T, theta)
    ref = O.State(phi, T, theta)
    for step in range(6):
        with np.errstate(all="ignore"):
            ref = O.step(ref, q, step)
        want = nans((ref.phi, ref.T, ref.theta))
        for name in ("fused", "two_pass", "graph"):
            s = runs[name]
            s.step(1)
            got = nans(s.fields() if isinstance(s, kb.Solver) else s.fields(0))
            for f, a, b in zip(("phi", "T", "theta"), got, want):
                assert np.array_equal(a, b), (name, step, f)
        if step % 3 == 2:
            runs["three"].step(3)
            for f, a, b in zip(("phi", "T", "theta"), nans(runs["three"].fields()), want):
                assert np.array_equal(a, b), ("three", step, f)
    runs["batch"].step(6)
    for f, a, b in zip(("phi", "T", "theta"), nans(runs["batch"].fields(0)), want):
        assert np.array_equal(a, b), ("batch", f)
    assert want[0].any() and want[2].any() and not want[0].all()
    for s in runs.values():
        s.close()
