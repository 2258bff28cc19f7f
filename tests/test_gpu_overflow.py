"""T that is finite when a launch of three steps starts and overflows inside it
(needs a GPU).

One hot cell in a field of +0 or 1: T is infinite after one step and NaN after
two or three, and a step from NaN makes phi NaN.  Whether those steps are one
launch or three, in a plain handle, a batch or the states an adjoint stores, the
fields are the same, and phi is NaN in the oracle's cells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# about 2^-13 and 2^-3 of the largest number: the 9-point sum times 1 / (3 dx^2), and the
# 9-point sum itself, overflow
HOT = {"f32": (1e35, 1e38), "f64": (1e305, 1e308)}


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


def state(nx, ny, prec, solid, hot, at):
    dt = np.float64 if prec == "f64" else np.float32
    phi, T = np.full((ny, nx), 1.0 if solid else 0.0, dt), np.zeros((ny, nx), dt)
    T[at[1], at[0]] = hot
    return phi, T


def same(a, b, what):
    """Equal bits; NaN where the other is NaN."""
    for name, x, y in zip(("phi", "T", "theta"), a, b):
        nan = np.isnan(x)
        assert np.array_equal(nan, np.isnan(y)), (what, name)
        assert np.array_equal(x[~nan].view(np.uint8), y[~nan].view(np.uint8)), (what, name)


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("solid", [0, 1])
# tiles of 8, 12, 16 (FP32) and 20 rows (FP32, 512 threads)
@pytest.mark.parametrize("prec,nx,ny", [("f32", 100, 70), ("f64", 100, 70), ("f32", 400, 400),
                                        ("f64", 400, 400), ("f32", 512, 512), ("f32", 1030, 771)])
def test_overflow_inside_a_launch(kb, O, prec, nx, ny, solid, boundary):
    p = kb.default_params(delta=0.04, aniso=6.0, noise_a=0.01, boundary=boundary, seed=1)
    q = O.default_params(**{k: getattr(p, k) for k in ("delta", "aniso", "noise_a", "boundary",
                                                       "seed")})
    # inside a tile, on both sides of a tile's edge, and at the grid's corner
    for hot in HOT[prec]:
        for at in ((50, 44), (31, 8), (64, 23), (0, 0), (nx - 1, ny - 1)):
            phi, T = state(nx, ny, prec, solid, hot, at)
            with np.errstate(all="ignore"):
                ref = O.run(O.State(phi.copy(), T.copy(), np.zeros_like(phi)), q, 3)
            with kb.Solver(nx, ny, prec, p) as a, kb.Solver(nx, ny, prec, p) as b:
                a.set_fields(phi, T)
                b.set_fields(phi, T)
                a.step(3)
                for _ in range(3):
                    b.step(1)
                assert np.isnan(ref.phi).any() or at != (50, 44)
                assert np.array_equal(np.isnan(a.phase()), np.isnan(ref.phi)), (hot, at)
                same(a.fields(), b.fields(), (hot, at))
                a.step(6)
                b.set_kernel("fused_dense")
                b.step(6)
                same(a.fields(), b.fields(), (hot, at, "later"))


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_overflow_inside_a_batch_launch(kb, prec):
    sizes = [(100, 70), (70, 33), (64, 64)]
    p = [kb.default_params(noise_a=0.01, boundary=m % 2, seed=m) for m in range(3)]
    for hot in HOT[prec]:
        with kb.Batch(sizes, p, prec) as a, kb.Batch(sizes, p, prec) as b:
            b.set_mode("graph", 2)         # 64 x 30 tiles, one step a launch
            for m, (nx, ny) in enumerate(sizes):
                for c in (a, b):
                    c.set_fields(m, *state(nx, ny, prec, m == 1, hot, (30 + m, 9)))
            a.step(6)
            b.step(6)
            for m in range(3):
                assert np.isnan(a.phase(m)).any()
                same(a.fields(m), b.fields(m), (hot, m))


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_overflow_inside_the_states_of_an_adjoint(kb, prec):
    """The states of a segment come from launches of three steps, in a plain
    handle and in a batch."""
    sizes = [(100, 70), (70, 33), (64, 64)]
    p = [kb.default_params(noise_a=0.01, boundary=m % 2, seed=m) for m in range(3)]
    for hot in HOT[prec]:
        st = [state(nx, ny, prec, m == 1, hot, (30 + m, 9)) for m, (nx, ny) in enumerate(sizes)]
        want = []
        for m, (nx, ny) in enumerate(sizes):
            with kb.Solver(nx, ny, prec, p[m]) as a, kb.Solver(nx, ny, prec, p[m]) as b:
                a.set_fields(*st[m])
                b.set_fields(*st[m])
                g, _, _ = a.adjoint(3, np.zeros_like(st[m][0]), 3)
                for _ in range(3):
                    b.step(1)
                want.append(b.fields())
                same(a.fields(), want[m], (hot, m))
                assert np.isnan(g["loss"]) and np.isnan(want[m][0]).any()
        with kb.Batch(sizes, p, prec) as a:
            for m in range(3):
                a.set_fields(m, *st[m])
            a.adjoint(3, [np.zeros_like(f[0]) for f in st], 3)
            for m in range(3):
                same(a.fields(m), want[m], (hot, m, "batch"))
