"""Tile status on the grids that keep one: more than 2^21 cells (needs a GPU).

2048 x 1100 cells are 160 chunks, too few for chunk lists, so every tile asks
its status words each step.  Every comparison is bitwise, against the launch
without status (fused_dense), which such grids step in the same tiles; nuclei
in a zero field, so that all kinds of tiles occur."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX, NY = 2048, 1100            # 32 x 37 tiles, the last row 20 rows high


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


def params(kb, boundary, **more):
    return kb.default_params(delta=0.04, aniso=6.0, K=2.0, theta0=0.2, noise_a=0.01,
                             boundary=boundary, seed=3, **more)


def same(a, b, what):
    for name, x, y in zip(("phi", "T", "theta"), a.fields(), b.fields()):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (what, name)


@pytest.mark.parametrize("boundary", [0, 1])
# aligned rows and rows staged cell by cell at the edges; the last, periodic, has tiles one
# cell wide and one row high, which no status can be kept for
@pytest.mark.parametrize("nx,ny,prec", [(NX, NY, "f32"), (NX, NY, "f64"), (2051, 1101, "f32"),
                                        (2049, 1051, "f32"), (2049, 1051, "f64")])
def test_status_matches_dense_bitwise(kb, nx, ny, prec, boundary):
    p = params(kb, boundary)
    with kb.Solver(nx, ny, prec, p) as a, kb.Solver(nx, ny, prec, p) as b:
        b.set_kernel("fused_dense")
        for s in (a, b):
            s.reset_seeds(6, 5.0, 3, 11)
        for n in (1, 1, 1, 40, 260):
            a.step(n)
            b.step(n)
            same(a, b, a.step_count)
        assert a.skip_stats() == {"listed_launches": 0, "stale_answers": 0}


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_status_after_writes_and_kernel_switches(kb, prec):
    """set_fields, resets, parameters, an adjoint and steps of the other kernels
    between steps that trust the status."""
    p = params(kb, 1)
    rng = np.random.default_rng(2)
    phi, T = np.zeros((NY, NX)), np.zeros((NY, NX))
    phi[950:960, 1700:1730] = 1.0      # where the old state is zero
    T[20:40, 1250:1290] = rng.random((20, 40)) * 0.3
    with kb.Solver(NX, NY, prec, p) as a, kb.Solver(NX, NY, prec, p) as b:
        b.set_kernel("fused_dense")

        def both(what, f, n):
            for s in (a, b):
                f(s)
                s.step(n)
            same(a, b, what)

        both("reset", lambda s: s.reset_disk(160, 150, 5.0), 30)
        both("set_fields", lambda s: s.set_fields(phi, T), 25)
        a.set_kernel("two_pass")
        both("two_pass", lambda s: s.set_kernel("two_pass"), 1)
        a.set_kernel("fused")
        b.set_kernel("fused_dense")
        both("switched back", lambda s: None, 20)
        # nuclei that only the other kernel steps: its tiles were +0 in both buffers before
        a.set_kernel("fused_dense")
        both("dense", lambda s: s.set_fields(phi[::-1], T[:, ::-1]), 5)
        a.set_kernel("fused")
        both("fused again", lambda s: None, 9)
        both("adjoint", lambda s: s.adjoint(5, phi, 2), 12)
        both("parameters", lambda s: s.set_params(K=1.2), 12)
        both("boundary", lambda s: s.set_params(boundary=0), 12)
        both("counter", lambda s: setattr(s, "step_count", 1003), 8)
        both("seeds", lambda s: s.reset_seeds(3, 4.0, 8, 7), 21)


@pytest.mark.parametrize("mode,g,n", [("graph", 2, 150), ("graph_lists", 2, 150), ("launch", 0, 5)])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_members_of_small_batches_keep_a_status(kb, prec, mode, g, n):
    """In graph mode, and in launches of calls too short for several steps a
    launch; one member's edge tiles are too thin for a status."""
    sizes = [(200, 130), (64, 64), (129, 61), (96, 250), (460, 250)]
    ps = [params(kb, k % 2, instance=k) for k in range(len(sizes))]
    with kb.Batch(sizes, ps, prec) as bt:
        bt.set_mode(mode, g)
        bt.reset_disk(-1, -1, -1, 5.0)
        for _ in range(150 // n):
            bt.step(n)
        got = [bt.fields(m) for m in range(len(sizes))]
    for (nx, ny), p, f in zip(sizes, ps, got):
        with kb.Solver(nx, ny, prec, p) as s:
            s.set_kernel("fused_dense")
            s.reset_disk(nx // 2, ny // 2, 5.0)
            s.step(150)
            for x, y in zip(f, s.fields()):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (nx, ny)
