"""The adjoint where it keeps words of all-zero tiles: FP32, more than 2048
tiles of 32 x 8 cells (needs a GPU).

Small members beside a large one ask for the words, the same grids alone do
not: everything agrees bit for bit.  A single grid that asks is compared with
itself shifted (periodic, no noise: every cell's arithmetic is the same), with a
batch member, with plain steps, and with FP64, which never asks.  Targets differ
from the final phi near the nuclei alone, so most tiles start as zero and
the adjoint reaches across their borders.  Sizes one past the tile in both
directions are the ones whose last tiles no word may speak for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEPS, EVERY = 24, 9


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


def disks(nx, ny, centres, r, dt=np.float32):
    """Disks that wrap around the edges."""
    phi = np.zeros((ny, nx), dt)
    y, x = np.ogrid[:ny, :nx]
    for cx, cy in centres:
        dx, dy = (x - cx + nx // 2) % nx - nx // 2, (y - cy + ny // 2) % ny - ny // 2
        phi[dx * dx + dy * dy <= r * r] = 1.0
    return phi


def params(kb, boundary, seed=1, noise=0.01):
    return kb.default_params(delta=0.05, aniso=6.0, K=1.7, theta0=0.15, noise_a=noise,
                             boundary=boundary, seed=seed)


def run(s, phi, target):
    s.set_fields(phi, np.zeros_like(phi))
    return s.adjoint(STEPS, target, EVERY, want_T0=True, want_phi0=True)


def test_members_that_ask_match_grids_that_do_not(kb):
    edges = [(33, 9), (65, 17), (97, 41), (129, 65), (225, 81), (64, 16), (70, 30), (3, 3), (5, 4),
             (771, 613)]
    sizes = [s for s in edges for _ in range(2)] + [(1000, 960)]   # both boundaries of each
    ps = [params(kb, m % 2, m) for m in range(len(sizes))]
    phi = [disks(nx, ny, [(1, 2), (nx // 2, ny // 2)], min(5, nx // 3)) for nx, ny in sizes]
    target = [disks(nx, ny, [(1, 2), (nx // 2, ny // 2)], min(7, nx // 2)) for nx, ny in sizes]
    with kb.Batch(sizes, ps, "f32") as b:
        for m, f in enumerate(phi):
            b.set_fields(m, f, np.zeros_like(f))
        g, dT = b.adjoint(STEPS, target, EVERY, want_T0=True)
    for m in range(len(sizes) - 1):
        with kb.Solver(*sizes[m], "f32", ps[m]) as s:
            one, one_T, _ = run(s, phi[m], target[m])
        assert one == g[m], (sizes[m], m)
        assert np.array_equal(one_T, dT[m]), (sizes[m], m)


@pytest.mark.parametrize("nx,ny", [(1025, 801), (1030, 771), (1056, 800)])
def test_shifted_grid_has_the_shifted_adjoint(kb, nx, ny):
    assert (-(-nx // 32)) * (-(-ny // 8)) > 2048
    p = params(kb, 0, noise=0.0)
    at = (nx // 2 + 3, ny // 2 + 1)
    phi, target = disks(nx, ny, [at], 6), disks(nx, ny, [(at[0] + 1, at[1])], 9)
    with kb.Solver(nx, ny, "f32", p) as s:
        g, dT, dphi = run(s, phi, target)
        for to in ((2, 1), (nx - 1, ny - 1), (0, ny // 3), (31, 7), (992, 400)):
            dx, dy = to[0] - at[0], to[1] - at[1]
            move = lambda f: np.roll(f, (dy, dx), (0, 1))
            h, hT, hphi = run(s, move(phi), move(target))
            assert np.array_equal(hT, move(dT)), to
            assert np.array_equal(hphi, move(dphi)), to
            # the same squares summed in another order, in FP64
            assert abs(h["loss"] - g["loss"]) <= 1e-12 * g["loss"], to
    assert (dT != 0).sum() > 40 * 40 and (dT == 0).any()


# 64 x 30 tiles fill the stored states of the first two, small tiles those of the third
@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("nx,ny,prec", [(1028, 1024, "f32"), (1449, 1448, "f64"),
                                        (1030, 771, "f32")])
def test_single_grid_matches_its_batch_member_and_plain_steps(kb, nx, ny, prec, boundary):
    dt = np.float64 if prec == "f64" else np.float32
    p = params(kb, boundary, 3)
    at = [(5, 3), (nx // 2, ny // 2), (nx - 40, ny - 9)]
    phi, target = disks(nx, ny, at, 6, dt), disks(nx, ny, at, 8, dt)
    with kb.Solver(nx, ny, prec, p) as s, kb.Solver(nx, ny, prec, p) as plain:
        g, dT, _ = run(s, phi, target)
        plain.set_fields(phi, np.zeros_like(phi))
        plain.step(STEPS)
        for x, y in zip(s.fields(), plain.fields()):
            assert np.array_equal(x, y)
    with kb.Batch([(40, 30), (nx, ny)], [params(kb, 1), p], prec) as b:
        b.set_fields(1, phi, np.zeros_like(phi))
        small = np.zeros((30, 40), dt)
        bg, bT = b.adjoint(STEPS, [small, target], EVERY, want_T0=True)
    assert bg[1] == g and np.array_equal(bT[1], dT)


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("nx,ny", [(1025, 801), (1028, 1024)])
def test_single_grid_matches_double_precision(kb, nx, ny, boundary):
    """As the FP32 adjoint of small grids: within 2e-2 of FP64's."""
    p = params(kb, boundary, 3)
    at = [(5, 3), (nx // 2, ny // 2), (nx - 40, ny - 9)]
    phi, target = disks(nx, ny, at, 6), disks(nx, ny, at, 8)
    with kb.Solver(nx, ny, "f32", p) as s, kb.Solver(nx, ny, "f64", p) as d:
        got = run(s, phi, target)
        want = run(d, phi.astype(float), target.astype(float))
    for k, v in want[0].items():
        assert abs(got[0][k] - v) <= 2e-2 * abs(v), k
    for x, y in zip(got[1:], want[1:]):
        assert np.linalg.norm(x - y) <= 2e-2 * np.linalg.norm(y)
