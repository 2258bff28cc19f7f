"""Resets by the number of nuclei (needs a GPU): up to eight travel with the
launch, up to what the reduction scratch holds (2389) go through it, more
through a buffer of their own.  phi is 1 exactly on the disks, and what the
fields held before is gone; on grids whose rows do and do not end on 16 bytes,
for one member of a batch and for all."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kb():
    import crystalgrowth_amd as kb
    if kb.device_count() < 1:
        pytest.fail("no GPU visible")
    return kb


def disks(nx, ny, cxy, r):
    y, x = (a.astype(float) for a in np.ogrid[:ny, :nx])
    phi = np.zeros((ny, nx))
    for cx, cy in cxy:
        phi[(x - cx) ** 2 + (y - cy) ** 2 <= r * r] = 1.0
    return phi


def is_reset(fields, want):
    return all(np.array_equal(f, w) for f, w in zip(fields, (want, 0 * want, 0 * want)))


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("nx,ny", [(256, 64), (257, 65), (31, 200)])
@pytest.mark.parametrize("count", [1, 2, 8, 9, 2389, 2390])
def test_disks_of_every_count(kb, count, nx, ny, prec):
    dirty = [np.full((ny, nx), 0.25)] * 3
    with kb.Solver(nx, ny, prec) as s:
        for r in (0.0, 3.5):
            s.set_fields(*dirty)
            cxy = s.reset_seeds(count, r, 1, 5)
            assert is_reset(s.fields(), disks(nx, ny, cxy, r)), r
    with kb.Batch([(nx, ny), (nx, ny), (nx, ny)], kb.default_params(), prec) as b:
        for m in range(3):
            b.set_fields(m, *dirty)
        b.reset_seeds(count, 3.5, 1, 5)
        for m in range(3):
            assert is_reset(b.fields(m), disks(nx, ny, cxy, 3.5)), m


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_one_member_leaves_the_others(kb, prec):
    sizes = [(33, 21), (64, 30), (5, 7)]
    with kb.Batch(sizes, kb.default_params(), prec) as b:
        for m, (nx, ny) in enumerate(sizes):
            for k, (x, y) in enumerate(sizes):
                b.set_fields(k, *[np.full((y, x), 0.25)] * 3)
            b.reset_disk(m, -1, -1, 2.0)
            for k, (x, y) in enumerate(sizes):
                if k == m:
                    assert is_reset(b.fields(k), disks(x, y, [(x // 2, y // 2)], 2.0))
                else:
                    assert all((f == 0.25).all() for f in b.fields(k)), (m, k)


def test_disks_far_outside(kb):
    with kb.Solver(70, 40) as s:
        big, low = 2 ** 31 - 1, -2 ** 31
        for cx, cy, r in ((big, low, 10.0), (low, big, 0.0), (35, big, 3e9), (low, low, 1e300),
                          (big, 20, 2.0 ** 31 - 30.5)):
            s.set_fields(*[np.full((40, 70), 0.25)] * 3)
            s.reset_disk(cx, cy, r)
            assert is_reset(s.fields(), disks(70, 40, [(cx, cy)], r)), (cx, cy, r)
