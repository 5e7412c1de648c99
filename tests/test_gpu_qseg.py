"""The pressure solve's iteration on small and middle grids (one block per
tile, one wave per eight levels) against the one-lane-per-column kernels: the
same values, sums and iteration counts, bit for bit.  Grids at the edges of
tiles, groups of four tiles, segments of eight levels and waves of one or
two segments, of every face class, with one-layer columns, surfaces that cross
layers and boundary columns that are not computational."""
import numpy as np
import pytest

from suntans_amd import cases, device

pytestmark = pytest.mark.gpu

# (cells per row, rows, levels): 64 cells per tile, 4 tiles per group
SIZES = [(2, 3, 8), (8, 4, 7), (31, 1, 9), (32, 1, 16), (16, 8, 17), (33, 4, 24), (40, 13, 63), (16, 9, 64), (16, 9, 65),
         (23, 11, 100), (9, 7, 127), (9, 7, 128), (64, 66, 12)]


def solve(st, mixed, tuning=(), fixed=None):
    dg = device.DeviceGrid(st)
    device.member_upload(dg, st)
    for k, v in tuning:
        dg.tune(k, v)
    if mixed:
        s = dg.q_solve_mixed(epsilon=1e-10, inner_tol=1e-4)
        n = (s["niters"], s["inner_iters"])
    else:
        s = dg.q_solve(epsilon=1e-10, fixed=fixed)
        n = s["niters"]
    q = dg.download("q", dg.sizes()["Nflat"])
    s2 = dg.q_solve(epsilon=1e-10)  # once more from the solution, on used buffers
    q2 = dg.download("q", dg.sizes()["Nflat"])
    dg.close()
    return q, n, q2, s["resid"]


def same(st, mixed=False, fixed=None):
    a = solve(st, mixed, (), fixed)
    b = solve(st, mixed, [("prec_unroll", 4)], fixed)
    assert a[1] == b[1] and a[3] == b[3]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("nx,ny,levels", SIZES, ids=["%dx%dx%d" % s for s in SIZES])
def test_sizes(gpu_available, nx, ny, levels):
    st = cases.tiny(nx + levels, nx=nx, ny=max(ny, 1), Nkmax=levels, min_layers=min(3, levels - 4))
    same(st)
    same(st, mixed=True)


@pytest.mark.parametrize("nx,ny,levels", [(128, 128, 70), (145, 142, 100), (181, 181, 100), (181, 181, 128)],
                         ids=["512 tiles", "644 tiles", "1024 tiles", "1024 deep"])
def test_around_the_size_limits(gpu_available, nx, ny, levels):
    """512 tiles and up to 1024, values of 10 to 34 MB in FP64 and half of
    that in FP32: both sides of the lines to the whole-column kernels."""
    st = cases.tiny(levels, nx=nx, ny=ny, Nkmax=levels)
    same(st, fixed=3)
    same(st, mixed=True)


@pytest.mark.parametrize("fixed", [1, 2, 3])
def test_fixed_iterations(gpu_available, fixed):
    same(cases.lock_exchange(seed=3), fixed=fixed)


SHAPES = {
    "quad": dict(planform="quad", nx=19, ny=13, Nkmax=21),
    "quadtri": dict(planform="quad", split_every=3, nx=19, ny=13, Nkmax=70),
    "hex": dict(planform="hex", nx=13, ny=9, Nkmax=15),
    "hex8": dict(planform="hex", split_every=4, maxfaces=7, nx=13, ny=9, Nkmax=40),
    "open": dict(nx=17, ny=11, Nkmax=20, open_marks=cases.open_ends()),
    "onelayer": dict(nx=17, ny=11, Nkmax=4, min_layers=0),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_shapes(gpu_available, name):
    st = cases.tiny(5, **SHAPES[name])
    same(st)
    same(st, mixed=True)


# members up to and past the limit of 1024 tiles (65536 cells)
MEMBERS = [SIZES[:7], SIZES[7:], [(129, 254, 9), (129, 255, 9), (2, 3, 8)]]


@pytest.mark.parametrize("sizes", MEMBERS, ids=["shallow", "deep", "limit"])
def test_batch_members(gpu_available, sizes):
    """A batch starts small members with these kernels.  Each member takes
    the solve's own iteration count within one (its sums are per tile, not per
    group of four) to the same q within 1e-10."""
    sts = [cases.tiny(nx + lv, nx=nx, ny=max(ny, 1), Nkmax=lv, min_layers=min(3, lv - 4)) for nx, ny, lv in sizes]
    one, many = [], []
    for st in sts:
        for to in (one, many):
            dg = device.DeviceGrid(st)
            device.member_upload(dg, st)
            to.append(dg)
    b = device.Batch()
    for again in range(2):  # the second time on used buffers
        for st, dg, mg in zip(sts, one, many):
            device.member_upload(dg, st)
            device.member_upload(mg, st)
        stats = b.q_solve(many, epsilon=1e-10)
        for dg, mg, s in zip(one, many, stats):
            w = dg.q_solve(epsilon=1e-10)
            n = dg.sizes()["Nflat"]
            qw, q = dg.download("q", n), mg.download("q", n)
            assert s["converged"] == w["converged"] == 1 and abs(s["niters"] - w["niters"]) <= 1
            assert np.linalg.norm(q - qw) <= 1e-10 * np.linalg.norm(qw)
    for st, dg, mg in zip(sts, one, many):
        device.member_upload(dg, st)
        device.member_upload(mg, st)
    # mixed: both end below a residual of 1e-10, so q is within 1e-8 (the
    # bound of the mixed form's other tests)
    stats = b.q_solve_mixed(many, epsilon=1e-10, inner_tol=1e-4)
    for dg, mg, s in zip(one, many, stats):
        w = dg.q_solve_mixed(epsilon=1e-10, inner_tol=1e-4)
        n = dg.sizes()["Nflat"]
        qw, q = dg.download("q", n), mg.download("q", n)
        assert s["converged"] == 1 and s["niters"] == w["niters"]
        assert abs(s["inner_iters"] - w["inner_iters"]) <= s["niters"]
        assert np.linalg.norm(q - qw) <= 1e-8 * np.linalg.norm(qw)
    for dg in one + many:
        dg.close()
    b.close()
