"""The kernels that small grids run (tuning key "small": segments of eight
levels, bands of levels, one block) against the kernels of large grids forced
onto the same grids, bit for bit: the stencils, both predictors, the flux
heights, the scalar step (sums, face values, column update with every Thomas
row count), and the pressure solve in both forms.  The other tests compare the
small kernels with the oracle, so this ties the large ones to it at every
depth and face class; the free-surface solve of large grids is compared with the
oracle itself."""
import numpy as np
import pytest

from suntans_amd import cases, device

import _impls

pytestmark = pytest.mark.gpu

# levels around the ends of segments, load groups and register heads
GRIDS = [dict(nx=nx, ny=ny, Nkmax=k) for nx, ny, k in
         [(3, 2, 7), (33, 1, 9), (16, 8, 10), (20, 13, 17), (16, 9, 33), (16, 9, 64), (11, 9, 100), (9, 7, 128)]] + [
    dict(planform="quad", split_every=3, nx=19, ny=13, Nkmax=21), dict(planform="quad", nx=9, ny=13, Nkmax=70),
    dict(planform="hex", nx=13, ny=9, Nkmax=15), dict(planform="hex", split_every=4, maxfaces=7, nx=13, ny=9, Nkmax=40),
    dict(nx=17, ny=11, Nkmax=4, min_layers=0), dict(nx=17, ny=11, Nkmax=12, open_marks=cases.open_ends())]
IDS = ["-".join(str(v) for v in k.values() if not callable(v)) for k in GRIDS]


def make(kw):
    kw = dict(kw)
    kw.setdefault("min_layers", min(3, kw["Nkmax"] - 4))
    return cases.tiny(kw["nx"] + kw["Nkmax"], **kw)


def loaded(st, small):
    """A device grid with every input field seeded."""
    rng = np.random.default_rng(3)
    dg = device.DeviceGrid(st)
    dg.tune("small", small)
    n, nw, ne = (len(st.get(f)) for f in ("dzz", "w", "u"))
    for f, m, a in (("u", ne, 0.1), ("utmp2", ne, 0.1), ("utmp", ne, 0.1), ("w", nw, 0.01), ("wtmp2", nw, 0.01),
                    ("wnew", nw, 0.01), ("s", n, 30), ("q", n, 1), ("qp", n, 1), ("Cn_W", nw, 1e-5),
                    ("Cn_W2", nw, 1e-5), ("tau_T", st.Ne, 1e-4), ("SfHp", ne, 1), ("SfHm", ne, 1)):
        dg.upload(f, rng.uniform(-a, a, m))
    for f, m, a in (("kappa_tv", n, 1e-3), ("nu_tv", n, 1e-3), ("nu_lax", n, 1e-4), ("CdB", st.Ne, 5e-3),
                    ("CdT", st.Ne, 2e-3)):
        dg.upload(f, rng.uniform(0, a, m))
    for f in ("dzz", "dzzold", "dzf", "D", "dv", "h", "htmp"):
        dg.upload(f, st.get(f))
    dg.upload("src", st.get("stmp"))
    dg.upload("active", (np.arange(st.Nc) % 5 > 0).astype(float))
    dg.upload("hcorr", np.zeros(st.Nc))
    dg.set_face_distances(device.face_distances(st))
    return dg, dict(n=n, w=nw, e=ne, c=st.Nc, f=st.Ne)


def both(st, call, fields):
    out = []
    for small in (1, 0):
        dg, size = loaded(st, small)
        got = call(dg)
        out.append([got] + [dg.download(f, size[k]) for f, k in fields])
        dg.close()
    assert out[0][0] == out[1][0]
    for x, y, f in zip(out[0][1:], out[1][1:], fields):
        assert np.array_equal(x, y, equal_nan=True), f


@pytest.mark.parametrize("kw", GRIDS, ids=IDS)
def test_stencils(gpu_available, kw):
    st = make(kw)
    both(st, lambda d: d.compute_qsource(0.55, 1.0, "stmp"), [("stmp", "n"), ("D", "f")])
    both(st, lambda d: d.corrector(1.0, "q", "qp"), [("u", "e"), ("w", "w"), ("qp", "n")])
    both(st, lambda d: d.continuity(0.55, "w"), [("w", "w")])
    both(st, lambda d: d.set_flux_height(st), [("dzf", "e")])


@pytest.mark.parametrize("kw", GRIDS, ids=IDS)
def test_predictors(gpu_available, kw):
    st = make(kw)
    for scheme in (0, 1, 2, 5):
        P = device.WPredParams(1.0, 0.55, 1e-4, 0.1, 5e-3, 1.0, scheme, 3, 3, 4, 0)
        both(st, lambda d: d.w_predict(P),
             [("w", "w"), ("wtmp", "w"), ("wc", "n"), ("stmp", "n"), ("Cn_W", "w"), ("Cn_W2", "w"), ("ue", "e")])
    P = device.UPredParams(1.0, 0.55, 9.81, 1e-4, 1.0, 0.5, 2)

    def predict(d):
        try:
            return d.u_predict(P)
        except RuntimeError as e:  # an edge level of two dry cells, on both sides
            return str(e)

    both(st, predict, [("utmp", "e"), ("utmp2", "e"), ("ue", "e"), ("D", "f"), ("wtmp2", "w")])


@pytest.mark.parametrize("tvd", [0, 1, 4])
@pytest.mark.parametrize("kw", GRIDS, ids=IDS)
def test_scalar_step(gpu_available, kw, tvd):
    st = make(kw)
    for step in (1, 3):
        both(st, lambda d: [d.update_scalars(0.55, 1.0, 1e-4, tvd, step=step + i) for i in range(2)],
             [("s", "n"), ("Cn", "n"), ("SfHp", "e"), ("SfHm", "e")])


@pytest.mark.parametrize("kw", GRIDS, ids=IDS)
def test_pressure(gpu_available, kw):
    st = make(kw)
    both(st, lambda d: d.q_solve(epsilon=1e-10)["niters"], [("q", "n")])
    both(st, lambda d: d.q_solve_mixed(epsilon=1e-10, inner_tol=1e-4)["inner_iters"], [("q", "n")])


def test_batch(gpu_available):
    """A batch of small members whose kernels are those of large batches."""
    sts = [make(kw) for kw in GRIDS if "open_marks" not in kw]
    out = []
    for small in (1, 0):
        dgs = [loaded(st, small)[0] for st in sts]
        b = device.Batch()
        b.compute_qsource(dgs, 0.55, 1.0, "stmp")
        b.correct(dgs, 0.55, 1.0, "q", "qp")
        b.update_scalars(dgs, [(0.55, 1.0, 1e-4, (4, 0, 1)[i % 3], 2) for i in range(len(dgs))])
        b.sync()
        out.append([dg.download(f, len(st.get(like))) for st, dg in zip(sts, dgs)
                    for f, like in (("stmp", "dzz"), ("u", "u"), ("w", "w"), ("qp", "dzz"), ("s", "dzz"))])
        for dg in dgs:
            dg.close()
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("precond", [0, 1])
@pytest.mark.parametrize("kw", [dict(nx=20, ny=17, Nkmax=5), dict(planform="quad", nx=30, ny=25, Nkmax=5),
                                dict(planform="hex", nx=30, ny=25, Nkmax=5),
                                dict(planform="hex", split_every=4, maxfaces=7, nx=30, ny=25, Nkmax=5)],
                         ids=["tri", "quad", "hex", "hex8"])
def test_free_surface(gpu_available, kw, precond):
    """The two-launch iteration against the oracle on grids that one block
    would solve: equal counts, h within 1e-10; the mixed form within 1e-8."""
    st = cases.tiny(5, min_layers=1, **kw)
    st.set("D", cases.depth_integrated_D(st))
    st.set_prop(hprecond=precond, epsilon=1e-10, maxiters=3000)
    o, a = _impls.oracle(), st.clone()
    o.cgsolve(a)
    want = a.get("h")
    dg = device.DeviceGrid(st)
    dg.tune("small", 0)
    g = st.get_prop
    for mixed in ((False, True) if precond else (False,)):  # the mixed form's test is absolute without it
        for f in ("D", "htmp", "h"):
            dg.upload(f, st.get(f))
        if mixed:
            r = dg.h_solve_mixed(g("grav"), g("theta"), g("dt"), epsilon=1e-10, precond=precond, max_outer=30)
        else:
            r = dg.h_solve(g("grav"), g("theta"), g("dt"), maxiters=3000, precond=precond, epsilon=1e-10)
            assert r["niters"] == o.stats("h")[0]
        assert r["converged"]
        assert np.linalg.norm(dg.download("h", st.Nc) - want) <= (1e-8 if mixed else 1e-10) * np.linalg.norm(want)
    dg.close()
