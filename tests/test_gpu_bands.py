"""The level-wise kernels by bands of levels and by segments, and the transfers
by 32-level blocks, on grids whose columns end around the edges of those: the
stencils, both predictors and the flux heights against the oracle bit for bit,
fields of every layout there and back."""
import numpy as np
import pytest

from suntans_amd import cases, device

import _impls

pytestmark = pytest.mark.gpu

LEVELS = [7, 8, 9, 16, 17, 31, 32, 33, 64, 65, 97, 128]


def grid(levels, **kw):
    return cases.tiny(levels, nx=11, ny=9, Nkmax=levels, min_layers=min(3, levels - 4), **kw)


@pytest.mark.parametrize("levels", LEVELS)
def test_transfers(gpu_available, levels):
    st = grid(levels)
    dg = device.DeviceGrid(st)
    rng = np.random.default_rng(levels)
    for name, like in (("q", "dzz"), ("w", "w"), ("u", "u"), ("h", "h"), ("D", "D")):
        a = rng.normal(size=len(st.get(like)))
        dg.upload(name, a)
        assert np.array_equal(dg.download(name, len(a)), a), name
    dg.close()


@pytest.mark.parametrize("planform", ["tri", "hex"])
@pytest.mark.parametrize("levels", LEVELS)
def test_stencils_and_predictors(gpu_available, levels, planform):
    o, d = _impls.oracle(), _impls.dropin()
    st = grid(levels, planform=planform)
    cases.upredictor_inputs(st, np.random.default_rng(5))
    cases.wpredictor_inputs(st, np.random.default_rng(17), nonlinear=2)
    st.set("D", cases.depth_integrated_D(st))

    def both(call, fields):
        a, b = st.clone(), st.clone()
        call(o, a)
        call(d, b)
        for f in fields:
            assert np.array_equal(a.get(f), b.get(f), equal_nan=True), (call, f)

    both(lambda i, s: i.compute_qsource(s), ("stmp", "D"))
    both(lambda i, s: i.corrector(s), ("u", "w", "q"))
    both(lambda i, s: i.continuity(s), ("w",))
    both(lambda i, s: i.wpredictor(s), ("w", "wtmp", "wc", "stmp", "Cn_W", "Cn_W2", "ut"))
    both(lambda i, s: i.upredictor_begin(s), ("utmp", "ut", "D", "wtmp2", "utmp2"))
    # last: it changes dzf, which the clones share
    dzf = st.get("dzf")
    a = st.clone()
    o.set_flux_height(a)
    want = a.get("dzf").copy()
    st.set("dzf", dzf)
    b = st.clone()
    d.set_flux_height(b)
    assert np.array_equal(b.get("dzf"), want)


@pytest.mark.parametrize("planform", ["tri", "quad", "hex"])
def test_batch_stencils_and_scalars(gpu_available, planform):
    """The same passes over a batch of grids of all these depths, and the TVD
    face passes, against the oracle bit for bit."""
    o = _impls.oracle()
    sts = [grid(levels, planform=planform) for levels in LEVELS]
    th, dt = sts[0].get_prop("theta"), sts[0].get_prop("dt")
    step, scal = [], []
    for i, st in enumerate(sts):
        rng = np.random.default_rng(i)
        st.set("qc", rng.normal(size=st.get("qc").shape))
        st.set("q", rng.normal(size=st.get("q").shape))
        st.set_prop(TVDsalt=3 + i % 2, n=2)
        dg = device.DeviceGrid(st)
        device.member_upload_step(dg, st)
        dg.upload("q", st.get("qc"))
        step.append(dg)
        dg = device.DeviceGrid(st)
        device.member_upload_tvd(dg, st)
        scal.append(dg)
    b = device.Batch()
    b.compute_qsource(step, th, dt)
    b.correct(step, th, dt)
    b.update_scalars(scal, [(st.get_prop("theta"), st.get_prop("dt"), st.get_prop("kappa_s"), 3 + i % 2, 2)
                            for i, st in enumerate(sts)])
    b.sync()
    for st, dg, sg in zip(sts, step, scal):
        m = st.wet_mask()
        a = st.clone()
        o.update_salinity(a)
        assert np.array_equal(sg.download("s", len(m))[m], a.get("s")[m])
        a = st.clone()
        a.set_prop(theta=th, dt=dt)
        o.compute_qsource(a)
        assert np.array_equal(dg.download("src", len(m))[m], a.get("stmp")[m])
        o.corrector(a)
        o.continuity(a)
        for f, g in (("qp", "q"), ("w", "w"), ("u", "u")):
            assert np.array_equal(dg.download(f, len(a.get(g))), a.get(g)), f
        dg.close()
        sg.close()
    b.close()
