"""Grids above 4096 tiles of cells, at the kernels that such grids run by
default (whole columns, two launches per free-surface iteration), through the
reference-signature drop-ins against the oracle: the stencils, both predictors,
the flux heights and the scalar step bit for bit, the free surface within
1e-10 and an equal count."""
import numpy as np
import pytest

from suntans_amd import cases

import _impls

pytestmark = pytest.mark.gpu

# the scalar step's column update keeps 9 rows in registers, so columns of up to 14
# levels end in its head, at its edge and below it
GRIDS = {"tri": dict(nx=364, ny=361, Nkmax=14), "quad": dict(planform="quad", nx=514, ny=512, Nkmax=11),
         "hex": dict(planform="hex", nx=514, ny=512, Nkmax=6, min_layers=1)}


@pytest.fixture(scope="module", params=sorted(GRIDS))
def st(request):
    s = cases.tiny(31, **GRIDS[request.param])
    assert s.Nc > 4096 * 64
    cases.upredictor_inputs(s, np.random.default_rng(5))
    cases.wpredictor_inputs(s, np.random.default_rng(17), nonlinear=2)
    s.set("D", cases.depth_integrated_D(s))
    s.set_prop(TVDsalt=4, n=2)
    return s


CALLS = {
    "source": (lambda i, s: i.compute_qsource(s), ("stmp", "D")),
    "corrector": (lambda i, s: i.corrector(s), ("u", "w", "q")),
    "continuity": (lambda i, s: i.continuity(s), ("w",)),
    "wpredictor": (lambda i, s: i.wpredictor(s), ("w", "wtmp", "wc", "stmp", "Cn_W", "Cn_W2", "ut")),
    "upredictor": (lambda i, s: i.upredictor_begin(s), ("utmp", "ut", "D", "wtmp2", "utmp2")),
    "scalars": (lambda i, s: i.update_salinity(s), ("s", "SfHp", "SfHm")),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_bitwise(gpu_available, st, name):
    call, fields = CALLS[name]
    a, b = st.clone(), st.clone()
    call(_impls.oracle(), a)
    call(_impls.dropin(), b)
    wet = st.edge_wet_mask()
    for f in fields:
        x, y = a.get(f), b.get(f)
        if f.startswith("SfH"):
            x, y = x[wet], y[wet]
        assert np.array_equal(x, y, equal_nan=True), f


def test_free_surface(gpu_available, st):
    st = st.clone()
    st.set_prop(hprecond=1, epsilon=1e-10, maxiters=2000)
    a, b = st.clone(), st.clone()
    o, d = _impls.oracle(), _impls.dropin()
    o.cgsolve(a)
    d.cgsolve(b)
    assert o.stats("h")[0] == d.stats("h")[0]
    assert np.linalg.norm(b.get("h") - a.get("h")) <= 1e-10 * np.linalg.norm(a.get("h"))


def test_z_flux_heights(gpu_available, st):
    """Last: it changes dzf, which the clones share."""
    dzf = st.get("dzf").copy()
    a = st.clone()
    _impls.oracle().set_flux_height(a)
    want = a.get("dzf").copy()
    st.set("dzf", dzf)
    b = st.clone()
    _impls.dropin().set_flux_height(b)
    assert np.array_equal(b.get("dzf"), want)
