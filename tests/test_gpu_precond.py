"""The preconditioner of the solves (inverse pivots, register head and LDS
stage) at column depths around the ends of its stages: 40 + 16 levels in
FP64, 48 + 16 in FP32.  The batched engine runs that head at every size; the
single-grid solve with prec_head 0 runs the plain sweep.  Both form the same
values, the engine summing its dot products per tile, so that q moves by
roundings of the dots only: 1e-12."""
import numpy as np
import pytest

from suntans_amd import cases, device

import _impls

pytestmark = pytest.mark.gpu


def build(levels):
    st = cases.tiny(levels, nx=11, ny=9, Nkmax=levels, min_layers=1)
    dg = device.DeviceGrid(st)
    device.member_upload(dg, st)
    return st, dg


@pytest.mark.parametrize("levels", [5, 39, 40, 41, 55, 56, 57, 63, 64, 65, 72])
def test_head_against_plain_sweep(gpu_available, levels):
    st, dg = build(levels)
    n = dg.sizes()["Nflat"]
    dg.tune("prec_head", 0)
    s0 = dg.q_solve(epsilon=1e-10)
    q0 = dg.download("q", n)
    dg.upload("q", st.get("qc"))
    b = device.Batch()
    s1 = b.q_solve([dg], epsilon=1e-10)[0]
    q1 = dg.download("q", n)
    assert s0["converged"] and s1["converged"] and abs(s0["niters"] - s1["niters"]) <= 1
    # one iteration more or less moves q by its residual; equal counts by roundings
    tol = 1e-12 if s0["niters"] == s1["niters"] else 1e-8
    assert np.linalg.norm(q1 - q0) <= tol * np.linalg.norm(q0)
    dg.upload("q", st.get("qc"))
    s2 = b.q_solve_mixed([dg], epsilon=1e-10, inner_tol=1e-4)[0]
    q2 = dg.download("q", n)
    b.close()
    dg.close()
    # both stop at a true residual of 1e-10
    assert s2["converged"]
    assert np.linalg.norm(q2 - q0) <= 1e-8 * np.linalg.norm(q0)


@pytest.mark.parametrize("kw", [dict(nx=190, ny=180, Nkmax=6), dict(planform="quad", nx=270, ny=250, Nkmax=6),
                                dict(planform="hex", nx=270, ny=250, Nkmax=6)], ids=["tri", "quad", "hex"])
def test_default_kernels_above_1024_tiles(gpu_available, kw):
    """The kernels a solve of a little over 1024 tiles takes by default
    (cached stores, register head, the plain or the exchange operator)
    against the plain ones, bit for bit."""
    st = cases.tiny(9, **kw)
    assert (st.Nc + 63) // 64 > 1024
    out = []
    for tuning in ((), (("xchg", 0), ("unroll", 1), ("prec_head", 0))):
        dg = device.DeviceGrid(st)
        device.member_upload(dg, st)
        for k, v in tuning:
            dg.tune(k, v)
        n = dg.q_solve(epsilon=1e-10)["niters"]
        out.append((n, dg.download("q", dg.sizes()["Nflat"])))
        dg.upload("q", st.get("qc"))
        n = dg.q_solve_mixed(epsilon=1e-10, inner_tol=1e-4)["inner_iters"]
        out[-1] += (n, dg.download("q", dg.sizes()["Nflat"]))
        dg.close()
    assert out[0][0] == out[1][0] and out[0][2] == out[1][2]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][3], out[1][3])


def test_plain_operator_on_scattered_tiles(gpu_available, monkeypatch):
    """A grid of over 1536 tiles in which one tile gathers cells from all over
    (more cross-tile faces than the exchange holds) runs the plain operator
    by default: the same bits as at one level per group."""
    st = cases.tiny(9, nx=230, ny=220, Nkmax=7)
    xv, yv = st.get("xv").copy(), st.get("yv").copy()
    i = np.random.default_rng(1).permutation(st.Nc)[:64]
    xv[i], yv[i] = xv[i[0]], yv[i[0]]
    top = device.topology
    monkeypatch.setattr(device, "topology", lambda s: top(s, {"xv": xv, "yv": yv}))
    out = []
    for tuning in ((), (("xchg", 0), ("unroll", 1))):
        dg = device.DeviceGrid(st)
        device.member_upload(dg, st)
        for k, v in tuning:
            dg.tune(k, v)
        n = dg.q_solve(epsilon=1e-10)["niters"]
        out.append((n, dg.download("q", dg.sizes()["Nflat"])))
        dg.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("levels", [23, 24, 25, 33, 50])
def test_entry_above_1024_tiles(gpu_available, levels):
    """The Preconditioner entry with its 24-row register head (1024 tiles and
    more) against the oracle, bit for bit, at columns that end around the head
    and its load groups."""
    st = cases.tiny(levels, nx=190, ny=180, Nkmax=levels, min_layers=min(20, levels - 4))
    assert (st.Nc + 63) // 64 > 1024
    rng = np.random.default_rng(levels)
    n = len(st.get("dzz"))
    st.set("wtmp", rng.uniform(0.5, 2, len(st.get("wtmp"))))
    st.set("stmp", rng.normal(size=n))
    st.set("uold", 0.0)
    b = st.clone()
    _impls.oracle().preconditioner(st)
    _impls.dropin().preconditioner(b)
    m = st.wet_mask()
    assert np.array_equal(b.get("uold")[m], st.get("uold")[m])
