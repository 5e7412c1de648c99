"""The scalar step on small grids (inflow sums and face values by level bands,
the column update with a wave per 8 or 16 levels) against the kernels that walk
whole columns, bit for bit, at the edges of segments, waves and tiles, with
surfaces that cross layers (rising and falling) and every face class."""
import numpy as np
import pytest

from suntans_amd import cases, device

pytestmark = pytest.mark.gpu

GRIDS = [dict(nx=nx, ny=ny, Nkmax=k) for nx, ny, k in
         [(3, 2, 7), (8, 4, 8), (33, 1, 9), (16, 8, 16), (20, 13, 17), (16, 9, 63), (16, 9, 64), (16, 9, 65), (11, 9, 100),
          (9, 7, 128)]] + [
    dict(planform="quad", split_every=3, nx=19, ny=13, Nkmax=21), dict(planform="quad", nx=9, ny=13, Nkmax=70),
    dict(planform="hex", nx=13, ny=9, Nkmax=15), dict(planform="hex", split_every=4, maxfaces=7, nx=13, ny=9, Nkmax=40),
    dict(nx=17, ny=11, Nkmax=4, min_layers=0), dict(nx=17, ny=11, Nkmax=12, open_marks=cases.open_ends())]


def step(st, tvd, n, tuning=()):
    dg = device.DeviceGrid(st)
    for f in ("s", "u", "utmp2", "dzf", "dzz", "dzzold", "wnew", "wtmp2"):
        dg.upload(f, st.get(f))
    rng = np.random.default_rng(1)
    dg.upload("kappa_tv", rng.uniform(0, 1e-3, len(st.get("kappa_tv"))))
    act = np.ones(st.Nc)
    act[::5] = 0
    dg.upload("active", act)
    for k, v in tuning:
        dg.tune(k, v)
    for i in range(2):
        dg.update_scalars(st.get_prop("theta"), st.get_prop("dt"), 1e-4, tvd, step=n + i)
    m, e = len(st.get("s")), len(st.get("u"))
    out = [dg.download("s", m), dg.download("Cn", m)]
    if tvd:
        out += [dg.download("SfHp", e), dg.download("SfHm", e)]
    dg.close()
    return out


@pytest.mark.parametrize("tvd", [0, 1, 3, 4])
@pytest.mark.parametrize("kw", GRIDS, ids=["-".join(str(v) for v in k.values() if not callable(v)) for k in GRIDS])
def test_segments_bitwise(gpu_available, kw, tvd):
    kw = dict(kw)
    kw.setdefault("min_layers", min(3, kw["Nkmax"] - 4))
    st = cases.tiny(kw["nx"] + kw["Nkmax"], **kw)
    for n in (1, 3):
        a = step(st, tvd, n)
        # whole columns throughout, with and without the head of Thomas rows
        for tuning in ([("small", 0)], [("small", 0), ("tvd_head", 0)]):
            for x, y in zip(a, step(st, tvd, n, tuning)):
                assert np.array_equal(x, y, equal_nan=True)
