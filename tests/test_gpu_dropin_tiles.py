"""barotropic_dynamics on tiles (small grids, and the biharmonic term on any)
against the stage-by-stage path, bit for bit, over tile edges in both
directions, with metrics uniform along x and per cell, a water flux and a
biharmonic viscosity that vary from cell to cell; and the march, with each kind
of metrics, just above the size at which it takes over."""
import numpy as np
import pytest

from _util import STATE, assert_bitwise
from inmsom_bt import BarotropicModel, make_basin, randomize_state

pytestmark = pytest.mark.gpu

ACC = ("ubrtr_i", "vbrtr_i", "ssh4gradx", "ssh4grady")


# columns around the 60-column tiles, rows around those of 4 and 8 rows written;
# the smallest basin; 333 x 301 has tiles of 12 rows, the smaller ones of 8; 660 x
# 640 is the march's without the biharmonic term
@pytest.mark.parametrize("ksw4", [0, 1])
@pytest.mark.parametrize("shape,metrics,nstep", [((7, 5), "uniform", 2), ((56, 28), "uniform", 1),
                                                 ((57, 29), "stretched", 3), ((117, 61), "stretched", 2),
                                                 ((285, 159), "uniform", 2), ((333, 301), "stretched", 1),
                                                 ((660, 640), "uniform", 1)])
def test_tiles_equal_stage_by_stage(shape, metrics, nstep, ksw4):
    print(f"drop-in tiles {shape} {metrics} nstep={nstep} ksw4={ksw4}", flush=True)
    b = randomize_state(make_basin(*shape, seed=31, sigma=min(5.0, 0.2 * min(shape)), metrics=metrics, lvisc_4=1e-3,
                                   hland=60.0 if min(shape) < 10 else 10.0), 12, wflux_amp=1e-5)
    rng = np.random.default_rng(6)
    sh = (b.ny, b.nx)
    inp = [1e3 * rng.standard_normal(sh), 1e3 * rng.standard_normal(sh), np.ascontiguousarray(b.wflux),
           b.mu * (1.0 + 0.3 * rng.random(sh)), b.mu4 * (1.0 + 0.3 * rng.random(sh))]
    out = {}
    for path in ("literal", "fused"):
        st = {k: np.ascontiguousarray(getattr(b, k)).copy() for k in ("u", "up", "v", "vp", "ssh", "sshp")}
        acc = {k: np.zeros(sh) for k in ACC}
        with BarotropicModel(b) as m:
            m.set_dropin_path(path)
            for _ in range(2):
                m.barotropic_dynamics(4.0 * nstep, nstep, ksw4, *st.values(), *acc.values(), *inp, m.rdis)
        out[path] = {**st, **acc}
    assert np.abs(out["fused"]["u"] - b.u).max() > 0.0
    assert_bitwise(out["fused"], out["literal"], STATE + ACC, f"{shape} {metrics} nstep={nstep} ksw4={ksw4}")


def _rows_basin(b):
    """b on a longitude-latitude grid: metrics that differ from row to row and
    from each other."""
    lat = np.radians(40.0 + 20.0 * np.arange(b.ny) / b.ny)[:, None]
    for i, k in enumerate(("dx", "dxt", "dxh", "dxb", "dy", "dyt", "dyh", "dyb")):
        c = np.cos(lat + 0.01 * i) if k[1] == "x" else 1.0 + 0.1 * np.sin(3.0 * lat + 0.2 * i)
        setattr(b, k, np.ascontiguousarray(np.broadcast_to(1000.0 * c, (b.ny, b.nx))))
    return b


# the march with its three kinds of metrics, where it takes over from the tiles
# (more than three rounds of 12-row tiles over 256 CUs, a third round less than a
# third full; one metric: more than one round) and the tiles just below: columns
# and rows that fill no strip, tile or chunk, wet cells next to the halo
@pytest.mark.parametrize("shape,metrics,nstep", [((691, 593), "stretched", 1), ((1013, 419), "stretched", 3),
                                                 ((691, 593), "rows", 1), ((1013, 419), "rows", 3),
                                                 ((691, 593), "uniform", 3), ((361, 299), "uniform", 1),
                                                 ((333, 301), "uniform", 2), ((541, 419), "rows", 2),
                                                 ((541, 419), "stretched", 1), ((601, 439), "rows", 1)])
def test_march_equals_stage_by_stage(shape, metrics, nstep):
    print(f"drop-in march {shape} {metrics} nstep={nstep}", flush=True)
    b = make_basin(*shape, seed=17, sigma=6.0, hland=1.0, metrics="stretched" if metrics == "stretched" else "uniform")
    b = randomize_state(b if metrics != "rows" else _rows_basin(b), 18, wflux_amp=1e-5)
    assert all((e == 0).any() for e in (b.lbasins[2], b.lbasins[-3], b.lbasins[:, 2], b.lbasins[:, -3]))
    rng = np.random.default_rng(7)
    sh = (b.ny, b.nx)
    if metrics == "stretched":
        b.rlh_s = b.rlh_s * (1.0 + 0.2 * rng.random(sh))
    inp = [1e3 * rng.standard_normal(sh), 1e3 * rng.standard_normal(sh), np.ascontiguousarray(b.wflux),
           b.mu * (1.0 + 0.3 * rng.random(sh)), np.zeros(sh)]
    out = {}
    for path in ("literal", "fused"):
        st = {k: np.ascontiguousarray(getattr(b, k)).copy() for k in ("u", "up", "v", "vp", "ssh", "sshp")}
        acc = {k: np.zeros(sh) for k in ACC}
        with BarotropicModel(b) as m:
            m.set_dropin_path(path)
            for _ in range(2):
                m.barotropic_dynamics(2.0 * nstep, nstep, 0, *st.values(), *acc.values(), *inp, m.rdis)
            assert m.dropin_path(0) == path
        out[path] = {**st, **acc}
    assert np.isfinite(out["literal"]["u"]).all() and np.abs(out["fused"]["u"] - b.u).max() > 0.0
    assert_bitwise(out["fused"], out["literal"], STATE + ACC, f"{shape} {metrics} nstep={nstep}")
