"""barotropic_dynamics on tiles (small grids, and the biharmonic term on any)
against the stage-by-stage path, bit for bit, over tile edges in both
directions, with metrics uniform along x and per cell, a water flux and a
biharmonic viscosity that vary from cell to cell; and the march just above the
size at which it takes over."""
import numpy as np
import pytest

from _util import STATE, assert_bitwise
from inmsom_bt import BarotropicModel, make_basin, randomize_state

pytestmark = pytest.mark.gpu

ACC = ("ubrtr_i", "vbrtr_i", "ssh4gradx", "ssh4grady")


# columns around the 60-column tiles, rows around the 4- and 8-row ones; the
# smallest basin; 660 x 640 is the march without the biharmonic term
@pytest.mark.parametrize("ksw4", [0, 1])
@pytest.mark.parametrize("shape,metrics,nstep", [((7, 5), "uniform", 2), ((56, 28), "uniform", 1),
                                                 ((57, 29), "stretched", 3), ((117, 61), "stretched", 2),
                                                 ((285, 159), "uniform", 2), ((660, 640), "uniform", 1)])
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
