"""The FP64 and FP32 modes' new velocity rounds its large term once.

Over a flat bottom of 255 m at rest level, with u a function of y and v of x,
no viscosity, drag or wind, the surface stays at rest and a substep's new
velocity is (255 u + 2 tau F) / 255 with a small F (advection and Coriolis).
The numerator, formed by one multiply-add, is rounded once and its quotient
once: half a unit in the velocity's last place each (255 is just below a power
of two), and 0.05 for the five roundings of 2 tau F / 255, at most 0.005 of a
velocity of 0.5 .. 1.  Rounding the product 255 u first makes it up to one unit
and a half."""
import numpy as np
import pytest

from inmsom_bt import BarotropicModel, make_basin

pytestmark = pytest.mark.gpu


def _basin(nxi, nyi, seed, kind):
    b = make_basin(nxi, nyi, seed=seed)
    wet = np.zeros((b.ny, b.nx), dtype=bool)
    wet[2:-2, 2:-2] = True
    rng = np.random.default_rng(seed)

    def speeds(n):
        return (rng.uniform(0.52, 0.98, n) * rng.choice([-1.0, 1.0], n)).astype(kind).astype(np.float64)

    b.lbasins = np.where(wet, 0, 1).astype(np.int32)
    b.hhq_rest = np.where(wet, 255.0, 0.0)
    b.mu, b.taux, b.tauy, b.ssh, b.sshp = (np.zeros((b.ny, b.nx)) for _ in range(5))
    b.cb_nl = 0.0
    b.u = np.where(wet & np.roll(wet, -1, 1), speeds(b.ny)[:, None], 0.0)
    b.v = np.where(wet & np.roll(wet, -1, 0), speeds(b.nx)[None, :], 0.0)
    b.up, b.vp = b.u.copy(), b.v.copy()
    return b


# tiles, and a march of 7 rows
@pytest.mark.parametrize("mode", ["fp64", "fp32"])
@pytest.mark.parametrize("rows", [0, 7])
def test_large_term_rounds_once(mode, rows):
    print(f"rounding {mode} rows={rows}", flush=True)
    kind = np.float32 if mode == "fp32" else np.float64
    b = _basin(261, 190, 5, kind)
    tau, d = 1.0, b.dx[0, 0]
    with BarotropicModel(b, rdis=np.zeros((b.ny, b.nx))) as m:
        m.set_launch(rows)
        m.run(1, mode, nstep=1, tau=tau)
        got = m.get_state()
    u, v, f = (np.asarray(a, dtype=np.longdouble) for a in (b.u, b.v, b.rlh_s))
    du, dv = u + np.roll(u, -1, 0), v + np.roll(v, -1, 1)  # on H points
    q, cor = dv * du, f * dv
    want_u = u + 2 * tau * (-(q - np.roll(q, 1, 0)) / d + cor + np.roll(cor, 1, 0)) / 4
    cor = f * du
    want_v = v + 2 * tau * (-(q - np.roll(q, 1, 1)) / d - cor - np.roll(cor, 1, 1)) / 4
    inner = (slice(6, -6), slice(6, -6))
    for k, x in (("u", want_u[inner]), ("v", want_v[inner])):
        ulp = np.spacing(np.abs(x).astype(kind)).astype(np.longdouble)
        err = float((np.abs(got[k][inner] - x) / ulp).max())
        print(f"  {k}: {err:.3f} ulp", flush=True)
        assert err <= 1.05, (k, err)
