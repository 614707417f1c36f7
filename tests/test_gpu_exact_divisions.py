"""Shared-divisor quotients (FP64_EXACT, the drop-in, the 3-D forcing) against the oracle, bit
for bit, where they could go wrong: states whose numerators lie at the format's limits
(denormals, the smallest normals, products that underflow, huge values that
overflow), waves that mix such cells with ordinary ones, divisors that are not
powers of two (nstep 3, 5, 7), and divisors so small that the step takes IEEE
divisions throughout."""
import numpy as np
import pytest

import oracle
from _util import STATE, assert_bitwise
from inmsom_bt import BarotropicModel, make_basin, randomize_state
from inmsom_bt.ensemble import Ensemble

pytestmark = pytest.mark.gpu


def _scaled(kind, shape, seed):
    """A basin whose fields' magnitudes are drawn over the exponents of `kind`,
    some cells staying ordinary."""
    b = randomize_state(make_basin(*shape, seed=seed, sigma=5.0), seed + 1)
    rng = np.random.default_rng(seed + 2)
    lo, hi = {"denormal": (-1074, -1000), "tiny": (-1030, -200), "all": (-1074, 0), "huge": (300, 1000),
              "zeros": (-1074, -1074)}[kind]
    for f in ("u", "up", "v", "vp", "ssh", "sshp"):
        a = np.array(getattr(b, f), dtype=np.float64)
        e = rng.integers(lo, hi + 1, size=a.shape)
        t = np.ldexp(1.0 + rng.random(a.shape), e) * np.where(rng.random(a.shape) < 0.5, -1.0, 1.0)
        if kind == "zeros":
            t = np.where(rng.random(a.shape) < 0.5, -0.0, 0.0)
        pick = rng.random(a.shape) < (0.02 if kind == "huge" else 0.7)
        if kind == "huge" and f in ("ssh", "sshp"):
            continue
        setattr(b, f, np.where((b.wet > 0) & pick, t, a))
    return b


CASES = [("denormal", (150, 40), 2, 40.0), ("tiny", (130, 37), 3, 40.0), ("all", (61, 50), 5, 40.0),
         ("zeros", (70, 30), 7, 40.0), ("huge", (64, 30), 2, 40.0), ("tiny", (62, 33), 2, 1e-25)]


@pytest.mark.parametrize("kind,shape,nstep,dt", CASES)
def test_exact_step_at_the_format_limits(kind, shape, nstep, dt):
    print(f"exact divisions {kind} {shape} nstep={nstep} dt={dt}", flush=True)
    b = _scaled(kind, shape, seed=61)
    b.dt = dt
    with np.errstate(all="ignore"):
        want = oracle.run(b, 2, nstep, out_steps=[2])[2]
    with BarotropicModel(b) as m:
        m.run(2, "fp64_exact", nstep=nstep)
        got = m.get_state()
    with Ensemble([b, b], mode="fp64_exact") as ens:
        ens.run(2, nstep=nstep)
        member = ens.get_state(1)
    for f in STATE:  # a NaN's sign and payload are the processor's own
        for g, what in ((got, "step"), (member, "member")):
            w, a = np.asarray(want[f]), np.asarray(g[f])
            assert np.array_equal(np.isnan(w), np.isnan(a)), (what, f)
            assert_bitwise({f: np.where(np.isnan(a), 0.0, a)}, {f: np.where(np.isnan(w), 0.0, w)}, (f,),
                           f"{kind} {what}")


@pytest.mark.parametrize("shape,nstep,chunk", [((150, 110), 5, 4), ((61, 70), 6, 1), ((300, 64), 7, 3)])
def test_exact_pairs_carry_depths(shape, nstep, chunk):
    """Substep pairs past the first read the filtered depths of the rows
    around their own while other work items write the next ones: two buffers,
    the oracle's state bit for bit."""
    print(f"exact pairs {shape} nstep={nstep} chunk={chunk}", flush=True)
    b = randomize_state(make_basin(*shape, seed=36, sigma=5.0), 11)
    want = oracle.run(b, 4, nstep, out_steps=[4])[4]
    with BarotropicModel(b) as m:
        m.set_launch(chunk)
        m.set_substeps_per_launch(2)
        m.run(4, "fp64_exact", nstep=nstep)
        assert_bitwise(m.get_state(), want, STATE, "step")
    with Ensemble([b, b], mode="fp64_exact") as ens:
        ens.set_substeps_per_launch(2)
        ens.run(4, nstep=nstep)
        assert_bitwise(ens.get_state(1), want, STATE, "member")


@pytest.mark.parametrize("lo,hi,frac,scale", [(-1074, -950, 0.7, 1.0), (-600, -100, 0.05, 1.0), (450, 500, 0.01, 1.0),
                                              (-20, 0, 1.0, 2.0 ** -70)])
def test_forcing_at_the_format_limits(lo, hi, frac, scale):
    """Velocities of level n-1 over the exponents lo .. hi at a fraction of the
    points, and metrics outside the divisors' range."""
    from test_gpu_forcing3d import _fields
    print(f"forcing 2^{lo}..2^{hi} at {frac}, metrics x {scale}", flush=True)
    b = randomize_state(make_basin(131, 45, seed=9, sigma=4.0, metrics="stretched"), 3)
    f = _fields(b, 5, seed=4)
    rng = np.random.default_rng(5)
    for k in ("uup", "vvp", "uup2d", "vvp2d"):
        t = np.ldexp(1.0 + rng.random(f[k].shape), rng.integers(lo, hi + 1, size=f[k].shape))
        f[k] = np.where((f[k] != 0.0) & (rng.random(f[k].shape) < frac), np.copysign(t, f[k]), f[k])
    for k in ("dx", "dy", "dxt", "dyt", "dxh", "dyh", "dxb", "dyb"):
        setattr(b, k, np.ascontiguousarray(getattr(b, k)) * scale)
    og = oracle.OracleGrid(b)
    with np.errstate(all="ignore"):
        want = oracle.forcing_3d(og, f, b.cb_nl, b.ebottom)
    with BarotropicModel(b) as m:
        got = m.forcing_3d(dict(f, taux=b.taux, tauy=b.tauy), f["dz"], f["rhsx2d"], f["rhsy2d"], f["pgx"], f["pgy"])
    for k in ("rhsx2d", "rhsy2d"):  # a NaN's sign and payload are the processor's own
        w, g = want[k], got[k]
        assert np.array_equal(np.isnan(w), np.isnan(g)), k
        assert_bitwise({k: np.where(np.isnan(g), 0.0, g)}, {k: np.where(np.isnan(w), 0.0, w)}, (k,), f"2^{lo}..2^{hi}")


@pytest.mark.parametrize("kind,nstep,dt", [("all", 3, 40.0), ("zeros", 2, 40.0), ("tiny", 1, 1e-25)])
def test_dropin_march_at_the_format_limits(kind, nstep, dt):
    """barotropic_dynamics on uniform metrics, a grid of the march's size."""
    print(f"drop-in march {kind} nstep={nstep} dt={dt}", flush=True)
    b = _scaled(kind, (700, 590), seed=71)
    og = oracle.OracleGrid(b)
    rd = og.rayleigh()
    rng = np.random.default_rng(6)
    rx, ry = rng.standard_normal((2, b.ny, b.nx)) * 1e3
    wf = rng.standard_normal((b.ny, b.nx)) * 1e-5
    acc = ("ubrtr_i", "vbrtr_i", "ssh4gradx", "ssh4grady")
    st = {k: np.ascontiguousarray(getattr(b, k)).copy() for k in ("u", "up", "v", "vp", "ssh", "sshp")}
    want, wacc = {k: v.copy() for k, v in st.items()}, {k: np.zeros_like(rx) for k in acc}
    with np.errstate(all="ignore"):
        oracle.barotropic_dynamics(og, dt, nstep, 0, want, wacc, rx, ry, wf, b.mu, b.mu4, rd)
    gacc = {k: np.zeros_like(rx) for k in acc}
    with BarotropicModel(b, rdis=rd) as m:
        m.barotropic_dynamics(dt, nstep, 0, *(st[k] for k in st), *(gacc[k] for k in acc), rx, ry, wf,
                              np.ascontiguousarray(b.mu), np.ascontiguousarray(b.mu4), rd)
    want.update(wacc)
    st.update(gacc)
    for k in want:  # a NaN's sign and payload are the processor's own
        w, g = want[k], st[k]
        assert np.array_equal(np.isnan(w), np.isnan(g)), k
        assert_bitwise({k: np.where(np.isnan(g), 0.0, g)}, {k: np.where(np.isnan(w), 0.0, w)}, (k,), kind)
