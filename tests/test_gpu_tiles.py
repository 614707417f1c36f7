"""The tiles of the fast modes on small grids: bit for bit what the march
gives (a launch shape of the caller's, here one row chunk, selects the march),
over tile edges in both directions, odd substep counts and calls that span
launches, for one basin and for an ensemble; and basins of different tile
sizes run by several threads at once."""
import threading

import pytest

from _util import STATE, assert_bitwise
from inmsom_bt import BarotropicModel, make_basin, randomize_state
from inmsom_bt.ensemble import Ensemble

pytestmark = pytest.mark.gpu


def _basin(nxi, nyi, seed=3):
    return randomize_state(make_basin(nxi, nyi, seed=seed, sigma=min(4.0, 0.2 * min(nxi, nyi))), seed + 1)


# array sizes around the 58-column tiles and the 2-, 6- and 10-row ones; the
# smallest; one just below the size at which the pipeline takes over
@pytest.mark.parametrize("mode", ["fp64", "fp32"])
@pytest.mark.parametrize("shape,nstep,steps", [((8, 6), 2, 3), ((54, 30), 2, 3), ((55, 31), 3, 3), ((113, 37), 1, 5),
                                               ((200, 91), 4, 2), ((271, 240), 5, 3), ((560, 520), 2, 2)])
def test_tiles_equal_march(mode, shape, nstep, steps):
    b = _basin(*shape)
    print(f"tiles {mode} {shape} nstep={nstep}", flush=True)
    out = []
    for chunk in (0, 5):
        with BarotropicModel(b) as m:
            m.set_launch(chunk)
            m.run(steps, mode, nstep=nstep, tau=5.0 * nstep)
            m.run(1, mode, nstep=nstep, tau=5.0 * nstep)
            out.append(m.get_state())
    assert_bitwise(out[0], out[1], STATE, f"tiles vs march {mode} {shape} nstep={nstep}")


# the last with more tiles than two rounds of the CUs: the march in FP64
@pytest.mark.parametrize("mode,nstep,many", [("fp32", 2, 1), ("fp64", 3, 1), ("fp32", 1, 1), ("fp64", 2, 30),
                                             ("fp32", 2, 30)])
def test_ensemble_tiles_equal_march(mode, nstep, many):
    basins = [_basin(x, y, seed=9 + k) for k, (x, y) in enumerate(((40, 90), (130, 33), (61, 62), (9, 7)))]
    basins = [b for b in basins for _ in range(many)]
    print(f"ensemble tiles {mode} nstep={nstep}", flush=True)
    out = []
    for rows, graph in ((0, True), (0, False), (7, False)):
        with Ensemble(basins, mode=mode) as ens:
            ens.set_launch(rows, 0)
            ens.run(9, nstep=nstep, tau=5.0 * nstep, graph=graph)
            out.append([ens.get_state(k) for k in range(len(basins))])
    for o in out[1:]:
        for k in range(len(basins)):
            assert_bitwise(o[k], out[0][k], STATE, f"member {k} {mode} nstep={nstep}")


@pytest.mark.parametrize("mode", ["fp64", "fp32"])
def test_tile_sizes_in_several_threads(mode):
    """Basins whose tiles differ in rows (and in LDS), each run by a thread of
    its own at once, give what each gives alone."""
    print(f"tiles of several sizes in threads, {mode}", flush=True)
    basins = [_basin(*shape, seed=21) for shape in ((64, 64), (256, 256), (512, 384))]
    out = [None] * len(basins)

    def run(k, reps):
        with BarotropicModel(basins[k]) as m:
            for _ in range(reps):
                m.run(3, mode, nstep=2)
            out[k] = m.get_state()

    for k in range(len(basins)):
        run(k, 20)
    alone = list(out)
    th = [threading.Thread(target=run, args=(k, 20)) for k in range(len(basins))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k, b in enumerate(basins):
        assert_bitwise(out[k], alone[k], STATE, f"{b.nx}x{b.ny} {mode}")
