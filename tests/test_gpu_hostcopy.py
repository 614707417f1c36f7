"""State to host arrays through pinned slots: every element of every array, over
the sizes where it could go wrong (below and above the limit of the staged
copy, the first copies without slots and the later ones with them, whole slots,
a last chunk of one element), FP64 and widened FP32, into pageable and pinned
arrays, from two contexts at once, and two members of one ensemble at once."""
import ctypes as C
import threading

import numpy as np
import pytest

from _util import STATE, assert_bitwise
from inmsom_bt import BarotropicModel, make_basin, randomize_state
from inmsom_bt import _capi
from inmsom_bt.ensemble import Ensemble
from inmsom_bt.hipmem import hip

pytestmark = pytest.mark.gpu


def _basin(nx, ny, seed):
    b = make_basin(nx - 4, ny - 4, seed=seed, sigma=5.0)
    assert (b.nx, b.ny) == (nx, ny)
    rng = np.random.default_rng(seed)
    for k in STATE:
        setattr(b, k, rng.standard_normal((ny, nx)))
    return b


# arrays of 8 B: 64 x 64; 512 x 512 is one slot of 2 MiB; 377 x 809 a slot and
# 42849 more; 511 x 513 one element less than a slot
@pytest.mark.parametrize("nx,ny", [(64, 64), (512, 512), (511, 513), (377, 809), (1030, 515)])
def test_state_reaches_the_host(nx, ny):
    print(f"host copy {nx}x{ny}", flush=True)
    b = _basin(nx, ny, seed=nx)
    want = {k: np.ascontiguousarray(getattr(b, k)) for k in STATE}
    f32 = {k: (want[k].astype(np.float32).astype(np.float64) if k in ("u", "v", "ssh") else want[k]) for k in STATE}
    with BarotropicModel(b) as m, Ensemble([b, randomize_state(b, 3)], mode="fp32") as ens:
        for rep in range(min(8, 2 + (32 << 20) // (36 * nx * ny))):  # past the copies made without slots
            assert_bitwise(m.get_state(), want, STATE, f"context, call {rep}")
            assert_bitwise(ens.get_state(0), f32, STATE, f"FP32 member, call {rep}")
        ptr, size = C.c_void_p(), nx * ny * 8
        assert hip().hipHostMalloc(C.byref(ptr), C.c_size_t(6 * size), C.c_uint(0)) == 0
        try:
            order = ("u", "up", "v", "vp", "ssh", "sshp")
            at = [C.cast(ptr.value + k * size, _capi._dp) for k in range(6)]
            _capi.check(_capi.lib().inmsom_bt_get_state(m._h, *at), "inmsom_bt_get_state")
            pin = {f: np.ctypeslib.as_array(at[k], (ny, nx)).copy() for k, f in enumerate(order)}
        finally:
            hip().hipHostFree(ptr)
        assert_bitwise(pin, want, STATE, "pinned arrays")


def test_two_contexts_at_once():
    print("host copy, two contexts at once", flush=True)
    basins = [_basin(700, 600, seed=s) for s in (1, 2)]
    got = [None, None]
    with BarotropicModel(basins[0]) as m0, BarotropicModel(basins[1]) as m1:
        def read(k, m):
            got[k] = [m.get_state() for _ in range(6)]
        th = [threading.Thread(target=read, args=(k, m)) for k, m in enumerate((m0, m1))]
        for t in th:
            t.start()
        for t in th:
            t.join()
    for k, b in enumerate(basins):
        for g in got[k]:
            assert_bitwise(g, {f: np.asarray(getattr(b, f)) for f in STATE}, STATE, f"context {k}")


@pytest.mark.parametrize("mode", ["fp64", "fp32"])
def test_two_members_at_once(mode):
    """Threads that each read a member of one ensemble get that member's
    state, whole, every time."""
    print(f"host copy, members of one ensemble at once, {mode}", flush=True)
    basins = [_basin(700, 600, seed=s) for s in (3, 4, 5)]
    want = []
    for b in basins:
        want.append({f: np.asarray(getattr(b, f)) for f in STATE})
        if mode == "fp32":
            want[-1].update({f: want[-1][f].astype(np.float32).astype(np.float64) for f in ("u", "v", "ssh")})
    got = [None] * len(basins)
    with Ensemble(basins, mode=mode) as ens:
        def read(k):
            got[k] = [ens.get_state(k) for _ in range(6)]
        th = [threading.Thread(target=read, args=(k,)) for k in range(len(basins))]
        for t in th:
            t.start()
        for t in th:
            t.join()
    for k, w in enumerate(want):
        for rep, g in enumerate(got[k]):
            assert_bitwise(g, w, STATE, f"member {k}, read {rep}")
