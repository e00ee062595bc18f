"""nsx_put_field / nsx_get_field: fields that cross in one chunk of layers, in
several and in ragged last ones, of every kind, periodic and walled: what
comes back is what went (bit for bit), periodic ghost rows are their
partners', rows that no rule fills stay as the caller left them."""
import ctypes

import numpy as np
import pytest

from nsx.abi import F
from nsx.case import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx, ny, nn, walls", [
    (2, 2, 2, None),          # small enough for the host to transpose
    (21, 11, 29, (1, 0, 0, 0)),  # the same with walls
    (32, 8, 30, None),        # 16,384 values: the most of those
    (33, 17, 31, (1, 0, 0, 0)),  # odd columns and layers, wall ghost rows
    (32, 16, 30, None),       # as many layers as a tile
    (90, 45, 67, None),       # 4.5 MB: two chunks, the last ragged
    (128, 64, 64, (0, 0, 0, 0)),  # three chunks
    (180, 91, 67, None),      # 18 MB: several threads copy
    (288, 229, 17, (1, 0, 0, 0)),  # 131,904 columns: three layers a chunk for four threads
    (400, 330, 16, None),     # 264,000 columns: one layer a chunk
])
def test_round_trip(nx, ny, nn, walls):
    from nsx.device import Context
    c = make_case(nx, ny, nn, seed=3, jitter=0.1, walls=walls)
    rng = np.random.default_rng(nx)
    G = Context(c)
    n0, nex = c.N_CELL0, c.N_CELLexact
    for name in ("UFN", "EDDY", "UFV", "UTFACE"):
        shape = G._shape(F[name])
        a = np.asfortranarray(rng.standard_normal(shape[::-1]).T)
        G.put(name, a)
        out = np.full(shape, -7.0, order="F")
        G._check(G.lib.nsx_get_field(G.h, F[name], ctypes.c_void_p(out.ctypes.data), 0))
        n = n0 if shape[0] == c.N_CELL else shape[0]
        assert np.array_equal(out[:n], a[:n]), name
        assert np.all(out[n:] == -7.0), name
        if shape[0] != c.N_CELL:
            continue
        G._check(G.lib.nsx_get_field(G.h, F[name], ctypes.c_void_p(out.ctypes.data), 1))
        partner = np.asarray(c.No_cp)[n0:nex, 2] - 1
        for g in range(n0, nex):
            wall = c.bcpc[g] == 1
            assert np.array_equal(out[g], a[g] if wall else a[partner[g - n0]]), (name, g)
        assert np.all(out[nex:] == -7.0), name
    G.close()


def test_small_mesh_takes_little():
    """The transfers' buffers follow the mesh: no megabytes on the device for
    fields of kilobytes (the allocator's own granule is 2 MB)."""
    from nsx.device import Context
    c = make_case(8, 6, 6, seed=3)
    G = Context(c)
    before = G.device_memory_used()
    G.put("UFN", c.u0)
    G.get("UFN")
    used = G.device_memory_used() - before
    G.close()
    assert used <= 2 << 20, used
