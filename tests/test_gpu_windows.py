"""The FP64 BiCGSTAB either side of the sizes where its launches change shape:
one window of 256 quads and less, a last window of one quad, as many windows as
take one a block (160) and one more, 512 and one more row of columns.  A random right-hand side
solved to 1e-12: the host-checked residual meets the reference's rule (2 eps
for the summation order), the pressure agrees with the vertical-mode solve's
(eps times the operator's condition number, below 1e5 here: 1e-7), and a
second run gives the same bits."""
import numpy as np
import pytest

from common import interior, ppe_residual, rel_err
from nsx.abi import PREC_FP64, PREC_MIXED, REFINE_MODAL
from nsx.case import make_case

pytestmark = pytest.mark.gpu

EPS = 1e-12


@pytest.mark.parametrize("nx, ny, nn, walls", [
    (2, 2, 2, None),           # 8 quads
    (16, 8, 2, None),          # 256: one window
    (43, 3, 2, (1, 0, 0, 0)),  # 258: two quads in the second
    (32, 16, 32, None),        # 36 windows, not a multiple of the XCDs
    (80, 85, 10, None),        # 160 windows: the most one window a block takes
    (72, 95, 10, None),        # 161: the general form
    (176, 124, 10, None),      # 512 windows
    (190, 115, 10, None),      # 513
])
def test_bicgstab_window_counts(nx, ny, nn, walls):
    from nsx.device import Context
    c = make_case(nx, ny, nn, seed=13, jitter=0.1, walls=walls, stretch=1.0)
    rhs = c.cell_field()
    rhs[:c.N_CELL0, 1:-1] = np.random.default_rng(nx).standard_normal((c.N_CELL0, c.NZ - 2))
    G = Context(c)
    G.set_params(eps=EPS)
    G.init_state()
    out = {}
    for prec in (PREC_FP64, PREC_MIXED):
        G.set_precision(prec, REFINE_MODAL, 0.1, 30)
        phi, _, info = G.bicgstab(c.cell_field(), rhs)
        assert info["exit"] == "converged", (prec, info)
        e1, e2 = ppe_residual(c, phi, rhs)
        assert min(e1, e2) < 2 * EPS, (prec, e1, e2)
        out[prec] = phi
        again, _, _ = G.bicgstab(c.cell_field(), rhs)
        assert np.array_equal(phi, again)
    G.close()
    assert rel_err(interior(c, out[PREC_FP64]), interior(c, out[PREC_MIXED])) <= 1e-7
