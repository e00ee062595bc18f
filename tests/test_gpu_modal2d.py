"""The vertical-mode solve (NSX_REFINE_MODAL) at the sizes where its parts end:
meshes of one, two and more levels of the 2D hierarchy, layers either side of
a 16-wide tile of the transforms, columns either side of a 16-column tile,
tables that need several panels, vectors that pass the LDS of a block, walls.
A random right-hand side solved to eps: the host-checked residual meets the
reference's rule (2 eps for the summation order), and the pressure agrees
with the FP64 BiCGSTAB's to what the two stopping errors allow (eps times the
operator's condition number, below 1e4 here: 1e-6)."""
import numpy as np
import pytest

from common import bc_case, interior, load_bc, ppe_residual, rel_err
from nsx.abi import PREC_MIXED, REFINE_MODAL
from nsx.case import make_case

pytestmark = pytest.mark.gpu

EPS = 1e-10


def _check(c, seed):
    from nsx.device import Context
    rng = np.random.default_rng(seed)
    rhs = c.cell_field()
    rhs[:c.N_CELL0, 1:-1] = rng.standard_normal((c.N_CELL0, c.NZ - 2))
    G = Context(c)
    G.set_params(eps=EPS)
    G.init_state()
    phi64, pv64, _ = G.bicgstab(c.cell_field(), rhs)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    phi, pv, info = G.bicgstab(c.cell_field(), rhs)
    again, _, _ = G.bicgstab(c.cell_field(), rhs)
    G.close()
    assert info["exit"] == "converged" and info["iters_fp32"] > 0, info
    e1, e2 = ppe_residual(c, phi, rhs)
    assert min(e1, e2) < 2 * EPS, (e1, e2)
    assert rel_err(interior(c, phi), interior(c, phi64)) <= 1e-6
    assert rel_err(pv, pv64) <= 1e-6
    assert np.array_equal(phi, again), "two runs of the same solve differ"


@pytest.mark.parametrize("nx, ny, nn", [
    (2, 2, 2),       # 8 columns, one level, two layers
    (8, 6, 15),      # 96 columns: the largest single level; one layer short of a tile
    (7, 7, 16),      # 98 columns: two levels, a column tile of two
    (13, 9, 17),     # one layer past a tile, odd columns
    (40, 21, 33),    # 1,680 columns, three levels
    (12, 8, 130),    # two panels
    (12, 8, 260),    # seventeen tiles: panels of the four that fit the LDS, the last with one
    (90, 41, 9),     # 7,380 columns: four levels, every vector in the block's LDS
    (110, 51, 6),    # 11,220 columns: two of the columns' four vectors in LDS
    (160, 76, 6),    # 24,320 columns, near the most that take a block per mode: none
    (160, 77, 6),    # 24,640: batched over the modes, ten of a tile's sixteen unused
    (201, 79, 17),   # odd columns, one mode past a tile
    (160, 80, 67),   # five tiles: thread groups that do not divide a block
])
def test_modal_sizes(nx, ny, nn):
    _check(make_case(nx, ny, nn, seed=11, jitter=0.1), seed=nx + nn)


@pytest.mark.parametrize("walls", [(1, 0, 0, 0), (0, 0, 0, 0), (0, 1, 1, 1)])
@pytest.mark.parametrize("nx, ny, nn", [(27, 15, 19), (159, 79, 7)])
def test_modal_walls_odd(nx, ny, nn, walls):
    _check(make_case(nx, ny, nn, seed=5, jitter=0.1, walls=walls), seed=3)


def test_modal_zero_and_solved_right_hand_sides():
    """A zero right-hand side and one solved already take no iterations; the pressure
    stays."""
    from nsx.device import Context
    c = bc_case(load_bc(), "duct", "steps")
    G = Context(c)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    G.init_state()
    zero = c.cell_field()
    phi, _, info = G.bicgstab(zero, zero)
    assert info["exit"] == "no solve" and info["iters"] == 0, info
    assert not np.any(interior(c, phi))
    rhs = c.cell_field()
    rhs[:c.N_CELL0, 1:-1] = np.random.default_rng(2).standard_normal((c.N_CELL0, c.NZ - 2))
    phi, _, info = G.bicgstab(zero, rhs)
    assert info["exit"] == "converged"
    again, _, info = G.bicgstab(phi, rhs)
    G.close()
    assert info["exit"] == "no solve" and info["iters"] == 0, info
    assert rel_err(interior(c, again), interior(c, phi)) <= 1e-12


@pytest.mark.parametrize("nn", [
    320,     # twenty tiles: four tiles' operands are the whole LDS
    1265,    # eighty tiles: one tile's operands are
    1300,    # not one tile's fit
])
def test_modal_deep_columns(nn):
    """The residual alone is checked: at these depths the operator's condition
    number, about the layers squared, leaves the pressures of two solves fewer
    common digits."""
    from nsx.device import Context
    c = make_case(3, 2, nn, seed=4, jitter=0.1)
    rhs = c.cell_field()
    rhs[:c.N_CELL0, 1:-1] = np.random.default_rng(nn).standard_normal((c.N_CELL0, c.NZ - 2))
    G = Context(c)
    G.set_params(eps=1e-8)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    G.init_state()
    phi, _, info = G.bicgstab(c.cell_field(), rhs)
    G.close()
    assert info["exit"] == "converged" and info["iters_fp32"] == info["iters"] > 0, info
    e1, e2 = ppe_residual(c, phi, rhs)
    assert min(e1, e2) < 2e-8, (e1, e2)


@pytest.mark.parametrize("bctop, bcbot", [(0, 1), (0, 0)])
@pytest.mark.parametrize("nx, ny, nn", [(40, 21, 33), (160, 77, 6)])
def test_modal_open_ends(nx, ny, nn, bctop, bcbot):
    """bctop or bcbot other than 1 leaves the end's coupling in the matrix, but
    every product mirrors the end layers, as get_Apk does: the operator stays
    the Neumann one that the modes are of, and two cycles solve it."""
    from nsx.device import Context
    c = make_case(nx, ny, nn, seed=6, jitter=0.1)
    c.bctop, c.bcbot = bctop, bcbot
    A, area = c.arrays, c.areaCell[:c.N_CELL0]
    if not bctop:
        A["AmCT"][:, -2] = area / c.dsig[-2]
    if not bcbot:
        A["AmCB"][:, 1] = area / c.dsig[0]
    A["AmC0"][:, 1:-1] = -1.0 * (A["AmCT"] + A["AmCB"] + A["AmC1"] + A["AmC2"] + A["AmC3"])[:, 1:-1]
    rhs = c.cell_field()
    rhs[:c.N_CELL0, 1:-1] = np.random.default_rng(nn).standard_normal((c.N_CELL0, c.NZ - 2))
    G = Context(c)
    G.set_params(eps=EPS)
    G.init_state()
    phi64, _, _ = G.bicgstab(c.cell_field(), rhs)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    phi, _, info = G.bicgstab(c.cell_field(), rhs)
    G.close()
    assert info["exit"] == "converged" and info["iters_fp32"] == info["iters"] > 0, info
    assert info["outer_passes"] == 2 and min(info["e1"], info["e2"]) < EPS, info
    assert rel_err(interior(c, phi), interior(c, phi64)) <= 1e-6


def _modes(c):
    """the vertical modes, columns of (NZ-2) x (NZ-2), and the layers' S"""
    n = c.NZ - 2
    t, S = 1.0 / c.dsig[1:n], c.dsigv[:n]
    T = np.zeros((n, n))
    for q in range(n - 1):
        T[q:q + 2, q:q + 2] += t[q] * np.array([[1.0, -1.0], [-1.0, 1.0]])
    r = 1.0 / np.sqrt(S)
    return r[:, None] * np.linalg.eigh(r[:, None] * T * r)[1], S


def _rhs_of_modes(c, parts):
    """the sum of amplitude x mode m x a random pattern of the columns"""
    phi, S = _modes(c)
    rhs = c.cell_field()
    for m, amplitude, seed in parts:
        f = np.random.default_rng(seed).standard_normal(c.N_CELL0)
        rhs[:c.N_CELL0, 1:-1] += amplitude * (f - f.mean())[:, None] * (S * phi[:, m])[None, :]
    return rhs


@pytest.mark.parametrize("easy_mode", [5, 2])
def test_modal_batched_does_not_remember(easy_mode):
    """A batched solve gives the bits of a fresh context's whatever the context
    solved before: an easy right-hand side (one high mode, few iterations)
    leaves few iterations queued for the next one."""
    from nsx.device import Context
    c = make_case(160, 77, 6, seed=11, jitter=0.1)
    hard = c.cell_field()
    hard[:c.N_CELL0, 1:-1] = np.random.default_rng(8).standard_normal((c.N_CELL0, c.NZ - 2))
    easy = _rhs_of_modes(c, [(easy_mode, 1.0, 9)])
    out = []
    for before in ([], [easy], [easy, easy, hard, easy]):
        G = Context(c)
        G.set_params(eps=EPS)
        G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
        G.init_state()
        its = [G.bicgstab(c.cell_field(), b)[2]["iters"] for b in before]
        phi, pv, info = G.bicgstab(c.cell_field(), hard)
        G.close()
        assert info["exit"] == "converged", info
        assert all(i < info["iters"] for i in its[:2]), (its, info)
        out.append((phi, pv, info["iters"], info["outer_passes"], info["e1"], info["e2"]))
    for o in out[1:]:
        assert o[2:] == out[0][2:], (o[2:], out[0][2:])
        assert np.array_equal(o[0], out[0][0]) and np.array_equal(o[1], out[0][1])


def test_modal_batched_timers_count_what_ran():
    """Of a solve that waits for more iterations the timers hold the cycles that
    ran, its 2D solves in two parts or more."""
    from nsx.device import Context
    c = make_case(160, 77, 6, seed=11, jitter=0.1)
    hard = c.cell_field()
    hard[:c.N_CELL0, 1:-1] = np.random.default_rng(8).standard_normal((c.N_CELL0, c.NZ - 2))
    G = Context(c)
    G.set_params(eps=EPS)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    G.init_state()
    G.bicgstab(c.cell_field(), _rhs_of_modes(c, [(5, 1.0, 9)]))
    G.timing(True)
    counts, swept = [], []
    for _ in range(2):
        G.timing_reset()
        info = G.bicgstab(c.cell_field(), hard)[2]
        for name in ("modal_fwd", "modal_bwd", "modal_spmv"):
            ms, n = G.timer(name)
            assert n == info["outer_passes"] and ms > 0, (name, n, info)
        counts.append(G.timer("modal_mg")[1])
        swept.append(G.timer("modal_swept")[1])
    G.close()
    assert counts[0] > counts[1] == info["outer_passes"], counts
    assert swept[0] == swept[1] >= info["iters"], swept


def test_modal_batched_finished_mode_stays():
    """Mode 1 ends before mode 0, which shares its group of four: its solution
    is the one it has beside mode 4, of the next group.  One cycle (the cap
    2 max_iters + 100 = 0), so that no later one hides a difference.  The two
    solves round differently in their sums and in the FP32 preconditioner,
    1e-7 of a step that is itself 2e-6 of the solution at the stop; steps
    taken after it made 1e-5."""
    from nsx.device import Context
    c = make_case(160, 77, 6, seed=11, jitter=0.1)
    phi, S = _modes(c)
    G = Context(c)
    G.set_params(eps=1e-6, max_iters=-50)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    G.init_state()
    x = []
    for other in (0, 4):
        p, _, info = G.bicgstab(c.cell_field(), _rhs_of_modes(c, [(1, 1.0, 3), (other, 100.0, 4)]))
        assert info["exit"] == "converged" and info["outer_passes"] == 1, info
        x.append(interior(c, p) @ (S * phi[:, 1]))
    G.close()
    assert rel_err(x[0], x[1]) <= 1e-10


def test_modal_contexts_of_two_sizes():
    """A small mesh's tables, made after a large one's, leave the large one's
    solves as they were (the kernels' LDS limits belong to the process)."""
    from nsx.device import Context
    cases = [make_case(90, 41, 9, seed=11, jitter=0.1), make_case(2, 2, 2, seed=11, jitter=0.1)]
    ctx, rhs, first = [], [], []
    for c in cases:
        G = Context(c)
        G.set_params(eps=EPS)
        G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
        G.init_state()
        r = c.cell_field()
        r[:c.N_CELL0, 1:-1] = np.random.default_rng(c.nx).standard_normal((c.N_CELL0, c.NZ - 2))
        ctx.append(G)
        rhs.append(r)
        first.append(G.bicgstab(c.cell_field(), r)[0])
    for G, c, r, phi in zip(ctx, cases, rhs, first):
        assert np.array_equal(G.bicgstab(c.cell_field(), r)[0], phi)
        G.close()


def test_modal_uneven_edges():
    """A mesh that nsx_commit takes: one cell lists a neighbour by two edges and
    is listed by one.  Its matrix is not symmetric and no solver converges;
    the solve ends as the FP64 one does, with a code and not with an error."""
    from nsx.device import Context
    c = make_case(13, 9, 6, seed=5, jitter=0.1, walls=(1, 0, 0, 0))
    A, cp, n0 = c.arrays, c.No_cp, c.N_CELL0
    i = next(q for q in range(n0 // 2, n0) if np.all(cp[q] <= n0) and np.all(cp[cp[q] - 1] <= n0))
    m = cp[i, 1] - 1
    f = list(cp[m]).index(i + 1)
    cp[i, 1] = cp[i, 0]
    cp[m, f] = next(g for g in cp[:n0].ravel() if g > n0 and c.bcpc[g - 1] == 1)
    A[f"AmC{f + 1}"][m] = 0.0
    A["AmC0"][m, 1:-1] = -1.0 * (A["AmCT"] + A["AmCB"] + A["AmC1"] + A["AmC2"] + A["AmC3"])[m, 1:-1]
    rhs = c.cell_field()
    rhs[:n0, 1:-1] = np.random.default_rng(1).standard_normal((n0, c.NZ - 2))
    G = Context(c)
    G.set_params(max_iters=50)
    G.init_state()
    _, _, i64 = G.bicgstab(c.cell_field(), rhs)
    G.set_precision(PREC_MIXED, REFINE_MODAL, 0.1, 30)
    _, _, info = G.bicgstab(c.cell_field(), rhs)
    G.close()
    assert info["exit"] == i64["exit"] == "max iterations", (info, i64)
