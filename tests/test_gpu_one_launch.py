"""Pressure solves in one launch against the solve in pieces (needs a gfx950 GPU).

Up to 131,072 rows (16,384 in a periodic domain) the CG runs as one launch
whose blocks meet at grid barriers; the pieces still serve larger systems,
the one_launch scalar at 0 and systems whose blocks have no 16-bit window.  The sizes lie on both sides of the lines between the kinds.
Both solves stop by the same test on the same residual, so they take the same
number of iterations up to the rounding of the sums, and the answer is judged
by its residual on the assembled matrix.
"""
import ctypes

import numpy as np
import pytest

from polymps_amd import configs
from polymps_amd.lib import Simulation

pytestmark = pytest.mark.gpu

PIECES, ONE_LAUNCH, NO_WINDOW, LATE, BACKOFF = range(5)   # solve_path


def _block(nx, ny, nz, thin=0):
    l0 = 0.6 / nx
    b = (nx * l0, ny * l0, nz * l0)
    w = configs.dam3d_inc(l0=l0, tank=(1.61, b[1], 2.0 * b[2]), block=b, seed=9, jitter=0.05, margin=18.4 * l0)
    if thin:   # of the particles above three layers every thin-th stays; none counts as surface
        above = w.pos.reshape(-1, 3)[:, 2] > 3.0 * l0
        keep = ~above | (np.arange(w.n) % thin == 0)
        w.pos = w.pos.reshape(-1, 3)[keep].reshape(-1)
        w.vel = w.vel.reshape(-1, 3)[keep].reshape(-1)
        w.types = w.types[keep]
        w.params.pnd_threshold = w.params.neigh_threshold = 0.0
    return w


def _solve(g, guess, pieces):
    g.set_scalar("one_launch", 0 if pieces else 1)
    g.set("ppe_x", guess)
    g.call("ppe_assemble")
    g.call("ppe_solve")
    return g.get("ppe_x"), int(g.scalar("solver_iter")), g.scalar("true_residual")


def _widest_window(g):
    """Slots of the widest window: per 256-row block the union of its rows'
    stencil rows, in the slot order of the buckets (every row has entries)."""
    p, pos = g.params, g.get("pos").reshape(-1, 3)
    nb = np.array([p.num_buckets_x, p.num_buckets_y, p.num_buckets_z])
    c = np.floor((pos - np.array(p.domain_min)) * p.inv_bucket_side + 1e-8).astype(int)
    key = (c[:, 2] * nb[1] + c[:, 1]) * nb[0] + c[:, 0]
    order = np.argsort(key, kind="stable")
    c = c[order]
    start = np.searchsorted(key[order], np.arange(nb.prod() + 1))
    widest = 0
    for a in range(0, len(c), 256):
        s = []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                q = c[a:a + 256] + [0, dy, dz]
                q = q[((q >= 0) & (q < nb)).all(axis=1)]
                if len(q):
                    row = (q[:, 2] * nb[1] + q[:, 1]) * nb[0]
                    s.append((start[row + np.maximum(q[:, 0] - 1, 0)].min(),
                              start[row + np.minimum(q[:, 0] + 1, nb[0] - 1) + 1].max()))
        size, last = 0, 0
        for lo, hi in sorted(s):
            size += max(0, hi - max(lo, last))
            last = max(last, hi)
        widest = max(widest, size)
    return widest


def _residual(m, b, x):
    rp, cols, vals = m
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    r = b - np.bincount(rows, vals * x[cols], len(b))
    return np.linalg.norm(r) / np.linalg.norm(b)


def _check(w, precision, path=ONE_LAUNCH):
    w.params.precision_mode = precision
    w.params.ppe_transpose = 0
    w.params.solver_tol = 1e-8
    n = len(w.types)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh, device=0)
    g.call("init")
    guess = 0.9 * g.get("press") + 1e-3 * configs.splitmix64_uniform(5, n)
    x0, it0, res0 = _solve(g, guess, True)
    assert g.scalar("solve_path") == PIECES
    x1, it1, res1 = _solve(g, guess, False)
    assert g.scalar("solve_path") == path
    m, b = g.ppe_matrix(), g.get("ppe_b")
    print(f"one launch {n} precision {precision}: {it0} and {it1} iterations, residuals {res0:.2e} {res1:.2e}", flush=True)
    assert it0 > 0 and abs(it1 - it0) <= 1 + it0 // 50
    # FP64 stops on the recurrence's residual, which drifts from the true one
    # by a few roundings of x per iteration: a hundredth of 1e-8 covers it
    # the reported residual is the matrix's, up to the rounding of its sums
    # (120 products of up to |a||x| ~ |b| each, eps 2.2e-16, against 1e-8)
    for x, res in ((x0, res0), (x1, res1)):
        assert res <= 1.01e-8
        assert abs(_residual(m, b, x) - res) <= 1e-3 * res + 1e-13
    press = g.get("press")
    assert np.array_equal(press, np.where(x1 < 0, 0.0, x1))
    # a second solve from the same guess gives the same bits: sums in a fixed order
    x2, it2, _ = _solve(g, guess, False)
    assert it2 == it1 and np.array_equal(x1, x2)
    return g


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(7, 5, 3), (32, 16, 32), (32, 27, 19), (64, 32, 32), (64, 41, 25), (64, 64, 32),
                                   (76, 69, 25)])
def test_sizes(built, shape, precision):
    w = _block(*shape)
    _check(w, precision, ONE_LAUNCH if w.n <= 131072 else PIECES)


@pytest.mark.parametrize("precision", [0, 1])
def test_profile_changes_no_result(built, precision):
    """Timing does not choose the solver: same path, same bits."""
    w = _block(32, 16, 16)
    w.params.precision_mode = precision
    print(f"profile {w.n} precision {precision}", flush=True)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh, device=0)
    g.call("init")
    guess = 0.9 * g.get("press")
    x0, it0, _ = _solve(g, guess, False)
    g.set_scalar("profile", 1)
    x1, it1, _ = _solve(g, guess, False)
    assert g.scalar("solve_path") == ONE_LAUNCH and g.scalar("spmv_launches") == 0
    assert it0 == it1 and np.array_equal(x0, x1)
    # the pieces are timed, with the same bits too
    p0, _, _ = _solve(g, guess, True)
    assert g.scalar("solve_path") == PIECES and g.scalar("spmv_launches") > 0
    g.set_scalar("profile", 0)
    p1, _, _ = _solve(g, guess, True)
    assert np.array_equal(p0, p1)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("l0", [0.02, 0.016])
def test_periodic(built, l0, precision):
    """The window is the whole vector (a periodic image lies across the domain)."""
    _check(configs.periodic_channel3d(l0=l0, size=(0.32, 0.4)), precision)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(220, 80, 6), (300, 80, 6)])
def test_wide_windows(built, shape, precision):
    """A thin layer above a dense one: its blocks look at all of that.  Up to
    65,536 rows such a window is staged in parts (three in FP64, two in FP32
    here), above the solve goes back to pieces."""
    w = _block(*shape, thin=300)
    small = len(w.types) <= 65536
    g = _check(w, precision, ONE_LAUNCH if small else NO_WINDOW)
    assert _widest_window(g) > (16384 if small else 9216)   # slots of the LDS


@pytest.mark.parametrize("precision", [0, 1])
def test_windows_come_back(built, precision):
    """A context that solved without windows solves the next system as a new
    context does, in one launch and to the same bits."""
    wide, narrow = _block(300, 80, 6, thin=300), _block(301, 80, 3)
    l0 = wide.params.part_dist
    narrow.pos = narrow.pos * (l0 / (0.6 / 301))   # the lattice of the wide block
    n = wide.n
    assert n == narrow.n
    wide.params.precision_mode = precision
    wide.params.ppe_transpose = 0
    print(f"windows come back {n} precision {precision}", flush=True)
    a = Simulation(wide.params, wide.types, wide.pos, wide.vel, mesh=wide.mesh, device=0)
    b = Simulation(a.params, wide.types, narrow.pos, wide.vel, mesh=wide.mesh, device=0)
    a.call("init")
    assert a.scalar("solve_path") == NO_WINDOW
    _solve(a, a.get("press"), False)
    assert a.scalar("solve_path") == NO_WINDOW
    zero = np.zeros(n)
    args = [np.ascontiguousarray(v) for v in (wide.types, narrow.pos, wide.vel, zero, zero)]
    a._check(a._lib.mps_upload_state(a._h, *[v.ctypes.data_as(ctypes.c_void_p) for v in args]))
    for g in (a, b):
        g.set("ppe_x", zero)
        g.call("init")
        assert g.scalar("solve_path") == ONE_LAUNCH
    for f in ("press", "ppe_x", "ppe_b"):
        assert np.array_equal(a.get(f), b.get(f)), f
    assert a.scalar("solver_iter") == b.scalar("solver_iter") > 0


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(64, 64, 64), (96, 64, 64), (97, 64, 64)])
def test_pieces(built, shape, precision):
    """Larger systems: the vector kernels take one row per thread up to 262,144
    rows and several above, and add the SpMV's sums themselves up to 393,216."""
    _check(_block(*shape), precision, PIECES)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(24, 6, 12), (64, 32, 32), (64, 41, 25)])
def test_blocks_that_do_not_meet(built, shape, precision):
    """A wait of one poll: blocks give up at their first barriers, all leave,
    and the solve runs in pieces with the same answer, as does the next one;
    the counters are at zero for the next launch, which meets again."""
    w = _block(*shape)
    w.params.precision_mode = precision
    w.params.ppe_transpose = 0
    print(f"one poll {w.n} precision {precision}", flush=True)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh, device=0)
    g.call("init")
    guess = 0.9 * g.get("press") + 1e-3 * configs.splitmix64_uniform(5, w.n)
    x0, it0, _ = _solve(g, guess, False)
    assert g.scalar("solve_path") == ONE_LAUNCH
    g.set_scalar("grid_spin", 1)
    x1, it1, res1 = _solve(g, guess, False)
    assert g.scalar("solve_path") == LATE and g.scalar("solve_repeats") == 1
    x3, _, _ = _solve(g, guess, False)
    assert g.scalar("solve_path") == BACKOFF and g.scalar("solve_repeats") == 1
    # by other kernels than a retry, from the residual the assembly left: the same system and
    # guess, both answers at a residual of 1e-8
    assert _residual(g.ppe_matrix(), g.get("ppe_b"), x3) <= 1.01e-8
    assert abs(it1 - it0) <= 1 and res1 <= 1.01e-8
    assert _residual(g.ppe_matrix(), g.get("ppe_b"), x1) <= 1.01e-8
    g.set_scalar("grid_spin", 65536)
    x2, it2, _ = _solve(g, guess, False)
    assert g.scalar("solve_path") == ONE_LAUNCH
    assert it2 == it0 and np.array_equal(x0, x2)
