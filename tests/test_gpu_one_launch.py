"""Pressure solves in one launch against the solve in pieces (needs a gfx950 GPU).

Up to 131,072 rows (16,384 in a periodic domain) the CG runs as one launch
whose blocks meet at grid barriers; the pieces still serve larger systems,
timed SpMV launches (the profile scalar) and systems whose blocks have no
16-bit window.  The sizes lie on both sides of the lines between the kinds.
Both solves stop by the same test on the same residual, so they take the same
number of iterations up to the rounding of the sums, and the answer is judged
by its residual on the assembled matrix.
"""
import numpy as np
import pytest

from polymps_amd import configs
from polymps_amd.lib import Simulation

pytestmark = pytest.mark.gpu


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
    g.set_scalar("profile", 1 if pieces else 0)
    g.set("ppe_x", guess)
    g.call("ppe_assemble")
    g.call("ppe_solve")
    return g.get("ppe_x"), int(g.scalar("solver_iter")), g.scalar("true_residual")


def _residual(m, b, x):
    rp, cols, vals = m
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    r = b - np.bincount(rows, vals * x[cols], len(b))
    return np.linalg.norm(r) / np.linalg.norm(b)


def _check(w, precision):
    w.params.precision_mode = precision
    w.params.ppe_transpose = 0
    w.params.solver_tol = 1e-8
    n = len(w.types)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh, device=0)
    g.call("init")
    guess = 0.9 * g.get("press") + 1e-3 * configs.splitmix64_uniform(5, n)
    x0, it0, res0 = _solve(g, guess, True)
    x1, it1, res1 = _solve(g, guess, False)
    m, b = g.ppe_matrix(), g.get("ppe_b")
    print(f"one launch {n} precision {precision}: {it0} and {it1} iterations, residuals {res0:.2e} {res1:.2e}", flush=True)
    assert it0 > 0 and abs(it1 - it0) <= 1 + it0 // 50
    # FP64 stops on the recurrence's residual, which drifts from the true one
    # by a few roundings of x per iteration: a hundredth of 1e-8 covers it
    assert res1 <= 1.01e-8
    # the reported residual is the matrix's, up to the rounding of its sums
    # (120 products of up to |a||x| ~ |b| each, eps 2.2e-16, against 1e-8)
    assert abs(_residual(m, b, x1) - res1) <= 1e-3 * res1 + 1e-13
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
    _check(_block(*shape), precision)


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
    g = _check(w, precision)
    assert g.scalar("ppe_window_blocks") < (len(w.types) + 255) // 256


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(64, 64, 64), (96, 64, 64), (97, 64, 64)])
def test_pieces(built, shape, precision):
    """Larger systems: the vector kernels take one row per thread up to 262,144
    rows and several above, and add the SpMV's sums themselves up to 393,216."""
    _check(_block(*shape), precision)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(24, 6, 12), (64, 32, 32), (64, 41, 25)])
def test_blocks_that_do_not_meet(built, shape, precision):
    """A wait of one poll: blocks give up at their first barriers, all leave,
    and the solve runs in pieces with the same answer; the counters are at
    zero for the next solve, which meets again."""
    w = _block(*shape)
    w.params.precision_mode = precision
    w.params.ppe_transpose = 0
    print(f"one poll {w.n} precision {precision}", flush=True)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh, device=0)
    g.call("init")
    guess = 0.9 * g.get("press") + 1e-3 * configs.splitmix64_uniform(5, w.n)
    x0, it0, _ = _solve(g, guess, False)
    g.set_scalar("grid_spin", 1)
    x1, it1, res1 = _solve(g, guess, False)
    assert abs(it1 - it0) <= 1 and res1 <= 1.01e-8
    assert _residual(g.ppe_matrix(), g.get("ppe_b"), x1) <= 1.01e-8
    g.set_scalar("grid_spin", 65536)
    x2, it2, _ = _solve(g, guess, False)
    assert it2 == it0 and np.array_equal(x0, x2)
