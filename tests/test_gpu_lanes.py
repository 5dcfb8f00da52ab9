"""Operators at every number of lanes per particle (needs a gfx950 GPU).

The neighbour sums run with 16, 4 or fewer lanes per particle, chosen by the
particle count.  Their terms are added in the reference's order whatever the
split, so each operator equals the oracle bit for bit; the sizes here lie on
both sides of the lines between the splits and leave wavefronts and batches
partly filled.
"""
import numpy as np
import pytest

from polymps_amd import configs
from polymps_amd.lib import MpsError, Simulation
from tests.parity_util import check, new_pair

pytestmark = pytest.mark.gpu


def _velocity(n, seed, dim):
    v = 2.0 * configs.splitmix64_uniform(seed, 3 * n).reshape(n, 3) - 1.0
    if dim == 2:
        v[:, 2] = 0.0
    return v.reshape(-1)


def _dam3d(nx, ny, nz):
    l0 = 0.6 / nx
    b = (nx * l0, ny * l0, nz * l0)
    # a strong jitter: some pairs closer than the collision distance, ragged neighbour counts
    w = configs.dam3d_inc(l0=l0, tank=(1.61, b[1], 2.0 * b[2]), block=b, seed=9, jitter=0.2)
    w.vel = _velocity(w.n, 31, 3)
    return w


@pytest.mark.parametrize("shape", [(7, 5, 3), (24, 6, 12), (32, 16, 16), (31, 17, 16), (64, 32, 40), (65, 32, 40)])
def test_polygon_wall_operators(built, shape):
    w = _dam3d(*shape)
    print(f"lanes {shape} {w.n}", flush=True)
    g, o = new_pair(w)

    def both(gop, oop, fields):
        g.call(gop)
        o.call(oop)
        check(g, o, fields, f"{w.n} {gop}")

    g.call("bucket_update"); o.call("update_buckets")
    both("viscosity", "viscosity", ["acc"])          # bucket walk
    g.call("build_neighbor_list")
    both("viscosity", "viscosity", ["acc"])          # list
    both("mesh_closest_point", "closest_point", ["riw2", "mirror"])
    both("mesh_update_near", "update_near_mesh", ["near_wall"])
    both("wall_npcd", "wall_npcd", ["npcd"])
    both("pnd_neigh_npcd", "pnd_neigh_npcd", ["num_neigh", "pnd_small", "npcd", "npcd2"])
    p = 1e4 * configs.splitmix64_uniform(77, w.n)
    g.set("press", p); o.set("press", p)
    both("correction_matrix", "correction_matrix", ["cm1", "cm2", "cm3"])
    both("vel_divergence", "vel_divergence", [])
    o.call("wall_vel_divergence")
    check(g, o, ["div_u"], f"{w.n} vel_divergence")
    both("press_gradient", "press_gradient", ["acc"])
    both("wall_press_gradient", "wall_press_gradient", ["acc", "force_wall"])
    both("wall_viscosity", "wall_viscosity", ["acc", "force_wall"])
    both("collision", "collision", ["vel"])
    assert np.any(g.get("vel") != w.vel)   # some pairs collided


@pytest.mark.parametrize("by", ["upload", "closest_point"])
def test_types_after_the_flags_are_dropped(built, by):
    """update_bc packs two flags next to the neighbours' types.  What makes the
    flags stale, an upload or new wall distances, leaves the types: dummy
    walls stay out of the matrix and walls keep their viscosity."""
    w = configs.dam2d_wc_long(l0=0.02, jitter=0.05)
    w.vel = _velocity(w.n, 33, 2)
    w.params.mps_type, w.params.pnd_type, w.params.knm_vs2 = 2, 0, 3e-6
    if by == "closest_point":   # particle walls inside a box mesh
        w.mesh = configs.mesh_arrays(*configs.box_mesh((-1.0, -1.0, -1.0), (2.0, 2.0, 1.0)))
    print(f"types after {by} {w.n}", flush=True)
    g, o = new_pair(w)
    g.call("init")
    o.call("init")
    assert (w.types != 0).any()
    if by == "upload":
        g.set("press", g.get("press"))
        g.set("ppe_x", g.get("ppe_x"))
    else:
        g.call("mesh_closest_point")
        o.call("closest_point")
    g.call("ppe_assemble")
    o.call("assemble_ppe")
    for x, y in zip(_sorted_coo(*g.ppe_matrix(), transpose=False), _sorted_coo(*o.ppe_matrix(), transpose=True)):
        assert np.array_equal(x, y)
    check(g, o, ["ppe_b"], "ppe_assemble")
    g.call("viscosity")
    o.call("viscosity")
    check(g, o, ["acc"], "viscosity")


@pytest.mark.parametrize("shape", [(7, 5, 3), (48, 12, 24), (65, 32, 40), (63, 33, 45)])
def test_queued_particles(built, shape):
    """A window of one word queues every particle with more than 32 candidates
    in a stencil row, almost all here; a queue of up to 16,384 takes a
    wavefront per particle, a longer one eight lanes.  Both give the lists of
    the full window: same entries, same sums in bits."""
    w = _dam3d(*shape)
    print(f"queue {shape} {w.n}", flush=True)
    out = []
    for words in (0, 1):
        g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh)
        if words:
            g.set_scalar("mask_words", words)
        g.call("bucket_update")
        g.call("build_neighbor_list")
        r = [g.scalar("list_entries"), g.scalar("list_entries_small"), g.scalar("list_max")]
        for op in ("viscosity", "pnd_neigh_npcd", "correction_matrix"):
            g.call(op)
        r += [g.get(f) for f in ("acc", "num_neigh", "pnd_small", "npcd", "cm1", "cm2", "cm3")]
        out.append(r)
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("l0", [0.02, 0.005, 0.0025, 0.00125])
def test_particle_wall_operators(built, l0):
    w = configs.dam2d_wc_long(l0=l0, jitter=0.1)
    w.vel = _velocity(w.n, 32, 2)
    print(f"lanes 2-D {w.n}", flush=True)
    g, o = new_pair(w)

    def both(gop, oops, fields):
        g.call(gop)
        for op in oops:
            o.call(op)
        check(g, o, fields, f"{w.n} {gop}")

    g.call("bucket_update"); o.call("update_buckets")
    g.call("build_neighbor_list")
    both("viscosity", ["viscosity"], ["acc"])
    both("pnd_neigh_npcd", ["pnd_neigh_npcd"], ["num_neigh", "pnd_small"])
    p = 1e4 * configs.splitmix64_uniform(78, w.n)
    pn = g.get("pnd_small")   # a PND as the step leaves it
    for s in (g, o):
        s.set("press", p)
        s.set("pndi", pn)
    both("correction_matrix", ["correction_matrix"], ["cm1", "cm2", "cm3"])
    both("pnd_diffusive", ["pnd_diffusive", "update_pnd", "mean_pnd_wall_dummy_surface"], ["pndi", "div_u", "diffusive"])
    both("update_bc", ["update_bc"], ["bc"])
    both("extrapolate_wall_dummy", ["extrapolate_wall_dummy"], ["press"])
    both("press_gradient", ["press_gradient"], ["acc"])
    both("collision", ["collision"], ["vel"])
    both("wall_dummy_velocity", ["wall_dummy_velocity"], ["vel"])   # bucket walks from here
    both("shifting", ["shifting"], ["pos"])


@pytest.mark.parametrize("l0", [0.01, 0.004, 0.0014])
def test_periodic_lists(built, l0):
    """Lists of a periodic domain by 64, 16 and 4 lanes per particle, seen
    through the sums over them (the neighbours across the seam among them)."""
    w = configs.periodic_channel2d(l0=l0, length=round(0.8 / l0) * l0, depth=round(0.2 / l0) * l0, mps_type=2,
                                   jitter=0.1)
    print(f"periodic lists {w.n}", flush=True)
    g, o = new_pair(w)
    g.call("bucket_update"); o.call("update_buckets")
    g.call("build_neighbor_list")
    for op, fields in (("viscosity", ["acc"]), ("pnd_neigh_npcd", ["num_neigh", "pnd_small", "npcd"]),
                       ("correction_matrix", ["cm1", "cm2", "cm3"])):
        g.call(op)
        o.call(op)
        check(g, o, fields, f"{w.n} {op}")


def _sorted_coo(rp, cols, vals, transpose):
    r = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    if transpose:
        r, cols = cols, r
    k = np.lexsort((cols, r))
    return r[k], cols[k], vals[k]


def _check_assembly(w, precision):
    w.params.precision_mode = precision
    g, o = new_pair(w)
    g.call("init")
    o.call("init")
    g.set("press", o.get("press"))
    guess = o.get("press") * 0.9
    for s in (g, o):
        s.set("ppe_x", guess)
    g.call("ppe_assemble")
    o.call("assemble_ppe")
    a = _sorted_coo(*g.ppe_matrix(), transpose=False)
    b = _sorted_coo(*o.ppe_matrix(), transpose=True)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    check(g, o, ["ppe_b"], f"{w.n} ppe_assemble")
    # the 16-bit window indices, through the solve in one launch
    g.call("ppe_solve")
    assert g.scalar("solve_path") == 1 and g.scalar("true_residual") <= 1e-8
    # the one-byte codes, through the solve in pieces: every block is served
    # from its window, and gathering from global memory gives the same bits
    g.set_scalar("one_launch", 0)
    x = []
    for window in (1, 0):
        g.set_scalar("ppe_window", window)
        g.set("ppe_x", guess)
        g.call("ppe_assemble")
        assert g.scalar("ppe_window_blocks") == window * ((w.n + 255) // 256)
        g.call("ppe_solve")
        assert g.scalar("solve_path") == 0 and g.scalar("true_residual") <= 1e-8
        x.append(g.get("ppe_x"))
    assert np.array_equal(*x) and np.any(x[0] != guess)


@pytest.mark.parametrize("shape", [(7, 5, 3), (32, 16, 16), (31, 17, 16), (64, 32, 32), (65, 32, 32)])
@pytest.mark.parametrize("precision", [0, 1])
def test_assembly(built, shape, precision):
    """The assembled system with 16, 4 and one lane per row: entries and
    right-hand side bit for bit, and the mixed solve's FP32 entries, codes and
    first residual through the solutions they give."""
    w = _dam3d(*shape)
    print(f"assembly {shape} {w.n} precision {precision}", flush=True)
    _check_assembly(w, precision)


@pytest.mark.parametrize("l0", [0.02, 0.0027, 0.0024])
@pytest.mark.parametrize("precision", [0, 1])
def test_assembly_2d(built, l0, precision):
    """The same in 2-D, with 4 lanes per row up to 20,480 rows and one above."""
    w = configs.dam2d_wc_long(l0=l0, tank=(round(1.0 / l0) * l0, round(0.6 / l0) * l0),
                              column=(round(0.25 / l0) * l0, round(0.5 / l0) * l0), jitter=0.05)
    w.params.mps_type, w.params.pnd_type, w.params.solver_tol = 2, 0, 1e-8
    print(f"assembly 2-D {w.n} precision {precision}", flush=True)
    _check_assembly(w, precision)


def test_wide_radius(built):
    """A large radius of 4.1 l0 takes mask rows of more than 512 candidates.
    Up to 81,920 particles the lists come from group walks, which need none;
    above, the build refuses unless the caller narrows the window."""
    w = _dam3d(24, 6, 12)
    w.params.re_l = 4.1
    print(f"wide radius {w.n}", flush=True)
    g, o = new_pair(w)
    assert g.scalar("list_capacity") > 512
    g.call("bucket_update"); o.call("update_buckets")
    g.call("build_neighbor_list")
    for op, fields in (("viscosity", ["acc"]), ("pnd_neigh_npcd", ["num_neigh", "pnd_small", "npcd"])):
        g.call(op)
        o.call(op)
        check(g, o, fields, op)
    w = _dam3d(24, 6, 12)
    w.params.re_l = 4.1
    _check_assembly(w, 1)
    w = _dam3d(78, 33, 32)
    w.params.re_l = 4.1
    print(f"wide radius {w.n}", flush=True)
    g = Simulation(w.params, w.types, w.pos, w.vel, mesh=w.mesh)
    with pytest.raises(MpsError, match="512 candidates"):
        g.call("init")
    g.set_scalar("mask_words", 16)
    g.call("init")
    assert g.scalar("list_max") > 200
