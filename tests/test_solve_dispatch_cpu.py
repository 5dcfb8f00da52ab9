"""Host side of the pressure solve without a GPU: what it allocates and which
kernels it launches, on a runtime that only notes both (host_runtime.cpp).

Each case runs in a process of its own, which loads that runtime in the place
of the real one before the library.
"""
import ctypes
import re
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


# ------------------------------------------------------- in the child process
class Runtime:
    def __init__(self, path):
        self.dll = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.dll.test_launched.restype = ctypes.c_char_p
        self.dll.test_allocations.restype = ctypes.c_long
        self.dll.test_live.restype = ctypes.c_long
        self.dll.test_status_bytes.argtypes = [ctypes.c_size_t]
        self.dll.test_fail_allocation.argtypes = [ctypes.c_long]
        text = (ROOT / "polymps_amd" / "csrc" / "mps_internal.h").read_text()
        names = re.sub(r"//.*", "", re.search(r"enum IScalar \{(.*?)\}", text, re.S).group(1))
        self.slots = {s.strip(): k for k, s in enumerate(names.split(","))}
        self.dll.test_status_bytes(4 * self.slots["NIS"])

    def status(self, **ints):
        self.dll.test_status_clear()
        for name, v in ints.items():
            self.dll.test_status_int(self.slots[name], v)

    def launches(self):
        out = self.dll.test_launched().decode().split()
        self.dll.test_forget_launches()
        return out


def _sim(nx=12, ny=6, nz=6, solver=0, precision=0):
    from polymps_amd import configs
    from polymps_amd.lib import Simulation
    l0 = 0.6 / nx
    b = (nx * l0, ny * l0, nz * l0)
    w = configs.dam3d_inc(l0=l0, tank=(1.61, b[1], 2.0 * b[2]), block=b)
    w.params.solver_type, w.params.precision_mode = solver, precision
    return Simulation(w.params, w.types, w.pos, w.vel)


def _solve(g):
    g.call("ppe_assemble")
    g.call("ppe_solve")


def allocations(rt, solver, precision, learned):
    """Whichever of its allocations fails, a solve reports it, and the next
    one makes every buffer that is missing."""
    from polymps_amd.lib import MpsError
    rt.status(I_CG_DONE=1)

    def run(g):
        if learned:
            g.gnn_init(0)
            g.set_scalar("learned_mode", 1)
        _solve(g)

    def made(fail):
        g = _sim(solver=solver, precision=precision)
        live, before = rt.dll.test_live(), rt.dll.test_allocations()
        rt.dll.test_fail_allocation(fail)
        failed = False
        try:
            run(g)
        except MpsError as e:
            assert "out of memory" in str(e), e
            failed = True
        rt.dll.test_fail_allocation(0)
        run(g)
        n = rt.dll.test_live() - live
        calls = rt.dll.test_allocations() - before
        g.close()
        return n, calls, failed

    clean, calls, failed = made(0)
    assert clean > 0 and not failed
    for k in range(1, calls + 1):
        n, _, failed = made(k)
        assert failed, k
        assert n == clean, f"allocation {k} of {calls} failed: {n} buffers afterwards, {clean} without a failure"
    assert rt.dll.test_live() == 0


ONE_LAUNCH = ("kCgOneLaunch", "kMxOneLaunch")


def meshes(rt, kind):
    """A wall mesh whose allocation fails is not installed half: the closest
    point search refuses it or does without its tree, and the next mesh and
    the context's end find no pointer of it."""
    from polymps_amd import configs
    from polymps_amd.lib import MpsError
    V, F = configs.channel_mesh(nhx=8, nhy=8)[:2]
    mesh = configs.mesh_arrays(V, F)
    assert len(mesh[1]) // 3 > 64   # with a tree

    def install(g):
        g.set_mesh_type(kind, *mesh)

    def made(fail):
        g = _sim()
        install(g)   # one to replace
        live, before = rt.dll.test_live(), rt.dll.test_allocations()
        rt.dll.test_fail_allocation(fail)
        failed = False
        try:
            install(g)
        except MpsError as e:
            assert "out of memory" in str(e), e
            failed = True
        calls = rt.dll.test_allocations() - before
        rt.dll.test_fail_allocation(0)
        rt.launches()
        refused = False
        try:
            g.closest_point_type(kind)
        except MpsError:
            refused = True
        got = rt.launches()
        if refused:
            assert not any(k.startswith("kClosestPoint") for k in got)
        else:
            assert ("kClosestPointBvh" in got) == (not failed)
        install(g)
        n = rt.dll.test_live() - live
        g.close()
        return n, calls, failed, refused

    n, calls, failed, refused = made(0)
    assert n == 0 and calls >= 3 and not failed and not refused
    for k in range(1, calls + 1):
        n, _, failed, refused = made(k)
        assert failed and n == 0, k
        assert refused or (kind == 0 and k > 3), k
    assert rt.dll.test_live() == 0


def path(rt, precision):
    """solve_path says what was launched: the one launch alone, or the pieces
    after it and why, or the pieces alone."""
    g = _sim(precision=precision)
    if precision:
        # a mixed solve in pieces reads |r|^2 and |b|^2 as 0 here and ends before its first pass
        pieces = "kTrueResidualFinish"
    else:
        pieces = "kCgSpmv"
    for ints, want in ((dict(), 1), (dict(I_GRID_LATE=1), 3), (dict(), 1), (dict(I_NOWIN=1), 2)):
        rt.status(I_CG_DONE=1, **ints)
        g.set_scalar("grid_spin", 4096)   # tries again after a give-up
        rt.launches()
        _solve(g)
        got = rt.launches()
        assert any(k.startswith(ONE_LAUNCH) for k in got)
        assert any(k == pieces for k in got) == (want != 1), (want, got)
        assert g.scalar("solve_path") == want
        # the assembly's residual serves the pieces unless blocks may have moved the guess
        first = "kTrueResidual" if precision else "kCgStart"
        assert got.count(first) == (1 if want == 3 else 0)
    g.close()
    rt.status(I_CG_DONE=1)
    g = _sim(solver=1)
    _solve(g)
    assert g.scalar("solve_path") == 0
    g.close()


def backoff(rt, precision):
    """After a barrier gave up the next solves run in pieces without a try, 4
    of them, then twice as many each time; a solve in one launch starts over."""
    g = _sim(precision=precision)
    assert g.scalar("grid_spin") == 4096
    paths = []

    def solves(n):
        for _ in range(n):
            rt.launches()
            _solve(g)
            paths.append(int(g.scalar("solve_path")))
            tried = any(k.startswith(ONE_LAUNCH) for k in rt.launches())
            assert tried == (paths[-1] != 4)

    rt.status(I_CG_DONE=1, I_GRID_LATE=1)
    solves(1 + 4 + 1 + 8 + 1 + 16 + 1)
    assert paths == [3] + 4 * [4] + [3] + 8 * [4] + [3] + 16 * [4] + [3]
    assert g.scalar("solve_repeats") == 4
    rt.status(I_CG_DONE=1)
    paths.clear()
    solves(32 + 2)
    assert paths == 32 * [4] + [1, 1]
    rt.status(I_CG_DONE=1, I_GRID_LATE=1)
    paths.clear()
    solves(6)
    assert paths == [3, 4, 4, 4, 4, 3]
    rt.status(I_CG_DONE=1)
    g.set_scalar("grid_spin", 100)
    paths.clear()
    solves(1)
    assert paths == [1] and g.scalar("grid_spin") == 100
    # the longest wait
    rt.status(I_CG_DONE=1, I_GRID_LATE=1)
    paths.clear()
    while paths.count(3) < 12:
        solves(1)
    late = [k for k, p in enumerate(paths) if p == 3]
    gaps = [b - a - 1 for a, b in zip(late, late[1:])]
    assert gaps == [4, 8, 16, 32, 64, 128, 256, 512, 1024, 1024, 1024]
    g.close()


def no_window(rt, precision):
    """After a launch that left for want of a window the pieces come first,
    until the assembly's flag is down again."""
    g = _sim(precision=precision)
    # what kCgStartFinish sets where it finds the flag down
    down = dict(I_CG_DONE=1 if precision else 6)
    up = dict(I_CG_DONE=1, I_NOWIN=1)
    for ints, want, tries in ((up, 2, 1), (up, 2, 0), (up, 2, 0), (down, 1, 1), (down, 1, 1), (up, 2, 1), (up, 2, 0)):
        rt.status(**ints)
        rt.launches()
        _solve(g)
        got = rt.launches()
        assert g.scalar("solve_path") == want
        assert sum(k.startswith(ONE_LAUNCH) for k in got) == tries
        # the assembly's residual serves whichever solves the system
        assert ("kTrueResidual" if precision else "kCgStart") not in got
    # a guess that moved after the assembly: its residual is computed for the pieces, and by the launch itself
    rt.status(**down)
    g.call("ppe_assemble")
    g.set_scalar("solver_failures", 0)
    rt.launches()
    g.call("ppe_solve")
    got = rt.launches()
    assert g.scalar("solve_path") == 1
    assert got.count("kTrueResidual" if precision else "kCgStart") == 1
    g.close()


def periodic(rt, precision):
    """A periodic domain's assembly makes no window tables or codes that no solve reads."""
    from polymps_amd import configs
    from polymps_amd.lib import Simulation
    rt.status(I_CG_DONE=1)
    w = configs.periodic_channel3d_polygon(l0=0.05, size=(0.3, 0.4))
    w.params.precision_mode = precision
    made = []
    for window in (0, 1):
        g = Simulation(w.params, w.types, w.pos, w.vel)
        g.set_scalar("ppe_window", window)
        live = rt.dll.test_live()
        rt.launches()
        _solve(g)
        got = rt.launches()
        assert "kPpeWindow" not in got and sum(k.startswith(ONE_LAUNCH) for k in got) == 1
        made.append(rt.dll.test_live() - live)
        g.close()
    assert made[0] == made[1]


def switches(rt, precision):
    """one_launch chooses the solver and the memory of its windows; profile does not."""
    from polymps_amd.lib import MpsError
    rt.status(I_CG_DONE=1)
    g = _sim(precision=precision)
    live = rt.dll.test_live()
    g.set_scalar("ppe_window", 0)
    g.set_scalar("one_launch", 0)
    for profile in (0, 1):
        g.set_scalar("profile", profile)
        rt.launches()
        _solve(g)
        assert not any(k.startswith(ONE_LAUNCH) for k in rt.launches())
        assert g.scalar("solve_path") == 0 and g.scalar("one_launch") == 0
    # neither windows nor the buffers of a solve in one launch (a mixed solve makes its eight, profile the entry sum)
    assert rt.dll.test_live() - live == (9 if precision else 1)
    g.set_scalar("one_launch", 1)
    for profile in (0, 1):
        g.set_scalar("profile", profile)
        rt.launches()
        _solve(g)
        assert sum(k.startswith(ONE_LAUNCH) for k in rt.launches()) == 1
        assert g.scalar("solve_path") == 1
    try:
        g.set_scalar("one_launch", 2)
        raise AssertionError("one_launch 2 was accepted")
    except MpsError:
        pass
    g.close()


def attributes(rt, precision):
    """A device that refuses the kernel's LDS size gets the solve in pieces."""
    rt.status(I_CG_DONE=1)
    for refuse in (0, 1):
        rt.dll.test_refuse_attributes(refuse)
        g = _sim(precision=precision)
        rt.launches()
        _solve(g)
        one = [k for k in rt.launches() if k.startswith(ONE_LAUNCH)]
        assert len(one) == (0 if refuse else 1), one
        g.close()


# ------------------------------------------------------------------ the tests
@pytest.fixture(scope="module")
def runtime(built, tmp_path_factory):
    out = tmp_path_factory.mktemp("runtime") / "libamdhip64.so.7"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(ROOT / "tests" / "host_runtime.cpp"), "-Wl,-soname,libamdhip64.so.7",
                    f"-Wl,--version-script={ROOT / 'tests' / 'host_runtime.map'}", "-o", str(out)], check=True)
    return out


def _child(runtime, case, *args):
    res = subprocess.run([sys.executable, __file__, str(runtime), case, *map(str, args)], capture_output=True,
                         text=True, timeout=300, cwd=ROOT)
    assert res.returncode == 0, (res.stdout + res.stderr)[-3000:]


@pytest.mark.parametrize("solver,precision,learned", [(0, 0, 0), (0, 1, 0), (1, 0, 0), (0, 0, 1)])
def test_allocation_failures(runtime, solver, precision, learned):
    _child(runtime, "allocations", solver, precision, learned)


@pytest.mark.parametrize("kind", [0, 2])
def test_mesh_allocation_failures(runtime, kind):
    _child(runtime, "meshes", kind)


@pytest.mark.parametrize("precision", [0, 1])
def test_solve_path(runtime, precision):
    _child(runtime, "path", precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_backoff(runtime, precision):
    _child(runtime, "backoff", precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_no_window(runtime, precision):
    _child(runtime, "no_window", precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_periodic_windows(runtime, precision):
    _child(runtime, "periodic", precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_switches(runtime, precision):
    _child(runtime, "switches", precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_refused_kernel_attributes(runtime, precision):
    _child(runtime, "attributes", precision)


if __name__ == "__main__":
    sys.path.insert(0, str(ROOT))
    globals()[sys.argv[2]](Runtime(sys.argv[1]), *map(int, sys.argv[3:]))
