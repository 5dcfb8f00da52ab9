"""The per-kernel byte model and table tool (no GPU)."""
import json
import re
import sqlite3
import subprocess

from polymps_amd import roofline as R


def test_kernel_names():
    assert R._key("void mpsgpu::kPpeAssemble<true, true, true>(mpsgpu::KArgs, double*)") == \
        "kPpeAssemble<true, true, true>"
    assert R._key("void mpsgpu::(anonymous namespace)::kViscosityNN<true>(mpsgpu::KArgs)") == "kViscosityNN<true>"
    assert R._key("mpsgpu::kMxSpmv(mpsgpu::KArgs, mpsgpu::CgPtrs)") == "kMxSpmv"
    assert R._key("__amd_rocclr_copyBuffer") == "__amd_rocclr_copyBuffer"


def test_every_model_entry_names_a_kernel(built):
    """A kernel that is renamed or gets other template arguments must not
    fall out of the table: every entry is some kernel of the library, and the
    kernels that carry a step have one."""
    out = subprocess.run(["nm", "-C", str(built)], capture_output=True, text=True, check=True).stdout
    kernels = {R._key(m.group(1)) for m in re.finditer(r"__device_stub__(\S.*)", out)}
    m = R.model({"n": 1, "L": 1, "LS": 1, "nnz": 1, "nesc": 1, "nlc": 1})
    found = {id(R.bytesOf(m, k)) for k in kernels}
    assert [k for k, v in m.items() if id(v) not in found] == []
    for k in ("kViscosity<true, 4, 4, 4>", "kPndNeighNPCD<true, 2, 2, 4>", "kCorrectionMatrix<true, 1, 2, 4>",
              "kPressGradient<true, 2, 2, 4>", "kCollisionPC<true, 2, 2, 4>", "kPpeAssemble<true, true, true, false>",
              "kPpeAssemble<true, true, true, true>", "kCgUpdate<float, false>", "kCgP<float>", "kBuildList<true>"):
        assert k in kernels and R.bytesOf(m, k)[0], k
    assert R.bytesOf(m, "kPpeAssemble<true, true, true, true>")[0] == R.bytesOf(
        m, "kPpeAssemble<true, true, true, false>")[0] + 2
    # a bucket walk is not a list launch
    assert R.bytesOf(m, "kViscosity<false, 4, 1, 1>")[0] is None


def test_spmv_bytes_match_the_library_formula():
    """The SpMV figures are the ones the library's profiling counts per
    launch with the LDS windows (spmvBytes in ppe.hip): FP32 5 nnz + 2 nlc +
    16 n, FP64 9 nnz + 2 nlc + 28 n (one-byte window codes, two-byte window
    escapes)."""
    s = {"n": 1000, "L": 120000, "LS": 30000, "nnz": 117000, "nesc": 900, "nlc": 9500}
    m = R.model(s)
    assert m["kMxSpmv"][0] == 5 * 117000 + 2 * 9500 + 16 * 1000
    assert m["kCgSpmv"][0] == 9 * 117000 + 2 * 9500 + 28 * 1000
    # every list consumer counts its list at 4 B per entry
    assert m["kViscosity<true>"][0] == 4 * 120000 + 140 * 1000
    assert m["kCorrectionMatrix<true>"][0] == 4 * 30000 + 136 * 1000


def test_working_dispatches_drop_gated_launches():
    d = [300_000] * 10 + [3_000] * 5
    assert R._working(d) == [300_000] * 10


def test_table_from_databases(tmp_path):
    """A table from minimal databases of the rocprofv3 views it reads."""
    tr = tmp_path / "t.db"
    c = sqlite3.connect(tr)
    c.execute("create table kernels (name text, duration integer)")
    c.executemany("insert into kernels values (?, ?)",
                  [("mpsgpu::kMxSpmv(mpsgpu::KArgs, mpsgpu::CgPtrs)", 250_000)] * 4)
    c.commit()
    pm = {}
    for cn, v in (("FETCH_SIZE", 500.0), ("WRITE_SIZE", 10.0)):
        p = tmp_path / f"{cn}.db"
        c = sqlite3.connect(p)
        c.execute("create table counters_collection (kernel_name text, duration integer, value real, "
                  "counter_name text)")
        c.executemany("insert into counters_collection values (?, ?, ?, ?)",
                      [("mpsgpu::kMxSpmv(mpsgpu::KArgs, mpsgpu::CgPtrs)", 250_000, v, cn),
                       ("__amd_rocclr_copyBuffer", 100_000, 1024.0 * (0.5 if cn == "FETCH_SIZE" else 1.0), cn)])
        c.commit()
        pm[cn] = p
    log = tmp_path / "line.log"
    log.write_text("noise\n" + json.dumps({"metric": "x", "sizes": {
        "particles": 1000, "list_entries": 120000, "list_entries_small": 30000,
        "nnz": 117000, "nnz_escaped": 900}}) + "\n")

    class A:
        trace, fetch, write, sq = str(tr), str(pm["FETCH_SIZE"]), str(pm["WRITE_SIZE"]), None
        copy_fetch, copy_write, copy_bytes, sizes, top = str(pm["FETCH_SIZE"]), str(pm["WRITE_SIZE"]), \
            1024.0 * 1024.0, str(log), 5
    out = R.table(A)
    row = [l for l in out.splitlines() if l.startswith("| kMxSpmv")][0].split("|")
    alg = 6 * 117000 + 4 * 900 + 16 * 1000
    assert row[6].strip() == f"{alg / 1e6:.0f}"
    # FETCH x 2 and WRITE x 1 from the copy: (500 * 2 + 10) KiB
    assert row[9].strip() == f"{(500 * 2 + 10) * 1024 / 1e6:.0f}"
