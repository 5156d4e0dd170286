"""Calls that fail on the host part of the way (an allocation, a launch, an error
left by other code) leave a system that the next call can use.  The library's
host code runs against a stand-in for the HIP runtime (cpp/hip_host_stub.cpp)
that fails a chosen call; kernels are recorded, not run.  No GPU."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRE = """
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_live_bytes.restype = stub.stub_most_items.restype = C.c_uint64
for f in ("calls", "live", "dirty_counts", "launches"):
    getattr(stub, "stub_" + f).restype = C.c_long
fail = lambda name, k=1: stub.stub_fail(name.encode(), C.c_long(k))
sys.path.insert(0, sys.argv[2])
import numpy as np
import particlebase_amd as pb

def raises(f, *a, **k):
    try:
        f(*a, **k)
    except pb.PBError:
        return True
    return False

def system(n=500, L=10.0, cells=None):
    s = pb.System(pb.Context(0), [n])
    s.set_cell([0, L] * 3)
    s.import_particles(np.zeros((n, 3)), np.ones(n))
    s.lj_set_params([1.0, 1.0], 1)
    s.lj_set_cutoff(6.25, shifted=True)
    if cells:
        s.setup_cells(cells)
    return s
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "cpp", "hip_host_stub.cpp")], check=True)

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRE + textwrap.dedent(code), out, os.path.dirname(HERE)],
                           capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stdout + p.stderr
    return run


@pytest.mark.parametrize("call", ["s.bin()", "s.lj_force()", "s.lj_run(0.001, 1)"])
@pytest.mark.parametrize("failure", ["stub.stub_pending_error()", "fail('k_scan')", "fail('k_scatter')",
                                     "fail('hipMalloc')"])
def test_sort_given_up_between_count_and_scatter(stub, call, failure):
    """The cells' counters are zero when the next sort counts (29791 cells: the
    scan allocates its block sums)."""
    stub(f"""
        s = system(500, 31.0, 1.0)
        s.lj_set_cutoff(1.0, shifted=True)
        {failure}
        raises(lambda: {call})
        stub.stub_fail(b"", C.c_long(0))
        for _ in range(2):
            s.bin()
            s.lj_force()
        assert stub.stub_launches(b"k_scatter") >= 4
        assert stub.stub_dirty_counts() == 0, stub.stub_dirty_counts()
    """)


ALLOCATING = {
    "cells": "s.setup_cells(1.0); s.bin()",
    "nlist": "s.setup_cells(2.5); s.coord_counts(6.25); s.nlist_build(6.25); s.lj_force_nlist()",
    "force": "s.lj_force()",
    "run": "s.lj_run(0.001, 1, energy_every=1); s.lj_run(0.001, 1, persistent=True)",
    "g(r)": "s.gr_hist(np.full(1, 0.1, np.float32), 50)",
    "sph": "s.setup_cells(1.0, periodic=False); s.sph_set_properties(one, one, 1.0); s.bin();"
           "s.sph_density(); s.sph_acceleration(); s.sph_inspect_density()",
    "wcsph": "s.setup_cells(1.0, periodic=False); s.sph_set_wcsph(0.5, 1.0, 10.0); s.bin();"
             "s.sph_density(); s.sph_acceleration()",
    "dem": "s.setup_cells(1.0, periodic=False); s.dem_set_properties(1e3, 0.5, 0.3, 0.1, 0.01, 0.4 * one);"
           "s.rot_set_inertia(0.4 * one); s.bin(); s.dem_calc_force(1e-4); s.dem_calc_force(1e-4);"
           "s.rot_step(1e-4)",
    "thermostat": "s.gt_step(0.001); s.mv2()",
}


@pytest.mark.parametrize("calls", list(ALLOCATING))
def test_failed_allocation(stub, calls):
    """Whichever allocation fails, the same calls made again end with all the
    device arrays of calls that never failed."""
    stub(f"""
        one = np.ones(500)
        def calls(s):
            {ALLOCATING[calls]}
        def mine(f):
            before = stub.stub_live(), stub.stub_live_bytes()
            f()
            return stub.stub_live() - before[0], stub.stub_live_bytes() - before[1]
        s = system()
        stub.stub_reset()
        want = mine(lambda: calls(s))
        n = stub.stub_calls(b"hipMalloc")
        assert n > 0
        for k in range(1, n + 1):
            s = system()
            def both():
                fail("hipMalloc", k)
                assert raises(calls, s), k
                calls(s)
            assert mine(both) == want, (k, n)
    """)


DEM = """
        one = np.ones(500)
        s = system(500, 10.0)
        s.setup_cells(1.0, periodic=False)
        s.dem_set_properties(1e3, 0.5, 0.3, 0.1, 0.01, 0.4 * one)
        s.rot_set_inertia(0.4 * one)
        s.bin()
        for _ in range(2):
            s.dem_calc_force(1e-4)
        s.dem_contacts()
"""


@pytest.mark.parametrize("kernel", ["k_dem_count", "k_scan", "k_dem_rows"])
def test_rewind_after_a_failed_contact_search(stub, kernel):
    """A search that fails has overwritten the rows of the matrix before the last:
    there is none to go back to."""
    stub(DEM + f"""
        fail("{kernel}")
        assert raises(s.dem_calc_force, 1e-4)
        s.dem_rewind()
        assert raises(s.dem_contacts)
        s.dem_calc_force(1e-4)
    """)


def test_contacts_whose_arrays_could_not_be_had(stub):
    """A restored matrix too large for its arrays (512) and for the memory: neither it
    nor the one before is there afterwards."""
    stub(DEM + """
        row = np.minimum(2 * np.arange(501), 998).astype(np.uint32)
        fail("hipMalloc")
        assert raises(s.dem_set_contacts, row, np.tile(np.arange(2, dtype=np.uint32), 499), np.zeros(998))
        assert raises(s.dem_contacts)
        s.dem_calc_force(1e-4)
    """)


@pytest.mark.parametrize("kernel,call", [("k_inverse_perm", "s.lj_force_nlist()"),
                                         ("k_dem_inv", "s.dem_calc_force(1e-4)")])
def test_inverse_order_that_was_not_made(stub, kernel, call):
    stub(f"""
        one = np.ones(500)
        s = system(500, 10.0, 2.5)
        if "{kernel}" == "k_dem_inv":
            s.dem_set_properties(1e3, 0.5, 0.3, 0.1, 0.01, 0.4 * one)
            s.rot_set_inertia(0.4 * one)
        s.bin()
        if "{kernel}" == "k_inverse_perm":
            s.nlist_build(6.25)
        stub.stub_reset()
        fail("{kernel}")
        assert raises(lambda: {call})
        {call}
        assert stub.stub_launches(b"{kernel}") == 1
    """)


def test_gr_noalloc_takes_nothing(stub):
    """pb_gr_hist_noalloc as the first call that moves data on its context: no device
    or pinned memory and no events are taken."""
    stub("""
        s = pb.System(pb.Context(0), [300])
        s.set_cell([0, 10.0] * 3)
        stub.stub_reset()
        step, hist = np.full(1, 0.1, np.float32), np.zeros(50, np.uint64)
        rc = s.lib.pb_gr_hist_noalloc(s.h, step.ctypes.data_as(C.POINTER(C.c_float)), 50,
                                      hist.ctypes.data_as(C.POINTER(C.c_uint64)))
        assert rc == pb.PB_OK
        assert [stub.stub_calls(x) for x in (b"hipMalloc", b"hipHostMalloc", b"hipEventCreate")] == [0, 0, 0]
    """)


@pytest.mark.parametrize("call", ["hipHostMalloc", "hipEventCreate"])
def test_context_that_could_not_be_made(stub, call):
    stub(f"""
        for k in (1, 2):
            fail("{call}", k)
            assert raises(pb.Context, 0), k
        system().get("r")
    """)


def test_list_of_the_largest_systems(stub):
    """Rows take a wavefront each: at 2^26 particles and more the work items of one
    launch would no longer fit in 32 bits."""
    stub("""
        n = (1 << 26) + 1
        s = pb.System(pb.Context(0), [n])
        s.set_cell([0, 10.0] * 3)
        s.lj_set_params([1.0, 1.0], 1)
        s.lj_set_cutoff(6.25)
        s.setup_cells(2.5)
        s.bin()
        s.coord_counts(6.25)
        s.nlist_build(6.25)
        s.lj_force_nlist()
        assert stub.stub_most_items() < 2 * n      # of all launches, whatever the lanes a row
    """)


@pytest.mark.parametrize("rmax", [4.0, 1e-7])        # two cells along an axis; too many cells
def test_refused_cells_leave_the_grid(stub, rmax):
    stub(f"""
        s = pb.System(pb.Context(0), [500])
        s.set_cell([0, 30.0, 0, 10.0, 0, 10.0])
        s.setup_cells(1.0)
        s.bin()
        before = s.cell_info()
        assert raises(s.setup_cells, {rmax})
        after = s.cell_info()
        assert all(np.array_equal(a, b) for a, b in zip(before, after)), after
        s.get_bins()
    """)


def test_cells_whose_arrays_could_not_be_had(stub):
    stub("""
        for k in range(1, 6):
            s = system(500, 10.0, 2.0)
            s.bin()
            fail("hipMalloc", k)
            assert raises(s.setup_cells, 1.0), k
            stub.stub_fail(b"", C.c_long(0))
            assert raises(s.bin) and raises(s.get_bins), k
            s.setup_cells(1.0)
            s.bin()
            fail("k_scatter")
            assert raises(s.bin) and raises(s.get_bins), k
    """)


def test_cell_order_after_a_failed_force(stub):
    """An LJ force that fails inside its own cell sort (here with more cells than the
    grid's) has given up the order that pb_bin made: calls that need it are errors
    until pb_bin ran again."""
    stub("""
        def fresh():
            s = system(500, 31.0, 5.0)
            s.lj_set_cutoff(1.0, shifted=True)
            s.bin()
            s.nlist_build(6.25)
            return s
        s = fresh()
        stub.stub_reset()
        s.lj_force()
        n = stub.stub_calls(b"hipMalloc")
        sort = [("hipMalloc", k) for k in range(1, n + 1)]
        sort += [(k, 1) for k in ("k_list_cellid", "k_scan", "k_scatter", "k_reorder")]
        lost = 0
        for what, k in sort:
            s = fresh()
            fail(what, k)
            assert raises(s.lj_force), (what, k)
            stub.stub_fail(b"", C.c_long(0))
            gone = raises(s.nlist_build, 6.25)
            assert gone == raises(s.get_bins), (what, k)
            lost += gone
            assert gone or what == "hipMalloc"
            s.bin()
            s.nlist_build(6.25)
        assert lost >= 6                          # two arrays of the cells, four kernels
    """)
