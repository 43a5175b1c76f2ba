"""The library's host code over tests/fake_hip.cpp (the HIP calls on host memory, no
kernels): what a call allocates, keeps, waits for and leaves behind when it fails.
Each case runs in a process of its own, so that the library binds to those calls."""
import ctypes as C
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HEAD = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
fake.fake_get.restype = fake.fake_pending.restype = fake.fake_streams.restype = C.c_int64
fake.fake_launches.restype = C.c_int64
fake.fake_faults.restype = C.c_char_p
(POINTS, DEVICE_LIMIT, PINNED_LIMIT, FAIL_MALLOC_FROM, NO_COMPACT, CLOCK_NS, PREV_AT, FIT_LIST_AT) = range(8)
(DEVICE_BYTES, DEVICE_PEAK, PINNED_BYTES, PINNED_PEAK, MALLOCS, LARGEST_PINNED, PAGEABLE, FITNESS_OLD) = range(8)
def put(what, v):
    fake.fake_set(C.c_int(what), C.c_int64(v))
get = lambda what: fake.fake_get(C.c_int(what))
sys.path.insert(0, {root!r})
import lowcost3dreconstruction_amd as lcr
lcr.init(0)
def failing(j, f, *a):
    # f with its j-th and later device allocations failing and nothing kept before;
    # whether it raised
    failing.t += 60
    put(CLOCK_NS, failing.t * 10**9)
    lcr.transform_points(cloud(3), np.eye(4))  # what was kept is too old by now
    put(FAIL_MALLOC_FROM, get(MALLOCS) + j)
    r = raises(f, *a)
    put(FAIL_MALLOC_FROM, 0)
    return r
failing.t = 0
def cloud(n):
    return np.random.default_rng(n).uniform(size=(n, 3)).astype(np.float32)
def raises(f, *a):
    try:
        f(*a)
    except lcr.LcrError:
        return True
    return False
"""
TAIL = """
faults = fake.fake_faults().decode()
assert not faults, faults
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", ROOT + "/tests/fake_hip.cpp", "-o", lib], check=True)

    def run(code):
        text = HEAD.format(lib=lib, root=ROOT) + textwrap.dedent(code) + TAIL
        # preloaded, it also stands before a C++ library that the interpreter brings in
        env = dict(os.environ, LD_PRELOAD=" ".join(filter(None, [os.environ.get("LD_PRELOAD"), lib])))
        r = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=120,
                           env=env)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_grown_counters_are_cleared_at_the_same_address(host):
    """A handle whose clouds grow: the larger table of cell counters may get the
    smaller one's address, and is cleared all the same."""
    host("""
    icp = lcr.IterativeClosestPoint()
    for n in (500, 800, 4000, 3000, 20000):
        put(POINTS, n)
        icp.setInputSource(cloud(n))
        icp.setInputTarget(cloud(n))
        icp.align()
    assert fake.fake_launches(b"k_cell_count") == 5
    """)


def test_new_proposal_has_every_weight_zero(host):
    """A proposal without set_weights: the BF16 copies that the forward reads are
    written too, whatever their blocks held."""
    host("""
    p = lcr.Proposal()
    p.forward(np.zeros((2, 40, 3), np.float32), np.zeros((2, 40, 3), np.float32))
    assert fake.fake_launches(b"k_enc_points") == 1
    """)


def test_new_proposal_is_ready_for_any_stream(host):
    """Cycles read a proposal's weights on their own streams: creating one leaves
    nothing in flight on its own."""
    host("""
    p = lcr.Proposal()
    assert fake.fake_pending() == 0
    """)


@pytest.mark.parametrize("what", ["cycle", "icp"])
def test_failed_run_leaves_nothing_in_flight(host, what):
    """A run that fails midway returns after the device is done with what it launched:
    the caller may destroy the proposal (whose buffers that work uses) or hand in
    other clouds next."""
    host(f"""
    put(POINTS, 500)
    clouds = [cloud(500)] * 3
    if {what!r} == "cycle":
        p = lcr.Proposal()
        c = lcr.Cycle(clouds, [(0, 1), (1, 2)], guesses=np.stack([np.eye(4)] * 2), proposal=p,
                      max_corr_dist=0.1, max_iterations=5)
        run = c.run
    else:
        icp = lcr.IterativeClosestPoint()
        icp.setInputSource(clouds[0])
        icp.setInputTarget(clouds[1])
        run = icp.align
    run()
    put(NO_COMPACT, 1)
    assert raises(run)
    assert fake.fake_pending() == 0
    put(NO_COMPACT, 0)
    run()
    """)


def test_fitness_after_new_parameters_takes_nothing_from_the_old_tiles(host):
    """A handle whose grid or tiles were laid out anew since its last align (other
    parameters, then correspondences) has neither matches nor tile lists for them."""
    m = C.CDLL(ROOT + "/lowcost3dreconstruction_amd/liblcr_mathcheck.so")
    host(f"""
    put(PREV_AT, {m.lcrm_icp_buffers_at(0)})
    put(FIT_LIST_AT, {m.lcrm_icp_buffers_at(1)})
    put(POINTS, 5000)
    icp = lcr.IterativeClosestPoint(tile=256)
    icp.setInputSource(cloud(5000))
    icp.setInputTarget(cloud(5000))
    icp.setMaxCorrespondenceDistance(0.1)
    icp.align()
    icp.getFitnessScore(0.01)
    assert get(FITNESS_OLD) == 3
    icp._p.tile = 64
    icp._push()
    icp.correspondences()
    icp.getFitnessScore(0.01)
    assert get(FITNESS_OLD) == 0
    icp.align()
    icp.getFitnessScore(0.01)
    assert get(FITNESS_OLD) == 3
    """)


def test_proposal_after_failed_allocations(host):
    """A batch or a training set that does not fit leaves the handle as it was made, or
    without a training set: never with sizes that its buffers do not have."""
    host("""
    def batch(b, n):
        return (np.zeros((b, n, 3), np.float32),) * 2
    failed = 0
    for j in range(1, 16):
        p = lcr.Proposal()
        p.forward(*batch(2, 200))
        failed += failing(j, p.forward, *batch(64, 3000))
        p.forward(*batch(2, 200))
        p.forward(*batch(64, 3000))
    assert 6 <= failed < 15, failed
    p = lcr.Proposal()
    p.dataset(*batch(3, 100), np.zeros((3, 6), np.float32))
    p.predict(0, 3)
    assert failing(1, p.dataset, *batch(300, 100), np.zeros((300, 6), np.float32))
    assert raises(p.predict, 0, 3) and raises(p.train, 1, 2)
    """)


@pytest.mark.parametrize("what", ["cycle", "icp"])
def test_run_after_failed_allocations(host, what):
    """A run whose buffers do not fit is set up again by the next one, whichever of the
    allocations failed."""
    m = C.CDLL(ROOT + "/lowcost3dreconstruction_amd/liblcr_mathcheck.so")
    host(f"""
    put(PREV_AT, {m.lcrm_icp_buffers_at(0)})
    put(FIT_LIST_AT, {m.lcrm_icp_buffers_at(1)})
    failed = 0
    for j in range(1, 60):
        put(POINTS, 4000)
        if {what!r} == "cycle":
            c = lcr.Cycle([cloud(4000)] * 3, [(0, 1), (1, 2)], max_corr_dist=0.1, max_iterations=5)
            run = c.run
        else:
            icp = lcr.IterativeClosestPoint()
            icp.setInputSource(cloud(4000))
            icp.setInputTarget(cloud(4000))
            icp.setMaxCorrespondenceDistance(0.1)
            run = icp.align
        failed += failing(j, run)
        run()
    assert failed >= 20, failed
    """)


@pytest.mark.parametrize("which", ["Source", "Target"])
def test_cloud_that_does_not_fit_is_not_set(host, which):
    """When the copy of a new cloud cannot be taken the handle has none on that side:
    the old one is not used under the new one's size."""
    host(f"""
    put(POINTS, 4000)
    icp = lcr.IterativeClosestPoint()
    icp.setInputSource(cloud(4000))
    icp.setInputTarget(cloud(4000))
    icp.align()
    put(PINNED_LIMIT, get(PINNED_BYTES) + 4096)
    assert raises(icp.setInput{which}, cloud(50000))
    put(PINNED_LIMIT, 0)
    assert raises(icp.align) and raises(icp.correspondences)
    icp.setInput{which}(cloud(50000))
    put(POINTS, 50000)
    icp.align()
    """)


def test_results_need_no_pinned_memory_of_their_size(host):
    """The staging of results stays at a few megabytes: beside the upload's copy (24
    bytes a point, a quarter more at most), a call on 2 M points takes little, and every
    byte of its results arrives."""
    host("""
    n = 2_000_003
    x = cloud(n)
    got = lcr.transform_points(x, np.eye(4), nrm=x)
    assert all((g.view(np.uint8) == 0xA5).all() for g in got)  # what a new block holds
    assert get(PINNED_PEAK) <= 24 * n * 5 // 4 + (9 << 20), get(PINNED_PEAK)
    """)


@pytest.mark.parametrize("limit", ["DEVICE_LIMIT", "PINNED_LIMIT"])
def test_a_large_call_takes_little_more_than_it_asks_for(host, limit):
    """Blocks are rounded up to size classes, by at most 16 MiB and only while there is
    room for it (12 M points and their normals: 24 bytes each of input and output, 32 of
    records, 4 of cloud numbers, five blocks; 24 bytes pinned and the results' ring),
    also where blocks of other sizes are kept."""
    host(f"""
    n = 12_000_000
    x = np.zeros((n, 3), np.float32)
    lcr.transform_points(x[:500_000], np.eye(4), nrm=x[:500_000])
    put({limit}, (24 + 24 + 32 + 4) * n + 5 * (16 << 20) if {limit} == DEVICE_LIMIT
        else 24 * n + (9 << 20))
    lcr.transform_points(x, np.eye(4), nrm=x)
    """)


def test_kept_memory_is_given_back(host):
    """lcr.release_memory() frees every kept block and stream, beside a live handle that
    goes on; idle blocks go at a later call, whichever kind of memory that one uses."""
    host("""
    def kept():
        return get(DEVICE_BYTES), get(PINNED_BYTES), fake.fake_streams()
    put(POINTS, 3000)
    lcr.normals(cloud(3000), 10)
    lcr.depth_fuse(np.full((4, 64, 64), 900, np.uint16), 2)
    assert min(kept()) > 0
    lcr.release_memory()
    assert kept() == (0, 0, 0)
    icp = lcr.IterativeClosestPoint()
    icp.setInputSource(cloud(3000))
    icp.setInputTarget(cloud(3000))
    icp.align()
    live = kept()
    lcr.normals(cloud(3000), 10)
    lcr.release_memory()
    assert all(a <= b for a, b in zip(kept(), live)) and min(kept()) > 0
    icp.align()
    del icp
    lcr.normals(cloud(3000), 10)
    before = kept()
    put(CLOCK_NS, 30 * 10**9)
    c = lcr.IterativeClosestPoint()
    c.setInputSource(cloud(300))  # takes pinned memory only
    assert kept()[0] == 0 and kept()[1] <= 8192 < before[1], (kept(), before)
    """)


def test_kept_memory_is_bounded(host):
    """Blocks that many live handles give back are kept up to a gigabyte on the device
    and 256 MiB of pinned memory; a call that fails midway keeps none of its own."""
    host("""
    put(POINTS, 150_000)
    cs = [lcr.Cycle([cloud(150_000)] * 2, [(0, 1)], max_corr_dist=0.05) for _ in range(12)]
    for c in cs:
        c.run()
    assert get(DEVICE_BYTES) > 1 << 30
    del cs, c
    assert 0 < get(DEVICE_BYTES) <= 1 << 30 and 0 < get(PINNED_BYTES) <= 256 << 20
    lcr.release_memory()
    assert failing(6, lcr.normals, cloud(150_000), 10)
    assert get(DEVICE_BYTES) <= 1 << 16, get(DEVICE_BYTES)
    """)


def test_autotune_times_runs_whose_graphs_are_captured(host):
    """No candidate's time holds the capture and instantiation of its graphs (three for
    an FP32 scan, two for the tile modes), which a user's later runs do not pay."""
    host("""
    put(POINTS, 3000)
    c = lcr.Cycle([cloud(3000)] * 3, [(0, 1), (1, 2)], max_corr_dist=0.1, max_iterations=5)
    t = c.autotune()
    assert t["candidates"] == 30
    assert t["default_ms"] == 0 and t["best_ms"] == 0, t
    """)


def test_predict_refuses_a_range_whose_end_overflows(host):
    host("""
    p = lcr.Proposal()
    p.dataset(np.zeros((3, 10, 3), np.float32), np.zeros((3, 10, 3), np.float32), np.zeros((3, 6), np.float32))
    out = np.zeros((512, 6), np.float32)
    fp = out.ctypes.data_as(C.POINTER(C.c_float))
    assert lcr.lib.lcr_proposal_predict(p._h, 2, 1, fp, None) == 0
    for first, count in ((2, 2), (0, 4), (3, 1), (2, 2**31 - 1), (2**31 - 1, 1), (2**31 - 1, 2**31 - 1)):
        assert lcr.lib.lcr_proposal_predict(p._h, first, count, fp, None) == -1, (first, count)
    """)


def test_resident_cycle_keeps_no_copy_of_its_upload(host):
    """Once a cycle's clouds are on the device in their own layout, the packed copies
    they came in (12 bytes a point pinned, as many on the device) go back."""
    host("""
    n = 100_000
    put(POINTS, n)
    c = lcr.Cycle([cloud(n)] * 2, [(0, 1)], max_corr_dist=0.05)
    c.run()
    held = get(DEVICE_BYTES)
    lcr.release_memory()
    assert get(PINNED_BYTES) < 12 * n, get(PINNED_BYTES)
    assert get(DEVICE_BYTES) <= held - 2 * 12 * n, (held, get(DEVICE_BYTES))
    c.run()
    """)
