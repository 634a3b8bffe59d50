"""The library's host code without a GPU: liblcs_hip.so on the recording
runtime of tests/host_runtime, in a process of its own.  What a call launches,
what it leaves pending when it returns and what it charges to its budget is
checked here; the kernels do not run."""
import json
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "platform-independent-lcs_amd")

PRELUDE = """
import ctypes, json, sys
rec = ctypes.CDLL({rec!r}, mode=ctypes.RTLD_GLOBAL)
rec.rec_launches.restype = ctypes.c_char_p
rec.rec_clock.restype = ctypes.c_double
rec.rec_live.restype = ctypes.c_size_t
sys.path.insert(0, {pkg!r})
import numpy as np
import lcs_amd
from lcs_amd import lib

def launches(name):
    return [tuple(map(int, l.split()[1:])) for l in rec.rec_launches().decode().splitlines() if name in l]

def zeros(n):
    return np.zeros(n, np.int32)
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the HIP headers")
    rec = str(tmp_path_factory.mktemp("runtime") / "librecording_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "host_runtime", "recording_hip.cpp"), "-o", rec], check=True)

    def run(code):
        """The value that `code` leaves in `result`."""
        script = PRELUDE.format(rec=rec, pkg=PKG) + code + "\nprint('RESULT', json.dumps(result))\n"
        done = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=60)
        assert done.returncode == 0, done.stderr
        return json.loads([l for l in done.stdout.splitlines() if l.startswith("RESULT ")][-1][7:])
    return run


def test_wide_short_pairs_are_cut(host):
    # tiles of the launch (grid.y of its seeding kernel): a wide pair is cut
    # though it has few cells, a square or tall one of that size is not
    sizes = [(64, 16384), (64, 100000), (1, 1000000), (512, 100000), (2000, 33000), (4000, 16400),
             (64, 16383), (300, 500), (4096, 4096), (8000, 8000), (100000, 64)]
    tiles = host(f"""
result = []
with lcs_amd.Context(0) as c:
    for m, n in {sizes}:
        rec.rec_clear()
        c.comb(zeros(m), zeros(n))
        result.append(launches('comb_prep_grid_kernel')[0][1])
""")
    assert all(t > 1 for t in tiles[:6]) and tiles[6:] == [1] * 5, tiles


def test_a_refused_pair_leaves_no_copy_queued(host):
    # the schedule is looked at after the strings are staged
    assert host("""
result = []
with lcs_amd.Context(0) as c:
    for m, sched in ((300, lcs_amd.schedule(3, 1, lcs_amd.VARIANT_CHAIN, 1)), (300, lcs_amd.schedule(4, 1, 99, 1)),
                     (300, lcs_amd.schedule(4, 9, lcs_amd.VARIANT_CHAIN, 1))):
        for call in (c.comb, c.comb_permutation):
            try:
                call(zeros(m), zeros(500), sched)
            except lcs_amd.LcsError:
                result.append(rec.rec_pending())
""") == [0] * 6


@pytest.mark.parametrize("n", [500, 100000])   # one tile; columns cut and merged
def test_the_time_reported_is_the_last_calls_own(host, n):
    # 1 ms a launch.  A device pair's time is read off its events later; a
    # batch or a product after it reports its own, a fixup (which reports
    # none) leaves the pair's
    got = host(f"""
def after(call, pair):
    with lcs_amd.Context(0) as c:
        if pair:
            dev = [np.zeros({n} + 300, np.int32) for _ in range(4)]
            lcs_amd._check("lcs_comb_device", lib().lcs_comb_device(
                c.handle, dev[0].ctypes.data, 300, dev[1].ctypes.data, {n}, None, dev[2].ctypes.data, dev[3].ctypes.data, None))
            if call is None:
                return c.info()[1]
        call(c)
        return c.info()[1]

def fixup(c):
    h, v = np.arange(70, dtype=np.int32), np.arange(70, 150, dtype=np.int32)
    c.comb_fixup(zeros(70), zeros(80), h, v, 0, 70, 0, 80)

batch = lambda c: c.batch_comb([zeros(100)] * 3, [zeros(200)] * 3, use_graph=False)
product = lambda c: c.braid_multiply(np.arange(50, dtype=np.int32), np.arange(60, dtype=np.int32), 20, False)
result = [after(batch, False), after(batch, True), after(product, False), after(product, True), after(None, True),
          after(fixup, True)]
""")
    assert got[0] == got[1] and got[2] == got[3] and got[4] == got[5] and min(got) > 0, got


def test_workspaces_of_one_pair_give_way_to_the_next(host):
    # strings, results and ring of the second pair fill the budget, so the
    # first one's tiles, permutations and byte copies have to go
    got = host("""
def need(m, n):
    return 8 * (m + n) + 16 * n + 100000

result = []
for first, second, sched in (((9000, 9000), (30000, 30000), lcs_amd.schedule(4, 1, lcs_amd.VARIANT_CHAIN, 1)),
                             ((60000, 60000), (100, 200000), lcs_amd.schedule(1, 1, lcs_amd.VARIANT_CHAIN, 1))):
    with lcs_amd.Context(0, hbm_budget=need(*second)) as c:
        for (m, n), s in ((first, None), (second, sched), (second, sched)):
            try:
                c.comb(zeros(m), zeros(n), s)
                result.append(0)
            except lcs_amd.LcsError as e:
                result.append(e.args)
""")
    assert got[1:3] == got[4:6] == [0, 0], got


def test_lcs_length_fits_where_its_rings_do(host):
    # half a byte a column for each pair's rings, the strings and a fixed part:
    # the codes (a byte or half a byte a column) are kept only where they fit
    need = {"300 x 500": 3912, "100000^2": 850808, "1000 of 50^2": 536256, "empty": 1332}
    got = host(f"""
need = {need!r}
calls = {{"300 x 500": (1, 300, 500), "100000^2": (1, 100000, 100000), "1000 of 50^2": (1000, 50, 50), "empty": (3, 0, 50)}}
result = []
for name, (pairs, m, n) in calls.items():
    for sigma in (4, 20):
        with lcs_amd.Context(0, hbm_budget=need[name]) as c:
            c.llcs_batch([zeros(m)] * pairs, [zeros(n)] * pairs, sigma)
            result.append(c.memory()[0] <= need[name])
""")
    assert got == [True] * 8


def test_an_index_dropped_on_another_thread_keeps_the_account(host):
    # the context's bytes stay those that the runtime has allocated for it,
    # with indexes dropped on one thread while another reserves and frees
    assert host("""
import queue, threading
result = []
for rounds in range(8):
    c = lcs_amd.Context(0)
    besides = rec.rec_live() - c.memory()[0]
    dropped = queue.Queue()

    def drop():
        for idx in iter(dropped.get, None):
            idx.close()

    thread = threading.Thread(target=drop, daemon=True)
    thread.start()
    perm = np.arange(300, dtype=np.int32)
    for i in range(1500):
        dropped.put(lcs_amd.DominanceIndex(c, perm))
        c.semilocal(perm, 20, 280, 0, zeros(4), zeros(4))   # a buffer of its own for the call
    dropped.put(None)
    thread.join()
    result.append(int(rec.rec_live() - c.memory()[0] - besides))
    c.close()
""") == [0] * 8


def test_a_context_waits_for_an_index_being_dropped(host):
    # the drop is inside its wait for the stream when the context is closed
    waited = host("""
import threading, time
c = lcs_amd.Context(0)
idx = lcs_amd.DominanceIndex(c, np.arange(300, dtype=np.int32))
rec.rec_slow_next_sync(1000)
drop = threading.Thread(target=idx.close, daemon=True)
drop.start()
time.sleep(0.2)
t = time.monotonic()
c.close()
result = time.monotonic() - t
drop.join()
""")
    assert waited > 0.5


def test_lds_limits_are_raised_on_every_device(host):
    # kernels that ask for more than 64 KB of LDS, on the first device and then
    # on a second one in the same process
    assert host("""
p = np.arange(3000, dtype=np.int32)
for device in (0, 1):
    with lcs_amd.Context(device) as c:
        c.braid_multiply(p, p, 2000, False)
        c.llcs_batch([zeros(100)], [zeros(100)], 4)
result = [rec.rec_lds_devices(k) for k in (b"llcs_chain_kernel", b"big_leaf_kernel", b"braid_core_lds_kernel")]
""") == [2, 2, 2]


def test_a_slice_has_a_bounded_number_of_workgroups(host):
    # each adds up the counts of those before it
    blocks = host("""
result = []
with lcs_amd.Context(0) as c:
    for size in (2047, 2048, 4096 * 2048 - 1, 4096 * 2048, 1 << 24):
        p = np.arange(size, dtype=np.int32)
        rec.rec_clear()
        c.braid_multiply(p, p[:100], 64, False)
        result += [g[0] for g in launches('slice_count_kernel') + launches('slice_scatter_kernel')]
""")
    assert blocks == [1, 1, 2, 2, 4096, 4096, 2049, 2049, 2731, 2731], blocks


def test_a_larger_product_needs_no_smaller_workspace(host):
    # a merge level reserves for its largest product, whichever has more
    # workgroups to a slice
    words = host("""
f = lib()._Z22lcsb_multiply_ws_wordsiiib
f.restype = ctypes.c_size_t
tile, most = 2048, 4096
sizes = [s + d for s in (tile, tile * most, 2 * tile * most, 3 * tile * most) for d in (-tile - 1, -tile, -1, 0, 1, tile)]
result = [[f(p, q, k, False) for p, q in zip(sizes, sizes)] for k in (1, 300)]
result += [[f(s, 400, 300, False) for s in sizes], [f(400, s, 300, False) for s in sizes]]
""")
    for row in words:
        assert row == sorted(row), row


def test_a_product_of_2048_strands_fits_where_it_did(host):
    # one workgroup's LDS holds the core where the budget does not hold the
    # workspace of a core spread over the GPU
    got = host("""
result = []
p = np.arange(4096, dtype=np.int32)
for budget in (0, 114776):
    with lcs_amd.Context(0, hbm_budget=budget) as c:
        rec.rec_clear()
        c.braid_multiply(p, p, 2048, True)
        result.append([len(launches('braid_core_lds_kernel')), len(launches('big_leaf_kernel'))])
""")
    assert got == [[0, 1], [1, 0]]


@pytest.mark.parametrize("size", [1, 5, 70000, (1 << 24) - 1, 1 << 24])
def test_products_refuse_what_is_no_permutation(host, size):
    # whichever loop checks: a value twice, one past the end, a negative one
    got = host(f"""
p, q = np.arange({size}, dtype=np.int32)[::-1].copy(), np.arange(1, dtype=np.int32)
result = []
with lcs_amd.Context(0) as c:
    for where, value in ((0, {size}), ({size} - 1, -1), ({size} // 2, None), (0, 1 if {size} > 2 else {size})):
        old = p[where]
        p[where] = old if value is None else value
        try:
            c.braid_multiply(p, q, 0, False)
            result.append('ok')
        except lcs_amd.LcsError as e:
            result.append('EINVAL' if 'EINVAL' in str(e) else str(e))
        p[where] = old
""")
    assert got == ["EINVAL", "EINVAL", "ok", "EINVAL"], got
