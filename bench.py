#!/usr/bin/env python3
"""Benchmark of the semi-local LCS seaweed hot path on one MI355X.

Default workload (one "step" = one full comb of the pair, inputs resident in
HBM): m = n = 2^20, A uniform over alphabet 4, B = A with 10% substitutions
and 2% single-symbol indels (seeded), output the int32 permutation of 2^21
strands.  Prints ONE JSON line with GCUPS, the integer-VALU roofline of the
comb kernel and a CPU baseline measured in the same run on this host.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--tile-m T]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [ROOT, os.path.join(ROOT, "platform-independent-lcs_amd")]

import numpy as np  # noqa: E402

import lcs_amd  # noqa: E402
from lcs_amd import hip as H  # noqa: E402

# MI355X: 256 CUs x 4 SIMD x 16 lanes = 64 int32 lane-ops per CU per clock,
# 2.4 GHz peak engine clock.  A cell is 4 VALU ops (cmp, min, cndmask, xor3).
PEAK_CLOCK_HZ = 2.4e9
OPS_PER_CELL = 4


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--log2n", type=int, default=20, help="m = n = 2^log2n")
    ap.add_argument("--tile-m", type=int, default=0)
    ap.add_argument("--waves-per-simd", type=int, default=0)
    ap.add_argument("--variant", type=int, default=0, help="0 auto, 1 register chain, 2 LDS band groups")
    ap.add_argument("--cpu-seconds", type=float, default=12.0, help="target CPU baseline sample length")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--check", action="store_true", help="cross-check two schedules bit-for-bit")
    ap.add_argument("--no-zipf", action="store_true", help="skip the m=2^14, n=2^22 Zipf leg")
    ap.add_argument("--no-semilocal", action="store_true", help="skip the semi-local query leg")
    ap.add_argument("--no-merge", action="store_true", help="skip the strips + steady-ant merge leg")
    ap.add_argument("--no-llcs", action="store_true", help="skip the bit-parallel LCS-length leg")
    ap.add_argument("--batch-pairs", type=int, default=10000, help="pairs of the batched leg (0: skip it)")
    ap.add_argument("--serve-requests", type=int, default=600, help="requests of the served leg (0: skip it)")
    ap.add_argument("--serve-rate", type=float, default=150.0, help="Poisson arrival rate (requests/s)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="only run 3 device-to-device copies of 256 MiB (HBM counter calibration) and exit")
    return ap.parse_args()


def host_cpus():
    """CPUs this process may run on: the affinity mask, cut to the cgroup's
    CPU quota when one is set (cpu.max), so no thread waits for a share."""
    n = len(os.sched_getaffinity(0))
    quota = None
    try:
        with open("/sys/fs/cgroup/cpu.max") as f:
            q, period = f.read().split()[:2]
            if q != "max":
                quota = max(1, int(int(q) // int(period)))
    except (OSError, ValueError):
        pass
    return (min(n, quota) if quota else n), n, quota


def _strip_rate(fn, m: int, b, target_s: float, min_cols: int):
    """Times fn(b[:cols]) on a full-height strip sized for ~target_s: the
    strip grows 4x until a run takes a quarter of the target (thread start-up
    and caches no longer dominate), then is sized from that run's rate."""
    cols = min(len(b), min_cols)
    while True:
        t0 = time.perf_counter()
        fn(b[:cols])
        dt = max(time.perf_counter() - t0, 1e-6)
        if dt >= target_s / 4 or cols >= len(b):
            break
        cols = min(len(b), cols * 4)
    cols = int(min(len(b), max(cols, cols * target_s / dt)))
    t0 = time.perf_counter()
    fn(b[:cols])
    return cols, time.perf_counter() - t0


def cpu_baseline(a, b, target_s: float):
    """The reference's CPU path restated in the oracle, timed on a
    full-height strip of the same pair and scaled to GCUPS:
      - value: the vectorised tiled comb (orc_comb_simd: the reference's
        Lcs_Semi_Tiled_MT shape, lcs_tiled.hpp:95-137, with the lanes of a
        sub-group owning rows, lcs_common.hpp:131-173, on AVX-512/AVX2 lanes)
        on every CPU this process may use;
      - scalar_block_wavefront: the scalar block wavefront (orc_comb_mt) on
        the same threads;
      - single_core: the sequential restatement of lcs_reference.hpp:5-69."""
    import oracle  # test infrastructure: the CPU baseline only
    threads, affinity, quota = host_cpus()
    m = len(a)
    cols, dt = _strip_rate(lambda bb: oracle.comb(a, bb, order="simd", threads=threads), m, b, target_s, 1024)
    cols_mt, dt_mt = _strip_rate(lambda bb: oracle.comb(a, bb, order="mt", threads=threads), m, b,
                                 target_s / 3, 256)
    cols1, dt1 = _strip_rate(lambda bb: oracle.comb(a, bb, order="rows"), m, b, target_s / 6, 16)
    isa = {1: "AVX2", 2: "AVX-512"}.get(2 if oracle.simd_isa_available(oracle.ISA_AVX512) else
                                        1 if oracle.simd_isa_available(oracle.ISA_AVX2) else 3, "scalar")
    return {"value": round(m * cols / dt / 1e9, 4), "unit": "GCUPS", "cores": threads, "kind": "port",
            "host_cpus": {"affinity": affinity, "cgroup_quota": quota},
            "sample": f"m={m} x first {cols} columns of the same pair ({m * cols:.3g} cells, {dt:.1f} s), "
                      f"oracle orc_comb_simd ({isa} stripes, lanes own rows), {threads} threads",
            "scalar_block_wavefront": {
                "value": round(m * cols_mt / dt_mt / 1e9, 4), "unit": "GCUPS", "cores": threads,
                "sample": f"m={m} x first {cols_mt} columns ({m * cols_mt:.3g} cells, {dt_mt:.1f} s), "
                          "oracle orc_comb_mt (scalar block wavefront)"},
            "single_core": {"value": round(m * cols1 / dt1 / 1e9, 4), "unit": "GCUPS", "cores": 1,
                            "sample": f"m={m} x first {cols1} columns ({m * cols1:.3g} cells, {dt1:.1f} s), "
                                      "oracle orc_comb_rows (sequential restatement of lcs_reference.hpp:5-69)"}}


def read_profile_value(path: str, prefix: str):
    """A number after `prefix` on a line of a committed profile summary."""
    try:
        with open(path) as f:
            for line in f:
                if prefix in line:
                    tail = line.split(prefix, 1)[1].strip()
                    return float(tail.split()[0])
    except (OSError, ValueError, IndexError):
        pass
    return None


def read_traffic(path: str):
    """HBM bytes per launch of the comb kernel from a committed rocprofv3
    --pmc summary (FETCH_SIZE + WRITE_SIZE, KiB per dispatch, scaled by the
    copy-kernel calibration factor stated in that file)."""
    try:
        with open(path) as f:
            for line in f:
                if line.startswith("traffic_bytes_per_launch:"):
                    return float(line.split(":", 1)[1])
    except OSError:
        pass
    return None


def calibrate_copy():
    """Three 256 MiB device-to-device copies: the reference kernel whose
    FETCH_SIZE / WRITE_SIZE readings scale the comb kernel's counters."""
    import ctypes
    h = H.hip()
    n = 64 << 20
    src, dst = H.DeviceArray(n), H.DeviceArray(n)
    h.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    for _ in range(3):
        assert h.hipMemcpy(dst.ptr, src.ptr, n * 4, 3) == 0   # hipMemcpyDeviceToDevice
    H.synchronize()
    print(json.dumps({"copied_bytes": n * 4, "copies": 3}), flush=True)


def learned_model(ctx, mode: int):
    """The cost model trained on the GPU on the autotuner's committed timing
    table of this device (None when no table is there)."""
    from lcs_amd import tuning
    if not os.path.exists(tuning.TABLES[mode]):
        return None, None
    table = tuning.load_table(mode)
    t0 = time.perf_counter()
    mlp = tuning.train(ctx, table)
    return mlp, {"table": os.path.relpath(tuning.TABLES[mode], ROOT), "shapes": len(table["rows"]),
                 "train_s": round(time.perf_counter() - t0, 2)}


def bench_batch(ctx, npairs: int):
    """10,000 pairs, m and n log-uniform in [256, 16384], alphabet 4, B = A
    mutated at a per-pair rate in [5%, 20%] (20% of it indels), resident in
    HBM.  Plain path: one lcs_comb_device call per pair (the drop-in's own
    schedule).  Batched path: lcs_batch_comb_device, every pair in one
    hipGraph launch, schedules from the library's built-in default (no
    model: the packed chain, 8 or 16 rows per lane by m, for every pair it
    can take; reported as batched_heuristic_*) and from the learned cost
    model.  Every batched result is compared with the plain path's, pair by
    pair."""
    from lcs_amd import tuning
    L = lcs_amd.lib()
    t0 = time.perf_counter()
    pairs = lcs_amd.workload_batch(npairs, seed=7)
    lay = lcs_amd.BatchLayout([p.a for p in pairs], [p.b for p in pairs])
    gen_s = time.perf_counter() - t0
    cells = float(np.sum(lay.m.astype(np.float64) * lay.n))
    da, db = H.DeviceArray.from_numpy(lay.a_all), H.DeviceArray.from_numpy(lay.b_all)
    dh0, dv0 = H.DeviceArray(lay.a_all.size), H.DeviceArray(lay.b_all.size)
    dh1, dv1 = H.DeviceArray(lay.a_all.size), H.DeviceArray(lay.b_all.size)

    def plain():
        for p in range(npairs):
            ao, bo = int(lay.a_off[p]) * 4, int(lay.b_off[p]) * 4
            rc = L.lcs_comb_device(ctx.handle, da.ptr.value + ao, int(lay.m[p]), db.ptr.value + bo, int(lay.n[p]),
                                   None, dh0.ptr.value + ao, dv0.ptr.value + bo, None)
            if rc:
                raise lcs_amd.LcsError("lcs_comb_device", rc)
        H.synchronize()

    plain()   # warm-up
    t0 = time.perf_counter()
    plain()
    plain_s = time.perf_counter() - t0
    ref_h, ref_v = dh0.numpy(), dv0.numpy()

    def batched(scheds):
        best, kms = 1e30, 0.0
        for _ in range(3):
            t1 = time.perf_counter()
            lcs_amd.batch_comb_device(ctx, lay, da.ptr, db.ptr, dh1.ptr, dv1.ptr, scheds)
            dt = time.perf_counter() - t1
            st = ctx.status()
            if st:
                raise lcs_amd.LcsError("lcs_ctx_status", st)
            if dt < best:
                best, kms = dt, ctx.info()[1]
        exact = bool(np.array_equal(dh1.numpy(), ref_h) and np.array_equal(dv1.numpy(), ref_v))
        return best, kms, exact

    heur_s, heur_kms, heur_exact = batched(None)
    out = {"workload": f"{npairs} pairs, m,n log-uniform [256,16384], alphabet 4, 5-20% mutations",
           "cells": cells, "gen_s": round(gen_s, 1),
           "plain_pairs_per_s": round(npairs / plain_s, 1), "plain_s": round(plain_s, 3),
           "batched_heuristic_pairs_per_s": round(npairs / heur_s, 1), "batched_heuristic_s": round(heur_s, 4),
           "batched_heuristic_kernel_ms": round(heur_kms, 3), "batched_heuristic_bit_exact": heur_exact}
    mlp, info = learned_model(ctx, 1)
    if mlp is not None:
        cands = tuning.table_candidates(tuning.load_table(1))
        scheds, idx = tuning.choose_schedules(mlp, lay.m, lay.n, [p.alphabet for p in pairs],
                                              [p.rate for p in pairs], cands)
        l_s, l_kms, l_exact = batched(scheds)
        out.update({"batched_learned_pairs_per_s": round(npairs / l_s, 1), "batched_learned_s": round(l_s, 4),
                    "batched_learned_kernel_ms": round(l_kms, 3), "batched_learned_bit_exact": l_exact,
                    "learned_choice_histogram": {f"tm{cands[i].tile_m}v{cands[i].variant}":
                                                 int(c) for i, c in zip(*np.unique(idx, return_counts=True))},
                    "cost_model": info})
        mlp.close()
        best_s = min(heur_s, l_s)
        tiles = [sc.tile_m for sc in scheds]
    else:
        out["cost_model"] = "no autotune table: heuristic schedules only"
        best_s = heur_s
        tiles = [0] * npairs
    # 16-bit strands, two pairs per wave (every pair here has m + n <= 32768)
    packed = [lcs_amd.schedule(tile_m=t, variant=lcs_amd.VARIANT_PACKED16) for t in tiles]
    p_s, p_kms, p_exact = batched(packed)
    out.update({"batched_packed16_pairs_per_s": round(npairs / p_s, 1), "batched_packed16_s": round(p_s, 4),
                "batched_packed16_kernel_ms": round(p_kms, 3), "batched_packed16_bit_exact": p_exact,
                "batched_packed16_tiles": "learned" if mlp is not None else "heuristic"})
    if p_exact:
        best_s = min(best_s, p_s)
    out["speedup_vs_plain"] = round(plain_s / best_s, 2)
    out["batched_gcups"] = round(cells / best_s / 1e9, 1)
    return out


def bench_zipf(ctx, steps: int = 3):
    """m = 2^14, n = 2^22, alphabet 26 with Zipf(1.1) frequencies, 64 planted
    5%-mutated copies of A in B.  The default schedule cuts b into column
    strips, combs them in one chain launch and merges the strip permutations
    with the GPU steady ant (k = m); the result is compared bit for bit with
    the same pair combed as one strip."""
    L = lcs_amd.lib()
    w = lcs_amd.workload_single("zipf_planted", seed=1)
    m, n = w.a.size, w.b.size
    da, db = H.DeviceArray.from_numpy(w.a), H.DeviceArray.from_numpy(w.b)
    dh, dv = H.DeviceArray(m), H.DeviceArray(n)

    def run(sched):
        rc = L.lcs_comb_device(ctx.handle, da.ptr, m, db.ptr, n, sched, dh.ptr, dv.ptr, None)
        if rc:
            raise lcs_amd.LcsError("lcs_comb_device", rc)
        H.synchronize()
        st = ctx.status()
        if st:
            raise lcs_amd.LcsError("lcs_ctx_status", st)

    run(None)
    t0 = time.perf_counter()
    for _ in range(steps):
        run(None)
    dt = (time.perf_counter() - t0) / steps
    h, v = dh.numpy(), dv.numpy()
    one = lcs_amd.schedule(strips=1)
    run(one)
    t0 = time.perf_counter()
    run(one)
    dt1 = time.perf_counter() - t0
    exact = bool(np.array_equal(h, dh.numpy()) and np.array_equal(v, dv.numpy()))
    cells = float(m) * n
    return {"workload": "m=2^14, n=2^22, alphabet 26 Zipf(1.1), 64 planted copies (5% subs)",
            "gcups": round(cells / dt / 1e9, 1), "ms": round(dt * 1e3, 2),
            "one_strip_gcups": round(cells / dt1 / 1e9, 1), "strips_vs_one_strip_bit_exact": exact,
            "llcs": int((v < m).sum())}


def bench_tiled_merge(ctx, da, db, m: int, n: int, h_ref, v_ref, strips=(1, 2, 4, 8)):
    """The m = n = 2^20 pair with S column strips combed in one chain launch
    and the strip permutations merged pairwise by the whole-GPU steady ant
    (k = m = 2^20, log2 S levels); S = 1 is the band chain alone.  Each
    result is compared bit for bit with the headline's."""
    L = lcs_amd.lib()
    dh, dv = H.DeviceArray(m), H.DeviceArray(n)
    out = {"workload": "single pair m=n=2^20, S column strips + steady-ant merges (k = m)"}
    for S in strips:
        sched = lcs_amd.schedule(strips=S)

        def run():
            rc = L.lcs_comb_device(ctx.handle, da.ptr, m, db.ptr, n, sched, dh.ptr, dv.ptr, None)
            if rc:
                raise lcs_amd.LcsError("lcs_comb_device", rc)
            H.synchronize()
            st = ctx.status()
            if st:
                raise lcs_amd.LcsError("lcs_ctx_status", st)
            return ctx.info()[1]

        run()
        ks = [run() for _ in range(2)]
        exact = bool(np.array_equal(dh.numpy(), h_ref) and np.array_equal(dv.numpy(), v_ref))
        k = min(ks)
        out[f"strips{S}"] = {"kernel_ms": round(k, 3), "gcups": round(float(m) * n / (k / 1e3) / 1e9, 1),
                             "chain_ms": round(ctx.chain_ms(), 3), "merge_levels": int(np.log2(S)),
                             "bit_exact_vs_headline": exact}
    dh.free()
    dv.free()
    return out


def bench_config1(ctx):
    """The reference's own CPU-runnable case: m = n = 4096 uniform over
    alphabet 4.  GPU: lcs_comb_device (best of 5 after a warm-up); CPU: the
    oracle's sequential comb (lcs_reference.hpp:5-69) and its vectorised
    tiled comb on the whole pair; all three outputs compared bit for bit."""
    import oracle  # test infrastructure: the CPU side of this leg only
    L = lcs_amd.lib()
    w = lcs_amd.workload_single("uniform4096", seed=1)
    m, n = w.a.size, w.b.size
    da, db = H.DeviceArray.from_numpy(w.a), H.DeviceArray.from_numpy(w.b)
    dh, dv = H.DeviceArray(m), H.DeviceArray(n)
    ks, walls = [], []
    for i in range(6):
        t0 = time.perf_counter()
        rc = L.lcs_comb_device(ctx.handle, da.ptr, m, db.ptr, n, None, dh.ptr, dv.ptr, None)
        if rc:
            raise lcs_amd.LcsError("lcs_comb_device", rc)
        H.synchronize()
        st = ctx.status()
        if st:
            raise lcs_amd.LcsError("lcs_ctx_status", st)
        if i:
            walls.append(time.perf_counter() - t0)
            ks.append(ctx.info()[1])
    h, v = dh.numpy(), dv.numpy()
    t0 = time.perf_counter()
    h1, v1 = oracle.comb(w.a, w.b, order="rows")
    seq_s = time.perf_counter() - t0
    threads = host_cpus()[0]
    t0 = time.perf_counter()
    h2, v2 = oracle.comb(w.a, w.b, order="simd", threads=threads)
    simd_s = time.perf_counter() - t0
    for d in (da, db, dh, dv):
        d.free()
    cells = float(m) * n
    return {"workload": "m=n=4096 uniform alphabet 4 (the reference's CPU-runnable case)",
            "gpu_ms": round(min(walls) * 1e3, 3), "gpu_kernel_ms": round(min(ks), 3),
            "gpu_gcups": round(cells / min(walls) / 1e9, 1),
            "cpu_sequential_ms": round(seq_s * 1e3, 1), "cpu_sequential_gcups": round(cells / seq_s / 1e9, 3),
            "cpu_vectorised_ms": round(simd_s * 1e3, 2), "cpu_vectorised_threads": threads,
            "bit_exact": bool(np.array_equal(h, h1) and np.array_equal(v, v1) and np.array_equal(h, h2)
                              and np.array_equal(v, v2)),
            "llcs": int((v < m).sum())}


def bench_semilocal(ctx, r2c, m: int, n: int, llcs: int, nq: int = 1 << 22):
    """Semi-local read-out on the permutation of the m=n=2^20 pair: build the
    dominance index from the device permutation, then answer nq random
    string-substring queries LCS(a, b[i:j)) from device buffers."""
    rng = np.random.default_rng(5)
    d_p = H.DeviceArray.from_numpy(r2c)
    build_ms = []
    for _ in range(3):
        H.synchronize()
        t0 = time.perf_counter()
        idx = lcs_amd.DominanceIndex(ctx, size=r2c.size, device_ptr=d_p.ptr.value)
        build_ms.append((time.perf_counter() - t0) * 1e3)
        if len(build_ms) < 3:
            idx.close()
    i, j = rng.integers(0, n + 1, nq), rng.integers(0, n + 1, nq)
    q0, q1 = np.minimum(i, j).astype(np.int32), np.maximum(i, j).astype(np.int32)
    q0[0], q1[0] = 0, n
    d0, d1, dout = H.DeviceArray.from_numpy(q0), H.DeviceArray.from_numpy(q1), H.DeviceArray(nq)
    times = []
    for _ in range(4):
        H.synchronize()
        t0 = time.perf_counter()
        idx.query_device(m, n, lcs_amd.SEMI_STRING_SUBSTRING, d0.ptr.value, d1.ptr.value, nq, dout.ptr.value)
        H.synchronize()
        times.append(time.perf_counter() - t0)
    got = dout.numpy()
    # the full window is the LCS; a sample agrees with the direct-count kernel
    direct = ctx.semilocal(r2c, m, n, lcs_amd.SEMI_STRING_SUBSTRING, q0[:8], q1[:8])
    ok = bool(got[0] == llcs and np.array_equal(direct, got[:8]))
    best = min(times[1:])
    out = {"workload": f"{nq} random LCS(a, b[i:j)) queries on P of the m=n=2^20 pair ({r2c.size} strands)",
           "index_build_ms": round(min(build_ms[1:]), 3), "index_mib": round(idx.nbytes / 2 ** 20, 2),
           "queries_per_s": round(nq / best, 0), "query_ms": round(best * 1e3, 3), "checks_pass": ok}
    idx.close()
    for d in (d_p, d0, d1, dout):
        d.free()
    return out


def bench_llcs(ctx, a, b, llcs_comb: int, steps: int = 3):
    """Score-only LCS length of the same m=n=2^20 pair by the bit-parallel
    kernel (one bit per cell); must equal the comb's LCS read-out."""
    da, db, dout = H.DeviceArray.from_numpy(a), H.DeviceArray.from_numpy(b), H.DeviceArray(1)
    ctx.llcs_device(da.ptr.value, a.size, db.ptr.value, b.size, 4, dout.ptr.value)   # warm
    H.synchronize()
    ks = []
    t0 = time.perf_counter()
    for _ in range(steps):
        ctx.llcs_device(da.ptr.value, a.size, db.ptr.value, b.size, 4, dout.ptr.value)
        H.synchronize()
        ks.append(ctx.info()[1])
    wall = (time.perf_counter() - t0) / steps
    got = int(dout.numpy()[0])
    for d in (da, db, dout):
        d.free()
    cells = float(a.size) * float(b.size)
    k = float(np.median(ks))
    return {"workload": f"LCS length of the m=n=2^{int(np.log2(a.size))} pair, bit-parallel (lcs_llcs_device)",
            "kernel_ms": round(k, 3), "gcups": round(cells / (k / 1e3) / 1e9, 1), "ms_per_call": round(wall * 1e3, 3),
            "llcs": got, "equals_comb": got == llcs_comb}


def bench_serve(ctx, nreq: int, rate: float):
    """Poisson arrivals of pair comparisons, lengths log-uniform in
    [1024, 262144], alphabet 4 or 20 (50/50), B from A by the same mutation
    model; admitted by an HBM budget into overlapping micro-batches, the
    schedule of each request chosen by the learned cost model.  Latency is
    submit-to-result on the host.  Beside the offered rate: the same
    requests all submitted at once (the server's capacity), higher offered
    rates (p99 at each), and the plain path under the same arrivals (one
    synchronous lcs_comb per request, in arrival order)."""
    from lcs_amd import tuning
    pairs = lcs_amd.workload_batch(nreq, seed=9, lo=1024, hi=262144, alphabet=(4, 20))
    srv = lcs_amd.Server(ctx, hbm_budget=8 << 30, max_inflight=4)
    mlp, info = learned_model(ctx, 0)
    if mlp is not None:
        srv.set_cost_model(mlp, tuning.table_candidates(tuning.load_table(0)))
    feats = tuning.features([p.a.size for p in pairs], [p.b.size for p in pairs], [p.alphabet for p in pairs],
                            [p.rate for p in pairs])
    gaps = np.random.default_rng(5).exponential(1.0, nreq)   # unit-rate Poisson gaps, scaled per run
    cells = float(sum(p.a.size * p.b.size for p in pairs))

    def served(r):
        """r requests/s (None: every request at t = 0); (wall s, latencies ms, stats, outputs)."""
        ids = []
        t0 = time.perf_counter()
        next_t = t0
        for p, f, gap in zip(pairs, feats, gaps):
            if r:
                next_t += gap / r
                while time.perf_counter() < next_t:
                    time.sleep(max(0.0, min(next_t - time.perf_counter(), 0.002)))
            ids.append(srv.submit(p.a, p.b, None, f))
        outs = [srv.wait(i, timeout_ms=120000) for i in ids]
        wall = time.perf_counter() - t0
        lat = np.array([srv.times(i)[1] for i in ids]) / 1e3
        st = srv.stats()
        for i in ids:
            srv.release(i)
        return wall, lat, st, outs

    def pct(lat):
        return round(float(np.percentile(lat, 50)), 2), round(float(np.percentile(lat, 99)), 2)

    wall, lat, st, outs = served(rate)
    # a sample of results against the same pair alone (bit-exact)
    exact = True
    for p, o in list(zip(pairs, outs))[:: max(1, nreq // 12)]:
        h1, v1, _ = ctx.comb(p.a, p.b)
        exact = exact and np.array_equal(o[0], h1) and np.array_equal(o[1], v1)
    p50, p99 = pct(lat)
    sat_wall, sat_lat, _, _ = served(None)
    sweep = {}
    for r in (2 * rate, 4 * rate):
        w2, l2, _, _ = served(r)
        sweep[f"{int(r)}/s"] = {"pairs_per_s": round(nreq / w2, 1), "p50_ms": pct(l2)[0], "p99_ms": pct(l2)[1]}
    srv.close()
    if mlp is not None:
        mlp.close()
    # the plain path under the same arrivals: one synchronous call per request
    plain_lat = []
    t0 = time.perf_counter()
    arrival = t0
    for p, gap in zip(pairs, gaps):
        arrival += gap / rate
        while time.perf_counter() < arrival:
            time.sleep(max(0.0, min(arrival - time.perf_counter(), 0.002)))
        ctx.comb(p.a, p.b)
        plain_lat.append((time.perf_counter() - arrival) * 1e3)
    plain_wall = time.perf_counter() - t0
    pp50, pp99 = pct(np.array(plain_lat))
    return {"workload": f"{nreq} requests, Poisson {rate}/s, lengths log-uniform [1024,262144], alphabet 4|20",
            "pairs_per_s": round(nreq / wall, 1), "gcups": round(cells / wall / 1e9, 1),
            "p50_ms": p50, "p99_ms": p99,
            "plain_pairs_per_s": round(nreq / plain_wall, 1), "plain_p50_ms": pp50, "plain_p99_ms": pp99,
            "capacity_pairs_per_s": round(nreq / sat_wall, 1),
            "capacity_gcups": round(cells / sat_wall / 1e9, 1),
            "capacity_p99_ms": pct(sat_lat)[1],
            "higher_rates": sweep,
            "micro_batches": st["batches"], "max_inflight": st["max_inflight"],
            "bit_exact_vs_alone_sample": bool(exact), "cost_model": info or "none (heuristic schedules)"}


def main():
    args = parse()
    if args.calibrate_copy:
        calibrate_copy()
        return
    if args.gpus != 1:
        print(f"bench.py runs on one GPU: --gpus {args.gpus} is not supported by this build "
              "(the multi-GPU sharding is a design only)", file=sys.stderr)
        sys.exit(2)
    size = 1 << args.log2n
    wl = lcs_amd.workload_single(f"mutated2^{args.log2n}", seed=1)
    a, b = wl.a, wl.b
    m, n = a.size, b.size
    ctx = lcs_amd.Context(0)
    cus, _ = ctx.info()
    sched = lcs_amd.schedule(tile_m=args.tile_m, waves_per_simd=args.waves_per_simd, variant=args.variant)
    da, db = H.DeviceArray.from_numpy(a), H.DeviceArray.from_numpy(b)
    dh, dv = H.DeviceArray(m), H.DeviceArray(n)
    L = lcs_amd.lib()

    def step():
        rc = L.lcs_comb_device(ctx.handle, da.ptr, m, db.ptr, n, sched, dh.ptr, dv.ptr, None)
        if rc:
            raise lcs_amd.LcsError("lcs_comb_device", rc)
        H.synchronize()
        # every timed step: a device-side wait that gave up would end the
        # launch early and be timed as a fast step
        st = ctx.status()
        if st:
            raise lcs_amd.LcsError("lcs_ctx_status", st)
        return ctx.info()[1], ctx.chain_ms()

    for _ in range(args.warmup):
        step()
    H.synchronize()
    kernel_ms = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        kernel_ms.append(step())
    H.synchronize()
    wall = time.perf_counter() - t0
    h, v = dh.numpy(), dv.numpy()
    # size-independent checks: the output is a bijection on [0, m+n)
    r2c, c2r = lcs_amd.from_strands(h, v)
    assert (r2c >= 0).all() and (c2r >= 0).all(), "output strands are not a permutation"
    llcs = int((v < m).sum())
    checked = None
    if args.check:
        alt = lcs_amd.schedule(tile_m=8 if (args.tile_m or 16) != 8 else 4)
        h2, v2, _ = ctx.comb(a, b, alt)
        checked = bool(np.array_equal(h, h2) and np.array_equal(v, v2))
    cells = float(m) * float(n)
    ms_step = wall / args.steps * 1e3
    gcups = cells * args.steps / wall / 1e9
    # the dominant kernel is the band chain (one launch combs every tile);
    # the rest of a step is the steady-ant merges of the tiles' permutations
    k_ms = float(np.mean([t for t, _ in kernel_ms]))
    chain_ms = float(np.mean([c for _, c in kernel_ms]))
    peak_ops = cus * 64 * PEAK_CLOCK_HZ
    achieved_ops = OPS_PER_CELL * cells / (chain_ms / 1e3)
    pmc_file = os.path.join(ROOT, "profiles", "comb_chain_mutated2^20_pmc.txt")
    traffic = read_traffic(pmc_file)
    clock_ghz = read_profile_value(pmc_file, "GRBM_GUI_ACTIVE / 8 XCDs / kernel time =")
    # end to end, as the reference times it: host strings in, permutation in
    # host memory (built on the GPU by lcs_comb_permutation); one untimed call
    # first reserves its device buffers
    ctx.comb_permutation(a, b, sched)
    t0 = time.perf_counter()
    r2c2, c2r2, _ = ctx.comb_permutation(a, b, sched)
    e2e = time.perf_counter() - t0
    e2e_same = bool(np.array_equal(r2c2, r2c) and np.array_equal(c2r2, c2r))
    out = {
        "metric": "GCUPS at m=n=2^20 (seaweed permutation, bit-exact)",
        "value": round(gcups, 2),
        "unit": "GCUPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_step, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int32",
        "data": "synthetic (seeded mt19937_64: uniform alphabet-4 A, B = A + 10% subs + 2% indels)",
        "config": {"workload": f"single pair m=n=2^{args.log2n}, tiled band-chain comb + steady-ant merge "
                               "(library default schedule: tiles by predicted time, 4 x 2 with seven merges at 2^20)",
                   "m": m, "n": n, "alphabet": 4, "tile_m": args.tile_m or None, "variant": args.variant or None,
                   "llcs": llcs},
        "roofline": {"bound": "valu", "achieved": round(achieved_ops / 1e12, 3), "peak": round(peak_ops / 1e12, 3),
                     "unit": "TOP/s (int32 lane-ops, 4 per cell)", "frac": round(achieved_ops / peak_ops, 4),
                     "traffic": traffic, "kernel": "comb_chain_kernel<16,32> (seed + chain + extract launch)",
                     "kernel_ms": round(chain_ms, 3), "kernel_gcups": round(cells / (chain_ms / 1e3) / 1e9, 2),
                     "step_kernels_ms": round(k_ms, 3),
                     "merge_share": round(max(0.0, 1.0 - chain_ms / k_ms), 4),
                     "measured_clock_ghz": clock_ghz,
                     "frac_at_measured_clock": (round(achieved_ops / (cus * 64 * clock_ghz * 1e9), 4)
                                                if clock_ghz else None)},
        "end_to_end": {"what": "lcs_comb_permutation: host strings in, PermutationMatrix rows in host memory",
                       "ms": round(e2e * 1e3, 3), "gcups": round(cells / e2e / 1e9, 2), "same_permutation": e2e_same},
    }
    if checked is not None:
        out["cross_schedule_bit_exact"] = checked
    if not args.no_cpu:
        out["config1"] = bench_config1(ctx)
    if not args.no_merge:
        out["tiled_merge"] = bench_tiled_merge(ctx, da, db, m, n, h, v)
    if not args.no_semilocal:
        out["semilocal"] = bench_semilocal(ctx, r2c, m, n, llcs)
    if not args.no_llcs:
        out["llcs_bitparallel"] = bench_llcs(ctx, a, b, llcs)
    if not args.no_zipf:
        out["zipf_planted"] = bench_zipf(ctx)
    if args.batch_pairs > 0:
        out["batched"] = bench_batch(ctx, args.batch_pairs)
    if args.serve_requests > 0:
        out["served"] = bench_serve(ctx, args.serve_requests, args.serve_rate)
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(a, b, args.cpu_seconds)
    print(json.dumps(out), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
