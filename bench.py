#!/usr/bin/env python3
"""Throughput of the trace-analysis path on one MI355X, plain and with the
learned EM initialiser.

A step is one 512-frame chunk of every ZMW of the pool through the whole
path (baseline filter, statistics aggregation, histogram, EM detection-model
estimation, Viterbi labeling, pulse accumulation) in the measurement
configuration: sigma EMA off and one model estimate per chunk, so every
stage runs on every chunk.  Workload: 2,097,152 ZMWs (32,768 lanes x 64) of
int16 traces, 16 chunks streamed (the first `warmup` chunks cover the
baseliner/DME start-up and are not timed).  All chunks are generated on the
GPU before timing starts, so inputs are resident in HBM.

Legs:
  plain    the drop-in path (reference EM, 20-iteration limit).
  learned  the same path with the learned EM start: 4,194,304 training pairs
           are generated by the plain pipeline on traces with per-ZMW SNR ~
           U[4, 20], the network is trained on the GPU (time reported, not in
           the timed region), then the pipeline runs with the EM capped at 3
           iterations and the plain EM as fallback.
  stress   4,194,304 ZMWs x 1024 frames at low SNR (sigma 25, amplitudes
           90/60/40/25), a +60 baseline step, 5% empty ZMWs: plain and
           learned throughput, fallback rate and label agreement (under
           "stress").
  batched  six pools of 131,072 ... 2,097,152 ZMWs with chunk lengths drawn from
           {256, 512, 1024}, autotuned kernel shapes, one captured hipGraph per
           chunk step, plain and learned-start (reported under "batched").
`value` is the plain leg's throughput: its frame labels agree with the
reference form of the oracle (DmeEmHost's own EM arithmetic) on >= 99.99% of
frames.  The learned leg is reported beside it with its label agreement with
the plain leg, counted on the GPU over every timed chunk, and the plain
pipeline's own agreement between a 20- and a 21-iteration EM limit (its
sensitivity to one more iteration).

Prints one JSON line.  The CPU baseline is the scalar C++ oracle timed on a
bounded sample on the host cores.
"""
import argparse
import ctypes
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
# Algorithmic bytes per ZMW-frame (MultiScaleLarge filter, F = 512):
#  baseline  = 2 in + 2 out + 2.78 filter windows in/out + 0.09 EMA/latent + 0.18 stats
#  histogram = 2 in + 1.17 (300 x u16 counters out) + 0.03 (bounds in, outlier counts in and out)
#              + 0.02 edge state:
#              in this cadence every add follows a reset, whose counters are known to be zero
#              and are not read (4.41 with the counters read back, a chunk that continues a
#              histogram)
ALG_BYTES = {"baseline": 7.05, "histogram": 3.22}
# HBM bytes per BaselineKernel launch at 32,768 lanes x 512 frames for each
# autotuner variant, from rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE runs of this
# benchmark, scaled by the same counters' readings for the library's copy kernel
# over 1 GiB (FETCH_SIZE x 2.0, WRITE_SIZE x 1.0):
# profiles/analyzer_kernels_32768lanes_f512_hbm_traffic.md.  Keyed by the variant:
# lanes per workgroup 1, 2, 4 (variant % 3) x frame groups in flight 1, 2 (variant >= 3).
BASELINE_TRAFFIC_BYTES = {0: (1899107.5 * 2.0 + 3912546.4) * 1024, 1: (1826757.8 * 2.0 + 3810264.3) * 1024,
                          2: (1830723.6 * 2.0 + 3814150.6) * 1024, 3: (1867174.7 * 2.0 + 3935758.5) * 1024,
                          4: (1988898.2 * 2.0 + 4063900.4) * 1024, 5: (1854085.6 * 2.0 + 3806584.1) * 1024}
# The histogram fast pass's, keyed by its autotuner variant (after the deferred reset, as the
# analyzer runs it: the counters start from zero and are only written); variants 1-15 (one wave
# per lane and the multi-wave forms) from an earlier run of the same commands; 0 is 19's kernel.
HIST_TRAFFIC_BYTES = {0: (1164363.9 * 2.0 + 1246209.0) * 1024, 1: (1074663.3 * 2.0 + 1940203.7) * 1024,
                      2: (1073285.7 * 2.0 + 1265043.3) * 1024, 3: (1073762.7 * 2.0 + 1392934.5) * 1024,
                      4: (1074528.2 * 2.0 + 1940203.7) * 1024, 5: (1073305.1 * 2.0 + 1265043.3) * 1024,
                      6: (1074254.5 * 2.0 + 1392934.5) * 1024, 7: (1076842.1 * 2.0 + 1940203.7) * 1024,
                      8: (1073376.1 * 2.0 + 1265043.3) * 1024, 9: (1086409.3 * 2.0 + 1392934.5) * 1024,
                      10: (1088198.2 * 2.0 + 1940203.7) * 1024, 11: (1086277.3 * 2.0 + 1392934.5) * 1024,
                      12: (1077730.0 * 2.0 + 1392934.5) * 1024, 13: (1085679.9 * 2.0 + 1265043.3) * 1024,
                      14: (1101751.8 * 2.0 + 1265043.3) * 1024, 15: (1102221.7 * 2.0 + 1392934.5) * 1024,
                      16: (1138660.5 * 2.0 + 1246208.2) * 1024, 17: (1164246.4 * 2.0 + 1246211.4) * 1024,
                      18: (1146681.8 * 2.0 + 1246216.1) * 1024, 19: (1164363.9 * 2.0 + 1246209.0) * 1024,
                      20: (1261457.9 * 2.0 + 1246210.8) * 1024, 21: (1100022.0 * 2.0 + 1246220.1) * 1024}
HIST_KERNELS = [(0, "HistAddFullKernel"), (1, "HistAddKernel"), (9, "HistAddWavesKernel"), (16, "HistAddFullKernel")]
# VALU-bound stages: algorithmic VALU lane-operations per ZMW-frame (labeler: 61 add /
# compare / select of the sparse recursion + 13 state scores + ROI; EM at one estimate per
# 512-frame chunk: 20 iterations x (301 x 5 x (exp + 8) + 300 x 5 x 12) = 4e5 per ZMW per
# estimate), against 256 CUs x 2.4 GHz x 128 lanes per CU cycle (2 wave64 VALU instructions)
# = 7.86e13 lane-operations/s.  The VALU instructions the kernels issue per lane-frame are
# the SQ_INSTS_VALU counts of profiles/analyzer_kernels_32768lanes_f512_sq_counters.md.
VALU_PEAK_LANE_OPS = 256 * 2.4e9 * 128
VALU_ALG_OPS = {"labels": 400.0, "dme": 4.0e5 / 512}
VALU_ISSUED_PER_LANE_FRAME = {"labels": 440.5, "dme": 821.4}
STAGES = ["baseline", "aggregate", "histogram", "dme", "labels", "pulses", "metrics"]


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def cpu_baseline(lanes, frames, chunks, timed_from, threads):
    """The oracle in its reference form (DmeEmHost's own EM arithmetic) on the
    same configuration, whole chunks through every stage."""
    import oracle as O
    import hw_amd as H
    from hw_amd import types as T
    O.threads(threads)
    cfg = H.bench_config(frames)
    p = H.tracegen_default()
    st = np.zeros(lanes, dtype=T.TRACEGEN_STATE)
    data = [O.tracegen(p, lanes, frames, c * frames, st, c == 0) for c in range(chunks)]
    an = O.Analyzer(cfg, 0, lanes, frames, em="reference")
    dts = (T.PULSE, T.STAT_ACC, T.BASELINER_STATS, T.LANE_MODEL)
    t0 = None
    for c in range(chunks):
        if c == timed_from:
            t0 = time.perf_counter()
        r = an(data[c], c * frames, dts, want=("pulses",))
        if r["rc"] != 0:
            raise RuntimeError("oracle analyzer failed")
    dt = time.perf_counter() - t0
    zf = lanes * 64 * frames * (chunks - timed_from)
    return zf / dt, dt


def timed_leg(H, cfg, bufs, L, F, warmup, steps, init=None, keep=False):
    """Runs warm-up chunks, then times `steps` chunks; returns a result dict (with the
    analyzer under "analyzer" when keep is set)."""
    an = H.BatchAnalyzer(0, L, F, cfg)
    if init is not None:
        an.set_initializer(init)
    an.set_profiling(True)
    for c in range(warmup):
        an(bufs[c], c * F)
        an.sync()
    H.sync()
    stage_ms = {s: [] for s in STAGES}
    t0 = time.perf_counter()
    for c in range(warmup, warmup + steps):
        an(bufs[c], c * F)
        ms = an.stage_ms()   # waits for this chunk's last event
        for s, v in zip(STAGES, ms):
            stage_ms[s].append(v)
    H.sync()
    dt = time.perf_counter() - t0
    fallback = an.fallback_count() if init is not None else None
    mean_ms = {s: float(np.mean(v)) for s, v in stage_ms.items()}
    zf = L * 64 * F
    res = {"value": zf * steps / dt, "dt": dt, "ms_per_step": dt * 1e3 / steps, "stage_ms": mean_ms,
           "em_iterations": an.em_iterations(), "fallback_last": fallback}
    if keep:
        res["analyzer"] = an
    return res


def host_input_leg(H, cfg, bufs, L, F, warmup, steps):
    """The plain pipeline with every chunk handed over in pinned host memory
    (hwpa_analyzer_process with on_device = 0): each call copies its chunk in on the
    analyzer's copy stream, overlapping the previous chunk's stages, and returns when
    the copy is done.  Timed like the plain leg, PCIe transfer included; beside it one
    2-byte-per-sample chunk copied host to device alone."""
    n = L * F * 64
    host = []
    for b in bufs[:warmup + steps]:
        h = H.host_pinned(n * 2)
        H.check(H.lib.hwpa_memcpy_dtoh(ctypes.c_void_p(h.data_ptr()), H.ptr(b), ctypes.c_size_t(n * 2)))
        host.append(h)
    d = H.dev_bytes(n * 2)
    H.check(H.lib.hwpa_memcpy_htod(H.ptr(d), ctypes.c_void_p(host[0].data_ptr()), ctypes.c_size_t(n * 2)))
    t0 = time.perf_counter()
    reps = 3
    for i in range(reps):
        H.check(H.lib.hwpa_memcpy_htod(H.ptr(d), ctypes.c_void_p(host[i % len(host)].data_ptr()),
                                       ctypes.c_size_t(n * 2)))
    copy_ms = (time.perf_counter() - t0) * 1e3 / reps
    del d
    an = H.BatchAnalyzer(0, L, F, cfg)
    for c in range(warmup):
        an(host[c], c * F, on_device=False)
    an.sync()
    t0 = time.perf_counter()
    for c in range(warmup, warmup + steps):
        an(host[c], c * F, on_device=False)
    an.sync()
    dt = time.perf_counter() - t0
    zf = L * 64 * F
    return {"value": zf * steps / dt, "ms_per_step": dt * 1e3 / steps, "steps": steps, "pinned": True,
            "copy_ms_per_chunk": copy_ms, "copy_gbs": n * 2 / (copy_ms * 1e-3) / 1e9}


def baz_leg(H, an, repeats=20):
    """BAZ packet encoding (production layout: bases only) of the analyzer's last chunk of
    pulses: size pass, scan and encode, timed over `repeats` calls from the same delta state."""
    pp, pc, mc = an.pulses_device()
    zmws = an.lanes * 64
    enc = H.BazEncoder(zmws)
    d_off, d_ev = H.dev_bytes((zmws + 1) * 8), H.dev_bytes(zmws * 4)
    enc.encode(pp, pc, mc, None, 0, d_off, d_ev)
    total = int(H.to_numpy(d_off, np.uint64, (zmws + 1,))[-1])
    events = int(H.to_numpy(d_ev, np.uint32, (zmws,)).sum())
    counts = H.fetch(pc, np.uint32, (zmws,))
    records = int(np.minimum(counts, mc).sum())
    d_out = H.dev_bytes(total + 16)
    for _ in range(3):
        enc.reset()
        enc.encode(pp, pc, mc, d_out, total, d_off, d_ev)
    H.sync()
    t0 = time.perf_counter()
    for _ in range(repeats):
        enc.reset()
        enc.encode(pp, pc, mc, d_out, total, d_off, d_ev)
    H.sync()
    ms = (time.perf_counter() - t0) * 1e3 / repeats
    # Algorithmic bytes: pulse records read once (20 B), stream written, per-ZMW delta state
    # read and written (16 B), offsets (8 B) and event counts (4 B) written.
    alg = records * 20 + total + zmws * (16 + 8 + 4)
    gbs = alg / (ms * 1e-3) / 1e9
    return {"zmws": zmws, "pulse_records": records, "bases_encoded": events, "stream_bytes": total,
            "bytes_per_base": total / max(events, 1), "ms_per_chunk": ms, "alg_bytes": alg, "achieved_gbs": gbs,
            "hbm_frac": gbs / HBM_PEAK_GBS}


def repack_leg(H, T, L, F, packet_blocks=50, repeats=10):
    """Block repacking of one chunk (L lanes x F frames, int16) from dense packets of
    packet_blocks blocks of 64 ZMWs x F frames, as a sensor source would deliver them:
    every sample read once and written once."""
    zmws = L * 64
    per = packet_blocks * 64
    src = H.dev_bytes(zmws * F * 2)
    packets = []
    for z0 in range(0, zmws, per):
        nb = min(packet_blocks, (zmws - z0) // 64)
        packets.append((src.view(z0 * F * 2, nb * 64 * F * 2), z0, 0, nb, F, 64))
    dst = H.dev_bytes(zmws * F * 2)
    r = H.Repacker(max_packets=len(packets))
    for _ in range(2):
        r.run(packets, T.ENCODING_INT16, dst, 0, 0, L, F)
    H.sync()
    t0 = time.perf_counter()
    for _ in range(repeats):
        r.run(packets, T.ENCODING_INT16, dst, 0, 0, L, F)
    H.sync()
    ms = (time.perf_counter() - t0) * 1e3 / repeats
    gbs = 2.0 * zmws * F * 2 / (ms * 1e-3) / 1e9
    return {"packets": len(packets), "packet_shape": [packet_blocks, F, 64], "bytes_moved": 2 * zmws * F * 2,
            "ms_per_chunk": ms, "achieved_gbs": gbs, "hbm_frac": gbs / HBM_PEAK_GBS}


def agreement(H, cfg_a, cfg_b, bufs, L, F, first, init_b=None, fallbacks=None):
    """Fraction of equal frame labels between two pipelines over chunks >= first.
    With `fallbacks` (a list), appends pipeline b's fallback ZMW count of every
    such chunk."""
    a = H.BatchAnalyzer(0, L, F, cfg_a)
    b = H.BatchAnalyzer(0, L, F, cfg_b)
    if init_b is not None:
        b.set_initializer(init_b)
    n = L * F * 64
    eq = tot = 0
    for c in range(len(bufs)):
        a(bufs[c], c * F)
        b(bufs[c], c * F)
        a.sync()
        b.sync()
        if c >= first and a.flags()[2] and b.flags()[2]:
            eq += H.count_equal_i16(a.labels_device(), b.labels_device(), n)
            tot += n
            if fallbacks is not None:
                fallbacks.append(b.fallback_count())
    return eq / tot if tot else None


STRESS_LANES, STRESS_FRAMES = 65536, 1024
# The stress distribution's generator settings (besides the seed and the step span).
STRESS_GEN = dict(baseline_sigma=25.0, amplitude=(90.0, 60.0, 40.0, 25.0), drift_per_chunk=0.0, step_drift=60.0,
                  empty_fraction=0.05)


def stress_leg(H, T, init, warmup=2, steps=4, seed=77, sensitivity=True):
    """Learned start under stress: 4,194,304 ZMWs x 1024-frame chunks, baseline
    sigma 25, amplitudes 90/60/40/25 (10% noise), no linear drift but a +60
    count baseline step at a uniformly drawn frame of the run, 5% of the ZMWs
    empty.  Times the plain and the learned pipeline, then runs both side by
    side for label agreement and the fallback count of every estimate."""
    L, F = STRESS_LANES, STRESS_FRAMES
    chunks = warmup + steps
    gen = H.tracegen_default(seed=seed, step_span=float(chunks * F), **STRESS_GEN)
    d_state = H.dev_bytes(L * T.TRACEGEN_STATE.itemsize)
    bufs = []
    for c in range(chunks):
        b = H.dev_bytes(L * F * 64 * 2)
        H.tracegen(gen, L, F, c * F, d_state, c == 0, b)
        bufs.append(b)
    H.sync()
    cfg = H.bench_config(F)
    cfgL = H.bench_config(F)
    cfgL.learned_init = 1
    plain = timed_leg(H, cfg, bufs, L, F, warmup, steps)
    learned = timed_leg(H, cfgL, bufs, L, F, warmup, steps, init=init)
    fb = []
    agree = agreement(H, cfg, cfgL, bufs, L, F, warmup, init_b=init, fallbacks=fb)
    Z = L * 64
    out = {"zmws": Z, "lanes": L, "frames_per_chunk": F, "chunks": chunks, "warmup": warmup, "steps": steps,
           "data": "sigma 25, amplitudes 90/60/40/25 (10%% noise), +60 step at a random frame, 5%% empty ZMWs, "
                   "seed %d" % seed,
           "plain_value": plain["value"], "plain_ms_per_step": plain["ms_per_step"],
           "learned_value": learned["value"], "learned_ms_per_step": learned["ms_per_step"],
           "speedup_vs_plain": learned["value"] / plain["value"],
           "plain_stage_ms": plain["stage_ms"], "learned_stage_ms": learned["stage_ms"],
           "fallback_rate": float(np.mean(fb)) / Z if fb else None,
           "fallback_zmws_per_estimate": fb, "label_agreement_vs_plain": agree}
    if sensitivity:
        cfg21 = H.bench_config(F)
        cfg21.em_iteration_limit = 21
        out["plain_20_vs_21_iterations_agreement"] = agreement(H, cfg, cfg21, bufs, L, F, warmup)
    return out


BATCH_LANES = [2048, 4096, 8192, 12288, 16384, 32768]


def batched_leg(H, T, init, warmup, steps, seed=2024, distinct=None, autotune=True):
    """Six pools (131,072 ... 2,097,152 ZMWs) with chunk lengths drawn from
    {256, 512, 1024}, all run one chunk step at a time through one captured
    hipGraph per step.  Every pool estimates its model once per 512 frames (or
    per chunk, for longer chunks), the cadence of the single-pool legs, so the
    pools' ZMW-frames cost what they cost there.  Every step's chunks are
    generated before timing (resident in HBM), consecutive chunks of each
    pool's traces unless `distinct` caps their number (then they repeat)."""
    rng = np.random.default_rng(seed)
    frames = [int(rng.choice([256, 512, 1024])) for _ in BATCH_LANES]
    pools = []
    for i, (L, F) in enumerate(zip(BATCH_LANES, frames)):
        cfg = H.bench_config(F, estimate_frames=512)
        cfg.learned_init = 1 if init is not None else 0
        pools.append((100 + i, L, F, cfg))
    b = H.Batch(pools)
    if init is not None:
        b.set_initializer(init)
    tune_s = 0.0
    if autotune:
        t0 = time.perf_counter()
        b.autotune(repeats=2)
        tune_s = time.perf_counter() - t0
    distinct = distinct or (warmup + steps)
    chunks = []
    for i, (_, L, F, _) in enumerate(pools):
        gen = H.tracegen_default(seed=seed + 17 * i)
        st = H.dev_bytes(L * T.TRACEGEN_STATE.itemsize)
        bufs = []
        for c in range(distinct):
            buf = H.dev_bytes(L * F * 64 * 2)
            H.tracegen(gen, L, F, c * F, st, c == 0, buf)
            bufs.append(buf)
        chunks.append(bufs)
    H.sync()
    for c in range(warmup):
        b.process([chunks[i][c % distinct] for i in range(len(pools))], [c * p[2] for p in pools])
    b.sync()
    t0 = time.perf_counter()
    for c in range(warmup, warmup + steps):
        b.process([chunks[i][c % distinct] for i in range(len(pools))], [c * p[2] for p in pools])
    b.sync()
    dt = time.perf_counter() - t0
    zf = sum(L * 64 * F for _, L, F, _ in pools) * steps
    out = {"value": zf / dt, "ms_per_step": dt * 1e3 / steps, "pools": [[L, F] for _, L, F, _ in pools],
           "zmws": sum(L * 64 for _, L, _, _ in pools), "steps": steps, "warmup": warmup,
           "graph": b.graph_stats(), "autotune_s": tune_s,
           "tuned": [[H.tune_get(k, L, F) for k in range(4)] for _, L, F, _ in pools],
           "distinct_chunks_per_pool": distinct}
    if init is not None:
        out["fallback_zmws_last_step"] = sum(b.pool(i).fallback_count() for i in range(len(pools)))
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=12)
    ap.add_argument("--warmup", type=int, default=4)
    ap.add_argument("--lanes", type=int, default=32768)
    ap.add_argument("--frames", type=int, default=512)
    ap.add_argument("--cpu-lanes", type=int, default=64)
    ap.add_argument("--cpu-chunks", type=int, default=16)
    ap.add_argument("--no-host-input", action="store_true",
                    help="skip the leg that hands chunks over in pinned host memory")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--plain-only", action="store_true")
    ap.add_argument("--train-pairs", type=int, default=4 * 1024 * 1024)
    ap.add_argument("--train-epochs", type=int, default=10)
    ap.add_argument("--no-agreement", action="store_true")
    ap.add_argument("--no-batched", action="store_true")
    ap.add_argument("--batched-steps", type=int, default=10)
    ap.add_argument("--no-stress", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the path shards by pool with no exchange, "
              "so --gpus %d is not run (use --gpus 1)" % args.gpus, file=sys.stderr)
        return 2
    if args.warmup < 4:
        log("warmup raised to 4 chunks (baseliner start-up 1024 frames + first estimate)")
        args.warmup = 4

    import hw_amd as H
    from hw_amd import types as T

    L, F = args.lanes, args.frames
    chunks = args.warmup + args.steps
    cfg = H.bench_config(F)
    gen = H.tracegen_default()
    log("generating %d chunks of %d lanes x %d frames on the GPU" % (chunks, L, F))
    d_state = H.dev_bytes(L * T.TRACEGEN_STATE.itemsize)
    bufs = []
    for c in range(chunks):
        b = H.dev_bytes(L * F * 64 * 2)
        H.tracegen(gen, L, F, c * F, d_state, c == 0, b)
        bufs.append(b)
    H.sync()
    copy_ms, copy_gbs = H.copy_bandwidth(1 << 30, 10)
    log("copy kernel: 1 GiB in %.3f ms = %.0f GB/s read+write" % (copy_ms, copy_gbs))
    t0 = time.perf_counter()
    tuned = H.autotune(cfg, L, F, repeats=6)   # the labeler's variants differ by ~2%: more launches per timing
    tune_s = time.perf_counter() - t0
    log("autotune (%.1f s): histogram, baseline, labels, pulses variants %s" % (tune_s, tuned["chosen"]))

    plain = timed_leg(H, cfg, bufs, L, F, args.warmup, args.steps, keep=True)
    log("plain: %.3g ZMW-frames/s, %.2f ms/chunk, stage ms %s" % (
        plain["value"], plain["ms_per_step"], {k: round(v, 3) for k, v in plain["stage_ms"].items()}))
    baz = baz_leg(H, plain.pop("analyzer"))
    repack = repack_leg(H, T, L, F)
    host_in = None
    if not args.no_host_input:
        hs = min(args.steps, 6)
        host_in = host_input_leg(H, cfg, bufs, L, F, args.warmup, hs)
        log("host input (pinned, PCIe included): %.3g ZMW-frames/s, %.2f ms/chunk; one chunk copied in %.2f ms "
            "(%.1f GB/s)" % (host_in["value"], host_in["ms_per_step"], host_in["copy_ms_per_chunk"], host_in["copy_gbs"]))
    log("repack: %d packets -> %d lanes x %d frames in %.3f ms, %.0f GB/s read+write" % (
        repack["packets"], L, F, repack["ms_per_chunk"], repack["achieved_gbs"]))
    log("BAZ encoding: %d bases -> %d bytes (%.2f B/base) in %.3f ms, %.0f GB/s algorithmic" % (
        baz["bases_encoded"], baz["stream_bytes"], baz["bytes_per_base"], baz["ms_per_chunk"], baz["achieved_gbs"]))

    learned = None
    train_info = None
    if not args.plain_only:
        from hw_amd import learned as Lr
        # Half of the pairs from the bench distribution with per-ZMW SNR ~ U[4, 20], half from
        # the stress distribution (sigma 25, analog ratios 90/60/40/25 with the brightest at
        # SNR ~ U[2, 8], +60 baseline steps, 5% empty ZMWs, 1024-frame chunks).
        zpe = L * 64
        half = args.train_pairs // 2
        pairs = Lr.PairSet(args.train_pairs)
        t0 = time.perf_counter()
        Lr.generate_pairs(L, 2 + max(1, (half + zpe - 1) // zpe) + 1, seed=424242, snr=(4.0, 20.0), frames=F,
                          pairs=pairs, min_conf=0.0, log=log, limit=half)
        Lr.generate_pairs(L // 2, 2 + max(1, (args.train_pairs - half + zpe // 2 - 1) // (zpe // 2)) + 1,
                          seed=434343, snr=(2.0, 8.0), frames=STRESS_FRAMES, pairs=pairs, min_conf=0.0, log=log,
                          gen_overrides=dict(STRESS_GEN, step_span=float(8 * STRESS_FRAMES)))
        gen_s = time.perf_counter() - t0
        init = H.Initializer(seed=1)
        losses, train_s = Lr.train(init, pairs, epochs=args.train_epochs, batch=4096, lr=2e-3, log=log)
        train_info = {"pairs": pairs.n, "valid_fraction": pairs.valid_fraction(), "generate_s": gen_s,
                      "train_s": train_s, "epochs": args.train_epochs, "batch": 4096,
                      "loss_first": losses[0][1], "loss_last": losses[-1][1]}
        pairs = None
        cfgL = H.bench_config(F)
        cfgL.learned_init = 1
        learned = timed_leg(H, cfgL, bufs, L, F, args.warmup, args.steps, init=init)
        log("learned: %.3g ZMW-frames/s, %.2f ms/chunk, stage ms %s, fallback %s of %d" % (
            learned["value"], learned["ms_per_step"], {k: round(v, 3) for k, v in learned["stage_ms"].items()},
            learned["fallback_last"], L * 64))
        # A second operating point: the same network with the EM capped at 3 iterations.
        cfg3 = H.bench_config(F)
        cfg3.learned_init = 1
        cfg3.learned_em_iteration_limit = 3
        cap3 = timed_leg(H, cfg3, bufs, L, F, args.warmup, args.steps, init=init)
        log("learned, EM cap 3: %.3g ZMW-frames/s, %.2f ms/chunk, fallback %s" % (
            cap3["value"], cap3["ms_per_step"], cap3["fallback_last"]))
        if not args.no_agreement:
            learned["label_agreement"] = agreement(H, cfg, cfgL, bufs, L, F, args.warmup, init_b=init)
            cap3["label_agreement"] = agreement(H, cfg, cfg3, bufs, L, F, args.warmup, init_b=init)
            cfg21 = H.bench_config(F)
            cfg21.em_iteration_limit = 21
            learned["plain_20_vs_21_iterations_agreement"] = agreement(H, cfg, cfg21, bufs, L, F, args.warmup)
            log("label agreement learned vs plain %.6f; plain 20 vs 21 EM iterations %.6f" % (
                learned["label_agreement"], learned["plain_20_vs_21_iterations_agreement"]))

    stress = None
    if learned is not None and not args.no_stress:
        bufs = None
        log("stress: %d ZMWs x %d frames, learned vs plain" % (STRESS_LANES * 64, STRESS_FRAMES))
        stress = stress_leg(H, T, init, sensitivity=not args.no_agreement)
        log("  plain %.3g, learned %.3g ZMW-frames/s (%.2fx), fallback %.4f, agreement %.6f, plain 20 vs 21 %s" % (
            stress["plain_value"], stress["learned_value"], stress["speedup_vs_plain"], stress["fallback_rate"],
            stress["label_agreement_vs_plain"], stress.get("plain_20_vs_21_iterations_agreement")))

    batched = None
    if not args.no_batched:
        log("batched pools: plain")
        batched = {"plain": batched_leg(H, T, None, 12, args.batched_steps)}
        log("  %.3g ZMW-frames/s, %.1f ms/step, graph %s" % (batched["plain"]["value"], batched["plain"]["ms_per_step"],
                                                            batched["plain"]["graph"]))
        if learned is not None:
            log("batched pools: learned")
            batched["learned"] = batched_leg(H, T, init, 12, args.batched_steps, autotune=False)
            log("  %.3g ZMW-frames/s, %.1f ms/step, fallback %s" % (
                batched["learned"]["value"], batched["learned"]["ms_per_step"],
                batched["learned"]["fallback_zmws_last_step"]))
            batched["learned_vs_plain_single_pool"] = batched["learned"]["value"] / plain["value"]

    # The headline is the plain pipeline: its labels agree with the reference form of
    # the oracle on >= 99.99% of frames (tests/test_gpu_reference.py); the learned start's
    # agreement with the plain pipeline is below that, so its rate is reported beside it.
    head = plain
    mean_ms = plain["stage_ms"]
    zf_step = L * 64 * F
    bl_gbs = ALG_BYTES["baseline"] * zf_step / (mean_ms["baseline"] * 1e-3) / 1e9
    hist_gbs = ALG_BYTES["histogram"] * zf_step / (mean_ms["histogram"] * 1e-3) / 1e9

    cpu = None
    if not args.no_cpu:
        threads = min(16, os.cpu_count() or 1)
        log("timing the CPU oracle on %d lanes x %d chunks with %d threads" % (args.cpu_lanes, args.cpu_chunks,
                                                                             threads))
        cpu_value, cpu_dt = cpu_baseline(args.cpu_lanes, F, args.cpu_chunks, 0, threads)
        cpu = {"value": cpu_value, "unit": "ZMW-frames/s", "cores": threads, "kind": "port",
               "sample": "the CPU workload of %d ZMWs (%d lanes x 64) x %d frames (%d chunks of %d, all timed, "
                         "%.1f s): the oracle's reference form of the plain pipeline (DmeEmHost's EM arithmetic), "
                         "same configuration, one thread per core" % (
                             args.cpu_lanes * 64, args.cpu_lanes, args.cpu_chunks * F, args.cpu_chunks, F, cpu_dt)}

    workload = ("plain pipeline (reference EM), %d ZMWs (%d lanes x 64) x %d-frame int16 chunks, %d chunks "
                "streamed, one estimate per chunk" % (L * 64, L, F, chunks))
    out = {
        "metric": "ZMW-frames/s on 1 GPU, plain vs learned-DME init, at matched label agreement",
        "value": head["value"],
        "unit": "ZMW-frames/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": head["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int16+f32",
        "data": "synthetic (seeded GPU generator: N(0,12^2) baseline, +-40 counts/chunk drift, "
                "amplitudes 180/120/80/50, geometric widths 8 / gaps 20)",
        "config": {"workload": workload, "lanes": L, "frames_per_chunk": F, "chunks": chunks,
                   "filter": "MultiScaleLarge", "init": "plain EM"},
        "roofline": {"bound": "hbm", "kernel": "BaselineKernel", "achieved": bl_gbs, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": bl_gbs / HBM_PEAK_GBS,
                     "traffic": BASELINE_TRAFFIC_BYTES.get(tuned["chosen"][1]) if (L, F) == (32768, 512) else None,
                     "alg_bytes_per_zmw_frame": ALG_BYTES["baseline"], "copy_kernel_gbs": copy_gbs},
        "histogram_roofline": {"kernel": [n for v, n in HIST_KERNELS if tuned["chosen"][0] >= v][-1],
                               "variant": tuned["chosen"][0], "bound": "hbm", "achieved": hist_gbs,
                               "peak": HBM_PEAK_GBS, "unit": "GB/s",
                               "frac": hist_gbs / HBM_PEAK_GBS, "alg_bytes_per_zmw_frame": ALG_BYTES["histogram"],
                               "traffic": HIST_TRAFFIC_BYTES.get(tuned["chosen"][0]) if (L, F) == (32768, 512)
                               else None},
        "valu_rooflines": {k: {"kernel": {"labels": "LabelKernel", "dme": "DmeEstimateKernel"}[k], "bound": "valu",
                               "achieved": VALU_ALG_OPS[k] * zf_step / (mean_ms[k] * 1e-3),
                               "peak": VALU_PEAK_LANE_OPS, "unit": "lane-ops/s",
                               "frac": VALU_ALG_OPS[k] * zf_step / (mean_ms[k] * 1e-3) / VALU_PEAK_LANE_OPS,
                               "alg_ops_per_zmw_frame": VALU_ALG_OPS[k],
                               "issued_valu_per_lane_frame": VALU_ISSUED_PER_LANE_FRAME[k],
                               "issue_frac": VALU_ISSUED_PER_LANE_FRAME[k] * zf_step / 64 / (mean_ms[k] * 1e-3)
                               / (VALU_PEAK_LANE_OPS / 64)}
                           for k in ("labels", "dme")},
        "autotune": {"seconds": tune_s, "histogram_ms": tuned["histogram"], "baseline_ms": tuned["baseline"],
                     "labels_ms": tuned["labels"], "pulses_ms": tuned["pulses"], "chosen": tuned["chosen"]},
        "stage_ms": head["stage_ms"],
        "dominant_stage": max(head["stage_ms"], key=head["stage_ms"].get),
        "plain": {"value": plain["value"], "ms_per_step": plain["ms_per_step"], "stage_ms": plain["stage_ms"],
                  "em_iterations_last_chunk": plain["em_iterations"]},
        "cpu_baseline": cpu,
        "baz_encoding": baz,
        "host_input": host_in,
        "repack": repack,
    }
    if learned is not None:
        out["learned"] = {"value": learned["value"], "ms_per_step": learned["ms_per_step"],
                          "stage_ms": learned["stage_ms"], "speedup_vs_plain": learned["value"] / plain["value"],
                          "fallback_zmws_last_chunk": learned["fallback_last"],
                          "label_agreement_vs_plain": learned.get("label_agreement"),
                          "plain_20_vs_21_iterations_agreement": learned.get("plain_20_vs_21_iterations_agreement"),
                          "em_iteration_cap": cfgL.learned_em_iteration_limit,
                          "em_convergence_tolerance": cfgL.learned_conv_tol, "training": train_info,
                          "em_cap_3": {"value": cap3["value"], "ms_per_step": cap3["ms_per_step"],
                                       "speedup_vs_plain": cap3["value"] / plain["value"],
                                       "fallback_zmws_last_chunk": cap3["fallback_last"],
                                       "label_agreement_vs_plain": cap3.get("label_agreement")}}
    if batched is not None:
        out["batched"] = batched
    if stress is not None:
        out["stress"] = stress
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
