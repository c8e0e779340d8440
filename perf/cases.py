"""Performance cases of the trace-analysis library, through its public entry points.

A case is a dict of plain values.  Its "kind" names what a user's program does
with the library; sizes are lanes of 64 ZMWs and frames per chunk.  Sizes come
from the benchmark's pools (2,048 ... 32,768 lanes, chunks of 256, 512 or 1024
frames), the tests' (a few lanes, uneven chunk lengths) and the integration
guide's (4,096 lanes x 512 frames); traces are the library's own seeded
generator's, with the signal-to-noise range, drift and share of empty ZMWs the
benchmark and the tests use.
"""
import ctypes

import numpy as np
import torch

import hw_amd as H
from hw_amd import learned as Lr
from hw_amd import types as T

LANE = T.LANE
STATS_BYTES = T.BASELINER_STATS.itemsize
HIST_BYTES = T.LANE_HIST.itemsize
MODEL_BYTES = T.LANE_MODEL.itemsize
# Filter windows, sample history and scalars of the large multi-scale baseline filter, per lane.
FILTER_STATE_BYTES = 47400
# One EM estimate of one ZMW: 20 iterations over 301 bin boundaries of 5 components.
EM_FLOPS_PER_ZMW = 4.0e5
# 13-state scorer and sparse recursion, per ZMW-frame.
LABEL_FLOPS = 400.0
BASELINE_FLOPS = 40.0
PULSE_FLOPS = 20.0
HIST_FLOPS = 8.0
MLP_FLOPS_PER_ROW = 2.0 * (128 * 256 + 256 * 256 + 256 * 12)


def listed():
    return [
        # The whole per-chunk analysis of the production pool, 2,097,152 ZMWs, one model estimate
        # per chunk, kernel shapes autotuned beforehand: the benchmark's headline workload.
        {"name": "pool-production", "kind": "pool", "lanes": 32768, "frames": 512, "enc": "int16", "input": "device",
         "cadence": "chunk", "tuned": True},
        # One pool of the integration guide's size as the reference's host calls it: 8-bit samples handed
        # over in page-locked host memory, the reference's estimation interval (4000 frames), not tuned.
        {"name": "pool-host-uint8", "kind": "pool", "lanes": 4096, "frames": 512, "enc": "uint8", "input": "pinned",
         "cadence": "reference", "tuned": False},
        # A small pool (a partly filled chip, a test run): what counts is how long one chunk takes.
        {"name": "pool-small", "kind": "pool", "lanes": 48, "frames": 512, "enc": "int16", "input": "device",
         "cadence": "chunk", "tuned": False},
        # Several uneven pools with different chunk lengths, one captured graph per chunk step.
        {"name": "pools-graph", "kind": "batch", "pools": 6, "lanes": 2048, "shape_seed": 11, "tuned": False},
        # The baseline filter stage on its own, a ragged number of lanes and long chunks.
        {"name": "baseline-stage", "kind": "baseline", "lanes": 9001, "frames": 1024, "enc": "int16", "filter": 0},
        # Statistics and histogram accumulation between two estimates: resets, then two chunks merged and
        # binned (a 1000-frame estimation interval).
        {"name": "accumulate-stage", "kind": "accumulate", "lanes": 6000, "frames": 512, "chunks": 2},
        # Model estimation (the EM fit) of one pool.
        {"name": "estimate-stage", "kind": "estimate", "lanes": 2048, "frames": 512},
        # Frame labels and pulses of one pool with a fixed model, a ragged pool and an uneven chunk.
        {"name": "call-stage", "kind": "call", "lanes": 1111, "frames": 496, "max_calls": 48},
        # Estimation started by the trained network, the low-confidence ZMWs re-estimated.
        {"name": "learned-estimate", "kind": "learned", "lanes": 4096, "frames": 512},
        # One optimisation step of the network, its gradients watched (batch size of the training recipe).
        {"name": "train-step", "kind": "train", "batch": 4096},
        # Packet encoding of one chunk's pulses for the output file.
        {"name": "encode-pulses", "kind": "baz", "lanes": 8192, "max_calls": 48, "internal": False},
        # Dense sensor packets into one pool's lane-major chunk.
        {"name": "repack-packets", "kind": "repack", "lanes": 4096, "frames": 512, "enc": "int16",
         "packet_blocks": 50, "block_width": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["pool", "pool", "batch", "baseline", "accumulate", "estimate", "call", "learned", "train", "baz",
                       "repack"])
    frames = rng.choice([256, 512, 512, 1024, 16 * rng.randint(8, 64)])
    if kind == "pool":
        pinned = rng.random() < 0.3
        return {"kind": "pool", "lanes": _log_int(rng, 16, 4096 if pinned else 12000), "frames": frames,
                "enc": rng.choice(["int16", "uint8"]), "input": "pinned" if pinned else "device",
                "cadence": rng.choice(["chunk", "reference"]), "tuned": False}
    if kind == "batch":
        return {"kind": "batch", "pools": rng.randint(2, 6), "lanes": _log_int(rng, 32, 2048),
                "shape_seed": rng.randrange(1 << 16), "tuned": False}
    if kind == "baseline":
        return {"kind": "baseline", "lanes": _log_int(rng, 16, 16000), "frames": frames,
                "enc": rng.choice(["int16", "uint8"]), "filter": rng.randint(0, 5)}
    if kind == "accumulate":
        return {"kind": "accumulate", "lanes": _log_int(rng, 16, 16000), "frames": frames, "chunks": rng.randint(1, 4)}
    if kind == "estimate":
        return {"kind": "estimate", "lanes": _log_int(rng, 16, 16000), "frames": frames}
    if kind == "call":
        return {"kind": "call", "lanes": _log_int(rng, 16, 16000), "frames": frames + rng.choice([0, 0, 1, -7]),
                "max_calls": rng.choice([48, 48, 24, 96])}
    if kind == "learned":
        return {"kind": "learned", "lanes": _log_int(rng, 16, 12000), "frames": frames}
    if kind == "train":
        return {"kind": "train", "batch": 64 * _log_int(rng, 4, 256)}
    if kind == "baz":
        return {"kind": "baz", "lanes": _log_int(rng, 16, 16000), "max_calls": rng.choice([48, 48, 24, 96]),
                "internal": rng.random() < 0.4}
    return {"kind": "repack", "lanes": _log_int(rng, 16, 12000), "frames": rng.choice([128, 256, 512, 1024]),
            "enc": rng.choice(["int16", "uint8"]), "packet_blocks": rng.randint(3, 60),
            "block_width": rng.choice([64, 64, 128])}


# ---- inputs ----------------------------------------------------------------------


def _empty(nbytes):
    return torch.empty(int(nbytes), dtype=torch.uint8, device="cuda")


def _zeros(nbytes):
    return torch.zeros(int(nbytes), dtype=torch.uint8, device="cuda")


class _Borrowed:
    """Device memory of the library as torch sees it (no copy); `owner` is kept alive."""

    def __init__(self, ptr, shape, typestr, owner):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}
        self.owner = owner


def _view(ptr, shape, typestr, owner):
    return torch.as_tensor(_Borrowed(ptr, shape, typestr, owner), device="cuda")


def _result(an, getter, shape, typestr):
    p = ctypes.c_void_p()
    H.check(getter(an.h, ctypes.byref(p)))
    return _view(p.value, shape, typestr, an)


def _traces(lanes, frames, chunks, seed, enc="int16"):
    """Consecutive chunks of seeded traces, [lanes, frames, 64], on the GPU."""
    gen = H.tracegen_default(seed=seed, snr_lo=6.0, snr_hi=18.0, empty_fraction=0.05)
    state = _empty(lanes * T.TRACEGEN_STATE.itemsize)
    out = []
    for c in range(chunks):
        tr = torch.empty((lanes, frames, LANE), dtype=torch.int16, device="cuda")
        H.tracegen(gen, lanes, frames, c * frames, state, c == 0, tr)
        if enc == "uint8":
            tr = (torch.div(tr, 2, rounding_mode="floor") + 64).clamp_(0, 255).to(torch.uint8)
        out.append(tr)
    H.sync()
    return out


def _config(frames, cadence, enc):
    if cadence == "chunk":
        cfg = H.bench_config(frames)
    else:
        cfg = H.default_config(sigma_ema_scale_strides=0.0)   # the reference's interval, a short start-up
    if enc == "uint8":
        cfg.movie.pedestal = 64
    return cfg


def _stats_leaves(stats, lanes):
    """The fields of a statistics record by type: moments and autocorrelation buffers, buffer
    indices, extrema, then the baseline and background moments."""
    b = stats.view(lanes, STATS_BYTES)
    return {"autocorr": b[:, :3328].view(torch.float32), "index": b[:, 3328:3456],
            "extrema": b[:, 3456:3712].view(torch.int16), "moments": b[:, 3712:].view(torch.float32)}


def _hist_leaves(hist, lanes):
    b = hist.view(lanes, HIST_BYTES)
    return {"bounds": b[:, :512].view(torch.float32), "counts": b[:, 512:].view(torch.int16)}


def _front(lanes, frames, seed):
    """Three chunks through the stages before an estimate: the last chunk's baselined traces, the
    histogram and statistics to estimate from, and the start-up models."""
    cfg = H.bench_config(frames)
    bl = H.Baseliner(cfg, lanes)
    stats, agg = _empty(lanes * STATS_BYTES), _empty(lanes * STATS_BYTES)
    hist, edge = _empty(lanes * HIST_BYTES), _empty(lanes * H.edge_state_bytes())
    models = _empty(lanes * MODEL_BYTES)
    base = torch.empty((lanes, frames, LANE), dtype=torch.int16, device="cuda")
    H.edge_state_init(edge, lanes)
    H.stats_reset(agg, lanes)
    for c, tr in enumerate(_traces(lanes, frames, 3, seed)):
        bl.run(tr, frames, base, stats)
        if c == 1:
            H.stats_merge(agg, stats, lanes)
            H.hist_reset(cfg, hist, agg, lanes)
            H.dme_init_models(cfg, agg, models, lanes)
            H.stats_reset(agg, lanes)
        elif c == 2:
            H.stats_merge(agg, stats, lanes)
            H.hist_add(hist, edge, base, frames, models, lanes)
    H.sync()
    return {"cfg": cfg, "base": base, "stats": stats, "agg": agg, "hist": hist, "edge": edge, "models": models}


_tuned = set()    # shapes tuned in this process (the library's table is process-wide)
_net = []         # the network, shared by the states of this process


def _network():
    """A network for the library, trained elsewhere (by torch, in 32 bits) on pairs of the plain pipeline with
    the training recipe's loss, output map and schedule."""
    if _net:
        return _net[0]
    pairs = Lr.generate_pairs(1024, 9, seed=101, snr=(4.0, 20.0), min_conf=0.0,
                              gen_overrides={"empty_fraction": 0.05})
    n = pairs.n
    x = _view(pairs.x.data_ptr(), (n, H.MLP_IN), "<i2", pairs).view(torch.bfloat16).float()
    t = _view(pairs.t.data_ptr(), (n, H.MLP_OUT), "<f4", pairs).clone()
    v = _view(pairs.v.data_ptr(), (n,), "|u1", pairs).float()
    t[v == 0, :11] = 0.0
    tv = t[v > 0][:, :6]
    offset, scale = tv.mean(0), tv.std(0).clamp(min=1e-3)
    w = torch.tensor(Lr.LL_WEIGHTS, device="cuda") * scale ** 2 / Lr.LL_FRAMES
    g = torch.Generator().manual_seed(1)
    params = []
    for n_out, n_in in ((256, 128), (256, 256), (12, 256)):
        params.append(((2.0 * torch.rand(n_out, n_in, generator=g) - 1.0) * (6.0 / n_in) ** 0.5).cuda())
        params.append(torch.zeros(n_out, device="cuda"))
    for p in params:
        p.requires_grad_()
    opt = torch.optim.Adam(params, lr=2e-3)
    batch, epochs = 4096, 10
    steps = epochs * (n // batch)
    for k in range(steps):
        for group in opt.param_groups:
            group["lr"] = 1e-4 + 1.9e-3 * 0.5 * (1.0 + float(np.cos(np.pi * k / steps)))
        at = (k % (n // batch)) * batch
        y = _forward(params, x[at:at + batch])
        opt.zero_grad()
        _loss(y, t[at:at + batch], v[at:at + batch], offset, scale, torch.cat([w, torch.ones(2, device="cuda")])).backward()
        opt.step()
    init = H.Initializer(seed=1)
    init.set_params(torch.cat([p.detach().reshape(-1) for p in params]).cpu().numpy())
    init.set_output_map(offset.tolist(), scale.tolist(), w.tolist() + [1.0, 1.0])
    _net.append(init)
    return init


def _forward(params, x):
    h = torch.relu(x @ params[0].t() + params[1])
    h = torch.relu(h @ params[2].t() + params[3])
    return h @ params[4].t() + params[5]


def _loss(y, t, valid, offset, scale, w):
    sq = (w[:6] * (y[:, :6] - (t[:, :6] - offset) / scale) ** 2).sum(1)
    ce = -w[6] * (t[:, 6:11] * torch.log_softmax(y[:, 6:11], 1)).sum(1)
    gate = w[7] * torch.nn.functional.binary_cross_entropy_with_logits(y[:, 11], t[:, 11], reduction="none")
    return ((sq + ce) * valid + gate).mean()


def _prepare_pool(case, seed):
    L, F, enc = case["lanes"], case["frames"], case["enc"]
    cfg = _config(F, case["cadence"], enc)
    if case["tuned"] and (L, F) not in _tuned:
        H.autotune(cfg, L, F, repeats=4)
        _tuned.add((L, F))
    an = H.BatchAnalyzer(0, L, F, cfg)
    pp, _, mc = an.pulses_device()
    pulses = _view(pp.data_ptr(), (L * LANE, mc, 5), "<i4", an)
    pulses.zero_()
    _result(an, H.lib.hwpa_result_metrics, (L, 137 * LANE), "|u1").zero_()
    chunks = _traces(L, F, 3, seed, enc)
    if case["input"] == "pinned":
        chunks = [c.cpu().pin_memory() for c in chunks]
    torch.cuda.synchronize()
    s = {"an": an, "chunks": chunks, "frame": 0, "k": 0, "dev": case["input"] == "device",
         "enc": T.ENCODING_UINT8 if enc == "uint8" else T.ENCODING_INT16}
    # Start-up of the baseline filter and the first estimates.
    warm = 4 if case["cadence"] == "chunk" else 2 + (1024 + 2 * 4000) // F
    for _ in range(warm):
        _chunk(s)
    s["out"] = _pool_leaves(an)
    torch.cuda.synchronize()
    return s


def _pool_leaves(an):
    L, F = an.lanes, an.frames
    pp, pc, mc = an.pulses_device()
    met = _result(an, H.lib.hwpa_result_metrics, (L, 137 * LANE), "|u1")
    return {"pulses": _view(pp.data_ptr(), (L * LANE, mc, 5), "<i4", an),
            "counts": _view(pc.data_ptr(), (L * LANE,), "<i4", an),
            "labels": _result(an, H.lib.hwpa_result_labels, (L, F, LANE), "<i2"),
            "baselined": _result(an, H.lib.hwpa_result_baselined, (L, F, LANE), "<i2"),
            "models": _result(an, H.lib.hwpa_result_models, (L, MODEL_BYTES // 2), "<f2"),
            "score": _result(an, H.lib.hwpa_result_viterbi_score, (L, LANE), "<f4"),
            "metric_counts": met[:, 64:960].view(torch.int16), "metric_signals": met[:, 960:5056].view(torch.float32)}


def _chunk(s):
    c = s["chunks"][s["k"] % len(s["chunks"])]
    s["an"](c, s["frame"], on_device=s["dev"], encoding=s["enc"])
    s["frame"] += s["an"].frames
    s["k"] += 1


def _batch_shapes(case):
    r = np.random.default_rng(case["shape_seed"])
    top = case["lanes"]
    lanes = [top] + [max(3, int(top * 2.0 ** -r.uniform(0.2, 4.0))) for _ in range(case["pools"] - 1)]
    return [(n, int(r.choice([256, 512, 1024]))) for n in lanes]


def _prepare_batch(case, seed):
    specs, chunks = [], []
    for i, (L, F) in enumerate(_batch_shapes(case)):
        specs.append((100 + i, L, F, H.bench_config(F, estimate_frames=512)))
        chunks.append(_traces(L, F, 2, seed + 17 * i))
    b = H.Batch(specs)
    for i in range(len(specs)):
        an = b.pool(i)
        pp, _, mc = an.pulses_device()
        _view(pp.data_ptr(), (an.lanes * LANE, mc, 5), "<i4", an).zero_()
        _result(an, H.lib.hwpa_result_metrics, (an.lanes, 137 * LANE), "|u1").zero_()
    torch.cuda.synchronize()
    s = {"b": b, "chunks": chunks, "frames": [p[2] for p in specs], "k": 0}
    for _ in range(12):
        _batch_step(s)
    out = {}
    for i in range(len(specs)):
        leaves = _pool_leaves(b.pool(i))
        out.update({"%s%d" % (n, i): leaves[n] for n in ("pulses", "counts", "labels", "models", "score")})
    s["out"] = out
    b.sync()
    return s


def _batch_step(s):
    k = s["k"]
    s["b"].process([c[k % len(c)] for c in s["chunks"]], [k * f for f in s["frames"]])
    s["k"] = k + 1


def _network_inputs(batch, seed):
    """Histogram-like network inputs, targets and validity flags, from the seed alone (CPU)."""
    g = torch.Generator().manual_seed(seed)

    def uni(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=g)

    bl, sd = uni(14.0, 26.0, batch, 1), uni(2.0, 3.0, batch, 1)
    snr = uni(4.0, 20.0, batch, 1)
    rel = torch.tensor([[1.0, 0.67, 0.44, 0.28]])
    mu = bl + snr * sd * rel
    w = torch.softmax(torch.randn(batch, 5, generator=g) * 0.3 + torch.tensor([2.5, 0.0, 0.0, 0.0, 0.0]), 1)
    x = torch.arange(128.0).view(1, 128)
    dens = w[:, :1] * torch.exp(-0.5 * ((x - bl) / sd) ** 2) / sd
    for a in range(4):
        s = torch.sqrt(sd ** 2 + (0.1 * (mu[:, a:a + 1] - bl)) ** 2 + 1.0)
        dens = dens + w[:, a + 1:a + 2] * torch.exp(-0.5 * ((x - mu[:, a:a + 1]) / s) ** 2) / s
    counts = torch.poisson(dens * 204.0, generator=g)
    feat = (16.0 * counts / counts.sum(1, keepdim=True).clamp(min=1.0)).to(torch.bfloat16)
    valid = torch.rand(batch, generator=g) < 0.9
    t = torch.cat([bl, 2.0 * torch.log(sd), mu, w, valid.float().view(-1, 1)], 1)
    params = []
    for n_out, n_in in ((256, 128), (256, 256), (12, 256)):
        params += [uni(-1.0, 1.0, n_out * n_in) * (6.0 / n_in) ** 0.5, torch.zeros(n_out)]
    offset = t[:, :6].mean(0)
    scale = t[:, :6].std(0)
    return feat, t, valid, torch.cat(params), offset, scale


NET_WEIGHTS = [1.0, 1.5, 0.2, 0.2, 0.2, 0.2, 1.0, 1.0]


def _pulse_records(zmws, max_calls, seed):
    """One chunk's pulse records [zmws, max_calls] (20 bytes each) and counts, as an analyzer leaves them."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    n = (zmws, max_calls)
    width = 1 + torch.floor(torch.log(rand(*n).clamp_(min=1e-6)) / np.log(1 - 1 / 8.0)).to(torch.int32)
    gap = 1 + torch.floor(torch.log(rand(*n).clamp_(min=1e-6)) / np.log(1 - 1 / 20.0)).to(torch.int32)
    start = 51200 + torch.cumsum(gap + width, 1, dtype=torch.int32) - width
    rec = torch.empty((*n, 5), dtype=torch.int32, device="cuda")
    mean = (rand(*n) * 2500 + 300).to(torch.int32)
    rec[..., 0] = start
    rec[..., 1] = width | (mean << 16)
    rec[..., 2] = (mean + 20) | ((mean + 300) << 16)
    rec[..., 3] = (rand(*n) * 4e5).view(torch.int32)
    label = (rand(*n) * 4).to(torch.int32)
    reject = (rand(*n) < 0.07).to(torch.int32)
    rec[..., 4] = label | (reject << 8)
    counts = (18 + 4.5 * torch.randn(zmws, generator=g, device="cuda")).round().clamp(0, max_calls).to(torch.int32)
    counts[rand(zmws) < 0.05] = 0
    rec *= (torch.arange(max_calls, device="cuda").view(1, -1) < counts.view(-1, 1)).to(torch.int32).unsqueeze(-1)
    return rec, counts


# ---- the cases ---------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pool":
        return dict(_prepare_pool(case, seed), kind=kind)
    if kind == "batch":
        return dict(_prepare_batch(case, seed), kind=kind)
    if kind == "train":
        feat, t, valid, params, offset, scale = _network_inputs(case["batch"], seed)
        init = H.Initializer(seed=1)
        init.set_params(params.numpy())
        init.set_output_map(offset.tolist(), scale.tolist(), NET_WEIGHTS)
        return {"kind": kind, "init": init, "batch": case["batch"], "x": feat.cuda(), "t": t.cuda(),
                "valid": valid.to(torch.uint8).cuda(), "grads": torch.empty(H.MLP_PARAMS, device="cuda"),
                "loss": torch.empty(1, device="cuda"), "step_loss": torch.empty(1, device="cuda")}
    L = case["lanes"]
    if kind == "baz":
        zmws = L * LANE
        rec, counts = _pulse_records(zmws, case["max_calls"], seed)
        enc = H.BazEncoder(zmws, internal=case["internal"])
        off, ev = torch.empty(zmws + 1, dtype=torch.int64, device="cuda"), torch.empty(zmws, dtype=torch.int32,
                                                                                     device="cuda")
        enc.encode(rec, counts, case["max_calls"], None, 0, off, ev)
        # The program's stream buffer has room for any chunk; what is past the stream stays zero.
        room = zmws * (320 if case["internal"] else 96)
        assert int(off[-1]) <= room
        return {"kind": kind, "enc": enc, "rec": rec, "counts": counts, "mc": case["max_calls"], "room": room,
                "off": off, "ev": ev, "data": _zeros(room)}
    F = case["frames"]
    if kind == "repack":
        u8 = case["enc"] == "uint8"
        g = torch.Generator(device="cuda").manual_seed(seed)
        dtype, bw = (torch.uint8, case["block_width"]) if u8 else (torch.int16, case["block_width"])
        zmws, per, nf = L * LANE, case["packet_blocks"] * bw, 128
        packets, keep = [], []
        for f0 in range(0, F, nf):
            for z0 in range(0, zmws, per):
                nb = -(-min(per, zmws - z0) // bw)
                d = torch.randint(0, 256, (nb * nf * bw * (1 if u8 else 2),), dtype=torch.uint8, device="cuda",
                                  generator=g)
                keep.append(d)
                packets.append((d, z0, f0, nb, nf, bw))
        return {"kind": kind, "r": H.Repacker(max_packets=len(packets)), "packets": packets, "L": L, "F": F,
                "enc": T.ENCODING_UINT8 if u8 else T.ENCODING_INT16,
                "out": torch.zeros((L, F, LANE), dtype=dtype, device="cuda")}
    if kind == "baseline":
        cfg = _config(F, "reference", case["enc"])
        cfg.filter_type = case["filter"]
        s = {"kind": kind, "bl": H.Baseliner(cfg, L), "L": L, "F": F, "k": 0, "chunks": _traces(L, F, 2, seed, case["enc"]),
             "enc": T.ENCODING_UINT8 if case["enc"] == "uint8" else T.ENCODING_INT16,
             "out": torch.empty((L, F, LANE), dtype=torch.int16, device="cuda"), "stats": _zeros(L * STATS_BYTES)}
        for _ in range(2):
            run(s)
        return s
    if kind == "call":
        cut = F
        F = 16 * -(-F // 16)
        f = _front(L, F, seed)
        cfg = f["cfg"]
        cfg.max_calls_per_zmw = case["max_calls"]
        H.dme_estimate(cfg, f["hist"], f["agg"], f["models"], (F, 2 * F), (2 * F, 3 * F), L)
        n = L * LANE
        s = {"kind": kind, "L": L, "F": cut, "base": f["base"][:, :cut].contiguous(), "models": f["models"], "frame": 0,
             "lab": H.Labeler(cfg, L, cut), "pul": H.Pulser(cfg, L),
             "labels": torch.empty((L, cut, LANE), dtype=torch.int16, device="cuda"),
             "latent": torch.empty((L, T.LATENT_FRAMES, LANE), dtype=torch.int16, device="cuda"),
             "score": torch.empty((L, LANE), device="cuda"),
             "pulses": torch.zeros((n, case["max_calls"], 5), dtype=torch.int32, device="cuda"),
             "counts": torch.zeros(n, dtype=torch.int32, device="cuda"),
             "ovf": torch.zeros(n, dtype=torch.int32, device="cuda"),
             "bl": torch.zeros((L, T.STAT_ACC.itemsize // 4), device="cuda")}
        run(s)
        return s
    f = _front(L, F, seed)
    f.update(kind=kind, L=L, F=F)
    if kind == "accumulate":
        f["chunks"] = case["chunks"]
        f["agg2"], f["hist2"] = _zeros(L * STATS_BYTES), _zeros(L * HIST_BYTES)
    else:
        f["start"] = f["models"].clone()
        f["iters"] = torch.zeros(L, dtype=torch.int32, device="cuda")
        if kind == "learned":
            f["cfg"].learned_init = 1
            f["net"] = _network()
    return f


def run(s):
    kind = s["kind"]
    if kind == "pool":
        _chunk(s)
        return s["out"]
    if kind == "batch":
        _batch_step(s)
        return s["out"]
    if kind == "train":
        s["init"].gradients(s["x"], s["t"], s["batch"], s["grads"], s["loss"], d_valid=s["valid"])
        s["init"].train_step(s["x"], s["t"], s["batch"], 1e-4, d_loss=s["step_loss"], d_valid=s["valid"])
        return {"grads": s["grads"], "loss": s["loss"], "step_loss": s["step_loss"]}
    if kind == "baz":
        s["enc"].reset()
        s["enc"].encode(s["rec"], s["counts"], s["mc"], s["data"], s["room"], s["off"], s["ev"])
        return {"data": s["data"], "offsets": s["off"], "events": s["ev"]}
    if kind == "repack":
        s["r"].run(s["packets"], s["enc"], s["out"], 0, 0, s["L"], s["F"])
        return s["out"]
    L, F = s["L"], s["F"]
    if kind == "baseline":
        s["bl"].run(s["chunks"][s["k"] % 2], F, s["out"], s["stats"], encoding=s["enc"])
        s["k"] += 1
        return {"out": s["out"], **_stats_leaves(s["stats"], L)}
    if kind == "call":
        s["lab"].run(s["base"], F, s["models"], s["labels"], s["latent"], s["score"])
        s["pul"].run(s["labels"], s["latent"], s["base"], F, s["frame"] - T.LATENT_FRAMES, s["models"], s["pulses"],
                     s["counts"], s["ovf"], s["bl"])
        s["frame"] += F
        return {n: s[n] for n in ("labels", "latent", "score", "pulses", "counts", "ovf", "bl")}
    if kind == "accumulate":
        H.stats_reset(s["agg2"], L)
        H.hist_reset(s["cfg"], s["hist2"], s["agg"], L)
        for _ in range(s["chunks"]):
            H.stats_merge(s["agg2"], s["stats"], L)
            H.hist_add(s["hist2"], s["edge"], s["base"], F, s["models"], L)
        return {**_stats_leaves(s["agg2"], L), **_hist_leaves(s["hist2"], L)}
    # An estimate updates the models it starts from: each pass starts from the same ones.
    s["models"].copy_(s["start"])
    span = ((F, 2 * F), (2 * F, 3 * F))
    out = {"models": s["models"].view(torch.float16)}
    if kind == "learned":
        out["fallback"] = H.dme_estimate_learned(s["cfg"], s["net"], s["hist"], s["agg"], s["models"], *span, L)
    else:
        H.dme_estimate(s["cfg"], s["hist"], s["agg"], s["models"], *span, L, s["iters"])
        out["iterations"] = s["iters"]
    return out


def work(case):
    kind = case["kind"]
    if kind == "batch":
        parts = [_pool_work(L, F, 2, 1.0 if F >= 512 else 0.5, 48) for L, F in _batch_shapes(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "train":
        # Forward and backward twice (gradients, then the step); inputs, targets, parameters and moments.
        return {"bytes": 2.0 * case["batch"] * (256 + 48 + 1) + 8.0 * H.MLP_PARAMS * 4,
                "flops": 2.0 * 3.0 * MLP_FLOPS_PER_ROW * case["batch"]}
    L = case["lanes"]
    Z = L * LANE
    if kind == "baz":
        # About 17 records of 20 bytes and 2.2 (internal: 8) bytes a record of stream, offsets and states per ZMW.
        return {"bytes": Z * (17.0 * 20 + 17.0 * (8.0 if case["internal"] else 2.2) + 28), "flops": Z * 17.0 * 10}
    F = case["frames"]
    ZF = float(Z) * F
    es = 1 if case.get("enc") == "uint8" else 2
    if kind == "pool":
        return _pool_work(L, F, es, 1.0 if case["cadence"] == "chunk" else min(1.0, F / 4000.0), 48)
    if kind == "repack":
        return {"bytes": 2.0 * ZF * es, "flops": 0.0}
    if kind == "baseline":
        return {"bytes": ZF * (es + 2) + L * (2.0 * FILTER_STATE_BYTES + STATS_BYTES), "flops": ZF * BASELINE_FLOPS}
    if kind == "accumulate":
        n = case["chunks"]
        return {"bytes": n * ZF * 2 + L * (1.0 * HIST_BYTES + MODEL_BYTES + 3.0 * STATS_BYTES), "flops": n * ZF * HIST_FLOPS}
    if kind == "call":
        return {"bytes": ZF * 4 + L * (MODEL_BYTES + 2.0 * 5500) + Z * (20.0 * F / 28 + 8),
                "flops": ZF * (LABEL_FLOPS + PULSE_FLOPS)}
    est = {"bytes": L * (1.0 * HIST_BYTES + STATS_BYTES + 2.0 * MODEL_BYTES), "flops": Z * EM_FLOPS_PER_ZMW}
    if kind == "learned":
        # Capped iterations for all, the full count for about a fifth.
        est["flops"] = Z * (EM_FLOPS_PER_ZMW * 0.45 + MLP_FLOPS_PER_ROW)
    return est


def _pool_work(L, F, es, estimates, max_calls):
    """One chunk through every stage: the samples in, labels, baselined traces and pulses out, the carried state
    of the filter, the statistics and the histogram."""
    ZF = float(L) * LANE * F
    return {"bytes": ZF * (es + 4) + L * LANE * min(max_calls, F / 28.0) * 20.0 +
            L * (2.0 * FILTER_STATE_BYTES + 2.0 * STATS_BYTES + 1.0 * HIST_BYTES),
            "flops": ZF * (BASELINE_FLOPS + HIST_FLOPS + LABEL_FLOPS + PULSE_FLOPS) +
            estimates * L * LANE * EM_FLOPS_PER_ZMW}


def exact(case, seed):
    """64-bit values of the network's gradients and loss.  The other kinds return whole numbers (samples, labels,
    counts, packets) and, beside them, sums and fits whose 64-bit values depend on those rounded samples or on
    which iteration a threshold stops at, so they have no value of their own."""
    if case["kind"] != "train":
        return None
    feat, t, valid, params, offset, scale = _network_inputs(case["batch"], seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, t, v = (a.to(dev).double() for a in (feat, t, valid))
    p = params.to(dev).double()
    sizes = [(256, 128), (256,), (256, 256), (256,), (12, 256), (12,)]
    parts, at = [], 0
    for shape in sizes:
        n = int(np.prod(shape))
        parts.append(p[at:at + n].view(shape).clone().requires_grad_())
        at += n
    w = torch.tensor(NET_WEIGHTS, dtype=torch.float64, device=dev)
    loss = _loss(_forward(parts, x), t, v, offset.to(dev).double(), scale.to(dev).double(), w)
    grads = torch.autograd.grad(loss, parts)
    one = loss.detach().view(1)
    return {"grads": torch.cat([g.reshape(-1) for g in grads]), "loss": one, "step_loss": one}
