"""Benchmark of the gfx950 attention path on BASELINE.json's configs.

python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload NAME] [--no-cpu]

A step is one attention call over resident synthetic inputs (seeded i.i.d.
N(0,1) f32, query pre-scaled by 1/sqrt(d) as the engine does). The JSON line's
value is the headline workload: single-token decode over a 32K-entry f32 KV
cache (BASELINE config 2 at full causal width), in algorithmic GB/s. The other
configs are measured in the same run and reported under "configs". The CPU
baseline is the oracle restatement of the reference's exact attention
(oracle/), threaded as the engine threads it, on a bounded sample.
"""
import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0        # MI355X HBM3E, GB/s
MIN_TIMED_MS = 5.0           # shortest timed region of a non-headline workload
MAX_STEPS = 1000
FP32_MFMA_PEAK_TFS = 157.3   # MI355X dense fp32 matrix, TFLOP/s
FP64_MFMA_PEAK_TFS = 78.6    # MI355X dense fp64 matrix, TFLOP/s


def load_package():
    import importlib.util
    name = "power_cpu_llm_amd"
    if name in sys.modules:
        return sys.modules[name]
    spec = importlib.util.spec_from_file_location(
        name, os.path.join(ROOT, "power-cpu-llm_amd", "__init__.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


# name: (qheads, kvheads, dim, nq, nkeys, causal, window, first_query, kind, unit-norm K)
WORKLOADS = {
    "decode_2k": (16, 8, 256, 1, 2048, True, 0, 2047, "decode", False),
    "decode_32k_window1024": (16, 8, 256, 1, 32768, True, 1024, 32767, "decode", False),
    # the sliding layer at a position that is not the last of a 256-key
    # chunk (255 positions of every 256): its 1024-key window starts and ends
    # inside chunks and covers five of them
    "decode_window1024_unaligned": (16, 8, 256, 1, 32668, True, 1024, 32667, "decode", False),
    "decode_32k": (16, 8, 256, 1, 32768, True, 0, 32767, "decode", False),
    "decode_128k_d512": (16, 2, 512, 1, 131072, True, 0, 131071, "decode", True),
    # the same global-layer decode (16/2/512, unit-norm K) at shorter caches
    "decode_2k_d512": (16, 2, 512, 1, 2048, True, 0, 2047, "decode", True),
    "decode_4k_d512": (16, 2, 512, 1, 4096, True, 0, 4095, "decode", True),
    "decode_8k_d512": (16, 2, 512, 1, 8192, True, 0, 8191, "decode", True),
    "decode_32k_d512": (16, 2, 512, 1, 32768, True, 0, 32767, "decode", True),
    # the reference's own attention throughput probe
    # (src/kernels/quantized/int8/tests.rs:770-809): 8 queries over every key
    # (no mask) of a sliding-layer and a global-layer geometry, device-resident
    # and through the AttentionMulti entry over host arrays (the engine's call)
    "probe_sliding_q8": (16, 8, 256, 8, 1279, False, 0, 0, "decode", False),
    "probe_global_q8": (16, 2, 512, 8, 3194, False, 0, 0, "decode", False),
    "probe_sliding_q8_host": (16, 8, 256, 8, 1279, False, 0, 0, "host", False),
    "probe_global_q8_host": (16, 2, 512, 8, 3194, False, 0, 0, "host", False),
    "prefill_4k_window1024": (16, 8, 256, 4096, 4096, True, 1024, 0, "prefill", False),
    "prefill_4k": (16, 8, 256, 4096, 4096, True, 0, 0, "prefill", False),
    "canvas_256x2304": (16, 8, 256, 256, 2304, False, 0, 2048, "canvas", False),
    # the global-layer geometry of Gemma-4 / DiffusionGemma (16 query heads,
    # 2 KV heads, head dim 512) through the same prefill and canvas paths
    "prefill_4k_d512": (16, 2, 512, 4096, 4096, True, 0, 0, "prefill", True),
    "canvas_256x2304_d512": (16, 2, 512, 256, 2304, False, 0, 2048, "canvas", True),
    # speculative verification (encode_speculative: the previous token and 7
    # drafts, causal over the cache and themselves)
    "verify_32k_q8": (16, 8, 256, 8, 32768, True, 0, 32760, "decode", False),
    # one decode step through the device-resident layer cache: append the
    # token's K/V row, attend over the 32K cache in place, roll back
    "decode_32k_cache": (16, 8, 256, 1, 32768, True, 0, 32767, "cache", False),
    # the head-transform prologue over a 4K-token prompt (norms and rotation
    # of 16 Q, 8 K and 8 V heads per token), and a whole decode step from raw
    # projections: transform, cache append and attention in one call (the
    # transform inside the pipelined decode's launch)
    "transform_4k": (16, 8, 256, 4096, 0, True, 0, 0, "transform", False),
    "decode_32k_step": (16, 8, 256, 1, 32768, True, 0, 32767, "step", False),
    # the same step for a sliding-window layer (window 1024 over a 32K
    # prompt: the spread decode)
    "decode_window_step": (16, 8, 256, 1, 32768, True, 1024, 32767, "step", False),
    # the whole attention layer of one decode token on the device: the step
    # above, then the output block on its attended row (LAYER_HIDDEN wide)
    "decode_32k_layer": (16, 8, 256, 1, 32768, True, 0, 32767, "layer", False),
    # the attention output block (projection of the 16 x 256 attended heads
    # to a 2816-wide hidden row, post-norm, residual) for one decode token and
    # for a 4K-token prompt; here `nkeys` is the hidden width
    "output_decode": (16, 8, 256, 1, 2816, False, 0, 0, "output", False),
    "output_4k": (16, 8, 256, 4096, 2816, False, 0, 0, "output", False),
    # the engine's own call of the 32K decode: the AttentionF32 entry over
    # pageable host arrays, so each call copies K and V over PCIe (the rate
    # that includes the copies, never the headline)
    "decode_32k_host": (16, 8, 256, 1, 32768, True, 0, 32767, "host", False),
    # the same call as the engine fans one position out over its workers
    # (src/engine/attention.rs:755-777): 16 concurrent calls of one query
    # head each, each copying only the KV head it reads
    "decode_32k_host_fanout": (16, 8, 256, 1, 32768, True, 0, 32767, "host", False),
}
HEADLINE = "decode_32k"
# host-array workloads timed in a default run (the others only when named)
DEFAULT_HOST = ("probe_sliding_q8_host", "probe_global_q8_host")
# BASELINE.json's configs (and the reference's probe shapes): each carries a
# CPU baseline beside its GPU figure
CPU_LEGS = ("decode_2k", "decode_32k_window1024", "decode_32k", "decode_128k_d512",
            "prefill_4k_window1024", "prefill_4k", "canvas_256x2304", "probe_sliding_q8",
            "probe_global_q8")
# rows of a prefill or canvas the CPU leg computes: every n-th query row
# (on all threads; on one thread)
ROW_SAMPLE = {"prefill_4k": (16, 128), "prefill_4k_window1024": (16, 128),
              "canvas_256x2304": (8, 64)}
# hidden width of the layer workload's output block (that of output_decode)
LAYER_HIDDEN = 2816
# the metric's second half: f32 prefill attention at 4K tokens (the global
# layer; the sliding-window layer is reported beside it)
PREFILL = ("prefill_4k", "prefill_4k_window1024")
PREFILL_SAMPLE_STEP = 16      # CPU baseline: every 16th query row of the prompt
PREFILL_SAMPLE_STEP_1CORE = 128


def traffic_bytes(name):
    """HBM bytes per launch of the workload's streaming kernel(s), from the
    committed rocprofv3 counter summary (profiles/hbm_traffic_counters.md: a
    line `traffic_bytes <workload> <bytes>`), or None when not measured."""
    path = os.path.join(ROOT, "profiles", "hbm_traffic_counters.md")
    if not os.path.exists(path):
        return None
    for line in open(path):
        f = line.split()
        if len(f) == 3 and f[0] == "traffic_bytes" and f[1] == name:
            return int(f[2])
    return None


def nq_of(name):
    return WORKLOADS[name][3]


def allowed_pairs(nq, nkeys, causal, window, first_query):
    """Allowed (query, key) pairs of one head (first_key = 0)."""
    if not causal:
        return nq * nkeys
    total = 0
    for i in range(nq):
        qp = first_query + i
        hi = min(qp, nkeys - 1)
        lo = max(0, qp - window + 1) if window else 0
        total += max(hi - lo + 1, 0)
    return total


def work(name):
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    if kind == "transform":
        # raw Q/K/V rows read, prepared rows written, (sin, cos) table rows read
        heads = qh + 2 * kvh
        return 0, nq * (2 * heads * dim * 4 + dim * 4), 0
    if kind == "output":
        # weights and attended rows read, residual read, result written
        width, hidden = qh * dim, nkeys
        return 2 * nq * width * hidden, 4 * (width * hidden + nq * width + 2 * nq * hidden), 0
    if kind == "layer":
        # the attention step, then the output block on its attended rows
        flops, bytes_, pairs = work_attention(qh, kvh, dim, nq, nkeys, causal, window, fq)
        width = qh * dim
        return (flops + 2 * nq * width * LAYER_HIDDEN,
                bytes_ + 4 * (width * LAYER_HIDDEN + nq * width + 2 * nq * LAYER_HIDDEN), pairs)
    return work_attention(qh, kvh, dim, nq, nkeys, causal, window, fq)


def work_attention(qh, kvh, dim, nq, nkeys, causal, window, fq):
    pairs = allowed_pairs(nq, nkeys, causal, window, fq)
    flops = 4 * dim * pairs * qh
    # decode bytes: attended K and V rows of every KV head, plus Q and O
    if causal:
        lo = max(0, fq - window + 1) if window else 0
        attended = min(fq + nq - 1, nkeys - 1) - lo + 1
    else:
        attended = nkeys
    bytes_ = 4 * (2 * attended * kvh * dim + 2 * nq * qh * dim)
    return flops, bytes_, pairs


def make_inputs(torch, name, seed):
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, unit = WORKLOADS[name]
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(0x5EED0000 + seed)
    q = torch.randn((nq, qh, dim), generator=gen, device=dev, dtype=torch.float32)
    k = torch.randn((nkeys, kvh, dim), generator=gen, device=dev, dtype=torch.float32)
    v = torch.randn((nkeys, kvh, dim), generator=gen, device=dev, dtype=torch.float32)
    if unit:
        k = k / k.norm(dim=-1, keepdim=True)
    scale = np.float32(1.0 / math.sqrt(dim))
    q = q * float(scale)  # the engine's f32 pre-scale of the query
    return q.contiguous(), k.contiguous(), v.contiguous()


def desc_for(ctx, name, q, k, v, out, k_canvas=None, v_canvas=None, kernel=0):
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    kw = dict(q=q.data_ptr(), q_stride=qh * dim, nq=nq, qheads=qh, kvheads=kvh, dim=dim,
              kh_first=0, kh_end=kvh, causal=int(causal), window=window, first_key=0,
              first_query=fq, out=out.data_ptr(), o_stride=qh * dim, kernel=kernel)
    if k_canvas is not None:
        n0 = nkeys - nq
        kw.update(k0=k.data_ptr(), v0=v.data_ptr(), n0=n0, k1=k_canvas.data_ptr(),
                  v1=v_canvas.data_ptr(), n1=nq)
    else:
        kw.update(k0=k.data_ptr(), v0=v.data_ptr(), n0=nkeys)
    return ctx.desc(**kw)


# Layer caches and head transforms of finished workloads, kept until the
# process ends: destroying them would free device memory mid-run, after which
# every later workload in the process streams more slowly (see main()).
RETAINED = []

# Each timed launch reads a different input set, and one cycle through the sets
# touches at least this many bytes: more than twice the MI355X's 256 MB
# last-level cache, so no launch finds its K/V there (a model's layers each
# have their own cache; re-reading one small set would measure the cache).
CYCLE_BYTES = 2 << 30
MAX_SETS = 64


def time_workload(torch, pcl, ctx, name, steps, warmup, seed=0, kernel=0):
    """Per-launch time (ms) from HIP events on the launch stream, and the
    per-kernel-role times from the library's own event spans."""
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    set_bytes = 4 * (2 * nkeys * kvh * dim + 2 * nq * qh * dim)
    nsets = max(2, min(MAX_SETS, -(-CYCLE_BYTES // set_bytes)))
    if kind == "cache":
        return time_cache_workload(torch, pcl, ctx, name, steps, warmup, nsets, seed)
    if kind in ("step", "layer"):
        return time_cache_workload(torch, pcl, ctx, name, steps, warmup, nsets, seed,
                                   transform=True, output=(kind == "layer"))
    if kind == "transform":
        return time_transform_workload(torch, pcl, ctx, name, steps, warmup, seed)
    if kind == "output":
        return time_output_workload(torch, pcl, ctx, name, steps, warmup, seed)
    if kind == "host":
        return time_host_workload(torch, pcl, name, steps, warmup, seed)
    sets = []
    for i in range(nsets):
        q, k, v = make_inputs(torch, name, seed + 1000 * i)
        out = torch.empty((nq, qh, dim), device="cuda:0", dtype=torch.float32)
        kc = vc = None
        if kind == "canvas":
            # canvas K/V live apart from the fixed prompt prefix (two segments)
            kc, vc = k[nkeys - nq:].clone(), v[nkeys - nq:].clone()
            k, v = k[:nkeys - nq].contiguous(), v[:nkeys - nq].contiguous()
        d = desc_for(ctx, name, q, k, v, out, kc, vc, kernel)
        sets.append(({"q": q, "k": k, "v": v, "out": out, "kc": kc, "vc": vc}, d))
    d0 = sets[0][1]
    ctx.reserve(ctx.workspace_bytes(d0))
    kernel = pcl.KERNEL_NAMES.get(ctx.resolve_kernel(d0), "?")
    for i in range(max(warmup, nsets)):
        ctx.launch(sets[i % nsets][1])
    torch.cuda.synchronize()
    if ctx.sync() != 0:
        raise RuntimeError("device error flag set for %s" % name)
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for i in range(steps):
        ctx.launch(sets[i % nsets][1])
    stop.record()
    torch.cuda.synchronize()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    ev = start.elapsed_time(stop) / steps
    err = ctx.sync()
    if err:
        raise RuntimeError("device error flag %d for %s" % (err, name))
    # the same launches again with the library's per-kernel event spans
    ctx.set_timing(True)
    for i in range(steps):
        ctx.launch(sets[i % nsets][1])
    (ms_stream, ms_comb), (n_stream, n_comb) = ctx.timing()
    ctx.set_timing(False)
    roles = {"stream_ms": ms_stream / max(n_stream, 1),
             "combine_ms": ms_comb / n_comb if n_comb else 0.0}
    host = sets[(steps - 1) % nsets][0]
    return ev, wall, kernel, host, roles, nsets


def time_host_workload(torch, pcl, name, steps, warmup, seed):
    """Wall time (ms) of pcl_hip_attention_f32_heads, the entry the engine
    binds as its AttentionF32 pointer, over pageable host arrays: the copies of
    Q, K and V to the device, the attention and the copy of the output back."""
    import ctypes
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    q, k, v = make_inputs(torch, name, seed)
    hq, hk, hv = (np.ascontiguousarray(x.cpu().numpy().reshape(-1)) for x in (q, k, v))
    del q, k, v
    out = np.empty(nq * qh * dim, np.float32)
    lib = pcl.load()
    fptr = ctypes.POINTER(ctypes.c_float)

    fanout = name.endswith("_fanout")

    def one(h0, h1):
        # all keys allowed: the decode position is the last key (no mask)
        if nq > 1:
            # AttentionMulti over every KV head (the probe's attention_multi)
            if not lib.pcl_hip_attention_f32_multi_kv(
                    hq.ctypes.data_as(fptr), nq, qh * dim, hk.ctypes.data_as(fptr),
                    hv.ctypes.data_as(fptr), qh, kvh, dim, nkeys, None, nkeys, None,
                    out.ctypes.data_as(fptr), qh * dim, 0, kvh):
                raise RuntimeError("pcl_hip_attention_f32_multi_kv failed for %s" % name)
        elif not lib.pcl_hip_attention_f32_heads(
                hq.ctypes.data_as(fptr), hk.ctypes.data_as(fptr), hv.ctypes.data_as(fptr),
                qh, kvh, dim, nkeys, None, None,
                out[h0 * dim:].ctypes.data_as(fptr), h0, h1):
            raise RuntimeError("pcl_hip_attention_f32_heads failed for %s" % name)

    if fanout:
        import concurrent.futures
        pool = concurrent.futures.ThreadPoolExecutor(qh)

        def call():
            list(pool.map(lambda h: one(h, h + 1), range(qh)))
    else:
        def call():
            one(0, qh)

    for _ in range(max(warmup, 1)):
        call()
    t0 = time.perf_counter()
    for _ in range(steps):
        call()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    if fanout:
        pool.shutdown()
    roles = {"stream_ms": 0.0, "combine_ms": 0.0}
    return wall, wall, "host+auto", {"q": torch.from_numpy(hq)}, roles, 1


def make_transform(torch, pcl, ctx, qh, kvh, dim):
    g = torch.Generator()
    g.manual_seed(0x5EED0600)
    qs = (1 + 0.1 * torch.randn(dim, generator=g)).numpy()
    ks = (1 + 0.1 * torch.randn(dim, generator=g)).numpy()
    return pcl.HeadTransform(ctx, qh, kvh, dim, qs, ks, 1e-6, 10000.0)


def time_transform_workload(torch, pcl, ctx, name, steps, warmup, seed):
    """The head transform of nq tokens at positions 0.. (raw rows seeded
    N(0,1)); HIP events around the launches."""
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    t = make_transform(torch, pcl, ctx, qh, kvh, dim)
    set_bytes = 8 * nq * (qh + 2 * kvh) * dim
    nsets = max(2, min(MAX_SETS, -(-CYCLE_BYTES // set_bytes)))
    sets = []
    dev = torch.device("cuda:0")
    for i in range(nsets):
        gen = torch.Generator(device=dev)
        gen.manual_seed(0x5EED0700 + seed + i)
        raw = [torch.randn((nq, h * dim), generator=gen, device=dev) for h in (qh, kvh, kvh)]
        outs = [torch.empty_like(x) for x in raw]
        sets.append((raw, outs))

    def step(i):
        raw, outs = sets[i % nsets]
        t.prepare(raw[0].data_ptr(), raw[1].data_ptr(), raw[2].data_ptr(), nq, 0,
                  outs[0].data_ptr(), outs[1].data_ptr(), outs[2].data_ptr())

    for i in range(max(warmup, nsets)):
        step(i)
    torch.cuda.synchronize()
    if ctx.sync():
        raise RuntimeError("device error flag set for %s" % name)
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for i in range(steps):
        step(i)
    stop.record()
    torch.cuda.synchronize()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    ev = start.elapsed_time(stop) / steps
    if ctx.sync():
        raise RuntimeError("device error flag set for %s" % name)
    RETAINED.append(t)
    roles = {"stream_ms": ev, "combine_ms": 0.0}
    return ev, wall, "head_transform", None, roles, nsets


def time_output_workload(torch, pcl, ctx, name, steps, warmup, seed):
    """The output block of nq tokens (weights [hidden][qheads*dim], seeded
    N(0, 1/width)); each timed call reads its own weight and input set."""
    qh, kvh, dim, nq, hidden, causal, window, fq, kind, _ = WORKLOADS[name]
    width = qh * dim
    set_bytes = 4 * (width * hidden + nq * width + 3 * nq * hidden)
    nsets = max(2, min(MAX_SETS, -(-CYCLE_BYTES // set_bytes)))
    dev = torch.device("cuda:0")
    sets = []
    for i in range(nsets):
        gen = torch.Generator(device=dev)
        gen.manual_seed(0x5EED0800 + seed + i)
        w = torch.randn((hidden, width), generator=gen, device=dev) * (1.0 / math.sqrt(width))
        x = torch.randn((nq, width), generator=gen, device=dev)
        res = torch.randn((nq, hidden), generator=gen, device=dev)
        scale = 1 + 0.1 * torch.randn(hidden, generator=gen, device=dev)
        proj = torch.empty((nq, hidden), device=dev)
        out = torch.empty((nq, hidden), device=dev)
        sets.append((w, x, res, scale, proj, out))

    def step(i):
        w, x, res, scale, proj, out = sets[i % nsets]
        ctx.attention_output(x.data_ptr(), nq, width, w.data_ptr(), hidden, scale.data_ptr(),
                             1e-6, res.data_ptr(), proj.data_ptr(), out.data_ptr())

    for i in range(max(warmup, nsets)):
        step(i)
    torch.cuda.synchronize()
    if ctx.sync():
        raise RuntimeError("device error flag set for %s" % name)
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for i in range(steps):
        step(i)
    stop.record()
    torch.cuda.synchronize()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    ev = start.elapsed_time(stop) / steps
    if ctx.sync():
        raise RuntimeError("device error flag set for %s" % name)
    if nq == 1 and width % 4 == 0 and width <= 16384:
        kernel = "project_row_lds"
    else:
        kernel = ("project_rows" if nq <= 5 else "project_few" if nq <= 32 else
                  "project_tiles")
    return ev, wall, kernel, None, {"stream_ms": ev, "combine_ms": 0.0}, nsets


def time_cache_workload(torch, pcl, ctx, name, steps, warmup, nsets, seed, transform=False,
                        output=False):
    """Decode steps through pcl.LayerCache: per step, append one token's K/V
    after nkeys-1 cached rows (as device rows, or with transform=True from the
    token's raw Q/K/V projections through the head transform, in one
    pcl_kv_cache_attend_token call that folds the transform into the
    pipelined decode's launch), attend over the cache's rows in place (its
    encoder descriptor),
    with output=True run the output block (LAYER_HIDDEN-wide projection,
    post-norm, residual) on the attended row, and roll the step back. Each
    input set is its own cache and output weights."""
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    t = make_transform(torch, pcl, ctx, qh, kvh, dim) if transform else None
    width = qh * dim
    dev = torch.device("cuda:0")
    sets = []
    for i in range(nsets):
        q, k, v = make_inputs(torch, name, seed + 1000 * i)
        cache = pcl.LayerCache(ctx, kvh, dim, nkeys + 1, window, 1 << 40)
        cache.reserve_rows(nkeys + 1)  # no growth (and no free) on the appends
        cache.append(k.data_ptr(), v.data_ptr(), nkeys - 1)
        cache.commit()
        out = torch.empty((nq, qh, dim), device="cuda:0", dtype=torch.float32)
        kt, vt = k[nkeys - 1:].clone(), v[nkeys - 1:].clone()
        host = {"q": q, "k": k, "v": v, "out": out, "kt": kt, "vt": vt}
        if transform:
            host["raw_q"] = q.clone()
            host["q_prepared"] = torch.empty_like(q)
        if output:
            gen = torch.Generator(device=dev)
            gen.manual_seed(0x5EED0900 + seed + i)
            host["w"] = torch.randn((LAYER_HIDDEN, width), generator=gen,
                                    device=dev) * (1.0 / math.sqrt(width))
            host["res"] = torch.randn((nq, LAYER_HIDDEN), generator=gen, device=dev)
            host["post"] = 1 + 0.1 * torch.randn(LAYER_HIDDEN, generator=gen, device=dev)
            host["proj"] = torch.empty((nq, LAYER_HIDDEN), device=dev)
            host["result"] = torch.empty((nq, LAYER_HIDDEN), device=dev)
        sets.append((host, cache))
    torch.cuda.synchronize()

    def step(i):
        host, cache = sets[i % nsets]
        if transform:
            # the token's transform, cache append and attention in one call
            # (the transform folded into the decode's launch where it can be)
            pending = cache.attend_token(t, host["raw_q"].data_ptr(), host["kt"].data_ptr(),
                                         host["vt"].data_ptr(), host["q_prepared"].data_ptr(),
                                         host["out"].data_ptr())
            d = cache.encoder_desc(pending, q=host["q_prepared"].data_ptr(), q_stride=qh * dim,
                                   nq=nq, qheads=qh, kh_first=0, kh_end=kvh,
                                   out=host["out"].data_ptr(), o_stride=qh * dim)
        else:
            pending = cache.append(host["kt"].data_ptr(), host["vt"].data_ptr(), 1)
            d = cache.encoder_desc(pending, q=host["q"].data_ptr(), q_stride=qh * dim, nq=nq,
                                   qheads=qh, kh_first=0, kh_end=kvh,
                                   out=host["out"].data_ptr(), o_stride=qh * dim)
            ctx.launch(d)
        if output:
            ctx.attention_output(host["out"].data_ptr(), nq, width, host["w"].data_ptr(),
                                 LAYER_HIDDEN, host["post"].data_ptr(), 1e-6,
                                 host["res"].data_ptr(), host["proj"].data_ptr(),
                                 host["result"].data_ptr())
        cache.rollback(pending)
        return d

    d0 = step(0)
    ctx.reserve(ctx.workspace_bytes(d0))
    kernel = pcl.KERNEL_NAMES.get(ctx.resolve_kernel(d0), "?")
    for i in range(max(warmup, nsets)):
        step(i)
    torch.cuda.synchronize()
    if ctx.sync() != 0:
        raise RuntimeError("device error flag set for %s" % name)
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for i in range(steps):
        step(i)
    stop.record()
    torch.cuda.synchronize()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    ev = start.elapsed_time(stop) / steps
    if ctx.sync():
        raise RuntimeError("device error flag set for %s" % name)
    ctx.set_timing(True)
    for i in range(steps):
        step(i)
    (ms_stream, ms_comb), (n_stream, n_comb) = ctx.timing()
    ctx.set_timing(False)
    roles = {"stream_ms": ms_stream / max(n_stream, 1),
             "combine_ms": ms_comb / n_comb if n_comb else 0.0}
    host = sets[(steps - 1) % nsets][0]
    RETAINED.append((sets, t))
    return ev, wall, kernel, host, roles, nsets


def host_inputs(name, host):
    """Q, K, V of a timed input set as flat host arrays (a canvas's two K/V
    segments joined in key order)."""
    q = host["q"].cpu().numpy().reshape(-1)
    k, v = host["k"].cpu().numpy(), host["v"].cpu().numpy()
    if host.get("kc") is not None:
        k = np.concatenate([k, host["kc"].cpu().numpy()])
        v = np.concatenate([v, host["vc"].cpu().numpy()])
    return q, k.reshape(-1), v.reshape(-1)


def reference_gmacs(name, sec):
    """The reference probe's own rate (int8/tests.rs:800-806): 2 nq qheads
    nkeys dim multiply-adds (scores and P.V) per call."""
    qh, kvh, dim, nq, nkeys = WORKLOADS[name][:5]
    return 2.0 * nq * qh * nkeys * dim / sec / 1e9


def cpu_baseline(name, host, threads, budget_s=20.0):
    """The oracle's exact path (port of p9_ref_attention_heads), engine
    threading, timed on a bounded sample: whole calls of the workload,
    repeated (median); the same on one core and the binary32 twin (port of
    pa_attention_f32_heads, the portable-int8 backends' path)."""
    from oracle import binding as orc
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    q, k, v = host_inputs(name, host)

    def timed(nthreads, reps, budget, binary32=False):
        times, out = [], None
        t_end = time.perf_counter() + budget
        while len(times) < 1 or (time.perf_counter() < t_end and len(times) < reps):
            t0 = time.perf_counter()
            ok, out = orc.threaded(q, nq, k, v, qh, kvh, dim, nkeys, causal, 0, fq, window,
                                   threads=nthreads, binary32=binary32)
            times.append(time.perf_counter() - t0)
            if not ok:
                raise RuntimeError("oracle error")
        return float(np.median(times)), len(times), out

    med, runs, out = timed(threads, 50, budget_s)
    gpu = host["out"].cpu().numpy().reshape(-1)
    maxerr = float(np.max(np.abs(gpu - out)))
    med1, runs1, _ = timed(1, 5, budget_s / 2)
    med32, runs32, _ = timed(threads, 5, budget_s / 4, binary32=True)
    _, bytes_, _ = work(name)
    cpu = {"value": bytes_ / med / 1e9, "unit": "GB/s", "cores": threads, "kind": "port",
           "sample": "%d whole %s calls (exact f64 path, engine head split), median %.4f s"
                     % (runs, name, med),
           "value_1core": bytes_ / med1 / 1e9,
           "sample_1core": "%d whole calls on one thread, median %.4f s" % (runs1, med1),
           "value_binary32": bytes_ / med32 / 1e9,
           "sample_binary32": "%d whole calls of the binary32 twin (pa_attention_f32 path), "
                              "%d threads, median %.4f s" % (runs32, threads, med32),
           "gpu_vs_oracle_maxabs": maxerr}
    if nq > 1:
        cpu["GMAC/s"] = reference_gmacs(name, med)
        cpu["GMAC/s_1core"] = reference_gmacs(name, med1)
        cpu["GMAC/s_binary32"] = reference_gmacs(name, med32)
    return cpu


def cpu_baseline_rows(name, host, threads, budget_s=20.0):
    """The oracle's exact path over a prefill or canvas, as the engine runs
    one (contiguous query ranges per worker, each query its own call with
    its own mask), on a sample: every n-th query row (ROW_SAMPLE), timed
    whole and repeated; rates count the sampled rows' own algorithmic
    flops."""
    from oracle import binding as orc
    qh, kvh, dim, nq, nkeys, causal, window, fq, kind, _ = WORKLOADS[name]
    q, k, v = host_inputs(name, host)
    q = q.reshape(nq, qh * dim)
    gpu = host["out"].cpu().numpy().reshape(nq, qh * dim)
    step, step1 = ROW_SAMPLE[name]

    def sample_flops(stride):
        pairs = 0
        for i in range(0, nq, stride):
            pairs += allowed_pairs(1, nkeys, causal, window, fq + i)
        return 4 * dim * qh * pairs

    def run(stride, nthreads, reps):
        rows = np.ascontiguousarray(q[::stride])
        times, out = [], None
        t_end = time.perf_counter() + budget_s
        while len(times) < reps or (time.perf_counter() < t_end and len(times) < 2 * reps):
            t0 = time.perf_counter()
            ok, out = orc.threaded(rows.reshape(-1), rows.shape[0], k, v, qh, kvh, dim, nkeys,
                                   causal, 0, fq, window, threads=nthreads, query_step=stride)
            times.append(time.perf_counter() - t0)
            if not ok:
                raise RuntimeError("oracle error")
            if time.perf_counter() > t_end and len(times) >= reps:
                break
        return float(np.median(times)), len(times), out.reshape(rows.shape[0], -1)

    med, runs, out = run(step, threads, 3)
    maxerr = float(np.max(np.abs(gpu[::step] - out)))
    med1, _, _ = run(step1, 1, 3)
    if causal:
        masks = "their own causal%s masks" % (" + window %d" % window if window else "")
    else:
        masks = "every key, no mask"
    return {"value": sample_flops(step) / med / 1e12, "unit": "TFLOP/s",
            "cores": threads, "kind": "port",
            "sample": "every %dth query row of the %d queries (%d rows, all heads, %s), exact "
                      "f64 path, %d whole runs, median %.3f s"
                      % (step, nq, len(range(0, nq, step)), masks, runs, med),
            "value_1core": sample_flops(step1) / med1 / 1e12,
            "sample_1core": "every %dth query row on one thread, median %.3f s" % (step1, med1),
            "gpu_vs_oracle_maxabs": maxerr}


def cpu_leg(name, host, threads, budget_s):
    """The CPU baseline of one workload (whole decode calls, or sampled
    prefill/canvas rows), with the host's core counts and model."""
    kind = WORKLOADS[name][8]
    if kind in ("prefill", "canvas"):
        cpu = cpu_baseline_rows(name, host, threads, budget_s)
    else:
        cpu = cpu_baseline(name, host, threads, budget_s)
    cpu["affinity_cores"] = len(os.sched_getaffinity(0))
    cpu["cpu"] = cpu_model()
    return cpu


def cpu_share():
    """Host threads for the CPU baseline and the affinity mask's core count.
    The box grants this process a share of its cores (OMP_NUM_THREADS, 16 on
    the GPU box) that can be smaller than the affinity mask; the baseline
    uses the share and reports both."""
    affinity = len(os.sched_getaffinity(0))
    try:
        share = int(os.environ.get("OMP_NUM_THREADS", "0"))
    except ValueError:
        share = 0
    threads = min(share, affinity) if share > 0 else affinity
    return max(threads, 1), affinity


def roofline(name, r):
    """Roofline block of a workload's dominant kernel: the launches that
    stream K/V (the ordered combine excluded), timed by the library's event
    spans over the timed steps."""
    kind = WORKLOADS[name][8]
    stream_s = r["stream_kernel_ms"] * 1e-3
    if kind == "layer":
        # the layer's bytes span several kernels (the output block has no
        # timing span): the whole step is the timed unit
        stream_s = r["ms"] * 1e-3
    if kind == "output" and nq_of(name) > 32:
        ach = r["algorithmic_flops"] / stream_s / 1e12
        roof = {"bound": "mfma", "achieved": ach, "peak": FP64_MFMA_PEAK_TFS,
                "unit": "TFLOP/s", "frac": ach / FP64_MFMA_PEAK_TFS,
                "traffic": traffic_bytes(name)}
    elif kind in ("decode", "cache", "step", "layer", "transform", "output"):
        ach = r["algorithmic_bytes"] / stream_s / 1e9
        roof = {"bound": "hbm", "achieved": ach, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": ach / HBM_PEAK_GBS, "traffic": traffic_bytes(name)}
    else:
        ach = r["algorithmic_flops"] / stream_s / 1e12
        roof = {"bound": "mfma", "achieved": ach, "peak": FP32_MFMA_PEAK_TFS,
                "unit": "TFLOP/s", "frac": ach / FP32_MFMA_PEAK_TFS,
                "traffic": traffic_bytes(name)}
    roof["kernel"] = r["kernel"]
    return roof


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default=None, help="time only this workload")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--kernel", type=int, default=0,
                    help="pcl_kernel choice for every workload (0 = the library's choice)")
    ap.add_argument("--cpu-budget", type=float, default=20.0)
    ap.add_argument("--copy-calibration", action="store_true",
                    help="first run a plain 256 MiB device copy (the reference point for "
                         "HBM byte counters under rocprofv3 --pmc)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the attention path runs on a single MI355X here "
              "(multi-GPU sharding is a design note, not a measured path).", file=sys.stderr)
        sys.exit(2)

    import torch
    pcl = load_package()
    pcl.load()
    ctx = pcl.Context(0, torch.cuda.current_stream().cuda_stream)
    if args.copy_calibration:
        # a plain elementwise copy kernel of known size: reads and writes 256 MiB
        src = torch.ones(64 << 20, device="cuda:0", dtype=torch.float32)
        dst = torch.empty_like(src)
        for _ in range(3):
            torch.mul(src, 1.0, out=dst)
        torch.cuda.synchronize()
        del src, dst

    # the host-copy workload runs only when named (its copies would crowd the
    # device-resident figures and their kernel traces). The headline runs
    # first, and no workload returns device memory to the driver (torch keeps
    # freed tensors in its cache): after a process frees device memory, every
    # later decode in it streams ~5 % slower, even over buffers allocated
    # before the free (87.1 -> 91.2 us per 32K step on the same 2 GiB of input
    # sets), which is the harness's doing, not the kernel's.
    names = ([args.workload] if args.workload
             else [HEADLINE] + [n for n in WORKLOADS
                                if n != HEADLINE and WORKLOADS[n][8] != "host"] +
             list(DEFAULT_HOST))
    results = {}
    hosts = {}
    for name in names:
        steps = args.steps if name == HEADLINE else max(5, args.steps // 5)
        ev, wall, kernel, host, roles, nsets = time_workload(torch, pcl, ctx, name, steps,
                                                             args.warmup, kernel=args.kernel)
        if name != HEADLINE and ev * steps < MIN_TIMED_MS and WORKLOADS[name][8] != "host":
            # a short timed region is dominated by launch jitter: time again
            # over at least MIN_TIMED_MS (the headline keeps --steps exactly)
            del host
            steps = min(MAX_STEPS, int(math.ceil(MIN_TIMED_MS / max(ev, 1e-3))))
            ev, wall, kernel, host, roles, nsets = time_workload(
                torch, pcl, ctx, name, steps, args.warmup, kernel=args.kernel)
        flops, bytes_, pairs = work(name)
        kind = WORKLOADS[name][8]
        r = {"ms": ev, "wall_ms": wall, "kernel": kernel, "steps": steps, "input_sets": nsets,
             "stream_kernel_ms": roles["stream_ms"], "combine_ms": roles["combine_ms"],
             "algorithmic_bytes": bytes_, "algorithmic_flops": flops}
        r["GB/s"] = bytes_ / (ev * 1e-3) / 1e9
        r["TFLOP/s"] = flops / (ev * 1e-3) / 1e12
        if kind == "output" and nq_of(name) > 32:
            r["frac_mfma_fp64"] = r["TFLOP/s"] / FP64_MFMA_PEAK_TFS
        elif kind == "host":
            r["pcie_inclusive_GB/s"] = r["GB/s"]
        elif kind in ("decode", "cache", "step", "layer", "transform", "output"):
            r["frac_hbm"] = r["GB/s"] / HBM_PEAK_GBS
        else:
            r["frac_mfma"] = r["TFLOP/s"] / FP32_MFMA_PEAK_TFS
        if nq_of(name) > 1 and name.startswith("probe_"):
            r["GMAC/s"] = reference_gmacs(name, ev * 1e-3)
        results[name] = r
        if name in CPU_LEGS or name == args.workload:
            hosts[name] = host
        else:
            del host
        print("# %s: %.4f ms (%s; stream %.4f + combine %.4f ms) %.1f GB/s %.2f TFLOP/s"
              % (name, ev, kernel, roles["stream_ms"], roles["combine_ms"], r["GB/s"],
                 r["TFLOP/s"]), file=sys.stderr)

    head = args.workload or HEADLINE
    hr = results[head]
    kind = WORKLOADS[head][8]
    threads, affinity = cpu_share()
    # the CPU baseline beside each BASELINE config (the headline's with the
    # full budget, the others with a shorter one), after every GPU timing
    if not args.no_cpu:
        for name in results:
            if name not in hosts or hosts[name] is None:
                continue
            if name not in CPU_LEGS and name != args.workload:
                continue
            if WORKLOADS[name][8] not in ("decode", "prefill", "canvas"):
                continue
            budget = args.cpu_budget if name == head else min(args.cpu_budget, 8.0)
            results[name]["cpu_baseline"] = cpu_leg(name, hosts[name], threads, budget)
            print("# cpu %s: %s" % (name, results[name]["cpu_baseline"]["sample"]),
                  file=sys.stderr)
    cpu = results[head].get("cpu_baseline")
    qh, kvh, dim, nq, nkeys, causal, window, fq, _, _ = WORKLOADS[head]
    if kind == "host":
        # host buffers: the copies dominate; no kernel roofline applies
        value, unit = hr["GB/s"], "GB/s"
        metric = "decode-attn GB/s at 32K KV incl. host copies"
        roof = {"bound": "pcie", "achieved": value, "peak": None, "unit": "GB/s",
                "frac": None, "traffic": None}
        roof["kernel"] = hr["kernel"]
    elif kind in ("decode", "cache", "step", "layer", "transform") or (kind == "output" and nq <= 32):
        value, unit, metric = hr["GB/s"], "GB/s", "decode-attn HBM GB/s at 32K KV"
        roof = roofline(head, hr)
    else:
        value, unit, metric = hr["TFLOP/s"], "TFLOP/s", "prefill attn TFLOP/s"
        roof = roofline(head, hr)
    # the metric's prefill half: each 4K prefill with its own roofline, and the
    # CPU baseline of the global one on a sample of its rows
    prefill = {}
    for name in PREFILL:
        if name not in results:
            continue
        r = results[name]
        block = {"metric": "prefill attn TFLOP/s (% fp32 MFMA peak) at 4K tokens",
                 "value": r["TFLOP/s"], "unit": "TFLOP/s", "ms_per_step": r["ms"],
                 "steps": r["steps"], "roofline": roofline(name, r), "cpu_baseline": None}
        block["cpu_baseline"] = r.get("cpu_baseline")
        prefill[name] = block
    line = {
        "metric": metric, "value": value, "unit": unit, "n_gpus": 1, "steps": hr["steps"],
        "warmup": args.warmup, "ms_per_step": hr["ms"], "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": head, "query_heads": qh, "kv_heads": kvh, "head_dim": dim,
                   "queries": nq, "kv_entries": nkeys, "causal": causal, "window": window,
                   "q_prescale": "1/sqrt(head_dim)", "kernel": hr["kernel"]},
        "roofline": roof,
        "cpu_baseline": cpu,
        "prefill": prefill or None,
        "configs": {n: {k: (round(x, 5) if isinstance(x, float) else x) for k, x in r.items()}
                    for n, r in results.items()},
        "host_cores": {"share": threads, "affinity": affinity, "cpu": cpu_model()},
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
