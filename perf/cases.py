"""Timing cases of the attention path, through its public entry points.

Each case is a plain dict; `kind` names the call a program makes:

  attend     Context.launch over device-resident K and V: a decode token, a
             few positions at once (speculative verification), a prompt, or
             a bidirectional canvas over a cached prefix (two segments)
  step       LayerCache.attend_token: one decode token of a layer from its
             raw projections (head norms, rotation, cache append, attention)
  layer      the step, then the attention output block on its attended row
  transform  HeadTransform.prepare over a prompt's raw projections
  output     Context.attention_output over a prompt's attended rows
  host       HipKernels.attention_multi over host arrays with byte masks (the
             engine's own call when its cache is in host memory)

Sizes are those of bench.py and the tests: sliding layers of 16 query and 8
KV heads of 256 dims with a 1024-key window, global layers of 16 query and 2
KV heads of 512 dims, hidden width 2816; the drawn cases also take the other
head dims and lengths that the entries accept.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EPSILON = 1e-6
ROPE_BASE = 10000.0


def _package():
    name = "power_cpu_llm_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(ROOT, "power-cpu-llm_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _attend(name, heads, nq, keys, prefix=0, causal=True, window=0, unit_keys=False):
    qheads, kvheads, dim = heads
    case = {"kind": "attend", "qheads": qheads, "kvheads": kvheads, "dim": dim, "nq": nq,
            "keys": keys, "prefix": prefix, "causal": causal, "window": window,
            "unit_keys": unit_keys}
    if name:
        case["name"] = name
    return case


def _step(name, kind, heads, position, window, hidden):
    qheads, kvheads, dim = heads
    case = {"kind": kind, "qheads": qheads, "kvheads": kvheads, "dim": dim,
            "position": position, "window": window, "hidden": hidden}
    if name:
        case["name"] = name
    return case


def _host(name, heads, nq, keys):
    qheads, kvheads, dim = heads
    case = {"kind": "host", "qheads": qheads, "kvheads": kvheads, "dim": dim, "nq": nq,
            "keys": keys}
    if name:
        case["name"] = name
    return case


SLIDING = (16, 8, 256)
GLOBAL = (16, 2, 512)


def listed():
    return [
        # one decode token early in a conversation: launch latency counts
        _attend("decode_2k", SLIDING, 1, 2048),
        # the usual decode step of a sliding layer: a window that starts and
        # ends inside the kernels' key chunks
        _step("step_window", "step", SLIDING, 32667, 1024, 0),
        # a full-causal layer of one decode token at 32K, projections to
        # residual: what a long-context decode spends its time on
        _step("layer_32k", "layer", SLIDING, 32767, 0, 2816),
        # a global layer's decode at the longest context, and at a ragged
        # length in the middle of the range
        _attend("decode_128k_d512", GLOBAL, 1, 131072, unit_keys=True),
        _attend("decode_7k_d512", GLOBAL, 1, 7001, unit_keys=True),
        # eight positions at once over a cache in host memory
        _host("host_verify", SLIDING, 8, 1279),
        # a prompt: full causal, sliding with a ragged length, and a global
        # layer's
        _attend("prefill_4k", SLIDING, 4096, 4096),
        _attend("prefill_window_3001", SLIDING, 3001, 3001, window=1024),
        _attend("prefill_4k_d512", GLOBAL, 4096, 4096, unit_keys=True),
        # one denoising step of a 256-position canvas over a 2048-key prefix
        _attend("canvas_2304", SLIDING, 256, 2304, prefix=2048, causal=False),
        # the prompt's projections through the head norms and rotation
        {"name": "transform_4k", "kind": "transform", "qheads": 16, "kvheads": 8, "dim": 256,
         "tokens": 4096, "position": 0},
        # the prompt's attended rows through the output projection
        {"name": "output_2000", "kind": "output", "tokens": 2000, "width": 4096,
         "hidden": 2816},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: sizes over the logarithm of each range."""
    while True:
        kind = rng.choice(("decode", "decode", "verify", "prefill", "prefill", "chunked",
                           "canvas", "step", "layer", "transform", "output", "host"))
        heads = rng.choice((SLIDING, SLIDING, GLOBAL, (32, 8, 128), (16, 4, 64)))
        window = rng.choice((0, 0, 1024))
        unit = heads[2] == 512
        if kind == "decode":
            case = _attend(None, heads, 1, _log(rng, 100, 131072), window=window, unit_keys=unit)
        elif kind == "verify":
            case = _attend(None, heads, rng.randint(2, 16), _log(rng, 200, 32768), window=window,
                           unit_keys=unit)
        elif kind == "prefill":
            n = _log(rng, 64, 4096)
            case = _attend(None, heads, n, n, window=window, unit_keys=unit)
        elif kind == "chunked":
            n = _log(rng, 64, 1024)
            case = _attend(None, heads, n, n + _log(rng, 256, 8192), window=window,
                           unit_keys=unit)
        elif kind == "canvas":
            n, prefix = rng.choice((64, 128, 256)), _log(rng, 256, 4096)
            case = _attend(None, heads, n, n + prefix, prefix=prefix, causal=False,
                           unit_keys=unit)
        elif kind in ("step", "layer"):
            case = _step(None, kind, heads, _log(rng, 100, 32768), window,
                         2816 if kind == "layer" else 0)
        elif kind == "transform":
            case = {"kind": kind, "qheads": heads[0], "kvheads": heads[1], "dim": heads[2],
                    "tokens": _log(rng, 16, 4096), "position": _log(rng, 1, 8192)}
        elif kind == "output":
            case = {"kind": kind, "tokens": _log(rng, 1, 2000),
                    "width": heads[0] * heads[2], "hidden": 2816}
        else:
            case = _host(None, heads, rng.randint(1, 8), _log(rng, 64, 3194))
        if heads[2] == 512 and case.get("keys", 0) > 8192 and case.get("nq", 1) > 256:
            continue
        if case["kind"] in ("attend", "host") and case["nq"] > case["keys"]:
            continue
        cost = work(case)
        if cost["flops"] <= 2.8e11 and cost["bytes"] <= 1.08e9:
            return case


# ---- one pass ---------------------------------------------------------------

_contexts = {}


def _context():
    """The program's one context, on torch's current stream."""
    stream = torch.cuda.current_stream().cuda_stream
    if stream not in _contexts:
        _contexts[stream] = _package().Context(torch.cuda.current_device(), stream)
    return _contexts[stream]


class _DeviceRow:
    """A cache row's device memory. The tensor over it keeps this object, and
    so the cache that owns the memory, alive."""

    def __init__(self, cache, pointer, count):
        self.cache = cache
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4",
                                         "data": (pointer, False), "version": 2}


def _cache_row(cache, pointer, count):
    row = _DeviceRow(cache, pointer, count)
    tensor = torch.as_tensor(row, device="cuda")
    # two references without the tensor's: the local and the call's argument
    assert sys.getrefcount(row) > 2 and tensor.data_ptr() == pointer
    return tensor


def _normals(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _attend_inputs(case, seed):
    """(q pre-scaled by 1/sqrt(dim) as the engine does, k, v): rows as they
    leave the head norms; a global layer's K rows have unit norm."""
    gen = torch.Generator("cuda").manual_seed(seed)
    scale = float(np.float32(1.0 / math.sqrt(case["dim"])))
    q = _normals(gen, case["nq"], case["qheads"], case["dim"]) * scale
    k = _normals(gen, case["keys"], case["kvheads"], case["dim"])
    v = _normals(gen, case["keys"], case["kvheads"], case["dim"])
    if case.get("unit_keys"):
        k = k / k.norm(dim=-1, keepdim=True)
    return q.contiguous(), k.contiguous(), v.contiguous()


def _scales(seed, dim):
    rng = np.random.default_rng(seed)
    return ((1.0 + 0.1 * rng.standard_normal(dim)).astype(np.float32),
            (1.0 + 0.1 * rng.standard_normal(dim)).astype(np.float32))


def _step_inputs(case, seed):
    """Cached rows before the token (the retained ones), and the token's raw
    projections."""
    gen = torch.Generator("cuda").manual_seed(seed)
    position, window = case["position"], case["window"]
    kept = min(position, window - 1) if window else position
    width = case["kvheads"] * case["dim"]
    k, v = _normals(gen, kept, width), _normals(gen, kept, width)
    raw_q = _normals(gen, case["qheads"] * case["dim"])
    raw_k, raw_v = _normals(gen, width), _normals(gen, width)
    return k, v, raw_q, raw_k, raw_v


def _output_inputs(tokens, width, hidden, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    attended = _normals(gen, tokens, width) * 0.1
    weights = _normals(gen, hidden, width) * (1.0 / math.sqrt(width))
    post_scale = 1.0 + 0.1 * _normals(gen, hidden)
    residual = _normals(gen, tokens, hidden)
    return attended, weights, post_scale, residual


def _transform_inputs(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    n, width = case["tokens"], case["kvheads"] * case["dim"]
    return (_normals(gen, n, case["qheads"] * case["dim"]), _normals(gen, n, width),
            _normals(gen, n, width))


def _host_inputs(case, seed):
    rng = np.random.default_rng(seed)
    nq, keys = case["nq"], case["keys"]
    scale = np.float32(1.0 / math.sqrt(case["dim"]))
    width = case["kvheads"] * case["dim"]
    queries = [rng.standard_normal(case["qheads"] * case["dim"], dtype=np.float32) * scale
               for _ in range(nq)]
    k = rng.standard_normal(keys * width, dtype=np.float32)
    v = rng.standard_normal(keys * width, dtype=np.float32)
    masks = [np.arange(keys) <= keys - nq + i for i in range(nq)]
    return queries, k, v, masks


def _project(state, attended, case, tokens, width):
    """The output block's tensors and call arguments in `state`."""
    weights, post_scale, residual = state["weights"], state["post_scale"], state["residual"]
    state["projected"] = torch.empty(tokens, case["hidden"], device="cuda")
    state["result"] = torch.empty(tokens, case["hidden"], device="cuda")
    state["project"] = (attended.data_ptr(), tokens, width, weights.data_ptr(), case["hidden"],
                        post_scale.data_ptr(), EPSILON, residual.data_ptr(),
                        state["projected"].data_ptr(), state["result"].data_ptr())


def prepare(case, seed):
    pcl = _package()
    state = {"kind": case["kind"]}
    if case["kind"] == "host":
        queries, k, v, masks = _host_inputs(case, seed)
        state.update(kernels=pcl.HipKernels(), queries=queries, k=k, v=v, masks=masks,
                     kvheads=case["kvheads"], dim=case["dim"])
        return state
    ctx = state["ctx"] = _context()
    if case["kind"] == "attend":
        q, k, v = _attend_inputs(case, seed)
        out = torch.empty_like(q)
        row = case["kvheads"] * case["dim"]
        first = case["prefix"] or case["keys"]
        # a canvas' own rows are another buffer than the prefix's cache
        k1, v1 = k[first:].clone(), v[first:].clone()
        k0, v0 = (k[:first].clone(), v[:first].clone()) if case["prefix"] else (k, v)
        state.update(q=q, k0=k0, v0=v0, k1=k1, v1=v1, out=out)
        state["desc"] = ctx.desc(
            q=q.data_ptr(), q_stride=case["qheads"] * case["dim"], nq=case["nq"],
            k0=k0.data_ptr(), v0=v0.data_ptr(), n0=first,
            k1=k1.data_ptr() or None, v1=v1.data_ptr() or None, n1=case["keys"] - first,
            qheads=case["qheads"], kvheads=case["kvheads"], dim=case["dim"], kh_first=0,
            kh_end=case["kvheads"], causal=int(case["causal"]), window=case["window"],
            first_key=0, first_query=case["keys"] - case["nq"], q_scale=1.0,
            out=out.data_ptr(), o_stride=case["qheads"] * case["dim"])
        assert row * case["keys"] == k.numel()
        ctx.reserve(ctx.workspace_bytes(state["desc"]))
    elif case["kind"] in ("step", "layer"):
        qheads, kvheads, dim = case["qheads"], case["kvheads"], case["dim"]
        position, window, width = case["position"], case["window"], kvheads * dim
        k, v, raw_q, raw_k, raw_v = _step_inputs(case, seed)
        kept = k.shape[0]
        query_scale, key_scale = _scales(seed, dim)
        transform = pcl.HeadTransform(ctx, qheads, kvheads, dim, query_scale, key_scale, EPSILON,
                                      ROPE_BASE, sliding=True)
        cache = pcl.LayerCache(ctx, kvheads, dim, position + 4096, window,
                               (2 * kept + 8192) * width * 8)
        cache.reserve_rows(kept + 4096 + 64)
        # tokens that have left the window again, then the retained ones
        passed = position - kept
        filler = torch.zeros(min(passed, 2048), width, device="cuda") if passed else None
        while passed:
            n = min(passed, 2048)
            cache.append(filler.data_ptr(), filler.data_ptr(), n)
            cache.commit()
            passed -= n
        if kept:
            cache.append(k.data_ptr(), v.data_ptr(), kept)
            cache.commit()
        out = torch.empty(qheads * dim, device="cuda")
        q_out = torch.empty(qheads * dim, device="cuda")
        state.update(cache=cache, transform=transform, raw=(raw_q, raw_k, raw_v), out=out,
                     q_out=q_out, scale=float(np.float32(1.0 / math.sqrt(dim))), pending=None)
        # where the token's K and V rows land, and the program's workspace
        state["pending"] = _token(state)
        keys, values, rows, _ = cache.view()
        offset = 4 * (rows - 1) * width
        state["k_row"] = _cache_row(cache, keys + offset, width)
        state["v_row"] = _cache_row(cache, values + offset, width)
        if case["kind"] == "layer":
            _, state["weights"], state["post_scale"], state["residual"] = _output_inputs(
                1, qheads * dim, case["hidden"], seed + 1)
            _project(state, out, case, 1, qheads * dim)
        torch.cuda.current_stream().synchronize()
    elif case["kind"] == "transform":
        raw = _transform_inputs(case, seed)
        query_scale, key_scale = _scales(seed, case["dim"])
        state["transform"] = pcl.HeadTransform(ctx, case["qheads"], case["kvheads"], case["dim"],
                                               query_scale, key_scale, EPSILON, ROPE_BASE,
                                               sliding=True)
        state["raw"] = raw
        state["made"] = tuple(torch.empty_like(x) for x in raw)
        state["tokens"], state["position"] = case["tokens"], case["position"]
        # the rotation table up to the prompt's end, kept with the transform
        state["transform"].query(raw[0].data_ptr(), 1, case["position"] + case["tokens"] - 1,
                                 state["made"][0].data_ptr())
    else:
        attended, state["weights"], state["post_scale"], state["residual"] = _output_inputs(
            case["tokens"], case["width"], case["hidden"], seed)
        state["attended"] = attended
        _project(state, attended, case, case["tokens"], case["width"])
    return state


def _token(state):
    raw_q, raw_k, raw_v = state["raw"]
    return state["cache"].attend_token(state["transform"], raw_q.data_ptr(), raw_k.data_ptr(),
                                       raw_v.data_ptr(), state["q_out"].data_ptr(),
                                       state["out"].data_ptr(), q_scale=state["scale"])


def run(state):
    kind = state["kind"]
    if kind == "attend":
        state["ctx"].launch(state["desc"])
        return state["out"]
    if kind in ("step", "layer"):
        # the same position again: the last pass's token is taken back first
        state["cache"].rollback(state["pending"])
        state["pending"] = _token(state)
        made = [state["out"], state["q_out"], state["k_row"], state["v_row"]]
        if kind == "layer":
            state["ctx"].attention_output(*state["project"])
            made += [state["projected"], state["result"]]
        return made
    if kind == "transform":
        raw_q, raw_k, raw_v = state["raw"]
        q, k, v = state["made"]
        state["transform"].prepare(raw_q.data_ptr(), raw_k.data_ptr(), raw_v.data_ptr(),
                                   state["tokens"], state["position"], q.data_ptr(),
                                   k.data_ptr(), v.data_ptr())
        return [q, k, v]
    if kind == "output":
        state["ctx"].attention_output(*state["project"])
        return [state["projected"], state["result"]]
    return state["kernels"].attention_multi(state["queries"], state["k"], state["v"],
                                            state["kvheads"], state["dim"], state["masks"])


# ---- what a pass cannot do without ------------------------------------------

def _pairs(nq, keys, causal, window):
    """Allowed (query, key) pairs, and the keys that any query reads."""
    if not causal:
        return nq * keys, keys
    hi = np.arange(keys - nq + 1, keys + 1)
    lo = np.maximum(hi - window, 0) if window else np.zeros(nq, np.int64)
    return int((hi - lo).sum()), int(keys - lo[0])


def work(case):
    kind = case["kind"]
    if kind in ("attend", "host"):
        pairs, read = _pairs(case["nq"], case["keys"], case.get("causal", True),
                             case.get("window", 0))
        row = case["qheads"] * case["dim"]
        values = 2 * read * case["kvheads"] * case["dim"] + 2 * case["nq"] * row
        masks = case["nq"] * case["keys"] if kind == "host" else 0
        return {"bytes": 4 * values + masks, "flops": 4 * row * pairs}
    if kind in ("step", "layer"):
        kept = case["position"]
        if case["window"]:
            kept = min(kept, case["window"] - 1)
        row, width = case["qheads"] * case["dim"], case["kvheads"] * case["dim"]
        # cached rows; raw q, k, v and the rows made from them; the output
        values = 2 * kept * width + 3 * row + 4 * width
        flops = 4 * row * (kept + 1)
        if kind == "layer":
            values += case["hidden"] * row + 4 * case["hidden"]
            flops += 2 * case["hidden"] * row
        return {"bytes": 4 * values, "flops": flops}
    if kind == "transform":
        row = (case["qheads"] + 2 * case["kvheads"]) * case["dim"]
        return {"bytes": 4 * case["tokens"] * (2 * row + case["dim"]),
                "flops": 8 * case["tokens"] * row}
    n, width, hidden = case["tokens"], case["width"], case["hidden"]
    return {"bytes": 4 * (n * width + hidden * width + 3 * n * hidden + hidden),
            "flops": 2 * n * width * hidden}


def tolerance(case):
    """About four times the largest error that exact() shows at these sizes:
    attention's 32-bit scores, probabilities and sums (6.5e-7 measured), and
    one rounding to 32 bits of the head transform's and the output block's
    64-bit sums (5.5e-8)."""
    if case["kind"] in ("transform", "output"):
        return {"rel": 2.2e-7}
    return {"rel": 2.6e-6}


# ---- the same outputs in 64 bits --------------------------------------------

def _attention64(q, k, v, group, first_query, causal, window):
    """q [nq][qheads][dim], k and v [keys][kvheads][dim] of the device, query
    i at key position first_query + i."""
    nq, qheads, dim = q.shape
    out = torch.empty(nq, qheads, dim, device=q.device, dtype=torch.float64)
    kp = torch.arange(k.shape[0], device=q.device)
    for kv in range(k.shape[1]):
        k64, v64 = k[:, kv].double(), v[:, kv].double()
        for h in range(kv * group, (kv + 1) * group):
            for i0 in range(0, nq, 1024):
                i1 = min(i0 + 1024, nq)
                s = q[i0:i1, h].double() @ k64.T
                if causal:
                    qp = torch.arange(first_query + i0, first_query + i1, device=q.device)[:, None]
                    ok = kp <= qp
                    if window:
                        ok &= qp - kp < window
                    s = s.masked_fill(~ok, -math.inf)
                out[i0:i1, h] = torch.softmax(s, dim=-1) @ v64
    return out


def _rotation64(position, count, dim):
    """The cosines and sines of f32 angles: a rotation's angle is the f32
    product of the position and an f32 frequency."""
    j = np.arange(dim // 2, dtype=np.float64)
    exponent = (np.float32(2.0) * j.astype(np.float32) / np.float32(dim)).astype(np.float64)
    power = np.power(ROPE_BASE, exponent).astype(np.float32)
    frequency = np.float32(1.0) / power
    positions = np.arange(position, position + count).astype(np.float32)
    angle = (positions[:, None] * frequency[None, :]).astype(np.float64)
    return (torch.from_numpy(np.cos(angle)).cuda()[:, None, :],
            torch.from_numpy(np.sin(angle)).cuda()[:, None, :])


def _norm64(x):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True)
                          + float(np.float32(EPSILON)))


def _transform64(raw, scale, heads, dim, position):
    """Rows [n][heads * dim] through the norm, the scale and the rotation
    (scale None: the norm alone)."""
    x = _norm64(raw.double().reshape(-1, heads, dim))
    if scale is not None:
        x = x * torch.from_numpy(scale).cuda().double()
        cos, sin = _rotation64(position, x.shape[0], dim)
        a, b = x[..., :dim // 2], x[..., dim // 2:]
        x = torch.cat((a * cos - b * sin, a * sin + b * cos), dim=-1)
    return x


def _output64(attended, weights, post_scale, residual):
    projected = attended.double() @ weights.double().T
    return [projected, residual.double() + _norm64(projected) * post_scale.double()]


def exact(case, seed):
    kind = case["kind"]
    if kind == "attend":
        q, k, v = _attend_inputs(case, seed)
        return _attention64(q, k, v, case["qheads"] // case["kvheads"],
                            case["keys"] - case["nq"], case["causal"], case["window"])
    if kind == "host":
        queries, k, v, _ = _host_inputs(case, seed)
        shape = (-1, case["kvheads"], case["dim"])
        q = torch.from_numpy(np.stack(queries)).reshape(case["nq"], case["qheads"], -1)
        made = _attention64(q.cuda(), torch.from_numpy(k).cuda().reshape(shape),
                            torch.from_numpy(v).cuda().reshape(shape),
                            case["qheads"] // case["kvheads"], case["keys"] - case["nq"], True, 0)
        return [row.reshape(-1).cpu().numpy() for row in made]
    if kind == "transform":
        raw_q, raw_k, raw_v = _transform_inputs(case, seed)
        query_scale, key_scale = _scales(seed, case["dim"])
        made = ((raw_q, query_scale, case["qheads"]), (raw_k, key_scale, case["kvheads"]),
                (raw_v, None, case["kvheads"]))
        return [_transform64(x, scale, heads, case["dim"], case["position"]).reshape(x.shape)
                for x, scale, heads in made]
    if kind == "output":
        return _output64(*_output_inputs(case["tokens"], case["width"], case["hidden"], seed))
    k, v, raw_q, raw_k, raw_v = _step_inputs(case, seed)
    query_scale, key_scale = _scales(seed, case["dim"])
    qheads, kvheads, dim, position = (case["qheads"], case["kvheads"], case["dim"],
                                      case["position"])
    q = _transform64(raw_q, query_scale, qheads, dim, position)
    k_row = _transform64(raw_k, key_scale, kvheads, dim, position)
    v_row = _transform64(raw_v, None, kvheads, dim, position)
    scale = float(np.float32(1.0 / math.sqrt(dim)))
    keys = torch.cat((k.double().reshape(-1, kvheads, dim), k_row))
    values = torch.cat((v.double().reshape(-1, kvheads, dim), v_row))
    out = _attention64(q * scale, keys, values, qheads // kvheads, keys.shape[0] - 1, False, 0)
    made = [out.reshape(-1), q.reshape(-1), k_row.reshape(-1), v_row.reshape(-1)]
    if kind == "layer":
        _, weights, post_scale, residual = _output_inputs(1, qheads * dim, case["hidden"],
                                                          seed + 1)
        made += _output64(out.reshape(1, -1), weights, post_scale, residual)
    return made
