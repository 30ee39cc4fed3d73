"""What is timed: the work that an inference engine has this library do, through its public entry points.

Four kinds of case, in the three head shapes of the benchmark and the tests:

* ``decode``: one token per sequence over contiguous caches or a page pool, one or more layers;
* ``prefill``: prompts, or the rest of prompts whose beginning is cached, over the same storages;
* ``proj``: a Q8_0 weight projection of one token, a decode batch or a prompt chunk;
* ``layer``: a whole attention layer, Q/K/V projections, RoPE, the KV write, attention and the output
  projection, of a decode step or a prompt.

Inputs are N(0, 1) (K scaled where the soft-cap has to act), weights N(0, 1/cols) in Q8_0, as in the benchmark.
Lengths and page tables follow from the case, values from the seed. Device buffers are torch tensors whose
addresses the entry points take.
"""
import ctypes
import math
import random

import numpy as np
import torch

from glint_amd.attn import GpuBackend

PAGE = 16

# (query heads, KV heads, head_dim, model width): SmolLM-135M, Llama-3-8B and Gemma-2-9B
SHAPES = {"smol": (9, 3, 64, 576), "llama": (32, 8, 128, 4096), "gemma": (16, 8, 256, 3584)}

ROPE_BASE = 10000.0
SOFTCAP = 50.0

_backend = None


def backend():
    """One backend for the process, as an engine keeps one."""
    global _backend
    if _backend is None:
        _backend = GpuBackend(0)
    return _backend


class Dev:
    """A torch tensor as the device buffer that the entry points take."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


# ------------------------------------------------------------------ the cases

def decode_case(shape, dtype="f32", paged=False, batch=1, lo=512, hi=512, prefix=0, window=0, softcap=False,
                k_mul=1.0, layers=1, graph=False):
    return {"kind": "decode", "shape": shape, "dtype": dtype, "paged": paged, "batch": batch, "lo": lo, "hi": hi,
            "prefix": prefix, "window": window, "softcap": softcap, "k_mul": k_mul, "layers": layers, "graph": graph}


def prefill_case(shape, dtype="f32", paged=False, precision="f32", batch=1, lo=512, hi=512, cached=0, window=0,
                 softcap=False, k_mul=1.0):
    return {"kind": "prefill", "shape": shape, "dtype": dtype, "paged": paged, "precision": precision, "batch": batch,
            "lo": lo, "hi": hi, "cached": cached, "window": window, "softcap": softcap, "k_mul": k_mul}


def proj_case(rows, cols, n_vec, layers=1):
    return {"kind": "proj", "rows": rows, "cols": cols, "n_vec": n_vec, "layers": layers}


def layer_case(shape, phase, dtype="f32", batch=1, lo=512, hi=512, layers=1, graph=False):
    return {"kind": "layer", "shape": shape, "phase": phase, "dtype": dtype, "batch": batch, "lo": lo, "hi": hi,
            "layers": layers, "graph": graph}


def listed():
    return [
        # a small model's decode step on its own, one sequence: nothing but launches and latency, so the
        # step's 30 layers are a captured graph
        dict(decode_case("smol", lo=512, hi=512, layers=30, graph=True), name="decode_smol_f32_512"),
        # one user's decode step with the default f32 cache: 32 layers back to back
        dict(decode_case("llama", lo=4096, hi=4096, layers=32), name="decode_llama_f32_4096"),
        # a server's decode step, one layer: 64 ragged sequences over a Q8_0 page pool with a shared prefix
        dict(decode_case("llama", "q8", True, batch=64, lo=128, hi=8192, prefix=256), name="decode_llama_q8_b64"),
        # a sliding-window layer and a global one, soft-capped, head_dim 256
        dict(decode_case("gemma", "q8", True, batch=32, lo=2048, hi=8192, window=4096, softcap=True, k_mul=3.0,
                         layers=2), name="decode_gemma_q8_b32"),
        # a lightly loaded server: the whole attention layer for four sequences, four layers in a captured graph
        dict(layer_case("llama", "decode", "q8", batch=4, lo=200, hi=2000, layers=4, graph=True),
             name="layer_decode_llama_q8_b4"),
        # prompts of a batch at the default precision
        dict(prefill_case("llama", batch=4, lo=2048, hi=2048), name="prefill_llama_f32_4x2048"),
        # the same with bf16 inputs to the matrix products
        dict(prefill_case("llama", precision="bf16", batch=4, lo=2048, hi=2048), name="prefill_llama_bf16_4x2048"),
        # chat-sized ragged prompts over a Q8_0 pool, soft-capped, in a sliding window that most stay inside
        dict(prefill_case("gemma", "q8", True, batch=6, lo=31, hi=700, window=512, softcap=True, k_mul=3.0),
             name="prefill_gemma_q8_ragged"),
        # a new turn after a cached conversation: few query rows over a long Q8_0 past
        dict(prefill_case("llama", "q8", True, "bf16", batch=1, lo=217, hi=217, cached=3800),
             name="prefill_llama_q8_suffix"),
        # the fused Q/K/V projection of one token, eight layers' weights in turn
        dict(proj_case(6144, 4096, 1, layers=8), name="proj_qkv_1"),
        # and of a 64-sequence decode batch
        dict(proj_case(6144, 4096, 64, layers=4), name="proj_qkv_64"),
        # a prompt's whole attention layer at the default precision: projections of many tokens, RoPE, KV write
        dict(layer_case("llama", "prefill", batch=1, lo=997, hi=997), name="layer_prefill_llama_f32_997"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    limit = 2.7e9  # of the largest listed case
    while True:
        kind = rng.choice(("decode", "decode", "prefill", "prefill", "proj", "layer"))
        shape = rng.choice(tuple(SHAPES))
        if kind == "decode":
            gemma = shape == "gemma"
            paged = rng.random() < 0.7
            hi = _log_int(rng, 16, 8192)
            batch = _log_int(rng, 1, 64) if paged else 1
            lo = rng.randint(max(1, hi // 16), hi) if batch > 1 else hi
            c = decode_case(shape, rng.choice(("f32", "q8")), paged, batch=batch, lo=lo, hi=hi,
                            prefix=min(rng.choice((0, 0, 100, 256)), lo) if batch > 1 else 0,
                            window=rng.choice((0, 1024, 4096)) if gemma else 0, softcap=gemma, k_mul=3.0 if gemma else 1.0,
                            layers=rng.choice((2, 4)) if paged else rng.choice((8, 16, 30)), graph=rng.random() < 0.4)
        elif kind == "prefill":
            gemma = shape == "gemma"
            hi = _log_int(rng, 17, 2048)
            c = prefill_case(shape, rng.choice(("f32", "q8")), rng.random() < 0.6, rng.choice(("f32", "bf16")),
                             batch=rng.randint(1, 6), lo=rng.randint(max(1, hi // 8), hi), hi=hi,
                             cached=rng.choice((0, 0, _log_int(rng, 30, 6000))),
                             window=rng.choice((0, 512, 4096)) if gemma else 0, softcap=gemma, k_mul=3.0 if gemma else 1.0)
        elif kind == "proj":
            rows, cols = rng.choice(((6144, 4096), (4096, 4096), (1024, 4096), (960, 576), (576, 576), (8192, 3584),
                                     (3584, 4096)))
            n_vec = _log_int(rng, 1, 2048)
            c = proj_case(rows, cols, n_vec, layers=4 if n_vec <= 64 else 1)
        elif rng.random() < 0.5:
            hi = _log_int(rng, 40, 4000)
            batch = _log_int(rng, 1, 48)
            c = layer_case(shape, "decode", rng.choice(("f32", "q8")), batch=batch, lo=rng.randint(max(1, hi // 8), hi),
                           hi=hi, layers=2, graph=rng.random() < 0.6)
        else:
            hi = _log_int(rng, 17, 1500)
            c = layer_case(shape, "prefill", batch=rng.randint(1, 3), lo=rng.randint(max(1, hi // 4), hi), hi=hi)
        w = work(c)
        if max(w["bytes"], w["flops"] / 50) <= limit:
            return c


# ------------------------------------------------------------------ what follows from a case alone

def _rng(case, what):
    return random.Random(what + "/" + "/".join("%s=%s" % (k, case[k]) for k in sorted(case) if k != "name"))


def lengths(case):
    """Tokens of each sequence: of a decode its context, of a prefill its new rows. Ragged ones reach both ends."""
    r = _rng(case, "lengths")
    n = [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    if case["batch"] > 1:
        n[0], n[-1] = case["hi"], case["lo"]
    return n


def contexts(case):
    """Positions that each sequence has in the cache, its new ones included."""
    cached = case.get("cached", 0)
    return [cached + n for n in lengths(case)]


def windows(case):
    """The sliding window of each layer: every other layer of a model that alternates is global."""
    w = case.get("window", 0)
    layers = case.get("layers", 1)
    return [w if layer % 2 == 0 else 0 for layer in range(layers)]


def page_table(case):
    """[B][pages] physical pages, a permutation of the pool, the prefix's whole pages shared; and the pool's size."""
    need = [(n + PAGE - 1) // PAGE for n in contexts(case)]
    shared = case.get("prefix", 0) // PAGE
    own = [n - min(shared, n) for n in need]
    perm = list(range(shared + sum(own)))
    _rng(case, "pages").shuffle(perm)
    table = np.zeros((len(need), max(need)), np.int32)
    at = shared
    for b, n in enumerate(need):
        table[b, :min(shared, n)] = perm[:min(shared, n)]
        table[b, min(shared, n):n] = perm[at:at + own[b]]
        at += own[b]
    return table, len(perm)


def kv_row_bytes(case):
    _, n_kv, d, _ = SHAPES[case["shape"]]
    return 2 * n_kv * d * 4 if case["dtype"] == "f32" else 2 * n_kv * (d // 32) * 34


def weight_bytes(rows, cols):
    return rows * (cols // 32) * 34


def _attention_work(case):
    """(KV bytes, q and output bytes, operations) of the case's attention calls."""
    n_heads, _, d, _ = SHAPES[case["shape"]]
    kv = qo = flops = 0
    decode = case["kind"] == "decode" or case.get("phase") == "decode"
    shared = case.get("prefix", 0) // PAGE * PAGE
    for w in windows(case):
        if decode:
            seen, common = 0, shared
            for n in contexts(case):
                start = max(0, n - w) if w else 0
                seen += n - max(start, min(shared, n))
                common = min(common, start)
                flops += 4 * n_heads * d * (n - start)
            kv += (seen + (shared - common)) * kv_row_bytes(case)
            qo += 2 * case["batch"] * n_heads * d * 4
        else:
            for n, end in zip(lengths(case), contexts(case)):
                first = end - n
                kv += (end - (max(0, first - w + 1) if w else 0)) * kv_row_bytes(case)
                qo += 2 * n * n_heads * d * 4
                pairs = sum(min(p + 1, w) if w else p + 1 for p in range(first, end))
                flops += 4 * n_heads * d * pairs
    return kv, qo, flops


def _layer_shapes(case):
    """(rows, cols) of the Q, K, V and output projections."""
    n_heads, n_kv, d, width = SHAPES[case["shape"]]
    return (n_heads * d, width), (n_kv * d, width), (n_kv * d, width), (width, n_heads * d)


def new_tokens(case):
    return case["batch"] if case["phase"] == "decode" else sum(lengths(case))


def work(case):
    if case["kind"] == "proj":
        r, c, n, layers = case["rows"], case["cols"], case["n_vec"], case["layers"]
        return {"bytes": layers * (weight_bytes(r, c) + 4 * n * (r + c)), "flops": layers * 2 * n * r * c}
    kv, qo, flops = _attention_work(case)
    if case["kind"] != "layer":
        return {"bytes": kv + qo, "flops": flops}
    n, width = new_tokens(case), SHAPES[case["shape"]][3]
    each = sum(weight_bytes(r, c) for r, c in _layer_shapes(case)) + 8 * n * width
    return {"bytes": kv + case["layers"] * each,
            "flops": flops + case["layers"] * sum(2 * n * r * c for r, c in _layer_shapes(case))}


def tolerance(case):
    """About four times the distance of the path from 64 bits, as measured: 4e-7 in 32 bits (sums of some thousand
    products, the exponentials between them), 3e-3 with bf16 matrix inputs. A layer over a Q8_0 pool quantises rows that
    it computed itself: a row's last bit can move a quant by one."""
    if case.get("precision") == "bf16":
        return {"rel": 1.2e-2, "max": 0.3}
    if case["kind"] == "layer" and case["dtype"] == "q8":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 2e-6, "max": 2e-4}


# ------------------------------------------------------------------ inputs

def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + what) & 0x7FFFFFFF)
    return g


def _normal(seed, what, shape, mul=1.0):
    t = torch.randn(shape, generator=_gen(seed, what), device="cuda", dtype=torch.float32)
    return t.mul_(mul) if mul != 1.0 else t


def quantize(x):
    """Q8_0 of f32 [..., 32 k]: (quants as f32, scales as f16), the quantiser's rules: the scale is max|x| / 127 (1 for
    an empty block), the quant x times its inverse, rounded half away from zero."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    top = b.abs().amax(-1, keepdim=True)
    one = torch.ones_like(top)
    d = torch.where(top > 0, top / (127.0 * one), one)  # a tensor divisor: a plain number would become a product
    r = b * (one / d)
    q = torch.trunc(r)
    q = (q + torch.where((r - q).abs() >= 0.5, torch.sign(r), torch.zeros_like(r))).clamp_(-127.0, 127.0)
    return q, d.squeeze(-1).half()


def dequantized(x):
    """f64 values of f32 rows as Q8_0 storage holds them."""
    q, d = quantize(x)
    return (q.double() * d.double().unsqueeze(-1)).reshape(x.shape)


def weights(seed, what, rows, cols):
    """GGML Q8_0 bytes of a rows x cols matrix, on the GPU."""
    q, d = quantize(_normal(seed, what, (rows, cols), 1.0 / math.sqrt(cols)))
    out = torch.empty((rows, cols // 32, 34), dtype=torch.uint8, device="cuda")
    out[..., :2] = d.unsqueeze(-1).view(torch.uint8)
    out[..., 2:] = q.to(torch.int8).view(torch.uint8)
    return out


def weights64(raw):
    d = raw[..., :2].contiguous().view(torch.float16).double()
    return (raw[..., 2:].contiguous().view(torch.int8).double() * d).reshape(raw.shape[0], -1)


def kv_rows(case, seed, layer):
    """K and V of a layer in the order of the storage's rows: positions of a contiguous cache, slots of a pool."""
    _, n_kv, d, _ = SHAPES[case["shape"]]
    if stored_in_pages(case):
        n = page_table(case)[1] * PAGE
    else:
        n = case["batch"] * max(contexts(case))
    return (_normal(seed, 10 * layer + 1, (n, n_kv * d), case.get("k_mul", 1.0)),
            _normal(seed, 10 * layer + 2, (n, n_kv * d)))


def stored_in_pages(case):
    return case["kind"] == "layer" or case["paged"]


def _storage(case, seed):
    """The filled cache or pool, and each layer's page table on the device."""
    be = backend()
    _, n_kv, d, _ = SHAPES[case["shape"]]
    layers = case.get("layers", 1)
    tables, stride = None, 0
    if stored_in_pages(case):
        table, pages = page_table(case)
        kv = be.create_page_pool(pages * layers, n_kv, d, case["dtype"])
        stride = table.shape[1]
        tables = [Dev(torch.from_numpy(table + layer * pages).cuda()) for layer in range(layers)]
    else:
        kv = be.create_kv_cache(layers, max(contexts(case)), n_kv, d, case["dtype"], n_seqs=case["batch"])
    for layer in range(layers):
        k, v = kv_rows(case, seed, layer)
        if stored_in_pages(case):
            rows = torch.arange(len(k), device="cuda", dtype=torch.int64) + layer * pages * PAGE
        else:
            n = max(contexts(case))
            rows = torch.cat([torch.arange(n, device="cuda", dtype=torch.int64) + kv.row_id(b, layer, 0)
                              for b in range(case["batch"])])
        torch.cuda.synchronize()
        for i in range(0, len(k), 1 << 16):
            part = slice(i, i + (1 << 16))
            kv.write_rows_device(Dev(rows[part]), Dev(k[part]), Dev(v[part]), len(rows[part]))
        be.sync()
    return kv, tables, stride


def _decode_args(case):
    """Per layer: host and device window starts and lengths."""
    ctx = np.array(contexts(case), np.int32)
    got = []
    for w in windows(case):
        start = np.maximum(0, ctx - w).astype(np.int32) if w else np.zeros_like(ctx)
        n = (ctx - start).astype(np.int32)
        got.append((start, n, Dev(torch.from_numpy(start).cuda()), Dev(torch.from_numpy(n).cuda())))
    return got


def _rope_pos(case):
    if case["phase"] == "decode":
        return np.array(contexts(case), np.int32) - 1
    return np.concatenate([np.arange(n, dtype=np.int32) for n in lengths(case)])


def prepare(case, seed):
    be = backend()
    s = {"case": case}
    if case["kind"] == "proj":
        s["w"] = [be.create_q8_weights(weights(seed, layer, case["rows"], case["cols"]).cpu().numpy(), case["rows"],
                                       case["cols"]) for layer in range(case["layers"])]
        s["x"] = [Dev(_normal(seed, 100 + layer, (case["n_vec"], case["cols"]))) for layer in range(case["layers"])]
        s["y"] = torch.zeros((case["layers"], case["n_vec"], case["rows"]), device="cuda")
        s["yd"] = [Dev(t) for t in s["y"]]
        torch.cuda.synchronize()
        return s
    n_heads, n_kv, d, width = SHAPES[case["shape"]]
    layers = case.get("layers", 1)
    s["kv"], s["tables"], s["stride"] = _storage(case, seed)
    decode = case["kind"] == "decode" or case.get("phase") == "decode"
    rows = case["batch"] if decode else sum(lengths(case))
    if decode:
        s["args"] = _decode_args(case)
    else:
        s["q_start"] = Dev(torch.tensor([0] + list(np.cumsum(lengths(case))), dtype=torch.int32, device="cuda"))
        s["offset"] = Dev(torch.full((case["batch"],), case.get("cached", 0), dtype=torch.int32, device="cuda"))
        s["max_q"] = max(lengths(case))
    s["out"] = torch.zeros((layers, rows, n_heads, d), device="cuda")
    s["outd"] = [Dev(t) for t in s["out"]]
    if case["kind"] == "layer":
        shapes = _layer_shapes(case)
        s["w"] = [[be.create_q8_weights(weights(seed, 1000 + 10 * layer + i, r, c).cpu().numpy(), r, c)
                   for i, (r, c) in enumerate(shapes)] for layer in range(layers)]
        s["x"] = [Dev(_normal(seed, 100 + layer, (rows, width))) for layer in range(layers)]
        for name, r in (("q", n_heads * d), ("k", n_kv * d), ("v", n_kv * d), ("y", width)):
            s[name] = torch.zeros((layers, rows, r), device="cuda")
            s[name + "d"] = [Dev(t) for t in s[name]]
        pos = _rope_pos(case)
        table, pages = page_table(case)
        owner = np.arange(rows) if decode else np.repeat(np.arange(case["batch"]), lengths(case))
        at = table[owner, pos // PAGE].astype(np.int64) * PAGE + pos % PAGE
        s["pos"] = Dev(torch.from_numpy(pos).cuda())
        s["at"] = [Dev(torch.from_numpy(at + layer * pages * PAGE).cuda()) for layer in range(layers)]
        s["rows"] = rows
    else:
        s["q"] = [Dev(_normal(seed, 100 + layer, (rows, n_heads, d))) for layer in range(layers)]
    torch.cuda.synchronize()
    if case.get("graph"):
        _step(s)  # sizes the scratch
        be.sync()
        s["graph"] = be.capture(lambda: _step(s, captured=True))
    return s


def _attend(s, layer, q, out, captured):
    be, case = backend(), s["case"]
    n_heads, _, d, _ = SHAPES[case["shape"]]
    scale = 1.0 / math.sqrt(d)
    cap = SOFTCAP if case.get("softcap") else None
    pages = {"page_table": s["tables"][layer], "page_table_stride": s["stride"]} if s["tables"] else {"layer": layer}
    if "args" in s:
        start, n, start_dev, n_dev = s["args"][layer]
        host = {} if captured else {"kv_start_host": start, "kv_len_host": n}
        be.decode(s["kv"], q, out, start_dev, n_dev, case["batch"], int(n.max()), n_heads, scale, cap, **pages, **host)
    else:
        be.prefill(s["kv"], q, out, s["q_start"], s["offset"], case["batch"], s["max_q"], n_heads, scale, cap,
                   sliding_window=windows(case)[layer], precision=case.get("precision", "f32"), **pages)


def _step(s, captured=False):
    be, case = backend(), s["case"]
    captured = captured or bool(case.get("graph"))
    if case["kind"] != "layer":
        for layer in range(case.get("layers", 1)):
            _attend(s, layer, s["q"][layer], s["outd"][layer], captured)
        return
    n_heads, n_kv, d, _ = SHAPES[case["shape"]]
    for layer in range(case["layers"]):
        wq, wk, wv, wo = s["w"][layer]
        x, q, k, v = s["x"][layer], s["qd"][layer], s["kd"][layer], s["vd"][layer]
        n = s["rows"]
        be.matvec_q8_0(wq, x, n, q)
        be.matvec_q8_0(wk, x, n, k)
        be.matvec_q8_0(wv, x, n, v)
        be.rope(q, n, n_heads, d, s["pos"], ROPE_BASE)
        be.rope(k, n, n_kv, d, s["pos"], ROPE_BASE)
        s["kv"].write_rows_device(s["at"][layer], k, v, n)
        _attend(s, layer, q, s["outd"][layer], captured)
        be.matvec_q8_0(wo, s["outd"][layer], n, s["yd"][layer])


def run(state):
    case = state["case"]
    if case["kind"] == "proj":
        for w, x, y in zip(state["w"], state["x"], state["yd"]):
            backend().matvec_q8_0(w, x, case["n_vec"], y)
        return {"y": state["y"]}
    if "graph" in state:
        state["graph"].replay()
    else:
        _step(state)
    if case["kind"] == "layer":
        return {k: state[k] for k in ("q", "k", "v", "out", "y")}
    return {"out": state["out"]}


# ------------------------------------------------------------------ the same in 64 bits

def _softmax_attention(q, k, v, first, window, scale, cap):
    """q [n][H][d] at positions first.., k and v [end][Hkv][d] from position 0, all f64."""
    n, n_heads, d = q.shape
    group = n_heads // k.shape[1]
    out = torch.empty_like(q)
    for i in range(0, n, 2048):
        rows = torch.arange(first + i, first + min(n, i + 2048), device=q.device).unsqueeze(1)
        keys = torch.arange(k.shape[0], device=q.device).unsqueeze(0)
        hidden = keys > rows
        if window:
            hidden = hidden | (keys <= rows - window)
        for h in range(n_heads):
            t = q[i:i + 2048, h] @ k[:, h // group].T.contiguous() * scale
            t = cap * torch.tanh(t / cap) if cap else t
            p = torch.softmax(t.masked_fill_(hidden, -math.inf), dim=1)
            out[i:i + 2048, h] = p @ v[:, h // group].contiguous()
    return out


def _rope64(x, pos):
    """x [n][H][d] f64 rotated by the angles that f32 frequencies and positions give."""
    d = x.shape[-1]
    i = np.arange(0, d, 2, dtype=np.float32) / np.float32(d)
    freq = np.float32(1.0) / np.power(np.float64(ROPE_BASE), i.astype(np.float64)).astype(np.float32)
    angle = torch.from_numpy((pos.astype(np.float32)[:, None] * freq).astype(np.float64)).cuda().unsqueeze(1)
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).reshape(x.shape)


def exact(case, seed):
    if case["kind"] == "proj":
        y = [_normal(seed, 100 + layer, (case["n_vec"], case["cols"])).double()
             @ weights64(weights(seed, layer, case["rows"], case["cols"])).T.contiguous()
             for layer in range(case["layers"])]
        return {"y": torch.stack(y)}
    n_heads, n_kv, d, width = SHAPES[case["shape"]]
    decode = case["kind"] == "decode" or case.get("phase") == "decode"
    rows = case["batch"] if decode else sum(lengths(case))
    ends = contexts(case)
    starts = [n - 1 for n in ends] if decode else [case.get("cached", 0)] * case["batch"]
    bound = np.concatenate(([0], np.cumsum([e - s for e, s in zip(ends, starts)])))
    got = {k: [] for k in ("q", "k", "v", "out", "y")}
    for layer, w in enumerate(windows(case)):
        k, v = kv_rows(case, seed, layer)
        k, v = (dequantized(k), dequantized(v)) if case["dtype"] == "q8" else (k.double(), v.double())
        if stored_in_pages(case):
            table = page_table(case)[0]
            where = [torch.from_numpy((table[b, np.arange(n) // PAGE].astype(np.int64) * PAGE + np.arange(n) % PAGE)).cuda()
                     for b, n in enumerate(ends)]
        else:
            where = [torch.arange(n, device="cuda") + b * max(ends) for b, n in enumerate(ends)]
        if case["kind"] == "layer":
            x = _normal(seed, 100 + layer, (rows, width)).double()
            mats = [weights64(weights(seed, 1000 + 10 * layer + i, r, c)) for i, (r, c) in enumerate(_layer_shapes(case))]
            q, kn, vn = (x @ m.T.contiguous() for m in mats[:3])
            pos = _rope_pos(case)
            q = _rope64(q.reshape(rows, n_heads, d), pos)
            kn = _rope64(kn.reshape(rows, n_kv, d), pos).reshape(rows, -1)
            at = torch.cat([where[b][s:] for b, s in enumerate(starts)])
            stored = (dequantized(kn.float()), dequantized(vn.float())) if case["dtype"] == "q8" else (kn, vn)
            k[at], v[at] = stored
        else:
            q = _normal(seed, 100 + layer, (rows, n_heads, d)).double()
        out = torch.empty_like(q)
        for b in range(case["batch"]):
            part = slice(int(bound[b]), int(bound[b + 1]))
            out[part] = _softmax_attention(q[part], k[where[b]].reshape(-1, n_kv, d), v[where[b]].reshape(-1, n_kv, d),
                                           starts[b], w, 1.0 / math.sqrt(d), SOFTCAP if case.get("softcap") else None)
        got["out"].append(out)
        if case["kind"] == "layer":
            got["q"].append(q.reshape(rows, -1))
            got["k"].append(kn)
            got["v"].append(vn)
            got["y"].append(out.reshape(rows, -1) @ mats[3].T.contiguous())
    return {k: torch.stack(v) for k, v in got.items() if v}
