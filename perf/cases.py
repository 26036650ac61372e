"""Performance cases: the calls that programs make of this package, with their sizes, inputs, oracles and tolerances.

Each case is a dict of plain values. Kinds:

- ``call``       one host-pointer product of one matrix (`CQMatrix.matvec`): the reference ABI's own call;
- ``stack``      a plan over many device-resident matrices (`Plan.run`), FP32 or int8 arithmetic: the projections
                 of a decode step for a batch of sequences;
- ``gemm``       the prompt GEMM of one matrix (`CQMatrix.gemm_device`);
- ``attention``  decode attention over the int8 cache (`KVCache.attention`);
- ``layer``      one decoder layer of a batch: Q|K|V, KV store and attention, O, MLP up and down, chained;
- ``engine``     a request to the single-sequence engine (`GpuEngine`): a prompt, then single-token steps.

Device work goes to one stream of this module, as a serving program would hold it. Weights and their device
handles, plans, caches and engines are made in `prepare`; `run` is one pass and returns the outputs' buffers.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from openneedle_amd import formats
from openneedle_amd.archive import Archive, synthetic_released
from openneedle_amd.cq import CQMatrix, Plan
from openneedle_amd.device import Stream
from openneedle_amd.engine import GpuEngine
from openneedle_amd.kv import KVCache


# ---- the cases --------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one LM-head-sized vector product through the drop-in ABI, host memory in and out
        dict(name="call_cq4_2048x512", kind="call", rows=2048, cols=512, bits=4, group=32, batch=1),
        # one decoder layer for a single conversation, and for a full serving batch, both at context 2048
        dict(name="layer_1", kind="layer", seqs=1, hidden=512, mlp=2048, context=2048),
        dict(name="layer_64", kind="layer", seqs=64, hidden=512, mlp=2048, context=2048),
        # decode at batch 1 over the projections of a large model: the headline weight stream
        dict(name="stack_fp32_cq4_b1", kind="stack", path="fp32", count=16, rows=8192, cols=8192, bits=4, group=32,
             batch=1),
        # 2-bit projections in the released precision map's groups, eight sequences at once, FP32 arithmetic
        dict(name="stack_fp32_cq2_b8", kind="stack", path="fp32", count=16, rows=4096, cols=4096, bits=2, group=128,
             batch=8),
        # int8 arithmetic at a small odd batch over matrices whose sides are no multiple of a tile
        dict(name="stack_int8_cq4_b5", kind="stack", path="int8", count=24, rows=5003, cols=3000, bits=4, group=64,
             batch=5),
        # int8 arithmetic at a batch of sixteen sequences
        dict(name="stack_int8_cq4_b16", kind="stack", path="int8", count=64, rows=4096, cols=4096, bits=4, group=32,
             batch=16),
        # grouped-query decode attention of sequences of different ages
        dict(name="attention_gqa_16", kind="attention", seqs=16, kvheads=8, per_kv=4, head_dim=128, length=4096,
             ragged=True),
        # a prompt of 512 tokens through one projection
        dict(name="gemm_512x8192x2048", kind="gemm", m=512, rows=8192, cols=2048, bits=4, group=32),
        # a long prompt of odd length through an MLP-sized projection
        dict(name="gemm_1999x11008x4096", kind="gemm", m=1999, rows=11008, cols=4096, bits=4, group=128),
        # a short request to the engine: a small prompt and a few dozen generated tokens
        dict(name="engine_request", kind="engine", prompt=32, steps=32, kv="fp32", matmul="fp32"),
        # a full prompt to the engine, logits of the last token
        dict(name="engine_prompt", kind="engine", prompt=512, steps=0, kv="fp32", matmul="fp32"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]; odd and even alike."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "stack", "stack", "stack", "gemm", "gemm", "attention", "layer", "engine"])
    if kind == "call":
        return dict(kind=kind, rows=_log(rng, 256, 8192), cols=_log(rng, 128, 4096), bits=rng.choice([2, 3, 4]),
                    group=rng.choice([32, 64, 128]), batch=_log(rng, 1, 8))
    if kind == "stack":
        path = rng.choice(["fp32", "int8"])
        rows, cols = _log(rng, 512, 8192), _log(rng, 512, 8192)
        batch = _log(rng, 1, 16 if path == "fp32" else 64)
        most = min(16 * 8192 ** 2, 16 * 8192 ** 2 * (4 if path == "fp32" else 32) // batch)
        count = max(1, min(64, _log(rng, 1 << 22, max(1 << 22, most)) // (rows * cols)))
        return dict(kind=kind, path=path, count=count, rows=rows, cols=cols,
                    bits=rng.choice([2, 4] if path == "int8" else [2, 3, 4]), group=rng.choice([32, 64, 128]),
                    batch=batch)
    if kind == "gemm":
        rows, cols = _log(rng, 512, 14336), _log(rng, 512, 8192)
        m = min(_log(rng, 16, 4096), max(16, 1999 * 11008 * 4096 // (rows * cols)))
        return dict(kind=kind, m=m, rows=rows, cols=cols, bits=rng.choice([2, 4]), group=rng.choice([32, 64, 128]))
    if kind == "attention":
        kvheads, per_kv, hd = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8]), rng.choice([32, 64, 128])
        length = _log(rng, 64, 8192)
        most = max(1, 16 * 8 * 128 * 4096 // (kvheads * hd * length))
        return dict(kind=kind, seqs=_log(rng, 1, min(64, most)), kvheads=kvheads, per_kv=per_kv, head_dim=hd,
                    length=length, ragged=rng.random() < 0.5)
    if kind == "layer":
        hidden = rng.choice([256, 512, 1024])
        return dict(kind=kind, seqs=_log(rng, 1, 64), hidden=hidden, mlp=hidden * rng.choice([2, 4]),
                    context=_log(rng, 64, 2048))
    return dict(kind="engine", prompt=_log(rng, 1, 512), steps=rng.randrange(0, 33),
                kv=rng.choice(["fp32", "int8"]), matmul=rng.choice(["fp32", "int8"]))


# ---- inputs -----------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _stream():
    return Stream()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _host_matrix(gen, rows, cols, bits, group):
    """(packed codes, fp16 norms) on the device, in the archive's row-major layout: uniform codes, norms as the
    archives of trained models hold them (tens of thousandths)."""
    padded = formats.padded_width(cols, group)
    packed = torch.randint(0, 256, (rows, padded * bits // 8), generator=gen, device="cuda", dtype=torch.uint8)
    norms = (torch.rand((rows, padded // group), generator=gen, device="cuda") * 0.045 + 0.005).half()
    return packed, norms


def _upload(gen, rows, cols, bits, group, int8=False):
    packed, norms = _host_matrix(gen, rows, cols, bits, group)
    torch.cuda.synchronize()
    m = CQMatrix(None, None, (rows, cols), bits, group, formats.codebook(bits, group),
                 device=(packed.data_ptr(), norms.data_ptr(), _stream()), int8=int8)
    _stream().synchronize()
    return m


LAYER_GROUP, LAYER_HEAD = 32, 64


def _layer_shapes(c):
    h, f = c["hidden"], c["mlp"]
    return dict(wq=(h, h), wk=(h, h), wv=(h, h), wo=(h, h), wu=(f, h), wd=(h, f))


def _engine_tokens(c, seed):
    r = np.random.default_rng(seed + 7919)
    return [int(t) for t in r.integers(2, 8192, c["prompt"] + c["steps"])]


def prepare(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "call":
        packed, norms = _host_matrix(g, c["rows"], c["cols"], c["bits"], c["group"])
        x = _normal(g, c["batch"], c["cols"]).cpu().numpy()
        m = CQMatrix(packed.cpu().numpy(), norms.cpu().numpy(), (c["rows"], c["cols"]), c["bits"], c["group"],
                     formats.codebook(c["bits"], c["group"]))
        return dict(case=c, m=m, x=x)
    if c["kind"] == "stack":
        int8 = c["path"] == "int8"
        mats = [_upload(g, c["rows"], c["cols"], c["bits"], c["group"], int8) for _ in range(c["count"])]
        x = _normal(g, c["count"], c["batch"], c["cols"])
        y = torch.empty((c["count"], c["batch"], c["rows"]), device="cuda")
        plan = Plan(mats, [t.data_ptr() for t in x], [t.data_ptr() for t in y], batch=c["batch"], int8=int8)
        torch.cuda.synchronize()
        return dict(case=c, plan=plan, x=x, y=y)
    if c["kind"] == "gemm":
        m = _upload(g, c["rows"], c["cols"], c["bits"], c["group"])
        x = _normal(g, c["m"], c["cols"])
        y = torch.empty((c["m"], c["rows"]), device="cuda")
        torch.cuda.synchronize()
        return dict(case=c, m=m, x=x, y=y)
    if c["kind"] == "attention":
        kv = KVCache(1, c["length"], c["kvheads"], c["head_dim"], c["seqs"])
        for c0, k, v in _cache_rows(g, c["seqs"], c["length"], c["kvheads"], c["head_dim"]):
            torch.cuda.synchronize()
            kv.store(0, k.data_ptr(), v.data_ptr(), k.shape[1], first_slot=c0, stream=_stream())
            _stream().synchronize()
        heads = c["kvheads"] * c["per_kv"]
        q = _normal(g, c["seqs"], heads, c["head_dim"])
        lengths = _lengths(g, c) if c["ragged"] else None
        out = torch.empty_like(q)
        torch.cuda.synchronize()
        return dict(case=c, kv=kv, q=q, out=out, lengths=lengths, heads=heads)
    if c["kind"] == "layer":
        n, cap = c["seqs"], c["context"]
        mats = {w: _upload(g, *s, 4, LAYER_GROUP, True) for w, s in _layer_shapes(c).items()}
        kvh = c["hidden"] // LAYER_HEAD
        kv = KVCache(1, cap, kvh, LAYER_HEAD, n)
        for c0, k, v in _cache_rows(g, n, cap - 1, kvh, LAYER_HEAD):
            torch.cuda.synchronize()
            kv.store(0, k.data_ptr(), v.data_ptr(), k.shape[1], first_slot=c0, stream=_stream())
            _stream().synchronize()
        buf = {b: torch.empty((n, c["mlp"] if b == "u" else c["hidden"]), device="cuda") for b in "qkvaoud"}
        buf["x"] = _normal(g, n, c["hidden"])

        def plan(ws, xs, ys):
            return Plan([mats[w] for w in ws], [buf[b].data_ptr() for b in xs], [buf[b].data_ptr() for b in ys],
                        batch=n, int8=True)

        plans = dict(qkv=plan(["wq", "wk", "wv"], "xxx", "qkv"), o=plan(["wo"], "a", "o"), up=plan(["wu"], "o", "u"),
                     down=plan(["wd"], "u", "d"))
        slot = torch.full((n,), cap - 1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return dict(case=c, plans=plans, kv=kv, buf=buf, slot=slot)
    engine = GpuEngine(_archive(seed), kv_cache=c["kv"], matmul=c["matmul"])
    return dict(case=c, engine=engine, tokens=_engine_tokens(c, seed))


def _archive(seed):
    return Archive(synthetic_released(seed=int(seed), tokenizer_bytes=0))


def _cache_rows(gen, seqs, slots, kvheads, hd):
    """(first slot, K, V) pieces of a cache's contents, `slots` tokens per sequence."""
    step = max(1, min(slots, (1 << 25) // (seqs * kvheads * hd)))
    for c0 in range(0, slots, step):
        n = min(step, slots - c0)
        yield c0, _normal(gen, seqs, n, kvheads, hd), _normal(gen, seqs, n, kvheads, hd)


def _lengths(gen, c):
    return torch.randint(max(1, c["length"] // 4), c["length"] + 1, (c["seqs"],), generator=gen, device="cuda",
                         dtype=torch.int32)


# ---- one pass ---------------------------------------------------------------------------------------------------
def run(state):
    c = state["case"]
    if c["kind"] == "call":
        return state["m"].matvec(state["x"])
    s = _stream()
    if c["kind"] == "stack":
        state["plan"].run(s)
        return state["y"]
    if c["kind"] == "gemm":
        state["m"].gemm_device(state["x"].data_ptr(), state["y"].data_ptr(), c["m"], s)
        return state["y"]
    if c["kind"] == "attention":
        lengths = state["lengths"]
        state["kv"].attention(0, state["q"].data_ptr(), state["out"].data_ptr(), state["heads"], c["length"],
                              d_lengths=None if lengths is None else lengths.data_ptr(), stream=s)
        return state["out"]
    if c["kind"] == "layer":
        p, b = state["plans"], state["buf"]
        p["qkv"].run(s)
        state["kv"].attention(0, b["q"].data_ptr(), b["a"].data_ptr(), c["hidden"] // LAYER_HEAD, c["context"],
                              stream=s, next=p["o"],
                              new=(b["k"].data_ptr(), b["v"].data_ptr(), state["slot"].data_ptr()))
        p["o"].run(s, prepared=True, next=p["up"])
        p["up"].run(s, prepared=True, next=p["down"])
        p["down"].run(s, prepared=True)
        return {k: b[k] for k in "qkvaoud"}
    e, tokens = state["engine"], state["tokens"]
    e.reset()
    logits, hidden = e.prefill(tokens[:c["prompt"]], last_only=True, hidden=True)
    out = [logits]
    for t in tokens[c["prompt"]:]:
        out.append(e.step(t)[0])
    return dict(logits=np.stack(out), hidden=hidden)


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _weights(rows, cols, bits, group):
    padded = formats.padded_width(cols, group)
    return rows * (padded * bits / 8 + padded // group * 2)


def work(case):
    c = case
    if c["kind"] in ("call", "stack", "gemm"):
        n, b = c.get("count", 1), c["m"] if c["kind"] == "gemm" else c["batch"]
        return dict(bytes=n * (_weights(c["rows"], c["cols"], c["bits"], c["group"])
                               + 4 * b * (c["rows"] + c["cols"])),
                    flops=2.0 * n * b * c["rows"] * c["cols"])
    if c["kind"] == "attention":
        fill = 0.625 if c["ragged"] else 1.0  # the mean of the lengths drawn between a quarter and the whole
        rows = c["seqs"] * c["kvheads"] * c["length"] * fill
        io = 2 * 4 * c["seqs"] * c["kvheads"] * c["per_kv"] * c["head_dim"]
        return dict(bytes=rows * 2 * (c["head_dim"] + 4) + io, flops=4.0 * rows * c["per_kv"] * c["head_dim"])
    if c["kind"] == "layer":
        n, shapes = c["seqs"], _layer_shapes(c).values()
        kv = n * c["context"] * 2 * (c["hidden"] + 4 * c["hidden"] // LAYER_HEAD)
        return dict(bytes=sum(_weights(*s, 4, LAYER_GROUP) for s in shapes) + kv + 4 * n * (7 * c["hidden"] + c["mlp"]),
                    flops=sum(2.0 * n * r * k for r, k in shapes) + 4.0 * n * c["context"] * c["hidden"])
    # released geometry: 27 layers of 2048 x 512 2-bit rows, 24 x 2048 fp32 lane rows, an 8192 x 512 4-bit head
    layer = 2048 * (512 / 4 + 8) + 24 * 2048 * 4
    head = 8192 * (512 / 2 + 8)
    cached = lambda pos: 27 * min(pos + 1, 256) * 2 * 256 * (4 if c["kv"] == "fp32" else 1)  # noqa: E731
    passes = 1 + c["steps"]
    nbytes = passes * (27 * layer + head) + cached(c["prompt"] - 1) + \
        sum(cached(c["prompt"] + i) for i in range(c["steps"])) + 4 * passes * 8192
    flops = (c["prompt"] + c["steps"]) * 27 * 2.0 * (2048 * 512 + 24 * 2048) + passes * 2.0 * 8192 * 512
    return dict(bytes=nbytes, flops=flops)


# ---- tolerances -------------------------------------------------------------------------------------------------
# About four times the error against 64 bits that each path shows, which is that of its data types.
def tolerance(case):
    c = case
    if c["kind"] == "gemm":  # fp16 operands, 32-bit sums
        return dict(rel=1.4e-3, max=1e-2)
    if c["kind"] == "attention":
        return dict(rel=4e-6, max=1e-4)
    if c["kind"] == "layer":  # an 8-bit input code of a later projection may fall on the other side of a rounding step
        return dict(rel=1e-2, max=0.1)
    if c["kind"] == "engine":
        if c["kv"] == "int8" or c["matmul"] == "int8":  # the same for K / V and activation codes, through 27 layers
            return dict(rel=1e-2, max=0.1)
        return dict(rel=3e-6, max=1e-4)
    if c["kind"] == "stack" and c["path"] == "int8":
        return dict(rel=1.4e-4, max=1e-2)
    return dict(rel=1.5e-6, max=1e-4)  # 32-bit sums


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------------------
def _codes(packed, bits, padded):
    if bits == 4:
        return torch.stack((packed & 15, packed >> 4), -1).reshape(packed.shape[0], padded)
    if bits == 2:
        return torch.stack([(packed >> s) & 3 for s in (0, 2, 4, 6)], -1).reshape(packed.shape[0], padded)
    stream = torch.stack([(packed >> s) & 1 for s in range(8)], -1).reshape(packed.shape[0], padded, bits)
    return sum(stream[..., b] << b for b in range(bits))


def _fwht(x, group):
    """x [..., n], n a multiple of group: the normalised Walsh-Hadamard transform of every group."""
    v, h = x.reshape(-1, group), 1
    while h < group:
        p = v.reshape(-1, group // (2 * h), 2, h)
        v = torch.stack((p[:, :, 0] + p[:, :, 1], p[:, :, 0] - p[:, :, 1]), 2).reshape(-1, group)
        h *= 2
    return (v / math.sqrt(group)).reshape(x.shape)


def _rotated(x, group):
    padded = formats.padded_width(x.shape[-1], group)
    return _fwht(torch.nn.functional.pad(x.double(), (0, padded - x.shape[-1])), group)


def _book(bits, group):
    return torch.from_numpy(formats.codebook(bits, group)).cuda().double()


def _product(packed, norms, bits, group, x, block=2048):
    """x [b, cols] times the matrix, in 64 bits; rows of the matrix in blocks."""
    r = _rotated(x, group)
    book, out = _book(bits, group), []
    for r0 in range(0, packed.shape[0], block):
        codes = _codes(packed[r0:r0 + block], bits, r.shape[1]).long()
        w = book[codes] * norms[r0:r0 + block].double().repeat_interleave(group, 1)
        out.append(r @ w.T)
    return torch.cat(out, 1)


def _product_int8(packed, norms, bits, group, x, block=2048):
    """The int8 path's arithmetic in 64 bits: activations quantised per group, centroids to 8 bits."""
    r = _rotated(x, group).reshape(x.shape[0], -1, group)
    top = r.abs().amax(-1, keepdim=True)
    scale = torch.where(top > 0, top / 127, torch.ones_like(top))
    r = (torch.round(r / scale).clamp(-127, 127) * scale).reshape(x.shape[0], -1)
    book = _book(bits, group)
    cs = book.abs().max() / 127
    book = torch.round(book / cs).clamp(-127, 127) * cs
    out = []
    for r0 in range(0, packed.shape[0], block):
        codes = _codes(packed[r0:r0 + block], bits, r.shape[1]).long()
        out.append(r @ (book[codes] * norms[r0:r0 + block].double().repeat_interleave(group, 1)).T)
    return torch.cat(out, 1)


def _quantised(rows):
    """Cache rows as the int8 cache holds them, in 64 bits. Its quantiser is defined in 32 bits: the quotients are
    rounded to 32 bits here too, so that the same codes come out."""
    top = rows.abs().amax(-1, keepdim=True)
    inv = torch.where(top > 0, (127.0 / top.double()).float(), torch.zeros_like(top))
    scale = torch.where(top > 0, (top.double() / 127.0).float(), torch.ones_like(top))
    return torch.round(rows * inv).clamp(-127, 127).double() * scale.double()


def _attend(q, k, v, lengths):
    """q [seqs, heads, hd], k / v [seqs, slots, kvheads, hd] in 64 bits."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for s in range(q.shape[0]):
        n = k.shape[1] if lengths is None else int(lengths[s])
        qs = q[s].double().reshape(k.shape[2], -1, q.shape[-1])
        score = torch.matmul(qs, k[s, :n].permute(1, 2, 0).contiguous()) / math.sqrt(q.shape[-1])
        out[s] = torch.matmul(torch.softmax(score, -1), v[s, :n].permute(1, 0, 2).contiguous()).reshape(out[s].shape)
    return out


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "call":
        packed, norms = _host_matrix(g, c["rows"], c["cols"], c["bits"], c["group"])
        return _product(packed, norms, c["bits"], c["group"], _normal(g, c["batch"], c["cols"]))
    if c["kind"] == "stack":
        mats = [_host_matrix(g, c["rows"], c["cols"], c["bits"], c["group"]) for _ in range(c["count"])]
        x = _normal(g, c["count"], c["batch"], c["cols"])
        product = _product_int8 if c["path"] == "int8" else _product
        return torch.stack([product(*m, c["bits"], c["group"], xi) for m, xi in zip(mats, x)])
    if c["kind"] == "gemm":
        packed, norms = _host_matrix(g, c["rows"], c["cols"], c["bits"], c["group"])
        return _product(packed, norms, c["bits"], c["group"], _normal(g, c["m"], c["cols"]))
    if c["kind"] == "attention":
        kv = [(_quantised(k), _quantised(v))
              for _, k, v in _cache_rows(g, c["seqs"], c["length"], c["kvheads"], c["head_dim"])]
        q = _normal(g, c["seqs"], c["kvheads"] * c["per_kv"], c["head_dim"])
        return _attend(q, torch.cat([k for k, _ in kv], 1), torch.cat([v for _, v in kv], 1),
                       _lengths(g, c) if c["ragged"] else None)
    if c["kind"] == "layer":
        n, kvh = c["seqs"], c["hidden"] // LAYER_HEAD
        mats = {w: _host_matrix(g, *s, 4, LAYER_GROUP) for w, s in _layer_shapes(c).items()}
        kv = [(_quantised(k), _quantised(v)) for _, k, v in _cache_rows(g, n, c["context"] - 1, kvh, LAYER_HEAD)]
        x = _normal(g, n, c["hidden"])
        o = {}
        for b in "qkv":
            o[b] = _product_int8(*mats["w" + b], 4, LAYER_GROUP, x)
        new = [_quantised(o[b].float().reshape(n, 1, kvh, LAYER_HEAD)) for b in "kv"]
        k, v = (torch.cat([p[i] for p in kv] + [new[i]], 1) for i in (0, 1))
        o["a"] = _attend(o["q"].reshape(n, kvh, LAYER_HEAD), k, v, None).reshape(n, -1)
        o["o"] = _product_int8(*mats["wo"], 4, LAYER_GROUP, o["a"])
        o["u"] = _product_int8(*mats["wu"], 4, LAYER_GROUP, o["o"])
        o["d"] = _product_int8(*mats["wd"], 4, LAYER_GROUP, o["u"])
        return o
    if c["kv"] == "int8" or c["matmul"] == "int8":
        return None  # a code on the other side of a rounding step in one layer shows in every later one
    return _engine_exact(c, seed)


def _engine_exact(c, seed):
    """The engine's model over the whole token sequence at once (needle2/csrc/engine.cpp:968-1044), in 64 bits."""
    archive = _archive(seed)
    m, dev = archive.metadata, "cuda"
    ids = _engine_tokens(c, seed)
    T, D, N, L = len(ids), m["d_model"], m["mhc_lanes"], m["num_layers"]
    H, KV, HD, window = m["num_heads"], m["num_kv_heads"], m["head_dim"], m["kv_window"]

    def tensor(name):
        return torch.from_numpy(np.ascontiguousarray(archive.tensors[name].dequantize(), np.float32)).to(dev).double()

    def matrix(name):
        """The record's dense weights in 64 bits."""
        r = archive.tensors[name]
        book = torch.from_numpy(r.cq_codebook()).to(dev).double()
        packed = torch.from_numpy(np.array(r.packed)).to(dev).reshape(r.shape[0], -1)
        norms = torch.from_numpy(np.array(r.norms)).to(dev).reshape(r.shape[0], -1).double()
        codes = _codes(packed, r.bits, formats.padded_width(r.shape[1], r.group_size)).long()
        return _fwht(book[codes] * norms.repeat_interleave(r.group_size, 1), r.group_size)[:, :r.shape[1]]

    def rms(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)

    def rope(x):
        half = HD // 2
        div = np.float32(m["rope_theta"]) ** (np.arange(half, dtype=np.float32) * 2 / np.float32(HD))
        angle = np.arange(T, dtype=np.float32)[:, None] / div.astype(np.float32)
        cos, sin = (torch.from_numpy(f(angle.astype(np.float64))).to(dev)[:, None] for f in (np.cos, np.sin))
        a, b = x[..., :half], x[..., half:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    def engram(site):
        tables, slots, sub = m["num_engram_tables"], m["engram_slots"], m["engram_sub_dim"]
        heads = tables // len(m["engram_orders"])
        weights = matrix(f"engram{site}.tables")
        rows = torch.zeros((T, tables * sub), dtype=torch.float64, device=dev)
        for t in range(T):
            for table in range(tables):
                order = m["engram_orders"][table // heads]
                if t + 1 < order:
                    continue
                acc = (0x9e3779b9 * (table + 1)) & 0xffffffff
                for j in range(order):
                    acc = ((acc ^ ids[t - j]) * 0x01000193) & 0xffffffff
                acc ^= acc >> 15
                rows[t, table * sub:(table + 1) * sub] = weights[table * slots + acc % slots]
        names = [n for n in archive.tensors if n.startswith(f"engram{site}.")]
        key, raw = rows @ matrix(names[1]).T, rows @ matrix(names[2]).T
        taps, value = tensor(names[3]), torch.zeros_like(raw)
        for tap in range(taps.shape[0]):
            back = tap * m["engram_conv_dilation"]
            if back < T and (not window or back < window):
                value[back:] += taps[tap] * raw[:T - back]
        return key, value

    def sinkhorn(a):
        a = torch.exp(a - a.amax((-1, -2), keepdim=True))
        for _ in range(20):
            a = a / a.sum(-1, keepdim=True)
            a = a / a.sum(-2, keepdim=True)
        return a

    names = list(archive.tensors)
    mhc = [n for n in names if n.startswith("mhc_")]
    a_pre, a_post, a_res, b_pre, b_post, b_res, p_pre, p_post, p_res = (
        tensor(n) for n in mhc)
    embedding = matrix("embedding")
    x = embedding[torch.tensor(ids, device=dev)][:, None].expand(T, N, D) * math.sqrt(D)
    at = torch.arange(T, device=dev)
    seen = (at[None] <= at[:, None]) & ((at[None] > at[:, None] - window) if window else True)
    hidden = []
    for l in range(L):
        (norm_in, wq, wk, wv, q_norm, k_norm, wg, wo, post_norm, attn_gate, pre_hada, d1, d2, d3) = [
            n for n in names if n.startswith(f"layer{l:02d}.")]
        nx = rms(x.reshape(T, N * D))
        own = torch.tensor([n == l % N for n in range(N)], device=dev)
        hpre = torch.sigmoid(a_pre[l] * (nx @ p_pre[l * N:(l + 1) * N].T) + b_pre[l] + torch.where(own, 4.0, -4.0))
        hpost = 2 * torch.sigmoid(a_post[l] * (nx @ p_post[l * N:(l + 1) * N].T) + b_post[l]
                                  + torch.where(own, 0.0, -4.0))
        route = sinkhorn((nx @ p_res[l * N * N:(l + 1) * N * N].T).reshape(T, N, N) * a_res[l] + b_res[l])
        u = (hpre[..., None] * x).sum(1)
        bx = u
        for site, layer in enumerate(m["engram_layers"]):
            if layer == l:
                key, value = engram(site)
                alpha = torch.sigmoid((rms(u) * rms(key)).sum(-1, keepdim=True) / math.sqrt(D))
                bx = bx + alpha * value
        z = rms(bx) * (1 + tensor(norm_in))
        q = rope(rms((z @ matrix(wq).T).reshape(T, H, HD)) * (1 + tensor(q_norm)))
        k = rope(rms((z @ matrix(wk).T).reshape(T, KV, HD)) * (1 + tensor(k_norm)))
        v = (z @ matrix(wv).T).reshape(T, KV, HD)
        att = torch.empty((T, H, HD), dtype=torch.float64, device=dev)
        for h in range(H):
            score = (q[:, h] @ k[:, h * KV // H].T) / math.sqrt(HD)
            att[:, h] = torch.softmax(score.masked_fill(~seen, -math.inf), -1) @ v[:, h * KV // H].contiguous()
        att = att.reshape(T, H * HD) * torch.sigmoid(z @ matrix(wg).T)
        proj = rms(att @ matrix(wo).T) * (1 + tensor(post_norm))
        bx = bx + torch.sigmoid(tensor(attn_gate)) * proj
        z = rms(bx) * (1 + tensor(pre_hada))
        hada = m["hada_n"]
        w = _fwht(torch.nn.functional.pad(z * tensor(d1)[:D], (0, hada - D)), hada) * tensor(d2)
        w = _fwht(w * torch.sigmoid(w), hada)[:, :D]
        bx = bx + tensor(d3)[:D] * w - u
        x = hpost[..., None] * bx[:, None] + torch.matmul(route, x)
        hidden.append(x.mean(1))
    zf = rms(hidden[-1]) * (1 + tensor("final_norm"))
    last = c["prompt"] - 1
    return dict(logits=zf[last:] @ embedding.T, hidden=torch.stack([h[last] for h in hidden]))
