"""Performance cases of the paged KV-cache path, called through the C-ABI of include/vspec_rocm.h.

A case is one call (or one pair of calls that a step makes together) as an engine makes it per
layer: descriptors, block tables, pools and output buffers are kept between calls, as a C caller
keeps them.  Kinds:

  decode   the attention of one decode step; with "append" the fused step that also writes the
           step's new token (vspec_rocm_paged_decode_step), else vspec_rocm_paged_decode_attention
  append   a prefill chunk written through the block tables (vspec_rocm_kv_append), with "rope"
           the rotary embedding of k and q fused in (vspec_rocm_kv_append_rope)
  mixed    the packed tokens of a continuous-batching step: prefill chunks of some sequences and
           one decode token of the others (vspec_rocm_kv_append_tokens)
  read     cached tokens read back in [T][H][D] order (vspec_rocm_kv_gather)
  compact  blocks moved together after eviction (vspec_rocm_kv_compact)

Contexts, chunk starts and moves come from the case and its "mix" number; data, tables and the
order of the blocks from the seed.
"""
import ctypes as C
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vspec-engine_amd", "python"))
import vspec_rocm as vr  # noqa: E402

KV = {"f32": vr.KV_F32, "f16": vr.KV_F16, "int4": vr.KV_INT4}
GQA = dict(q_heads=32, kv_heads=8, head_dim=128, block=16)  # the Qwen3-8B KV shape of bench.py


def listed():
    return [
        # bench.py's default workload: a full batch of equal 4k contexts, f16 cache
        dict(name="step-f16-b64-4k", kind="decode", kv="f16", batch=64, ctx_lo=4097, ctx_hi=4097, append=True, numerics="3bit", mix=0, **GQA),
        # continuous batching: every context has its own length
        dict(name="step-f16-b64-ragged", kind="decode", kv="f16", batch=64, ctx_lo=128, ctx_hi=8192, append=True, numerics="3bit", mix=4, **GQA),
        # a small server batch
        dict(name="step-f16-b16-2k", kind="decode", kv="f16", batch=16, ctx_lo=2049, ctx_hi=2049, append=True, numerics="3bit", mix=0, **GQA),
        # one interactive user
        dict(name="step-f16-b1-4k", kind="decode", kv="f16", batch=1, ctx_lo=4097, ctx_hi=4097, append=True, numerics="3bit", mix=0, **GQA),
        # the full batch on the quantised cache, and the small one
        dict(name="step-int4-b64-4k", kind="decode", kv="int4", batch=64, ctx_lo=4097, ctx_hi=4097, append=True, numerics="3bit", mix=0, **GQA),
        dict(name="step-int4-b16-2k", kind="decode", kv="int4", batch=16, ctx_lo=2049, ctx_hi=2049, append=True, numerics="3bit", mix=0, **GQA),
        # the reference cache's own element type: the small server batch, and its smallest
        # configuration (one sequence, 8 heads of 64, no grouping, plain numerics)
        dict(name="step-f32-b16-2k", kind="decode", kv="f32", batch=16, ctx_lo=2049, ctx_hi=2049, append=True, numerics="3bit", mix=0, **GQA),
        dict(name="decode-f32-b1-257", kind="decode", kv="f32", batch=1, ctx_lo=257, ctx_hi=257, append=False, numerics="plain", mix=0,
             q_heads=8, kv_heads=8, head_dim=64, block=16),
        # chunked prefill into a quantised cache that already holds long contexts
        dict(name="append-int4-b8-c512", kind="append", kv="int4", src="f16", batch=8, tokens=512, start_lo=16384, start_hi=32256, rope=False, mix=5, **GQA),
        # chunked prefill of an f16 cache with the rotary embedding of k and q
        dict(name="append-rope-f16-b4-c1024", kind="append", kv="f16", src="f16", batch=4, tokens=1024, start_lo=0, start_hi=8192, rope=True, mix=1, **GQA),
        # a cached context read back as fp32 rows, the form of the reference's read call
        dict(name="read-f32-f16-b8-ragged", kind="read", kv="f16", out="f32", batch=8, ctx_lo=1024, ctx_hi=8192, mix=3, **GQA),
        # compaction of the surviving three quarters of eight long quantised contexts
        dict(name="compact-int4-8594", kind="compact", kv="int4", moves=8594, mix=0, **GQA),
    ]


def draw(rng):
    def spread(lo, hi):  # whole numbers, even over their logarithm
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))

    kind = rng.choices(["decode", "append", "mixed", "read", "compact"], [12, 3, 1, 2, 1])[0]
    q_heads, kv_heads, head_dim = rng.choice([(32, 8, 128)] * 4 + [(16, 4, 128), (32, 4, 128), (8, 8, 64), (16, 4, 64), (12, 4, 128)])
    c = dict(kind=kind, kv=rng.choice(["f16", "f16", "int4", "int4", "f32"]), q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
             block=rng.choice([16, 16, 16, 32, 64]), mix=rng.randrange(1 << 20))
    row = 2 * kv_heads * _row_bytes(c)  # cache bytes of one token
    if kind == "decode":
        c["batch"] = spread(1, 128)
        c["ctx_hi"] = spread(16, max(16, min(32768, int(0.9e9 / row / c["batch"]))))
        c["ctx_lo"] = c["ctx_hi"] if rng.random() < 0.4 else max(1, c["ctx_hi"] // rng.choice([2, 8, 64]))
        c["append"] = rng.random() < 0.8
        c["numerics"] = rng.choice(["3bit", "3bit", "plain"])
    elif kind == "append":
        c["src"] = "f32" if c["kv"] == "f32" or rng.random() < 0.2 else "f16"
        c["batch"] = spread(1, 64)
        c["tokens"] = spread(1, max(1, 6000 // c["batch"]))
        c["start_lo"], c["start_hi"] = 0, spread(16, 8192)
        c["rope"] = rng.random() < 0.5
    elif kind == "mixed":
        c["src"] = "f32" if c["kv"] == "f32" else "f16"
        c["prefills"], c["decodes"] = rng.randint(1, 4), spread(1, 128)
        c["tokens"] = spread(16, 1024)
        c["start_lo"], c["start_hi"] = 0, spread(16, 8192)
    elif kind == "read":
        c["out"] = rng.choice(["raw", "f32"])
        c["batch"] = spread(1, 32)
        c["ctx_hi"] = spread(16, max(16, 32768 // c["batch"]))
        c["ctx_lo"] = c["ctx_hi"] if rng.random() < 0.4 else max(1, c["ctx_hi"] // 8)
    else:
        c["moves"] = spread(16, max(16, int(1.2e8 / row / c["block"])))
    return c


def _row_bytes(case):
    """Bytes of one token's row of one kv head in K or in V, scales included."""
    d = case["head_dim"]
    return {"f32": 4 * d, "f16": 2 * d, "int4": d // 2 + d // 16}[case["kv"]]


def _lens(case):
    r = random.Random(case["mix"])
    return [r.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["batch"])]


def _appended(case):
    """(sequence, start position, new tokens) of an append or mixed case, by sequence."""
    r = random.Random(case["mix"])
    if case["kind"] == "append":
        return [(b, r.randint(case["start_lo"], case["start_hi"]), case["tokens"]) for b in range(case["batch"])]
    n = case["prefills"] + case["decodes"]
    return [(b, r.randint(case["start_lo"], case["start_hi"]), case["tokens"] if b < case["prefills"] else 1) for b in range(n)]


def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + what)


def _token_dtype(case):
    return torch.float32 if case.get("src", "f32" if case["kv"] == "f32" else "f16") == "f32" else torch.float16


def _tokens(case, seed, what, shape):
    """Key and value rows as a model's projections give them: normal, in the source type."""
    g = _gen(seed, what)
    return [torch.randn(shape, generator=g, device="cuda").to(_token_dtype(case)) for _ in range(2)]


def _pool_and_tables(case, seed, lens, spare=1.2):
    """A pool with a fifth of its blocks free and the sequences' blocks scattered over it."""
    p = case["block"]
    need = [-(-t // p) for t in lens]
    blocks = int(math.ceil(spare * sum(need)))
    pool = vr.PagedPool(KV[case["kv"]], blocks, p, case["kv_heads"], case["head_dim"])
    perm = torch.randperm(blocks, generator=torch.Generator().manual_seed(int(seed) + 1)).to(torch.int32)
    tables = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    return pool, tables.cuda()


def _fill(case, seed, pool, tables, lens):
    """Sequence b's first lens[b] tokens, written as prefill writes them."""
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    for b, n in enumerate(lens):
        if n:
            k, v = _tokens(case, seed, 16 + b, (1, n, case["kv_heads"], case["head_dim"]))
            vr.kv_append(pool, tables[b:b + 1], zero, k, v)


def _int(xs):
    return torch.tensor(xs, dtype=torch.int32, device="cuda")


def _pool_bits(pool):
    """The pool's memory as whole numbers: its bytes are part of what a call leaves behind."""
    word = {vr.KV_F32: torch.int32, vr.KV_F16: torch.int16, vr.KV_INT4: torch.uint8}[pool.dtype]
    out = {"k": pool.k.view(word), "v": pool.v.view(word)}
    if pool.dtype == vr.KV_INT4:
        out.update(ks=pool.ks, vs=pool.vs, kf=pool.kf)
    return out


class State:
    """call(stream) makes one pass with everything that it needs kept in its closure."""

    def __init__(self, call, result):
        self.call, self.result = call, result


def prepare(case, seed):
    lib, kind = vr.lib(), case["kind"]
    heads, d = case["kv_heads"], case["head_dim"]
    if kind == "decode":
        lens = _lens(case)
        pool, tables = _pool_and_tables(case, seed, lens)
        _fill(case, seed, pool, tables, [n - 1 for n in lens] if case["append"] else lens)
        ctx = _int(lens)
        q = torch.randn((len(lens), case["q_heads"], d), generator=_gen(seed, 1), device="cuda")
        out = torch.empty_like(q)
        k, v = _tokens(case, seed, 2, (len(lens), heads, d))
        desc = vr.make_decode_desc(pool, tables, ctx, q, out, max(lens),
                                   vr.NUMERICS_3BIT if case["numerics"] == "3bit" else vr.NUMERICS_PLAIN,
                                   min_ctx_len=max(lens) if min(lens) == max(lens) else 0)
        ref, src = C.byref(desc), vr.KV_F32 if k.dtype == torch.float32 else vr.KV_F16
        keep = (pool, tables, ctx, q, out, k, v)
        if case["append"]:
            def call(stream, keep=keep, k=k.data_ptr(), v=v.data_ptr()):
                desc.stream = stream
                return lib.vspec_rocm_paged_decode_step(ref, k, v, src)
        else:
            def call(stream, keep=keep):
                desc.stream = stream
                return lib.vspec_rocm_paged_decode_attention(ref)
        return State(call, dict(out=out, **(_pool_bits(pool) if case["append"] else {})))
    if kind in ("append", "mixed"):
        new = _appended(case)
        pool, tables = _pool_and_tables(case, seed, [at + n for _, at, n in new])
        kv, width = C.byref(pool.desc()), tables.shape[1]
        src = vr.KV_F32 if case["src"] == "f32" else vr.KV_F16
        result = _pool_bits(pool)
        if kind == "mixed":
            k, v = _tokens(case, seed, 2, (sum(n for _, _, n in new), heads, d))
            item = _int([b for b, _, n in new for _ in range(n)])
            pos = _int([at + i for _, at, n in new for i in range(n)])
            return State(lambda stream: lib.vspec_rocm_kv_append_tokens(
                kv, k.shape[0], item.data_ptr(), pos.data_ptr(), tables.data_ptr(), len(new), width, k.data_ptr(), v.data_ptr(), src, stream), result)
        n = case["tokens"]
        k, v = _tokens(case, seed, 2, (len(new), n, heads, d))
        start = _int([at for _, at, _ in new])
        if not case["rope"]:
            return State(lambda stream: lib.vspec_rocm_kv_append(
                kv, len(new), tables.data_ptr(), width, start.data_ptr(), n, k.data_ptr(), v.data_ptr(), src, stream), result)
        cos, sin = _rope_tables(case)
        q = torch.randn((len(new), n, case["q_heads"], d), generator=_gen(seed, 1), device="cuda")
        result["q"] = q_out = torch.empty_like(q)
        return State(lambda stream: lib.vspec_rocm_kv_append_rope(
            kv, len(new), tables.data_ptr(), width, start.data_ptr(), n, k.data_ptr(), v.data_ptr(), src, cos.data_ptr(), sin.data_ptr(), d,
            cos.shape[0], q.data_ptr(), q_out.data_ptr(), case["q_heads"], stream), result)
    if kind == "read":
        lens = _lens(case)
        pool, tables = _pool_and_tables(case, seed, lens)
        _fill(case, seed, pool, tables, lens)
        kv, ctx = C.byref(pool.desc()), _int(lens)
        off = torch.tensor([sum(lens[:b]) for b in range(len(lens))], dtype=torch.int64, device="cuda")
        raw = case["out"] == "raw"
        int4_raw = raw and case["kv"] == "int4"
        shape = (sum(lens), heads, d // 2 if int4_raw else d)
        result = {n: torch.empty(shape, dtype=pool.k.dtype if raw else torch.float32, device="cuda") for n in ("k", "v")}
        if int4_raw:
            result.update({n: torch.empty((sum(lens), heads, d // 32), dtype=torch.int16, device="cuda") for n in ("ks", "vs")})
        outs = [result["k"].data_ptr(), result["v"].data_ptr()] + [result[n].data_ptr() if int4_raw else None for n in ("ks", "vs")]
        mode = vr.GATHER_RAW if raw else vr.GATHER_F32
        keep = (pool, result)
        return State(lambda stream, keep=keep: lib.vspec_rocm_kv_gather(
            kv, len(lens), tables.data_ptr(), tables.shape[1], ctx.data_ptr(), max(lens), off.data_ptr(), mode, *outs, stream), result)
    n = case["moves"]
    scattered = -(-4 * n // 3)  # live blocks lie scattered over the first 4/3 n, and move to a run behind them
    pool = vr.PagedPool(KV[case["kv"]], scattered + n, case["block"], heads, d)
    result, g = _pool_bits(pool), _gen(seed, 1)
    for name, t in result.items():
        t.random_(0, 1 << 16, generator=g) if name == "kf" else t.random_(generator=g)
    src = torch.randperm(scattered, generator=torch.Generator().manual_seed(int(seed)))[:n].to(torch.int32).cuda()
    dst = (scattered + torch.arange(n)).to(torch.int32).cuda()
    kv = C.byref(pool.desc())
    return State(lambda stream: lib.vspec_rocm_kv_compact(kv, n, src.data_ptr(), dst.data_ptr(), stream), result)


def run(state):
    if not state.call(torch.cuda.current_stream().cuda_stream):
        raise vr.VspecRocmError(vr.last_error())
    return state.result


def _rope_tables(case):
    positions = max(at + n for _, at, n in _appended(case))
    half = case["head_dim"] // 2
    freq = 1e6 ** (-torch.arange(half, dtype=torch.float64) / half)
    angle = torch.arange(positions, dtype=torch.float64)[:, None] * freq
    return angle.cos().float().cuda(), angle.sin().float().cuda()


def work(case):
    row, heads, d = _row_bytes(case), case["kv_heads"], case["head_dim"]
    src = 2 if _token_dtype(case) == torch.float16 else 4
    if case["kind"] == "decode":
        lens = _lens(case)
        old = sum(lens) - (len(lens) if case["append"] else 0)
        bytes_ = old * heads * 2 * row + sum(-(-t // case["block"]) for t in lens) * 4 + len(lens) * case["q_heads"] * d * 8
        if case["append"]:
            bytes_ += len(lens) * heads * 2 * (src * d + row)
        return {"bytes": bytes_, "flops": 4 * sum(lens) * case["q_heads"] * d}
    if case["kind"] in ("append", "mixed"):
        new = _appended(case)
        n = sum(t for _, _, t in new)
        bytes_ = n * heads * 2 * (src * d + row) + 8 * n
        if case.get("rope"):
            span = min(n, max(at + t for _, at, t in new) - min(at for _, at, _ in new))
            bytes_ += n * case["q_heads"] * d * 8 + span * d * 4
        return {"bytes": bytes_, "flops": n * heads * 2 * d}
    if case["kind"] == "read":
        n = sum(_lens(case))
        return {"bytes": n * heads * 2 * (row + (row if case["out"] == "raw" else 4 * d)), "flops": n * heads * 2 * d}
    return {"bytes": 4 * case["moves"] * heads * case["block"] * row, "flops": 0}


def tolerance(case):
    # appended, moved and read values are whole numbers or exact products: bit for bit
    if case["kind"] != "decode":
        return "exact"
    # int4 decodes round each weight x scale product to fp16 once (2^-12 of it), f32 sums otherwise;
    # about four times the error against exact() over the ranges (2e-4 and 1.3e-3; 4e-7 and 2.1e-6)
    return {"rel": 8e-4, "max": 5e-3} if case["kv"] == "int4" else {"rel": 2e-6, "max": 1e-5}


def _stored(case, x):
    """The values that the cache holds for token rows x, in 64 bits."""
    if case["kv"] == "f32":
        return x.double()
    if case["kv"] == "f16":
        return x.half().double()
    x = x.float().unflatten(-1, (-1, 32))  # groups of 32 share a scale: an eighth of the second largest magnitude
    rep = x.abs().topk(2, dim=-1).values[..., 1:]
    scale = torch.where(rep > 0, rep / 8, torch.ones_like(rep)).clamp(min=1e-6, max=65504.0).half().float()
    return ((x / scale).round().clamp(-8, 7).double() * scale.double()).flatten(-2)


def _limited(x, three_bit):
    """Rows clipped to 4.5 standard deviations (and to 16 in 3-bit mode)."""
    th = (4.5 * x.std(-1, correction=0, keepdim=True)).clamp(min=1e-6)
    th = th.clamp(max=16.0) if three_bit else th
    return x.clamp(-th, th)


def exact(case, seed):
    heads, d = case["kv_heads"], case["head_dim"]
    if case["kind"] == "decode":
        lens, three = _lens(case), case["numerics"] == "3bit"
        group = case["q_heads"] // heads
        q = _limited(torch.randn((len(lens), case["q_heads"], d), generator=_gen(seed, 1), device="cuda").double(), three)
        last = _tokens(case, seed, 2, (len(lens), heads, d))
        out = torch.empty_like(q)
        for b, n in enumerate(lens):
            old = n - 1 if case["append"] else n
            k, v = _tokens(case, seed, 16 + b, (1, old, heads, d)) if old else (last[0][:1, None][:, :0], last[1][:1, None][:, :0])
            k, v = k[0], v[0]
            if case["append"]:
                k, v = torch.cat([k, last[0][b][None]]), torch.cat([v, last[1][b][None]])
            k, v = _limited(_stored(case, k), three), _stored(case, v)
            k, v = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
            score = torch.bmm(q[b].view(heads, group, d), k) / math.sqrt(d)
            score = score.clamp(-24, 24) if three else score
            out[b] = torch.bmm(score.softmax(-1), v).view(-1, d)
        return {"out": out}
    if case["kind"] == "append" and case["rope"]:
        cos, sin = (t.double() for t in _rope_tables(case))
        new = _appended(case)
        q = torch.randn((len(new), case["tokens"], case["q_heads"], d), generator=_gen(seed, 1), device="cuda").double()
        at = torch.tensor([a for _, a, _ in new], device="cuda")[:, None] + torch.arange(case["tokens"], device="cuda")
        c, s = cos[at][:, :, None], sin[at][:, :, None]
        x, y = q[..., :d // 2], q[..., d // 2:]
        return {"q": torch.cat([x * c - y * s, x * s + y * c], -1)}
    if case["kind"] == "read" and case["out"] == "f32":
        k, v = zip(*(_tokens(case, seed, 16 + b, (n, heads, d)) for b, n in enumerate(_lens(case))))
        return {"k": _stored(case, torch.cat(k)), "v": _stored(case, torch.cat(v))}
    return None
