"""GPU tests of single kernel paths at the sizes where they can go wrong (tile edges,
remainders), against a general path of the library or a plain torch reference."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("no GPU visible for a gpu-marked test")
    return torch.device("cuda:0")


@pytest.mark.parametrize("kind,D,H,P", [("f16", 8, 3, 16), ("f16", 24, 2, 48), ("f16", 64, 1, 16), ("f16", 128, 8, 32),
                                        ("int4", 64, 3, 32), ("int4", 128, 2, 16), ("int4", 96, 2, 16)])
@pytest.mark.parametrize("mode", ["raw", "f32"])
def test_gather_units_equal_row_gather(gpu, kind, D, H, P, mode):
    """kv_gather (units of 4 tokens) against kv_gather_rows (token by token): contexts off
    multiples of 4, a bound below a context, an invalid block, gaps between the outputs of
    the sequences that must stay as they were."""
    import torch
    import vspec_rocm as vr

    dt = {"f16": vr.KV_F16, "int4": vr.KV_INT4}[kind]
    lens, bound, gap = [1, 2, 3, 4, 5, 4 * P + 3, 130, 0], 101, 3
    pool = vr.PagedPool(dt, 96, P, H, D, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(D + P)
    nblk = -(-max(lens) // P)
    tables = torch.randperm(96, generator=torch.Generator().manual_seed(1))[:len(lens) * nblk].view(len(lens), nblk).to(torch.int32)
    x = [torch.randn((len(lens), nblk * P, H, D), generator=g, device=gpu) for _ in range(2)]
    vr.kv_append(pool, tables, torch.zeros(len(lens), dtype=torch.int32), *x)
    tables[6, 1] = -1  # tokens P .. 2P - 1 of sequence 6 are not read
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    counts = [min(n, bound) for n in lens]
    off = [sum(counts[:b]) + gap * (b + 1) for b in range(len(lens))]
    total = sum(counts) + gap * (len(lens) + 1)
    raw = mode == "raw"
    out = {n: torch.full((total, H, D // 2 if raw and kind == "int4" else D), 7, device=gpu,
                         dtype=pool.k.dtype if raw else torch.float32) for n in "kv"}
    sc = {n: torch.full((total, H, max(D // 32, 1)), 7, device=gpu, dtype=torch.int16) for n in "kv"}
    import ctypes as C

    kv, tab = pool.desc(), tables.to(gpu)
    offd = torch.tensor(off, dtype=torch.int64, device=gpu)
    assert vr.lib().vspec_rocm_kv_gather(C.byref(kv), len(lens), tab.data_ptr(), nblk, ctx.data_ptr(), bound, offd.data_ptr(),
                                         vr.GATHER_RAW if raw else vr.GATHER_F32, out["k"].data_ptr(), out["v"].data_ptr(),
                                         sc["k"].data_ptr(), sc["v"].data_ptr(), torch.cuda.current_stream().cuda_stream), vr.last_error()
    # the same tokens through the row-list gather
    toks = [(b, t) for b, n in enumerate(counts) for t in range(n) if tables[b, t // P] >= 0]
    where = torch.tensor([off[b] + t for b, t in toks], device=gpu)
    pages = torch.tensor([int(tables[b, t // P]) for b, t in toks], dtype=torch.int32, device=gpu)
    slots = torch.tensor([t % P for _, t in toks], dtype=torch.int32, device=gpu)
    rows = {n: torch.empty((len(toks), H, D), device=gpu) for n in "kv"}
    assert vr.lib().vspec_rocm_kv_gather_rows(C.byref(kv), len(toks), pages.data_ptr(), slots.data_ptr(), rows["k"].data_ptr(),
                                              rows["v"].data_ptr(), torch.cuda.current_stream().cuda_stream)
    for n in "kv":
        got = out[n]
        if raw and kind == "int4":
            s = sc[n].view(torch.float16).float().repeat_interleave(32, -1)
            c = got.to(torch.int32)
            codes = torch.stack([((c & 15) ^ 8) - 8, ((c >> 4) ^ 8) - 8], -1).flatten(-2)
            got = codes.float() * s
        assert torch.equal(got[where].float(), rows[n])
        keep = torch.ones(total, dtype=torch.bool, device=gpu)
        keep[where] = False
        assert bool((out[n][keep] == 7).all())
        if raw and kind == "int4":
            assert bool((sc[n][keep] == 7).all())


@pytest.mark.parametrize("B,H", [(1, 8), (5, 8), (40, 16)])
def test_fused_step_many_short_items_d64(gpu, monkeypatch, B, H):
    """f16 pools with 64-element heads, several short work items per workgroup (more than the
    four whose new token is staged up front): the fused step leaves the bytes of kv_append."""
    import torch
    import vspec_rocm as vr

    monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", "0")
    D, P, T = 64, 16, 21
    g = torch.Generator(device=gpu).manual_seed(B)
    tables = torch.randperm(2 * B, generator=torch.Generator().manual_seed(B)).view(B, 2).to(torch.int32).to(gpu)
    kv = [torch.randn((B, T, H, D), generator=g, device=gpu).half() for _ in range(2)]
    new = [torch.randn((B, H, D), generator=g, device=gpu).half() for _ in range(2)]
    q = torch.randn((B, H, D), generator=g, device=gpu)
    pools = [vr.PagedPool(vr.KV_F16, 2 * B, P, H, D, device=gpu) for _ in range(2)]
    zero = torch.zeros(B, dtype=torch.int32)
    for pool in pools:
        vr.kv_append(pool, tables, zero, *kv)
    vr.kv_append(pools[0], tables, zero + T, *(x[:, None].contiguous() for x in new))
    vr.paged_decode_step(pools[1], tables, torch.full((B,), T + 1, dtype=torch.int32), q, *new)
    assert torch.equal(pools[0].k, pools[1].k) and torch.equal(pools[0].v, pools[1].v)


def _decode_setup(gpu, kind, lens, Hq, H, D, P, used=False, seed=0):
    import torch
    import vspec_rocm as vr

    dt = {"f32": vr.KV_F32, "f16": vr.KV_F16, "int4": vr.KV_INT4}[kind]
    nblk = max(1, -(-max(lens) // P))
    g = torch.Generator(device=gpu).manual_seed(seed + D + P + sum(lens))
    n = len(lens) * nblk
    tables = torch.randperm(n + 3, generator=torch.Generator().manual_seed(seed))[:n].view(len(lens), nblk).to(torch.int32).to(gpu)
    x = [torch.randn((len(lens), nblk * P, H, D), generator=g, device=gpu).half() for _ in range(2)]
    pools = []
    for _ in range(2):
        pool = vr.PagedPool(dt, n + 3, P, H, D, device=gpu)
        vr.kv_append(pool, tables, torch.zeros(len(lens), dtype=torch.int32), *x)
        pools.append(pool)
    q = torch.randn((len(lens), Hq, D), generator=g, device=gpu)
    new = [torch.randn((len(lens), H, D), generator=g, device=gpu).half() for _ in range(2)]
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    bu = None
    if used:  # some middle blocks partly filled; the last entry's count ends the span
        bu = torch.full((len(lens), nblk), P, dtype=torch.int32, device=gpu)
        bu[:, ::3] = max(1, P - 5)
        for b, t in enumerate(lens):
            if t:
                bu[b, (t - 1) // P] = (t - 1) % P + 1
    return vr, pools, tables, ctx, q, new, bu


def _same_pools(a, b):
    import torch

    return all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in
               ((a.k, b.k), (a.v, b.v), (a.ks, b.ks), (a.vs, b.vs), (a.kf, b.kf)) if x is not None)


@pytest.mark.parametrize("kind", ["f16", "int4"])
@pytest.mark.parametrize("lens,Hq,H,D,P,used", [
    ([1], 8, 8, 64, 16, False), ([16, 17, 0, 1], 8, 2, 128, 16, False), ([64, 65, 80, 81, 3], 6, 2, 64, 48, False),
    ([129], 24, 2, 128, 16, False), ([1000, 31, 515], 4, 2, 128, 32, True), ([300] * 5, 16, 4, 64, 16, True),
    ([4100, 77], 8, 2, 128, 16, False), ([130, 33, 700], 32, 2, 128, 16, True), ([47], 8, 1, 64, 48, False)])
def test_item_split_equals_balanced_split(gpu, monkeypatch, kind, lens, Hq, H, D, P, used):
    """One work item's part per workgroup, for several part counts, against the balanced split:
    the fused step's pool bytes are the same and the outputs differ only by rounding (f16: f32
    sums of weights <= 1 against |v| < 6 in another order, below 16 * 2^-24 * 6; int4 also
    rounds each weight x scale once to fp16 on either side, 2 * 2^-12 * 6)."""
    import torch

    vr, pools, tables, ctx, q, new, bu = _decode_setup(gpu, kind, lens, Hq, H, D, P, used)
    tol = 2 * 6 * 2.0 ** -12 if kind == "int4" else 6e-6
    for same in (False, True):
        if same and len(set(lens)) > 1:
            continue
        hint = dict(max_ctx_len=max(lens), min_ctx_len=max(lens) if same else 0, block_used=bu)
        for numerics in (vr.NUMERICS_PLAIN, vr.NUMERICS_3BIT):
            monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", "0")
            want = vr.paged_decode_step(pools[0], tables, ctx, q, *new, numerics=numerics, **hint)
            plain = vr.paged_decode(pools[0], tables, ctx, q, numerics=numerics, **hint)
            for parts in ("1", "2", "5", "64"):
                monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", parts)
                out = torch.full_like(q, float("nan"))
                vr.paged_decode_step(pools[1], tables, ctx, q, *new, numerics=numerics, out=out, **hint)
                assert _same_pools(*pools)
                assert float((out - want).abs().max()) <= tol
                out = vr.paged_decode(pools[1], tables, ctx, q, numerics=numerics, **hint)
                assert float((out - plain).abs().max()) <= tol


def test_item_split_keeps_the_workspace_plan(gpu, monkeypatch):
    """The item split fits the workspace that the balanced split's plan asks for, at every size
    below the one the caller sized its workspace for."""
    import ctypes as C

    vr, pools, tables, ctx, q, new, _ = _decode_setup(gpu, "f16", [2049] * 2, 8, 2, 128, 16)
    import torch

    out = torch.empty_like(q)
    big = vr.make_decode_desc(pools[0], tables, ctx, q, out, 2049)
    ws = torch.empty(vr.decode_workspace_bytes(big), dtype=torch.uint8, device=gpu)
    for bound in list(range(1, 400, 13)) + [640, 1000, 1024, 1500, 2000, 2049]:
        cl = torch.full((2,), bound, dtype=torch.int32, device=gpu)
        d = vr.make_decode_desc(pools[0], tables, cl, q, out, bound, workspace=ws)
        assert vr.lib().vspec_rocm_paged_decode_attention(C.byref(d)), vr.last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("lens,Hq,H,D,P,used,src", [
    ([1], 8, 8, 64, 16, False, "f16"), ([16, 17, 0, 1], 8, 2, 128, 16, False, "f32"), ([64, 65, 80, 81, 3], 6, 2, 64, 48, False, "f32"),
    ([257], 24, 2, 128, 16, False, "f16"), ([1000, 31, 515], 32, 4, 128, 32, True, "f32"), ([300] * 5, 16, 2, 64, 16, True, "f16")])
def test_f32_step_parts(gpu, monkeypatch, lens, Hq, H, D, P, used, src):
    """f32 pools: the fused step (token patched into the tile that holds it, by every group of
    query heads) against kv_append and the plain decode in one part, for several part counts:
    the same pool bytes; outputs within the rounding of f32 sums in another order (weights
    <= 1 against |v| < 6: 16 * 2^-24 * 6)."""
    import torch

    vr, pools, tables, ctx, q, new, bu = _decode_setup(gpu, "f32", lens, Hq, H, D, P, used)
    if src == "f32":
        new = [x.float() * 1.001 for x in new]
    live = [b for b, t in enumerate(lens) if t]
    at = torch.tensor([lens[b] - 1 for b in live], dtype=torch.int32)
    vr.kv_append(pools[0], tables[live].contiguous(), at, *(x[live][:, None].contiguous() for x in new))
    hint = dict(max_ctx_len=max(lens), block_used=bu)
    for numerics in (vr.NUMERICS_PLAIN, vr.NUMERICS_3BIT):
        monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", "1")
        want = vr.paged_decode(pools[0], tables, ctx, q, numerics=numerics, **hint)
        for parts in ("", "1", "2", "5", "64"):
            monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", parts)
            got = vr.paged_decode_step(pools[1], tables, ctx, q, *new, numerics=numerics, **hint)
            assert _same_pools(*pools)
            assert float((got - want).abs().max()) <= 6e-6


def _attend_valid(vr, pool, tables, spans, used, q, numerics):
    """Decode attention in 64 bits over the rows that the pool holds at the valid slots (read
    back as fp32 rows by kv_gather_rows)."""
    import ctypes as C
    import torch

    P, three = pool.block_tokens, numerics == vr.NUMERICS_3BIT
    H, D = pool.num_kv_heads, pool.head_dim

    def limited(x):
        th = (4.5 * x.std(-1, correction=0, keepdim=True)).clamp(min=1e-6)
        th = th.clamp(max=16.0) if three else th
        return x.clamp(-th, th)

    tab, use, out = tables.cpu(), used.cpu(), torch.zeros(q.shape, dtype=torch.float64)
    for b, span in enumerate(spans):
        at = [t for t in range(span) if t % P < int(use[b, t // P])]
        if not at:
            continue
        pages = torch.tensor([int(tab[b, t // P]) for t in at], dtype=torch.int32, device=q.device)
        slots = torch.tensor([t % P for t in at], dtype=torch.int32, device=q.device)
        k, v = (torch.empty((len(at), H, D), device=q.device) for _ in range(2))
        assert vr.lib().vspec_rocm_kv_gather_rows(C.byref(pool.desc()), len(at), pages.data_ptr(), slots.data_ptr(), k.data_ptr(),
                                                  v.data_ptr(), torch.cuda.current_stream().cuda_stream), vr.last_error()
        kc, vc, qc = limited(k.cpu().double()), v.cpu().double(), limited(q[b].cpu().double())
        for h in range(q.shape[1]):
            s = kc[:, h // (q.shape[1] // H)] @ qc[h] / D ** 0.5
            s = s.clamp(-24, 24) if three else s
            out[b, h] = s.softmax(0) @ vc[:, h // (q.shape[1] // H)]
    return out


@pytest.mark.parametrize("kind", ["f32", "f16", "int4"])
@pytest.mark.parametrize("Hq,H,D,P,blocks", [
    # used tokens of each block, the last one's span; tiles without a valid slot as a wave's only
    # tile, as its first of two, as a whole part, and as a whole sequence
    (8, 2, 128, 32, [[10, 32], [32, 16, 32, 3], [0, 0], [1]]), (8, 8, 64, 48, [[48, 5, 0, 48, 48, 20], [16, 47]]),
    (6, 2, 64, 16, [[0, 16, 0, 16, 3], [16, 0, 0, 0, 16, 16, 16, 16, 1], [0]]), (32, 4, 128, 64, [[5, 64, 64, 9, 64, 64, 40]])])
def test_decode_skips_tiles_without_valid_slots(gpu, monkeypatch, kind, Hq, H, D, P, blocks):
    """block_used counts that leave whole tiles empty, for several splits, against 64-bit
    attention over the valid rows (2e-5: the bar of the parity tests for f32 and f16; int4 also
    rounds each weight x scale once to fp16, 2^-12 of |v| < 8)."""
    import torch

    n = max(len(b) for b in blocks)
    spans = [(len(b) - 1) * P + b[-1] for b in blocks]
    vr, pools, tables, ctx, q, new, _ = _decode_setup(gpu, kind, [n * P] * len(blocks), Hq, H, D, P)
    used = torch.tensor([b + [0] * (n - len(b)) for b in blocks], dtype=torch.int32, device=gpu)
    ctx = torch.tensor(spans, dtype=torch.int32, device=gpu)
    tol = 8 * 2.0 ** -12 if kind == "int4" else 2e-5
    for numerics in (vr.NUMERICS_PLAIN, vr.NUMERICS_3BIT):
        want = _attend_valid(vr, pools[0], tables, spans, used, q, numerics)
        for parts in ("", "0", "1", "2", "5"):
            if parts:
                monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", parts)
            else:
                monkeypatch.delenv("VSPEC_ROCM_DECODE_ITEM_PARTS", raising=False)
            got = vr.paged_decode(pools[0], tables, ctx, q, numerics=numerics, block_used=used)
            assert float((got.cpu().double() - want).abs().max()) <= tol, (numerics, parts)
        # the step: each live sequence's last token replaced first
        monkeypatch.delenv("VSPEC_ROCM_DECODE_ITEM_PARTS")
        vr.paged_decode_step(pools[1], tables, ctx, q, *new, numerics=numerics, block_used=used)
        want = _attend_valid(vr, pools[1], tables, spans, used, q, numerics)
        got = vr.paged_decode_step(pools[1], tables, ctx, q, *new, numerics=numerics, block_used=used)
        assert float((got.cpu().double() - want).abs().max()) <= tol, numerics


@pytest.mark.parametrize("parts", ["1", "2"])
def test_f32_scores_far_below_zero(gpu, monkeypatch, parts):
    """f32 pools, plain numerics, every score below -1e30: the waves and the parts keep their
    relative weights (tokens of tile 2 score -8e32, the others twice that: the output is
    the mean of tile 2's V rows, up to 16 roundings of |v| < 6)."""
    import torch
    import vspec_rocm as vr

    monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", parts)
    T, D = 128, 64
    g = torch.Generator(device=gpu).manual_seed(3)
    u = torch.randint(0, 2, (D,), generator=g, device=gpu).float() * 2 - 1
    k = 2e16 * u.repeat(1, T, 1, 1)  # [1][T][1][D]
    k[:, 32:48] *= 0.5
    v = torch.randn((1, T, 1, D), generator=g, device=gpu)
    pool = vr.PagedPool(vr.KV_F32, T // 16, 16, 1, D, device=gpu)
    tables = torch.arange(T // 16, dtype=torch.int32).view(1, -1)
    vr.kv_append(pool, tables, torch.zeros(1, dtype=torch.int32), k, v)
    out = vr.paged_decode(pool, tables, torch.tensor([T], dtype=torch.int32), (-1e16 * u).view(1, 1, D).contiguous())
    want = v[0, 32:48, 0].double().mean(0)
    assert float((out[0, 0].double() - want).abs().max()) <= 16 * 2.0 ** -24 * 6


@pytest.mark.parametrize("sessions,rows,Hq,H,D,P", [
    ([14], 5, 8, 2, 128, 16), ([30, 1, 250], 3, 6, 2, 64, 32), ([63, 500], 4, 32, 4, 128, 48), ([47, 130], 32, 4, 1, 64, 16),
    ([15, 700, 63], 22, 8, 8, 64, 16)])
def test_f32_step_rows_that_share_blocks(gpu, monkeypatch, sessions, rows, Hq, H, D, P):
    """f32 pools, `rows` rows of the batch on one session's block table, each appending the
    session's next token (across a tile and a block; up to and above the 64 rows that the decode
    kernel looks after itself): every row sees the tokens of the rows before it, as after
    kv_append (the same pool bytes; outputs within the rounding of f32 sums in another order)."""
    import torch

    lens = [n + r + 1 for n in sessions for r in range(rows)]
    nblk = -(-max(lens) // P)
    vr, pools, tables, _, _, _, _ = _decode_setup(gpu, "f32", [nblk * P] * len(sessions), Hq, H, D, P)
    tables = tables.repeat_interleave(rows, 0).contiguous()
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(len(lens))
    q = torch.randn((len(lens), Hq, D), generator=g, device=gpu)
    for src in (torch.float32, torch.float16):
        new = [torch.randn((len(lens), H, D), generator=g, device=gpu).to(src) for _ in range(2)]
        vr.kv_append(pools[0], tables, ctx - 1, *(x[:, None].contiguous() for x in new))
        monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", "1")
        want = vr.paged_decode(pools[0], tables, ctx, q, numerics=vr.NUMERICS_3BIT)
        for parts in ("1", "", "3"):
            monkeypatch.setenv("VSPEC_ROCM_DECODE_ITEM_PARTS", parts)
            vr.kv_append(pools[1], tables, ctx - 1, *(x[:, None].neg().contiguous() for x in new))  # what the step replaces
            got = vr.paged_decode_step(pools[1], tables, ctx, q, *new, numerics=vr.NUMERICS_3BIT)
            assert _same_pools(*pools)
            assert float((got - want).abs().max()) <= 6e-6, (src, parts)


@pytest.mark.parametrize("pt", [16, 48, 512])
def test_f32_partition_tokens_is_the_part_size(gpu, pt):
    """f32 pools: with partition_tokens every part of an item holds that many tokens, whatever the
    longest context of the batch: the (max, sum) states in the workspace equal the exponential
    sums over exactly those tokens, and the other slots stay as they were (sums of up to 512
    exponentials <= 1 of scores with 2^-22 of error: 1e-5)."""
    import ctypes as C
    import torch

    lens, H, D, P = [1049, 130, 16], 2, 64, 16
    vr, pools, tables, ctx, q, _, _ = _decode_setup(gpu, "f32", lens, H, H, D, P)
    out = torch.empty_like(q)
    parts = -(-max(lens) // pt)
    d = vr.make_decode_desc(pools[0], tables, ctx, q, out, max(lens), partition_tokens=pt)
    assert vr.decode_workspace_bytes(d) == len(lens) * H * parts * (D + 2) * 4
    ws = torch.full((len(lens) * H * parts * (D + 2),), 7e7, device=gpu)
    d = vr.make_decode_desc(pools[0], tables, ctx, q, out, max(lens), partition_tokens=pt, workspace=ws)
    assert vr.lib().vspec_rocm_paged_decode_attention(C.byref(d)), vr.last_error()
    ml = ws[len(lens) * H * parts * D:].view(len(lens), H, parts, 2).cpu().double()
    k, _, _, _ = vr.kv_gather(pools[0], tables, ctx, out_mode=vr.GATHER_F32)
    k, at = k.cpu().double(), 0
    limit = lambda x: torch.minimum(torch.maximum(x, -4.5 * x.std(-1, correction=0, keepdim=True)), 4.5 * x.std(-1, correction=0, keepdim=True))  # noqa: E731
    for b, n in enumerate(lens):
        for h in range(H):
            s = limit(k[at:at + n, h]) @ limit(q[b, h].cpu().double()) / D ** 0.5
            ranges = range(0, n, pt) if n > pt else []  # an item in one part has no state
            for i, t in enumerate(ranges):
                want = s[t:t + pt].logsumexp(0)
                got = ml[b, h, i, 0] * 0.6931471805599453 + ml[b, h, i, 1].log()
                assert abs(float(got - want)) <= 1e-5, (b, h, i)
            assert bool((ml[b, h, len(ranges):] == 7e7).all())
        at += n


@pytest.mark.parametrize("rows", [7, 66])
def test_f32_step_in_hip_graph(gpu, rows):
    """f32 pools, items cut into parts, the append in the decode's launch (up to 64 rows) and ahead of
    it (more), captured: every replay, with the step's tokens replaced in the pool and eager work
    in between, equals the eager step bit for bit, pool bytes included."""
    import torch

    lens = [1 + (211 * b) % 900 for b in range(rows)]
    vr, pools, tables, ctx, q, new, _ = _decode_setup(gpu, "f32", lens, 8, 2, 128, 16)
    want = vr.paged_decode_step(pools[0], tables, ctx, q, *new, max_ctx_len=max(lens))
    out = torch.empty_like(q)
    d = vr.make_decode_desc(pools[1], tables, ctx, q, out, max(lens))
    ws = torch.empty(vr.decode_workspace_bytes(d), dtype=torch.uint8, device=gpu)
    assert ws.numel()
    s = torch.cuda.Stream()

    def step():
        vr.paged_decode_step(pools[1], tables, ctx, q, *new, max_ctx_len=max(lens), out=out, workspace=ws, stream=s.cuda_stream)

    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        step()
    for rep in range(4):
        vr.kv_append(pools[1], tables, ctx - 1, *(x[:, None].neg().contiguous() for x in new))  # what the step replaces
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        assert _same_pools(*pools), rep
        vr.paged_decode(pools[0], tables, ctx, q, max_ctx_len=max(lens))
