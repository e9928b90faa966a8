"""Paged attention of prompt rows and of decoded rows at the edges of their
tiles, pages and key parts, against fp64 on the CPU. Results are bf16, off by up to
2^-8 of themselves (half a step of 2^-7 at a power of two). The weights that meet
128-wide values of prompts are rounded to bf16 as well, each by up to 2^-8 of itself,
2^-9 on average: 2^-8 of the weighted sum of |v| is allowed, for decoded rows too,
whose weights have 16 bits (test_decode_weights). 64-wide heads keep 32-bit weights:
2^-18 for their exponentials, whose arguments are rounded products of up to 2^5."""
import math

import pytest
import torch

from xllm_service_amd import ops
from xllm_service_amd.ops import hybrid as H

pytestmark = pytest.mark.gpu
PAGE = 16


def make(lens, ctx, kv_heads, per, dim, seed, spare=3):
    """bf16 queries behind a wider row, caches over scattered pages, and the
    lengths, on the CPU."""
    g = torch.Generator().manual_seed(seed)
    need = [-(-(n + c) // PAGE) for n, c in zip(lens, ctx)]
    order = torch.randperm(sum(need) + spare, generator=g).to(torch.int32)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    pool = (sum(need) + spare, kv_heads, PAGE, dim)
    k, v = (torch.randn(pool, generator=g).to(torch.bfloat16)
            for _ in range(2))
    heads = kv_heads * per
    rows = torch.randn(sum(lens), (heads + 2) * dim, generator=g)
    return rows.to(torch.bfloat16), k, v, table


def want(q, k, v, table, lens, ctx, scale, window=0, keep_first=0,
         chunked=False, sink=None, cap=0.0, head_scale=None):
    """(result, weighted sum of |v|) in fp64; q [T, heads, dim]."""
    heads, dim = q.shape[1:]
    per = heads // k.shape[1]
    out, big, at = [], [], 0
    for s, (n, c) in enumerate(zip(lens, ctx)):
        pages = table[s, :-(-(n + c) // PAGE)].long()
        kk, vv = (x[pages].transpose(1, 2).reshape(-1, k.shape[1], dim)[:n + c]
                  .double().repeat_interleave(per, 1) for x in (k, v))
        z = torch.einsum("thd,lhd->htl", q[at:at + n].double(), kk) * scale
        if head_scale is not None:
            z = z * head_scale.double()[:, None, None]
        if cap:
            z = cap * torch.tanh(z / cap)
        pos, key = c + torch.arange(n)[:, None], torch.arange(n + c)[None]
        gone = key > pos
        if window:
            first = pos // window * window if chunked else pos - window + 1
            gone = gone | ((key < first) & (key >= keep_first))
        z = z.masked_fill(gone, -math.inf)
        m = z.amax(-1, keepdim=True)
        if sink is not None:
            m = torch.maximum(m, sink.double()[:, None, None])
        p = torch.exp(z - m)
        den = p.sum(-1, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink.double()[:, None, None] - m)
        p = p / den
        out.append(torch.einsum("htl,lhd->thd", p, vv))
        big.append(torch.einsum("htl,lhd->thd", p, vv.abs()))
        at += n
    return torch.cat(out), torch.cat(big)


def check(got, ref, big):
    off = (got.double().cpu() - ref).abs()
    assert torch.isfinite(got).all()
    weights = 2.0 ** (-8 if got.shape[-1] == 128 else -18)
    over = off - weights * big - 2.0 ** -8 * ref.abs() - 1e-6
    assert over.max() <= 0, f"off by {off.max():.3g}, over by {over.max():.3g}"


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lens,ctx,kv_heads,per", [
    ([1, 31, 32, 33], [0, 15, 16, 17], 3, 1),       # waves and pages
    ([63, 64, 65], [0, 1, 63], 2, 2),               # key tiles
    ([127, 128, 129, 1], [0, 0, 5, 64], 1, 1),      # row tiles
    ([18, 19, 37], [47, 300, 0], 4, 7),             # heads that share keys
    ([3, 1, 9], [2100, 1033, 4500], 2, 4),          # keys split over parts
    ([1], [9000], 1, 8),                            # over 64 tiles of one page
    ([1] * 70 + [5], [3] * 70 + [40], 2, 3),        # more than 64 sequences
])
def test_prefill_edges(dim, lens, ctx, kv_heads, per):
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(lens) + dim)
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)))
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)])
    dev = [t.cuda() for t in (k, v, table, cu.int(), sl.int())]
    qd = rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim))
    # the result goes into rows of a wider tensor; what is beside them stays
    wide = torch.full((sum(lens), (heads + 1) * dim), 7.0,
                      dtype=torch.bfloat16, device="cuda")
    out = wide[:, :heads * dim].unflatten(-1, (heads, dim))
    for sign in (1.0, -1.0):
        got = ops.paged_attn_prefill(qd, *dev, sign * scale, out=out)
        check(got, *want(q, k, v, table, lens, ctx, sign * scale))
    assert (wide[:, heads * dim:] == 7.0).all()


@pytest.mark.parametrize("lens,ctx,sign", [
    ([300, 1, 257, 32, 0, 333], [0, 2300, 17, 5, 9, 100], 1.0),  # row tiles
    ([60, 850], [4500, 0], -1.0),                   # over 64 tiles of keys
    ([13] * 70, [2100] + [3] * 69, 1.0),            # more than 64 sequences
])
def test_prefill_many_tiles(lens, ctx, sign, kv_heads=16, per=8):
    """Calls of two turns of workgroups and 2048 keys and more."""
    dim = 128
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(lens))
    heads, scale = kv_heads * per, sign * dim ** -0.5
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)))
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)])
    dev = [t.cuda() for t in (k, v, table, cu.int(), sl.int())]
    wide = torch.full((sum(lens), (heads + 1) * dim), 7.0,
                      dtype=torch.bfloat16, device="cuda")
    out = wide[:, :heads * dim].unflatten(-1, (heads, dim))
    got = ops.paged_attn_prefill(
        rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim)), *dev, scale,
        out=out)
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    check(got, *want(q, k, v, table, lens, ctx, scale))
    assert (wide[:, heads * dim:] == 7.0).all()


@pytest.mark.parametrize("lens,ctx,kv_heads,per,sign", [
    ([900, 1, 257, 32, 0, 433], [0, 2300, 17, 5, 9, 100], 16, 8, 1.0),
    ([900, 1, 257, 32, 0, 433], [0, 3100, 17, 5, 9, 100], 16, 8, 1.0),  # row tiles
    ([700, 333], [0, 2100], 15, 7, 1.0),            # tokens on both sides of a wave's
    ([600, 500], [1500, 0], 32, 3, -1.0),
    ([1100], [950], 88, 1, 0.0),                    # equal weights
    ([260] * 65 + [300], [0] * 65 + [1800], 4, 2, 1.0),
    ([260] * 65 + [300], [0] * 65 + [2800], 4, 2, 1.0),   # more than 64 sequences
    ([1150], [2100], 18, 8, 1.0),                   # before and behind the lines of the
    ([1150], [2100], 14, 8, 1.0),                   # rule: 648, 504
    ([1150], [1900], 18, 8, -1.0),                  # and 3072 keys
])
def test_prefill_long_chains(lens, ctx, kv_heads, per, sign):
    """Few sequences of many tokens, and many of some: eight waves in turn."""
    test_prefill_many_tiles(lens, ctx, sign, kv_heads, per)


@pytest.mark.parametrize("kv_heads,per,dim,lens,ctx,sign", [
    (1, 1, 128, [1, 127], [127, 0], 1.0),            # a tile for some waves only
    (3, 1, 64, [33, 31, 32], [96, 64, 65], -1.0),    # edges of row and key tiles
    (2, 7, 128, [9, 30, 0, 2], [640, 1, 64, 255], 1.0),
    (1, 5, 64, [40], [984], 1.0),                    # four turns of waves
    (1, 3, 128, [100, 5], [1948, 0], -1.0),          # eight
    (2, 1, 64, [3] * 70, [150] + [0] * 69, 1.0),     # more than 64 sequences
    (1, 1, 128, [127], [1393], 1.0),                 # before 1536 keys
    (1, 1, 128, [127], [1409], 1.0),                 # from there on too few rows
    (1, 1, 128, [128], [1408], -1.0),                # and enough
])
def test_prefill_few_rows(kv_heads, per, dim, lens, ctx, sign):
    """Waves of a workgroup that share out the keys of its rows."""
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(lens))
    heads, scale = kv_heads * per, sign * dim ** -0.5
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)))
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)])
    dev = [t.cuda() for t in (k, v, table, cu.int(), sl.int())]
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    wide = torch.full((sum(lens), (heads + 1) * dim), 7.0,
                      dtype=torch.bfloat16, device="cuda")
    out = wide[:, :heads * dim].unflatten(-1, (heads, dim))
    got = ops.paged_attn_prefill(
        rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim)), *dev, scale,
        out=out)
    check(got, *want(q, k, v, table, lens, ctx, scale))
    assert (wide[:, heads * dim:] == 7.0).all()


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("lens,keys,kv_heads,per", [
    ([40, 7], [130, 0], 2, 2),                       # waves that share the keys
    ([300, 50, 9], [60, 0, 300], 16, 8),             # whole chains
    ([900, 300, 5], [450, 0, 2300], 16, 8),
    ([900, 300, 5], [450, 0, 2300], 13, 8),          # eight waves in turn
])
def test_prefill_rows_without_keys(dim, lens, keys, kv_heads, per):
    """More new tokens than keys, or no keys at all: rows in front of the first key
    are zero, the others see what they see."""
    ctx = [n - m for n, m in zip(keys, lens)]
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, 31)
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)))
    dev = [t.cuda() for t in (k, v, table, cu.int(),
                              torch.tensor(keys, dtype=torch.int32))]
    got = ops.paged_attn_prefill(
        rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim)), *dev, scale)
    sees = torch.cat([torch.arange(n) + c >= 0 for n, c in zip(lens, ctx)])
    on = [i for i, n in enumerate(keys) if n > 0]
    left = [min(lens[i], keys[i]) for i in on]
    check(got[sees.cuda()], *want(q[sees], k, v, table[on], left,
                                  [max(ctx[i], 0) for i in on], scale))
    assert (got[~sees.cuda()] == 0).all()


@pytest.mark.parametrize("lens,ctx,kv_heads,per", [
    ([9], [120], 4, 1),                 # waves that share the keys
    ([80], [300], 16, 8),               # whole chains
    ([900], [1300], 16, 8),             # eight waves in turn
])
def test_prefill_sums_whole_weights(lens, ctx, kv_heads, per):
    """One key has the weight 1 and the only value, all others a weight that bf16
    would round by nearly 2^-8 of itself: what is left of a result's error is the
    rounding of v / sum, up to 2^-9 and of either sign, so that the mean over many
    is far below 2^-12; sums of rounded weights are off by 2^-9.2 and more."""
    dim, weight = 128, 0.5 + 2.0 ** -9 - 2.0 ** -16
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, 3)
    heads, first = kv_heads * per, table[0, 0].long()
    q = torch.zeros(lens[0], heads, dim, dtype=torch.bfloat16)
    q[..., 0] = 1.0
    k.zero_()
    k[first, :, 0, 0] = 1.0
    only = torch.rand(kv_heads, dim, generator=torch.Generator().manual_seed(
        per)).add_(1.0).to(torch.bfloat16)
    v.zero_()
    v[first, :, 0] = only
    got = ops.paged_attn_prefill(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor([0, lens[0]], dtype=torch.int32, device="cuda"),
        torch.tensor([lens[0] + ctx[0]], dtype=torch.int32, device="cuda"),
        -math.log(weight)).double().cpu()
    keys = ctx[0] + 1 + torch.arange(lens[0])
    ref = only.double().repeat_interleave(per, 0)[None] \
        / (1.0 + (keys.double() - 1.0) * weight)[:, None, None]
    off = got / ref - 1.0
    assert off.abs().max() < 2.0 ** -8
    assert off.mean().abs() < 2.0 ** -12


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("ctx", [[3, 0], [2600, 900]])      # whole; in parts
def test_prefill_leaves_other_rows(dim, ctx):
    """Rows of q and out outside of every prompt (cu_q) are not written."""
    lens, heads = [5, 9], 4
    rows, k, v, table = make(lens, ctx, 1, heads, dim, 21)
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    pad = torch.randn(2, heads, dim).to(torch.bfloat16)
    tail = torch.randn(6, heads, dim).to(torch.bfloat16)
    cu = torch.tensor([2, 7, 16], dtype=torch.int32)
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)], dtype=torch.int32)
    dev = [t.cuda() for t in (k, v, table, cu, sl)]
    qd, scale = torch.cat([pad, q, tail]).cuda(), dim ** -0.5
    ref, big = want(q, k, v, table, lens, ctx, scale)
    out = torch.full_like(qd, 7.0)
    ops.paged_attn_prefill(qd, *dev, scale, out=out)
    check(out[2:16], ref, big)
    assert (out[:2] == 7.0).all() and (out[16:] == 7.0).all()
    out = torch.full((22, heads * dim), 7.0, device="cuda")
    H.capped_attn(qd.flatten(1), *dev[:3], *dev[3:], heads, scale, 0.0, out)
    check(out[2:16].unflatten(-1, (heads, dim)), ref, big)
    assert (out[:2] == 7.0).all() and (out[16:] == 7.0).all()


def test_prefill_standout_scores():
    """Scores far apart: the running maximum moves within and across tiles."""
    lens, ctx = [40], [150]
    rows, k, v, table = make(lens, ctx, 1, 2, 128, 5)
    k[table[0, 4], 0, 3] *= 30.0
    k[table[0, 9], 0, 15] *= 60.0
    q = rows[:, :256].unflatten(-1, (2, 128))
    got = ops.paged_attn_prefill(
        q.contiguous().cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor([0, 40], dtype=torch.int32, device="cuda"),
        torch.tensor([190], dtype=torch.int32, device="cuda"), 0.3)
    check(got, *want(q, k, v, table, lens, ctx, 0.3))


def test_prefill_needs_no_host():
    """No list of tiles, no wait: the call can be captured, and a replay
    follows the lengths on the device."""
    rows, k, v, table = make([40, 24], [20, 0], 2, 2, 128, 9)
    q = rows[:, :512].unflatten(-1, (4, 128)).contiguous()
    dev = [t.cuda() for t in (q, k, v, table)]
    cu = torch.tensor([0, 40, 64], dtype=torch.int32, device="cuda")
    sl = torch.tensor([60, 24], dtype=torch.int32, device="cuda")
    out = torch.empty_like(dev[0])
    ops.paged_attn_prefill(*dev, cu, sl, 0.1, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.paged_attn_prefill(*dev, cu, sl, 0.1, out=out)
    for lens, ctx in (([40, 24], [20, 0]), ([30, 34], [10, 14])):
        cu.copy_(torch.tensor([0, lens[0], 64]))
        sl.copy_(torch.tensor([n + c for n, c in zip(lens, ctx)]))
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        check(out, *want(q, k, v, table, lens, ctx, 0.1))


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("keys,kv_heads,per", [
    ([1], 1, 1), ([15, 16, 17, 31, 32, 33], 2, 8),          # pages and tiles
    ([127, 128, 129, 255, 256, 257, 700], 4, 7),            # waves
    ([2049, 5, 4500], 3, 2), ([9001], 2, 4),                # parts
    ([40 + 7 * i for i in range(70)], 4, 3),                # many pairs
    ([33 + 61 * (i % 7) for i in range(29)] + [6000], 3, 2),  # one long one
    ([18000, 33], 1, 5),              # over 32 tiles of one wave
])
def test_decode_edges(dim, keys, kv_heads, per):
    ctx = [n - 1 for n in keys]
    rows, k, v, table = make([1] * len(keys), ctx, kv_heads, per, dim,
                             sum(keys) + dim)
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    sl = torch.tensor(keys, dtype=torch.int32)
    dev = [t.cuda() for t in (k, v, table, sl)]
    qd = rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim))
    wide = torch.full((len(keys), (heads + 1) * dim), 7.0,
                      dtype=torch.bfloat16, device="cuda")
    out = wide[:, :heads * dim].unflatten(-1, (heads, dim))
    for sign in (1.0, -1.0):
        got = ops.paged_attn_decode(qd, *dev, sign * scale, out=out)
        check(got, *want(q, k, v, table, [1] * len(keys), ctx, sign * scale))
    assert (wide[:, heads * dim:] == 7.0).all()


def test_narrow_prefill_has_gradients():
    """64-wide prompt rows: wanted gradients come from torch's operations."""
    lens, ctx, heads, dim = [5, 9], [3, 20], 4, 64
    rows, k, v, table = make(lens, ctx, 2, 2, dim, 23)
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim)).contiguous()
    cu = torch.tensor([0, 5, 14], dtype=torch.int32, device="cuda")
    sl = torch.tensor([8, 29], dtype=torch.int32, device="cuda")
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = ops.paged_attn_prefill(qd, kd, vd, table.cuda(), cu, sl, 0.1)
    assert out.requires_grad
    out.float().sum().backward()
    for t in (qd, kd, vd):
        assert t.grad is not None and (t.grad != 0).any()
    with torch.no_grad():
        got = ops.paged_attn_prefill(qd, kd, vd, table.cuda(), cu, sl, 0.1)
    check(got, *want(q, k, v, table, lens, ctx, 0.1))


@pytest.mark.parametrize("ctx", [[3, 0], [2600, 900]])      # whole; in parts
@pytest.mark.parametrize("flat", [False, True])
def test_prefill_shapes_of_results(ctx, flat):
    """Results as rows of heads * dim, with more rows than there are queries;
    caches of different sizes."""
    lens, heads, dim = [5, 9], 4, 128
    rows, k, v, table = make(lens, ctx, 1, heads, dim, 22)
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim)).contiguous()
    cu = torch.tensor([0, 5, 14], dtype=torch.int32)
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)], dtype=torch.int32)
    more = torch.cat([v, v[:2]])
    out = torch.full((20, heads * dim), 7.0, dtype=torch.bfloat16,
                     device="cuda")
    ops.paged_attn_prefill(
        *(t.cuda() for t in (q, k, more, table, cu, sl)), 0.1,
        out=out if flat else out.unflatten(-1, (heads, dim)))
    check(out[:14].unflatten(-1, (heads, dim)),
          *want(q, k, v, table, lens, ctx, 0.1))
    assert (out[14:] == 7.0).all()


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("odd", ["caches", "rows", "all"])
@pytest.mark.parametrize("decode", [True, False])
def test_any_alignment(dim, odd, decode):
    """Caches, queries and results at odd addresses (2 B) and row strides."""
    lens, ctx = ([1, 1], [70, 3000]) if decode else ([5, 20], [2100, 40])
    heads, scale = 8, dim ** -0.5
    rows, k, v, table = make(lens, ctx, 2, 4, dim, dim)
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)]).int().cuda()

    def shifted(t, on):
        if not on:
            return t.cuda()
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        flat[1:].copy_(t.flatten())
        return flat[1:].view(t.shape)
    kd, vd = (shifted(t, odd != "rows") for t in (k, v))
    extra = odd != "caches"
    wide = torch.full((sum(lens), heads * dim + extra), 7.0,
                      dtype=torch.bfloat16, device="cuda")
    qd = wide.clone()[:, extra:].unflatten(-1, (heads, dim)).copy_(q)
    out = wide[:, extra:].unflatten(-1, (heads, dim))
    if decode:
        got = ops.paged_attn_decode(qd, kd, vd, table.cuda(), sl, scale,
                                    out=out)
    else:
        got = ops.paged_attn_prefill(qd, kd, vd, table.cuda(), cu, sl, scale,
                                     out=out)
    check(got, *want(q, k, v, table, lens, ctx, scale))
    assert (wide[:, :extra] == 7.0).all()


@pytest.mark.parametrize("keys,per", [
    ([777], 4), ([200], 8), ([5001], 1), ([600 + 33 * i for i in range(24)], 4),
    ([40 + 70 * i for i in range(70)], 7)])
def test_decode_weights(keys, per):
    """The softmax weights of 128-wide heads have 16 bits: what the results are
    off by is their rounding to bf16 (half a step of 2^-7 of their power of two),
    and 2^-15 of the weighted sum of |v| for the weights and 32-bit sums."""
    ctx = [n - 1 for n in keys]
    rows, k, v, table = make([1] * len(keys), ctx, 4, per, 128, sum(keys))
    q = rows[:, :512 * per].unflatten(-1, (4 * per, 128))
    got = ops.paged_attn_decode(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor(keys, dtype=torch.int32, device="cuda"), 0.13)
    ref, big = want(q, k, v, table, [1] * len(keys), ctx, 0.13)
    over = (got.double().cpu() - ref).abs() - 2.0 ** -15 * big \
        - 2.0 ** (torch.floor(torch.log2(ref.abs())) - 8)
    assert over.max() <= 0, f"over by {over.max():.3g}"


@pytest.mark.parametrize("keys,kv_heads,per", [
    ([1, 16, 9], 12, 1), ([64] * 29 + [17, 3], 12, 1),       # shuffled
    ([17] * 24, 12, 1), ([65, 64, 1] * 10, 12, 2),           # streamed
    ([33 * i + 1 for i in range(64)], 12, 1),                # by two waves
    ([5000] + [40] * 29, 3, 1)])                             # never in parts
def test_narrow_decode_forms(keys, kv_heads, per):
    """64-wide heads on both sides of the lines between their forms."""
    ctx = [n - 1 for n in keys]
    rows, k, v, table = make([1] * len(keys), ctx, kv_heads, per, 64, sum(keys))
    q = rows[:, :kv_heads * per * 64].unflatten(-1, (kv_heads * per, 64))
    got = ops.paged_attn_decode(
        q.cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor(keys, dtype=torch.int32, device="cuda"), 0.125)
    check(got, *want(q, k, v, table, [1] * len(keys), ctx, 0.125))


def on_litter(call, size, fill):
    """call(), which asks for `size` bytes, on memory that holds `fill`, and that
    memory: the allocator gives a freed block between two that stay to the next one
    who asks for as much."""
    held = [torch.full((size // 8,), fill, dtype=torch.int64, device="cuda")
            for _ in range(8)]
    for i in range(len(held)):
        at, held[i] = held[i].data_ptr(), None
        call()
        held[i] = torch.empty(size // 8, dtype=torch.int64, device="cuda")
        if held[i].data_ptr() == at:
            return held[i]
    assert False, "scratch lies elsewhere"


def over_litter(call, out, sl, lengths, ref):
    """call() into out, for `lengths` in sl, over scratch of several values: alone,
    and in replays of a graph, to the same bits. The first lengths are split."""
    call()
    was = torch.cuda.memory_stats()["requested_bytes.all.allocated"]
    call()
    size = torch.cuda.memory_stats()["requested_bytes.all.allocated"] - was
    assert size > 0
    refs = {tuple(n): ref(n) for n in lengths}
    for fill in (0, -1, 0x7f7f7f7f7f7f7f01):
        out.fill_(3.0)
        scratch = on_litter(call, size, fill)
        assert (scratch != fill).any()             # parts were in it
        check(out, *refs[tuple(lengths[0])])
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            scratch = on_litter(call, size, fill)
        for now in lengths:
            sl.copy_(torch.tensor(now))
            out.fill_(3.0)
            graph.replay()
            got = out.clone()
            assert now != lengths[0] or (scratch != fill).any()
            call()
            assert torch.equal(got, out)
            check(got, *refs[tuple(now)])


@pytest.mark.parametrize("dim,keys,kv_heads,per", [
    (128, [12 * 32, 12 * 32 + 1, 17 * 32], 8, 4),     # where parts begin
    (128, [32 * 32 + 1, 65 * 32, 8 * 65 * 32 + 5], 1, 7),   # eight of them, more
    (64, [16 * 32, 16 * 32 + 1, 21 * 32, 31, 2000], 16, 1),
    (128, [23 * 32, 23 * 32 + 1, 3000, 40] * 3, 8, 3),      # 96 pairs
    (128, [24 * 32, 24 * 32 + 1, 3000, 40] * 3, 8, 1),
    (128, [40 * 32, 40 * 32 + 1, 4000, 9, 700] * 3, 8, 2),  # 120
    (128, [32 * 32 + 1, 4200, 900, 40] * 3, 8, 4),          # in a longer table
    (64, [19 * 32, 19 * 32 + 1, 2000, 700] * 2, 12, 1),
    (64, [39 * 32, 39 * 32 + 1, 2000, 9] * 4, 12, 2)])      # 192
def test_decode_parts_meet(dim, keys, kv_heads, per):
    """Sequences split into parts, whose last workgroup merges: over scratch that
    held anything before, and in replays of a captured step whose lengths change."""
    ctx = [n - 1 for n in keys]
    rows, k, v, table = make([1] * len(keys), ctx, kv_heads, per, dim, sum(keys))
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim)).contiguous()
    dev = [t.cuda() for t in (q, k, v, table)]
    sl = torch.tensor(keys, dtype=torch.int32, device="cuda")
    out = torch.empty_like(dev[0])
    over_litter(
        lambda: ops.paged_attn_decode(*dev, sl, scale, out=out), out, sl,
        [keys, keys, [max(1, n // 2) for n in keys], keys],
        lambda lens: want(q, k, v, table, [1] * len(lens), [n - 1 for n in lens],
                          scale))


def test_decode_standout_scores():
    rows, k, v, table = make([1, 1], [900, 350], 1, 2, 128, 5)
    k[table[0, 4], 0, 3] *= 30.0
    k[table[0, 50], 0, 15] *= 60.0
    k[table[1, 21], 0, 13] *= 90.0            # the last key of all
    q = rows[:, :256].unflatten(-1, (2, 128))
    got = ops.paged_attn_decode(
        q.contiguous().cuda(), k.cuda(), v.cuda(), table.cuda(),
        torch.tensor([901, 351], dtype=torch.int32, device="cuda"), 0.3)
    check(got, *want(q, k, v, table, [1, 1], [900, 350], 0.3))


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("width", [0, 1])
def test_decode_without_keys(dim, width):
    """Sequences of no keys, in tables with and without columns: zeros."""
    k = torch.randn(3, 2, PAGE, dim, device="cuda").to(torch.bfloat16)
    q = torch.randn(3, 8, dim, device="cuda").to(torch.bfloat16)
    table = torch.zeros(3, width, dtype=torch.int32, device="cuda")
    sl = torch.zeros(3, dtype=torch.int32, device="cuda")
    assert (ops.paged_attn_decode(q, k, k, table, sl, 0.1) == 0).all()
    for sink in (None, torch.zeros(8, device="cuda")):
        out = torch.full((3, 8, dim), 7.0, device="cuda")
        H.capped_attn(q.flatten(1), k, k, table, None, sl, 8, 0.1, 0.0, out,
                      sink=sink)
        assert (out == 0).all()


@pytest.mark.parametrize("dim,seqs,kv_heads,per", [
    (128, 12, 8, 4), (64, 12, 8, 4), (64, 32, 6, 4), (128, 32, 4, 1),
    (64, 16, 12, 1), (128, 100, 8, 2)])
def test_decode_without_keys_of_many(dim, seqs, kv_heads, per):
    """Tables without columns, pairs of sequence and key head by tens: zeros."""
    k = torch.randn(3, kv_heads, PAGE, dim, device="cuda").to(torch.bfloat16)
    q = torch.randn(seqs, kv_heads * per, dim, device="cuda").to(torch.bfloat16)
    table = torch.zeros(seqs, 0, dtype=torch.int32, device="cuda")
    sl = torch.zeros(seqs, dtype=torch.int32, device="cuda")
    out = torch.full_like(q, 7.0)
    ops.paged_attn_decode(q, k, k, table, sl, 0.1, out=out)
    assert (out == 0).all()


@pytest.mark.parametrize("tokens,keys,width,decode", [
    (40, 30, 64, False), (40, 0, 64, False),         # parts that meet
    (60, 20, 256, False),                            # parts of a kernel of merges
    (40, 30, 10, False), (300, 250, 40, False),      # few rows, a group of waves,
    (900, 700, 56, False),                           # two of them
    (1, 0, 64, True)])
def test_sinks_of_no_weight(tokens, keys, width, decode):
    """A sink of -inf: rows without keys are zero, the others as without it."""
    heads, kv_heads, dim, none = 32, 8, 128, min(keys, tokens) - tokens
    g = torch.Generator().manual_seed(tokens)
    k, v = (torch.randn(max(width, 1), kv_heads, PAGE, dim, generator=g)
            .to(torch.bfloat16).cuda() for _ in range(2))
    q = torch.randn(tokens, heads * dim, generator=g).to(torch.bfloat16).cuda()
    table = torch.arange(width, dtype=torch.int32, device="cuda")[None]
    cu = torch.tensor([0, tokens], dtype=torch.int32, device="cuda")
    sl = torch.tensor([keys], dtype=torch.int32, device="cuda")
    outs = []
    for value in (-math.inf, -1e30):
        sink = torch.full((heads,), value, device="cuda")
        out = torch.full((tokens, heads, dim), 7.0, device="cuda")
        H.capped_attn(q, k, v, table, None if decode else cu, sl, heads, 0.1, 0.0,
                      out, sink=sink)
        assert (out[:-none] == 0).all() and torch.isfinite(out).all()
        outs.append(out)
    assert torch.equal(*outs)


OPTIONS = {
    "plain": {},
    "window": dict(window=50),
    "window + kept": dict(window=33, keep_first=5),
    "window of one": dict(window=1, keep_first=70),
    "chunks": dict(window=48, chunked=True),
    "sink": dict(window=64, sink=True),
    "cap": dict(cap=5.0),
    "large cap": dict(cap=50.0),
    "head scales": dict(head_scale=True, cap=3.0, sink=True),
    "signs": dict(head_scale=True, window=100),
}


@pytest.mark.parametrize("opts", list(OPTIONS))
@pytest.mark.parametrize("dim,bf16_out", [(64, True), (128, False),
                                          (128, True)])
@pytest.mark.parametrize("lens,ctx,kv_heads,per,decode", [
    ([1, 33, 64, 130], [16, 31, 100, 0], 2, 4, False),
    ([5, 2], [1500, 3000], 1, 2, False),                   # parts
    ([1, 2, 5, 33] * 6, [100, 31, 400, 0] * 6, 2, 4, False),   # few keys, many
    ([1] * 5, [0, 15, 31, 127, 400], 3, 4, True),
    ([1, 1], [2000, 4095], 1, 32, True),                   # parts
    ([1] * 30, [20 + 31 * i for i in range(29)] + [3500], 3, 2, True),
])
def test_options(dim, bf16_out, lens, ctx, kv_heads, per, decode, opts):
    """Windows, kept keys, chunks, sinks, caps and head multipliers, fp32 and
    bf16 results, keys read as values; the weights have 32 bits."""
    opts = dict(OPTIONS[opts])
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(ctx) + dim)
    heads, T, scale = kv_heads * per, sum(lens), 1.5 * dim ** -0.5
    g = torch.Generator().manual_seed(3)
    for name in ("sink", "head_scale"):
        if opts.get(name):
            opts[name] = torch.randn(heads, generator=g)
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)], dtype=torch.int32)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32)
    q = rows[:, :heads * dim]
    for values in (v, k):
        kd = k.cuda()
        vd = kd if values is k else v.cuda()
        wide = torch.full((T, (heads + 1) * dim), 7.0, device="cuda",
                          dtype=torch.bfloat16 if bf16_out else torch.float32)
        out = wide[:, :heads * dim]
        H.capped_attn(rows.cuda()[:, :heads * dim], kd, vd, table.cuda(),
                      None if decode else cu.cuda(), sl.cuda(), heads, scale,
                      opts.get("cap", 0.0), out, opts.get("window", 0),
                      *(opts[x].cuda() if x in opts else None
                        for x in ("sink",)), opts.get("keep_first", 0),
                      opts["head_scale"].cuda() if "head_scale" in opts
                      else None, opts.get("chunked", False))
        ref, big = want(q.unflatten(-1, (heads, dim)), k, values, table, lens,
                        ctx, scale, **opts)
        off = (out.unflatten(-1, (heads, dim)).double().cpu() - ref).abs()
        over = off - 2.0 ** -17 * big - (2.0 ** -8 * ref.abs() if bf16_out
                                         else 0.0)
        assert over.max() <= 1e-6, f"off by {off.max():.3g}"
        assert (wide[:, heads * dim:] == 7.0).all()


@pytest.mark.parametrize("opts", ["window", "cap", "sink", "chunks", "window + kept"])
@pytest.mark.parametrize("dim,lens,ctx,kv_heads,per,decode", [
    (128, [1] * 6, [0, 14, 15, 16, 31, 47], 4, 4, True),
    (128, [1] * 4, [15, 63, 64, 100], 1, 32, True),
    (64, [1] * 5, [0, 15, 16, 31, 63], 2, 16, True),
    (128, [16, 1, 40], [0, 30, 7], 2, 8, False),
    (128, [48, 49, 33] * 5, [0, 0, 15] * 5, 8, 1, False),
    (64, [16, 1, 40], [0, 30, 7], 3, 2, False),
])
def test_options_over_few_keys(dim, lens, ctx, kv_heads, per, decode, opts):
    """Where one tile or two hold all keys, on both sides of what the kernels of 16
    rows a wave are left."""
    test_options(dim, False, lens, ctx, kv_heads, per, decode, opts)


@pytest.mark.parametrize("kv_heads,per,dim,lens,ctx,sign", [
    (8, 4, 128, [650], [0], 1.0),                    # waves in two groups
    (8, 4, 128, [60, 700, 1], [900, 0, 130], -1.0),  # tiles for one group only
    (12, 3, 128, [1500], [0], 1.0),                  # more workgroups than CUs
    (12, 1, 64, [448, 64, 65, 384] * 2 + [300], [0, 0, 1, 5] * 2 + [0], 1.0),
    (8, 4, 128, [260, 64, 33, 250, 1, 320, 300], [0, 90, 4, 3, 270, 0, 0], 1.0),
    (8, 4, 128, [40] * 40, [i % 5 * 60 for i in range(40)], 1.0),
])
def test_prefill_orders_and_groups(kv_heads, per, dim, lens, ctx, sign):
    """Row tiles in the order of their chains, in one turn, two and more; groups
    of waves that share out the keys of their rows."""
    test_prefill_few_rows(kv_heads, per, dim, lens, ctx, sign)


@pytest.mark.parametrize("kv_heads,per,dim", [(3, 3, 128), (5, 5, 64), (7, 6, 128),
                                               (1, 11, 64), (2, 25, 128), (1, 71, 64)])
def test_prefill_heads_of_no_power_of_two(kv_heads, per, dim):
    """Rows and workgroups are divided by head counts with a multiplication."""
    test_prefill_few_rows(kv_heads, per, dim, [257, 1, 0, 130, 333], [40, 700, 5, 0, 90],
                          1.0)


@pytest.mark.parametrize("kv_heads,per,dim,lens,ctx,sign", [
    (8, 4, 128, [200, 90, 333, 1, 150, 0, 257] * 3, [7, 60, 5] * 7, 1.0),   # over three
    (8, 4, 128, [200, 90, 333, 1, 150, 0, 257] * 2, [7, 60, 5, 9] * 3 + [3, 0], -1.0),
    (8, 4, 128, [260, 301, 330, 280, 270, 289], [0, 100, 3, 0, 0, 20], -1.0),   # under two
    (8, 4, 128, [64, 1, 0, 65, 33], [0, 9, 5, 0, 3], 1.0),                  # less than one
    (12, 1, 64, [406, 300, 430] * 2 + [33, 64] * 4, [0, 18] * 7, 1.0),      # of 64-wide heads
    (12, 1, 64, [58, 115, 97, 31, 64, 0, 60] * 2, [3, 1] * 7, -1.0),
])
def test_prefill_order_of_turns(kv_heads, per, dim, lens, ctx, sign):
    """Row tiles of one turn of the CUs as they are, of up to two folded, of more."""
    test_prefill_few_rows(kv_heads, per, dim, lens, ctx, sign)


@pytest.mark.parametrize("kv_heads,per,dim,lens,ctx,sign", [
    (2, 4, 128, [50, 60, 0, 130, 20], [2500, 100, 30, 0, 700], 1.0),
    (4, 4, 128, [3] * 68 + [64, 1], [0, 90] * 34 + [1300, 1100], -1.0),
    (3, 5, 128, [9, 77], [1015, 1016], 1.0),         # parts of eight tiles, and nine
    (1, 1, 128, [60, 1], [8200, 40], 1.0),          # sixteen parts
    (12, 1, 64, [100, 5, 33], [1500, 0, 450], 1.0),
    (8, 4, 128, [70], [3000], -1.0),                 # one sequence
    (8, 4, 128, [300], [2000], 1.0),                 # in parts of two groups
    (4, 7, 128, [1, 197, 0, 261], [900, 1750, 3, 524], 1.0),
    (8, 4, 128, [600, 20, 33], [0, 1500, 100], 1.0),
])
def test_prefill_parts_by_length(kv_heads, per, dim, lens, ctx, sign):
    """Keys split by a sequence's own length, over 64 sequences and more."""
    test_prefill_few_rows(kv_heads, per, dim, lens, ctx, sign)


@pytest.mark.parametrize("kv_heads,per,dim,lens,ctx", [
    (2, 4, 128, [50, 60, 9], [3900, 100, 700]),      # parts of a kernel of merges
    (8, 4, 128, [60, 200, 40], [4000, 100, 700]),    # six of two groups
    (8, 4, 128, [300], [2000]),                      # three of one sequence
    (12, 1, 64, [420], [900]),                       # one group
])
def test_prefill_parts_meet(kv_heads, per, dim, lens, ctx):
    """Parts that the last one merges: over scratch that held anything before, and
    in replays of a captured call whose lengths change, to the same bits."""
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(ctx))
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim)).contiguous()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    dev = [t.cuda() for t in (q, k, v, table)]
    keys = [[n + c // by for n, c in zip(lens, ctx)] for by in (1, 3)]
    sl = torch.tensor(keys[0]).int().cuda()
    out = torch.empty_like(dev[0])
    over_litter(
        lambda: ops.paged_attn_prefill(*dev, cu, sl, scale, out=out), out, sl,
        [keys[0], keys[0], keys[1], keys[0]],
        lambda now: want(q, k, v, table, lens, [m - n for m, n in zip(now, lens)],
                         scale))


@pytest.mark.parametrize("kv_heads,per,dim,lens,keys", [
    (4, 4, 128, [20, 33, 40, 31, 9], [3840, 3785, 3900, 3780, 100]),
    (2, 7, 128, [70, 30, 18, 1], [3264, 3901, 3584, 3905]),
    (1, 1, 128, [1, 128, 129, 5, 40, 64], [4096, 3840, 4090, 3901, 3111, 64]),
    (8, 4, 128, [60, 40], [4096, 3841]),
    # two groups of waves, the last part merges: four parts, six, eight, and one of 13 tiles
    (8, 4, 128, [60, 200, 40], [2113, 700, 90]),
    (8, 4, 128, [60, 200, 40], [4060, 300, 4033]),
    (8, 4, 128, [60, 200, 40, 1], [7100, 8190, 40, 6145]),
    (4, 7, 128, [40, 33, 120, 9], [832, 833, 400, 9]),
    # one group, up to four; in a turn by longer parts, or none
    (8, 4, 128, [500, 60, 90], [1800, 2049, 90]),
    (8, 4, 128, [618, 647], [1212, 1288]),
    (4, 4, 128, [1000, 1100], [1000, 1100]),
    (12, 1, 64, [300, 200, 129], [1800, 1537, 300]),
    # few rows of many key heads
    (32, 1, 128, [10, 12, 9], [2000, 700, 3454]),
])
def test_prefill_parts_of_several(kv_heads, per, dim, lens, keys):
    """Parts by each sequence's length, which the last one merges where row tiles are
    many. Calls alone and among others end their parts in different orders, and all of
    them have the same bits."""
    ctx = [n - m for n, m in zip(keys, lens)]
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, sum(keys))
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim)).contiguous()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    dev = [t.cuda() for t in (q, k, v, table)]
    sl = torch.tensor(keys).int().cuda()
    outs = [torch.empty_like(dev[0]) for _ in range(64)]
    for i, out in enumerate(outs):
        if i % 8 == 0:
            torch.cuda.synchronize()
        ops.paged_attn_prefill(*dev, cu, sl, scale, out=out)
    check(outs[0], *want(q, k, v, table, lens, ctx, scale))
    for out in outs[1:]:
        assert torch.equal(out, outs[0])


@pytest.mark.parametrize("opts", ["cap", "window", "sink"])
def test_prefill_parts_with_options(opts):
    test_prefill_options_of_forms([40, 3, 200], [1700, 5, 600], 2, 4, 900, opts)


def test_prefill_groups_without_keys():
    test_prefill_rows_without_keys(128, [700, 90, 5], [100, 660, 0], 8, 4)


@pytest.mark.parametrize("opts", ["cap", "head scales", "window", "sink"])
@pytest.mark.parametrize("lens,ctx,kv_heads,per,window", [
    ([400, 390], [260, 30], 8, 4, 630),              # waves in two groups
    ([30, 9, 128], [600, 0, 1], 2, 4, 700),          # few rows: up to 768 keys
    ([130], [900], 4, 4, 640),
])
def test_prefill_options_of_forms(lens, ctx, kv_heads, per, window, opts):
    name = opts + str(window)
    OPTIONS[name] = dict(OPTIONS[opts])
    if "window" in OPTIONS[name]:
        OPTIONS[name].update(window=window, keep_first=9)
    try:
        test_options(128, False, lens, ctx, kv_heads, per, False, name)
    finally:
        del OPTIONS[name]


def test_prefill_without_prompts():
    """cu_q of one entry, or of none, names no rows: out stays as it is."""
    rows, k, v, table = make([300], [0], 1, 4, 128, 34)
    q = rows[:, :512].unflatten(-1, (4, 128)).cuda()
    for n in (1, 0):
        empty = torch.zeros(n, dtype=torch.int32, device="cuda")
        out = torch.full_like(q, 7.0)
        ops.paged_attn_prefill(q, k.cuda(), v.cuda(), table[:0].cuda(), empty,
                               empty[:0], 0.1, out=out)
        assert (out == 7.0).all()


@pytest.mark.parametrize("seqs,kv_heads,per,keys,width", [
    (191, 4, 2, 70, 512), (192, 4, 2, 70, 512),      # parts | whole
    (191, 4, 2, 250, 16), (192, 4, 2, 250, 16), (192, 4, 2, 250, 17),  # waves
    (3, 2, 8, 32, 2), (3, 2, 8, 33, 3)])
def test_decode_forms(seqs, kv_heads, per, keys, width):
    """Both sides of the lines between parts and waves of 128-wide heads."""
    lens, ctx, scale = [1] * seqs, [(keys * (i + 1)) // seqs - 1 if keys > 40
                                    else keys - 1 for i in range(seqs)], 0.088
    ctx = [max(c, 0) for c in ctx]
    rows, k, v, table = make(lens, ctx, kv_heads, per, 128, 35)
    wide = torch.zeros(seqs, max(width, table.shape[1]), dtype=torch.int32)
    wide[:, :table.shape[1]] = table
    q = rows[:, :kv_heads * per * 128].unflatten(-1, (kv_heads * per, 128))
    sl = torch.tensor(ctx, dtype=torch.int32) + 1
    got = ops.paged_attn_decode(q.cuda(), k.cuda(), v.cuda(), wide.cuda(),
                                sl.cuda(), scale)
    check(got, *want(q, k, v, table, lens, ctx, scale))
