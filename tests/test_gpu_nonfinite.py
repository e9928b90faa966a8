"""A NaN or an infinite entry of a query, a key or a value reaches the same results
whether the keys are split over workgroups or not: those that 64-bit arithmetic
makes non-finite, and no others."""
import math

import pytest
import torch

from test_gpu_attention import make, want
from test_gpu_decay import features, recur
from xllm_service_amd import ops
from xllm_service_amd.ops import hybrid as H

pytestmark = pytest.mark.gpu

# new tokens, cached tokens, key heads, query heads per key head: too few keys
# or too many pairs to be split, then few pairs over many keys
DECODE = {"whole": ([1] * 3, [40, 300, 90], 2, 4),
          "split": ([1, 1], [2600, 900], 2, 4)}
PREFILL = {"whole": ([9, 33], [40, 70], 2, 4),
           "split": ([5, 3], [2600, 900], 1, 4)}


def plant(bad, where, rows, k, v, table, dim):
    """One entry: of the first query head's of the last row, or of the second
    cached key or value of the last sequence (which all its rows see)."""
    if where == "q":
        rows[-1, 5] = bad
    else:
        (k if where == "k" else v)[table[-1, 0], 0, 1, dim // 2] = bad


def agree(got, ref):
    got = got.double().cpu()
    assert torch.equal(torch.isfinite(got), torch.isfinite(ref))
    ok = torch.isfinite(ref)
    assert (got[ok] - ref[ok]).abs().max() < 0.05


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("how", ["whole", "split"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("entry", ["decode", "prefill", "capped decode",
                                   "capped prefill"])
def test_paged(entry, dim, how, where, bad):
    decode = "decode" in entry
    lens, ctx, kv_heads, per = (DECODE if decode else PREFILL)[how]
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, 7)
    plant(bad, where, rows, k, v, table, dim)
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)]).int().cuda()
    ref, _ = want(q, k, v, table, lens, ctx, scale)
    dev = [t.cuda() for t in (k, v, table)]
    qd = rows.cuda()[:, :heads * dim]
    if "capped" in entry:
        out = torch.zeros(sum(lens), heads, dim, device="cuda")
        H.capped_attn(qd, *dev, None if decode else cu, sl, heads, scale, 0.0,
                      out)
        agree(out, ref)
    elif decode:
        agree(ops.paged_attn_decode(qd.unflatten(-1, (heads, dim)), *dev, sl,
                                    scale), ref)
    else:
        agree(ops.paged_attn_prefill(qd.unflatten(-1, (heads, dim)), *dev, cu,
                                     sl, scale), ref)


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("dim,lens,ctx,kv_heads,per", [
    (128, [9, 33], [40, 170], 2, 4), (64, [9, 33], [40, 170], 2, 4),
    (128, [610, 500], [40, 1600], 32, 3)])
def test_prompts(dim, lens, ctx, kv_heads, per, where, bad):
    """Waves that share the keys of few rows, and eight of long prompts in turn."""
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, 7)
    plant(bad, where, rows, k, v, table, dim)
    heads, scale = kv_heads * per, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)]).int().cuda()
    dev = [t.cuda() for t in (k, v, table)]
    ref, _ = want(q, k, v, table, lens, ctx, scale)
    agree(ops.paged_attn_prefill(
        rows.cuda()[:, :heads * dim].unflatten(-1, (heads, dim)), *dev, cu, sl,
        scale), ref)


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("where", ["q", "k"])
@pytest.mark.parametrize("how", ["whole", "split"])
@pytest.mark.parametrize("dim", [64, 128, 96])
@pytest.mark.parametrize("decode", [True, False])
def test_capped_scores(decode, dim, how, where, bad):
    """Scores of every size meet the cap: a NaN stays one, an infinite one
    becomes the cap (96: the kernel for other widths)."""
    lens, ctx, kv_heads, per = (DECODE if decode else PREFILL)[how]
    rows, k, v, table = make(lens, ctx, kv_heads, per, dim, 8)
    plant(bad, where, rows, k, v, table, dim)
    heads, cap, scale = kv_heads * per, 3.0, dim ** -0.5
    q = rows[:, :heads * dim].unflatten(-1, (heads, dim))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)]).int().cuda()
    out = torch.zeros(sum(lens), heads, dim, device="cuda")
    H.capped_attn(rows.cuda()[:, :heads * dim],
                  *(t.cuda() for t in (k, v, table)),
                  None if decode else cu, sl, heads, scale, cap, out)
    agree(out, want(q, k, v, table, lens, ctx, scale, cap=cap)[0])


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("where", ["q", "key", "tail"])
@pytest.mark.parametrize("keys", [[30, 20], [90, 2600]])
def test_latent(keys, where, bad):
    g = torch.Generator().manual_seed(5)
    W, r, heads, scale = 576, 512, 16, 192 ** -0.5
    need = [-(-n // 16) for n in keys]
    cache = torch.randn(sum(need), 16, W, generator=g).to(torch.bfloat16)
    table = torch.zeros(2, max(need), dtype=torch.int32)
    table[0, :need[0]] = torch.arange(need[0])
    table[1, :need[1]] = torch.arange(need[0], sum(need))
    q = torch.randn(2, heads, W, generator=g).to(torch.bfloat16)
    if where == "q":
        q[1, 3, 7] = bad
    else:
        cache[table[1, 0], 1, 40 if where == "key" else 560] = bad
    out = torch.zeros(2, heads, r, device="cuda")
    H.latent_attn(q.cuda(), cache.cuda(), table.cuda(), None,
                  torch.tensor(keys, dtype=torch.int32, device="cuda"), scale,
                  r, out)
    ref = []
    for s, n in enumerate(keys):
        k = cache[table[s, :need[s]].long()].reshape(-1, W)[:n].double()
        ref.append(torch.softmax(q[s].double() @ k.t() * scale, -1) @ k[:, :r])
    agree(out, torch.stack(ref))


@pytest.mark.parametrize("how", ["whole", "split"])
@pytest.mark.parametrize("decode", [True, False])
def test_nan_factors(decode, how):
    """A NaN scale, or the NaN multiplier or sink of one head."""
    lens, ctx, kv_heads, per = (DECODE if decode else PREFILL)[how]
    rows, k, v, table = make(lens, ctx, kv_heads, per, 128, 9)
    heads = kv_heads * per
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0))).int().cuda()
    sl = torch.tensor([n + c for n, c in zip(lens, ctx)]).int().cuda()
    dev = [t.cuda() for t in (k, v, table)]
    q = rows.cuda()[:, :heads * 128]
    for cap in (0.0, 5.0):
        mult = torch.ones(heads, device="cuda")
        mult[2] = math.nan
        out = torch.zeros(sum(lens), heads, 128, device="cuda")
        for more in (dict(head_scale=mult), dict(sink=mult)):
            H.capped_attn(q, *dev, None if decode else cu, sl, heads, 0.1, cap,
                          out, **more)
            gone = torch.isnan(out)
            assert gone[:, 2].all() and gone.sum() == gone[:, 2].numel()
    q = q.unflatten(-1, (heads, 128))
    out = ops.paged_attn_decode(q, *dev, sl, math.nan) if decode else \
        ops.paged_attn_prefill(q, *dev, cu, sl, math.nan)
    assert torch.isnan(out).all()
    if decode:
        latent = torch.randn(dev[0].shape[0], 16, 512, device="cuda").to(
            torch.bfloat16)
        out = torch.zeros(len(lens), 8, 512, device="cuda")
        H.latent_attn(torch.ones_like(out, dtype=torch.bfloat16), latent,
                      dev[2], None, sl, math.nan, 512, out)
        assert torch.isnan(out).all()


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("T,at", [(100, 0), (100, 15), (100, 37),  # one chunk
                                  (300, 0), (300, 37), (300, 127), (300, 200)])
def test_decayed(T, at, where, bad):
    """One entry of one token: the tokens before it do not see it, and the state
    is lost where 64-bit arithmetic loses it."""
    g = torch.Generator().manual_seed(T + at)
    heads, D, V = 2, 64, 128
    a = torch.tensor([0.9, 0.99])
    x = torch.randn(T, heads * (2 * D + V), generator=g).to(torch.bfloat16)
    cut = (0, heads * D, 2 * heads * D, x.shape[1])
    x[at, cut["qkv".index(where)] + D + 5] = bad         # second head
    x, f = features(x)
    ref, after = recur(*(f[:, b:e].reshape(T, heads, -1)
                         for b, e in zip(cut, cut[1:])), a.double(),
                       torch.zeros(heads, D, V, dtype=torch.float64))
    i32 = dict(dtype=torch.int32, device="cuda")
    state = torch.zeros(1, heads, D, V, device="cuda")
    out = torch.zeros(T, heads, V, device="cuda")
    xd = x.cuda()
    H.decay_attn(*(xd[:, b:e] for b, e in zip(cut, cut[1:])), a.cuda(), state,
                 torch.zeros(1, **i32), torch.tensor([0, T], **i32),
                 torch.zeros(1, **i32), out, max_q_len=T)
    agree(out, ref)
    agree(state[0], after)
