"""Decoded and prompt rows of latent attention at rank 512, at the edges of pages,
tiles, windows and key parts, against fp64. The weights have 32 bits: an output may
be off by 2^-17 of the weighted sum of absolute values (exponents are rounded
products of up to 2^5)."""
import math

import pytest
import torch

from xllm_service_amd.ops import hybrid as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", [0, 64])
@pytest.mark.parametrize("heads", [1, 16, 21, 32])
@pytest.mark.parametrize("window", [0, 1, 40])
@pytest.mark.parametrize("keys", [[1, 15, 16, 17, 31, 32, 33, 64, 65, 100],
                                  [2100, 5], [300] * 40,
                                  [90] * 90 + [1500],
                                  [200, 40] * 44 + [1000],
                                  [500, 30] * 12 + [1100]])
def test_decode_edges(tail, heads, window, keys):
    g = torch.Generator().manual_seed(tail + heads + window + len(keys))
    W, r, scale = 512 + tail, 512, 192 ** -0.5
    need = [-(-n // 16) for n in keys]
    cache = torch.randn(sum(need) + 3, 16, W, generator=g).to(torch.bfloat16)
    order = torch.randperm(sum(need) + 3, generator=g).to(torch.int32)
    table = torch.zeros(len(keys), max(need) + 1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    q = torch.randn(len(keys), heads, W, generator=g).to(torch.bfloat16)
    if len(keys) == 2:                       # one key far above the others
        cache[table[0, 70], 3] *= 20.0
    for sign in (1.0, -1.0):
        out = torch.full((len(keys), heads, r), 9.0, device="cuda")
        H.latent_attn(q.cuda(), cache.cuda(), table.cuda(), None,
                      torch.tensor(keys, dtype=torch.int32, device="cuda"),
                      sign * scale, r, out, window)
        for s, n in enumerate(keys):
            k = cache[table[s, :need[s]].long()].reshape(-1, W)[:n].double()
            z = q[s].double() @ k.t() * (sign * scale)
            if window:
                z[:, :max(0, n - window)] = -math.inf
            p = torch.softmax(z, -1)
            off = (out[s].double().cpu() - p @ k[:, :r]).abs()
            over = off - 2.0 ** -17 * (p @ k[:, :r].abs())
            assert over.max() <= 1e-7, f"sequence {s}: off by {off.max():.3g}"


@pytest.mark.parametrize("op", ["latent", "capped"])
def test_fixed_parts(op, monkeypatch):
    """XLLM_LATENT_PARTS and XLLM_CAPPED_PARTS fix the parts of decoded rows: one
    part needs no workspace, 16 need one, and the results agree."""
    g = torch.Generator(device="cuda").manual_seed(4)
    keys, heads = 900, 8
    table = torch.randperm(60, generator=g, device="cuda").int().view(1, 60)
    sl = torch.tensor([keys], dtype=torch.int32, device="cuda")
    if op == "latent":
        cache = torch.randn(60, 16, 576, generator=g, device="cuda").to(
            torch.bfloat16)
        q = torch.randn(1, heads, 576, generator=g, device="cuda").to(
            torch.bfloat16)
        out = torch.zeros(1, heads, 512, device="cuda")

        def run():
            H.latent_attn(q, cache, table, None, sl, 0.07, 512, out)
    else:
        k, v = (torch.randn(60, 2, 16, 128, generator=g, device="cuda").to(
            torch.bfloat16) for _ in range(2))
        q = torch.randn(1, heads * 128, generator=g, device="cuda").to(
            torch.bfloat16)
        out = torch.zeros(1, heads, 128, device="cuda")

        def run():
            H.capped_attn(q, k, v, table, None, sl, heads, 0.08, 0.0, out)
    run()
    free = out.clone()
    used = {}
    for parts in (1, 16):
        monkeypatch.setenv(f"XLLM_{op.upper()}_PARTS", str(parts))
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        out.zero_()
        run()
        torch.cuda.synchronize()
        used[parts] = torch.cuda.max_memory_allocated() - before
        assert (out - free).abs().max() <= 1e-5
    assert used[1] == 0 and used[16] > 0, used


@pytest.mark.parametrize("tail", [0, 64])
@pytest.mark.parametrize("heads,new,old,window", [
    (16, [1, 8, 9, 40], [0, 31, 64, 15], 0),     # edges of row and key tiles
    (21, [7, 1, 30], [90, 33, 0], 40),           # heads that divide no row tile
    (32, [5], [1500], 0),                        # parts of one sequence
    (16, [3, 20, 2], [1100, 0, 400], 0),         # ... of several, and one without
    (32, [9, 4], [700, 1300], 500),              # ... in a window
    (1, [300, 2], [10, 5], 1),
    (16, [3] * 70, [40] * 70, 0),                # more sequences than lanes
    (16, [3] * 70, ([0, 40, 600] * 24)[:70], 0),     # ... and parts of them
    (16, [0, 5, 0, 33, 0], [40, 90, 0, 0, 7], 0),    # sequences of no new tokens
    (16, [5, 0, 33, 0], [900, 1300, 0, 40], 0),      # ... beside parts
    (40, [9, 1, 40], [100, 700, 0], 0),          # many heads
    (64, [20], [1500], 0),
    (32, [500, 300, 60], [0, 70, 800], 0)])      # a turn of the CUs and more
def test_prompt_edges(tail, heads, new, old, window):
    g = torch.Generator().manual_seed(tail + heads + window + len(new))
    W, r, scale = 512 + tail, 512, 192 ** -0.5
    keys = [n + o for n, o in zip(new, old)]
    need = [-(-n // 16) for n in keys]
    cache = torch.randn(sum(need) + 3, 16, W, generator=g).to(torch.bfloat16)
    order = torch.randperm(sum(need) + 3, generator=g).to(torch.int32)
    table = torch.zeros(len(keys), max(need) + 1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    q = torch.randn(sum(new), heads, W, generator=g).to(torch.bfloat16)
    cache[table[0, 0], 0] *= 20.0                # one key far above the others
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    for sign in (1.0, -1.0):
        out = torch.full((sum(new), heads, r), 9.0, device="cuda")
        H.latent_attn(q.cuda(), cache.cuda(), table.cuda(),
                      torch.tensor(cu, dtype=torch.int32, device="cuda"),
                      torch.tensor(keys, dtype=torch.int32, device="cuda"),
                      sign * scale, r, out, window)
        for s, n in enumerate(new):
            if n == 0:
                continue
            k = cache[table[s, :need[s]].long()].reshape(-1, W)[:keys[s]].cuda()
            k = k.double()
            z = q[cu[s]:cu[s + 1]].cuda().double() @ k.t() * (sign * scale)
            pos = old[s] + torch.arange(n, device="cuda")[:, None, None]
            at = torch.arange(keys[s], device="cuda")
            z = z.masked_fill((at > pos) | (window > 0) & (at <= pos - window),
                              -math.inf)
            p = torch.softmax(z, -1)
            off = (out[cu[s]:cu[s + 1]].double() - p @ k[:, :r]).abs()
            # A score is a sum of 36 products in a row, each rounded to 2^-24 of what
            # is summed, at most |q| |k|: errors of 6 such steps, as they add up at
            # random, are more than 2^-17 where the standout key is seen.
            most = (q[cu[s]:cu[s + 1]].cuda().double().abs() @ k.abs().t()).masked_fill(
                z == -math.inf, 0.0).amax(-1, keepdim=True) * scale
            bound = (6 * 2.0 ** -24 * most).clamp(min=2.0 ** -17)
            over = off - bound * (p @ k[:, :r].abs())
            assert over.max() <= 1e-7, f"sequence {s}: off by {off.max():.3g}"


@pytest.mark.parametrize("tail", [0, 64])
@pytest.mark.parametrize("heads,new,old", [
    (16, [301], [2900]), (32, [40, 6, 130], [3000, 2500, 2800]),   # parts
    (32, [300, 221, 400, 475, 250], [200, 39, 257, 100, 0])])
def test_prompt_tiles_of_128_rows(tail, heads, new, old):
    """Calls that row tiles of 64 would take longer for."""
    assert prompt_way(heads, new, old)[0] == 128
    test_prompt_edges(tail, heads, new, old, 0)


def prompt_way(heads, new, old, window=0):
    """Rows of a tile, 64-key tiles of a part at least (0: no parts), parts at most of
    what test_prompt_edges makes of these."""
    width = max(-(-(n + o) // 16) for n, o in zip(new, old)) + 1
    return H._hyb().latent_rows_way(sum(new), len(new), heads, width, window)


@pytest.mark.parametrize("tail", [0, 64])
@pytest.mark.parametrize("rows,heads,new,old", [
    (64, 16, [1100], [0]), (64, 16, [1300, 200], [0, 0]),
    (128, 32, [533], [2600]), (128, 32, [400, 30, 500], [1500, 3000, 600])])
def test_prompt_long_chains(tail, rows, heads, new, old):
    """Keys in one piece, more than the 1024 whose pages a wave asks for at a time."""
    assert prompt_way(heads, new, old)[:2] == (rows, 0)
    test_prompt_edges(tail, heads, new, old, 0)


@pytest.mark.parametrize("heads,new,old,window", [
    (32, [5], [1500], 0), (16, [3, 20, 2], [1100, 0, 400], 0),
    (32, [9, 4], [700, 1300], 500), (16, [3] * 70, ([0, 40, 600] * 24)[:70], 0),
    (16, [5, 0, 33, 0], [900, 1300, 0, 40], 0), (64, [20], [1500], 0),
    (16, [301], [2900], 0), (32, [40, 6, 130], [3000, 2500, 2800], 0)])
def test_prompts_in_parts(heads, new, old, window):
    """The calls above that are meant to have parts have them."""
    _, least, most = prompt_way(heads, new, old, window)
    assert least > 0 and most > 1


@pytest.mark.parametrize("r,tail,page", [(512, 64, 32), (512, 0, 8), (480, 64, 16),
                                         (272, 32, 16)])
@pytest.mark.parametrize("heads,window", [(16, 0), (17, 40), (64, 0)])
def test_prompts_of_other_sizes(r, tail, page, heads, window):
    """Wide rows of another rank, or in pages of another size."""
    g = torch.Generator().manual_seed(r + page + heads)
    W, new, old, scale = r + tail, [5, 40, 1, 16], [70, 0, 300, 33], 0.07
    keys = [n + o for n, o in zip(new, old)]
    need = [-(-n // page) for n in keys]
    cache = torch.randn(sum(need) + 2, page, W, generator=g).to(torch.bfloat16)
    order = torch.randperm(sum(need) + 2, generator=g).to(torch.int32)
    table = torch.zeros(len(keys), max(need), dtype=torch.int32)
    cu = [0]
    for i, n in enumerate(need):
        table[i, :n] = order[sum(need[:i]):sum(need[:i]) + n]
        cu.append(cu[-1] + new[i])
    q = torch.randn(sum(new), heads, W, generator=g).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device="cuda")
    out = torch.full((sum(new), heads, r), 9.0, device="cuda")
    H.latent_attn(q.cuda(), cache.cuda(), table.cuda(), torch.tensor(cu, **i32),
                  torch.tensor(keys, **i32), scale, r, out, window)
    for s, n in enumerate(new):
        k = cache[table[s, :need[s]].long()].reshape(-1, W)[:keys[s]].double()
        z = q[cu[s]:cu[s + 1]].double() @ k.t() * scale
        pos = old[s] + torch.arange(n)[:, None, None]
        at = torch.arange(keys[s])
        z = z.masked_fill((at > pos) | (window > 0) & (at <= pos - window), -math.inf)
        p = torch.softmax(z, -1)
        off = (out[cu[s]:cu[s + 1]].double().cpu() - p @ k[:, :r]).abs()
        most = (q[cu[s]:cu[s + 1]].double().abs() @ k.abs().t()).masked_fill(
            z == -math.inf, 0.0).amax(-1, keepdim=True) * scale
        bound = (6 * 2.0 ** -24 * most).clamp(min=2.0 ** -17)   # as above
        over = off - bound * (p @ k[:, :r].abs())
        assert over.max() <= 1e-7, f"sequence {s}: off by {over.max():.3g}"


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("heads,old", [(16, 0), (32, 70), (16, 1500)])
def test_prompt_nonfinite(heads, old, bad):
    """A new token's latent that is not finite is lost to the rows that see it, and to
    no token in front of its 64 rows; so is a NaN factor to all."""
    g = torch.Generator().manual_seed(heads + old)
    n, W, at = 24, 576, 9
    need = -(-(n + old) // 16)
    cache = torch.randn(need, 16, W, generator=g).to(torch.bfloat16)
    cache.view(-1, W)[old + at, 40] = bad
    table = torch.arange(need, dtype=torch.int32)[None].cuda()
    q = torch.randn(n, heads, W, generator=g).to(torch.bfloat16).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    out = torch.zeros(n, heads, 512, device="cuda")

    def run(scale):
        H.latent_attn(q, cache.cuda(), table, torch.tensor([0, n], **i32),
                      torch.tensor([n + old], **i32), scale, 512, out, 0)
        return torch.isfinite(out)
    fine = run(0.07)
    assert not fine[at:, :, 40].any()
    assert fine[:at * heads // 64 * 64 // heads].all()
    assert not run(math.nan).any()
