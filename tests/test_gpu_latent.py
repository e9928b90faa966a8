"""Decoded rows of latent attention at rank 512, at the edges of pages, tiles,
windows and key parts, against fp64. The weights have 32 bits: an output may
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
