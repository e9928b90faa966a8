"""Rotation and cache writes in 16 B pieces against the kernel for any alignment,
which few tokens and rows shifted by 8 bytes take: the same arithmetic, so the same
bits."""
import pytest
import torch

from xllm_service_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 5, 300, None])
@pytest.mark.parametrize("heads,kv_heads,dim", [(32, 8, 128), (28, 4, 128),
                                                (12, 12, 64), (3, 1, 80),
                                                (5, 2, 96), (1, 1, 16)])
@pytest.mark.parametrize("sections", [None, "eights", "odd"])
def test_both_kernels(T, heads, kv_heads, dim, sections):
    if T is None:                          # as few as the 16 B kernel takes
        T = 16384 // ((heads + 2 * kv_heads) * (dim // 16)) + 1
    g = torch.Generator(device="cuda").manual_seed(T + heads + dim)
    width = (heads + 2 * kv_heads) * dim
    data = torch.randn(T, width, generator=g, device="cuda").to(torch.bfloat16)
    table = torch.randn(512, dim, generator=g, device="cuda")
    pages = T // 16 + 2
    slots = torch.randperm(pages * 16, generator=g, device="cuda")[:T]
    slots[T // 2] = -1
    half = dim // 2
    if sections is None:
        shape, secs = (T,), None
    else:
        a = half // 2 // 8 * 8 if sections == "eights" else half // 3
        if a == 0:
            pytest.skip("half a head is too short for sections")
        shape, secs = (3, T), (a, half - a, 0)
    pos = torch.randint(512, shape, generator=g, device="cuda")
    outs = []
    for shift in (0, 4):
        flat = torch.zeros(T, width + 8, device="cuda", dtype=torch.bfloat16)
        rows = flat[:, shift:shift + width]
        rows.copy_(data)
        q, k, v = rows.split([heads * dim, kv_heads * dim, kv_heads * dim], 1)
        kc = torch.zeros(pages, kv_heads, 16, dim, device="cuda",
                         dtype=torch.bfloat16)
        vc = torch.zeros_like(kc)
        ops.fused_rope_cache(pos, q.unflatten(1, (heads, dim)),
                             k.unflatten(1, (kv_heads, dim)),
                             v.unflatten(1, (kv_heads, dim)), kc, vc, slots,
                             table, dim, mrope_sections=secs)
        outs.append((rows.clone(), kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert not torch.equal(outs[0][0][:, :heads * dim], data[:, :heads * dim])
