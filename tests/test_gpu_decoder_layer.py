"""A decoder layer as one native call against the calls of its modules: the same
kernels in the same order, so the same bits."""
import pytest
import torch

from xllm_service_amd import ops
from xllm_service_amd.engine.metadata import AttnMetadata
from xllm_service_amd.models.config import get_config
from xllm_service_amd.models.llama import LlamaDecoderLayer
from xllm_service_amd.ops import ref

pytestmark = pytest.mark.gpu


def _step(layer, cfg, prompts, decodes, first):
    """One pass over chunks of `prompts` tokens behind 20 cached ones and rows of
    `decodes` cached ones; fresh inputs and caches every time."""
    g = torch.Generator(device="cuda").manual_seed(3)
    T, pages = sum(prompts) + len(decodes), 64

    def bf(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(
            torch.bfloat16)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    caches = [bf(pages, cfg.num_kv_heads, 16, cfg.head_dim) for _ in "kv"]
    tables = torch.arange(pages, device="cuda", dtype=torch.int32).view(8, 8)
    pos = [p for n in prompts for p in range(20, 20 + n)] + list(decodes)
    seq = [i for i, n in enumerate(prompts) for _ in range(n)] \
        + list(range(len(prompts), len(prompts) + len(decodes)))
    slots = [int(tables[s, p // 16]) * 16 + p % 16 for s, p in zip(seq, pos)]
    cu = [0]
    for n in prompts:
        cu.append(cu[-1] + n)
    P = len(prompts)
    meta = AttnMetadata(
        num_prefill_tokens=cu[-1], num_decode_tokens=len(decodes),
        slot_mapping=torch.tensor(slots, device="cuda"),
        cu_q=i32(cu) if P else None,
        prefill_seq_lens=i32([20 + n for n in prompts]) if P else None,
        prefill_block_tables=tables[:P].contiguous() if P else None,
        decode_seq_lens=i32([n + 1 for n in decodes]) if decodes else None,
        decode_block_tables=tables[P:P + len(decodes)].contiguous()
        if decodes else None)
    cos_sin = ref.rope_table(cfg.head_dim, 256, cfg.rope_theta).cuda()
    x, residual = bf(T, cfg.hidden_size), bf(T, cfg.hidden_size)
    out = layer(x, None if first else residual,
                torch.tensor(pos, device="cuda"), caches, meta, cos_sin)
    return [*out, *caches]


@pytest.mark.parametrize("prompts,decodes,first", [
    ([5], [], True), ([40, 33], [17, 90, 3], False), ([], [31], False),
    ([70, 60], [], False)])
def test_native_layer(prompts, decodes, first, monkeypatch):
    cfg = get_config("llama-2k")
    with torch.device("cuda"):
        layer = LlamaDecoderLayer(cfg, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(1)
    for p in layer.parameters():
        p.data.normal_(0.0, 0.02, generator=g)
    calls = []
    native = ops.decoder_layer
    monkeypatch.setattr(ops, "decoder_layer",
                        lambda *a: calls.append(1) or native(*a))
    with torch.inference_mode():
        got = _step(layer, cfg, prompts, decodes, first)
        assert len(calls) == 1
        seen = []
        layer.mlp.down.register_forward_hook(lambda *a: seen.append(1))
        want = _step(layer, cfg, prompts, decodes, first)
        assert len(calls) == 1 and len(seen) == 1
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    with torch.no_grad():                     # gradients could be asked for
        _step(layer, cfg, prompts, decodes, first)
    assert len(calls) == 1
