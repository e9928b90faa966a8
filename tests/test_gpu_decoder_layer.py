"""Decoder layers as one native call against the calls of their modules. What enters
and leaves attention of a first layer is the same bits. Norms and gates between two
products are made by these, without some of the roundings, so that a layer's result
differs by a few independent errors of 2^-9: within 2^-7 in the 2-norm, 2^-6 after
three layers. Against 64 bits they are no further off than the modules."""
import dataclasses

import pytest
import torch

from xllm_service_amd import ops
from xllm_service_amd.engine.metadata import AttnMetadata
from xllm_service_amd.models.config import ModelConfig, get_config
from xllm_service_amd.models.llama import LlamaDecoderLayer, _native_layers
from xllm_service_amd.ops import ref

pytestmark = pytest.mark.gpu


def _step(layers, cfg, prompts, decodes, first, no_slot=(), held=list,
          mrope=False, by=None):
    """One pass over chunks of `prompts` tokens behind 20 cached ones and rows of
    `decodes` cached ones; fresh inputs and caches every time. `held`: what holds
    the caches of the layers; `mrope`: three rows of positions, each its own; `by`:
    what makes the pass in the layers' place."""
    g = torch.Generator(device="cuda").manual_seed(3)
    T = sum(prompts) + len(decodes)
    pages = 8 * max(10, len(prompts) + len(decodes))

    def bf(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(
            torch.bfloat16)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    caches = [[bf(pages, cfg.num_kv_heads, 16, cfg.head_dim) for _ in "kv"]
              for _ in layers]
    tables = torch.arange(pages, device="cuda", dtype=torch.int32).view(-1, 8)
    pos = [p for n in prompts for p in range(20, 20 + n)] + list(decodes)
    seq = [i for i, n in enumerate(prompts) for _ in range(n)] \
        + list(range(len(prompts), len(prompts) + len(decodes)))
    slots = [int(tables[s, p // 16]) * 16 + p % 16 for s, p in zip(seq, pos)]
    slots = [-1 if i in no_slot else s for i, s in enumerate(slots)]
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
    pos = torch.tensor(pos, device="cuda")
    if mrope:
        pos = torch.stack([pos, pos // 2, pos // 3 + 7])
    residual = None if first else residual
    if by is not None:
        return by(layers, cfg, x, residual, pos, caches, meta, cos_sin), caches
    done = _native_layers(layers, x, residual, pos, held(caches), meta, cos_sin)
    if done is None:
        done = x, residual
        for layer, kv in zip(layers, caches):
            done = layer(*done, pos, kv, meta, cos_sin)
    return done, caches


def _off(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


@pytest.mark.parametrize("name", ["llama-2k", "llama-4k"])
@pytest.mark.parametrize("prompts,decodes,first,n_layers", [
    ([5], [], True, 1), ([40, 33], [17, 90, 3], False, 1), ([], [31], False, 3),
    ([], [31] * 8, True, 3), ([70, 60], [], False, 1), ([33, 50, 90], [4], True, 3),
    ([100, 105, 107], [], True, 3)])
def test_native_layers(name, prompts, decodes, first, n_layers, monkeypatch):
    cfg = get_config(name)
    with torch.device("cuda"):
        layers = [LlamaDecoderLayer(cfg, torch.bfloat16)
                  for _ in range(n_layers)]
    g = torch.Generator(device="cuda").manual_seed(1)
    for n, p in torch.nn.ModuleList(layers).named_parameters():
        p.data.normal_(1.0 if "norm" in n else 0.0, 0.02, generator=g)
    calls = []
    native = ops.decoder_layers
    monkeypatch.setattr(ops, "decoder_layers",
                        lambda *a: calls.append(1) or native(*a))
    with torch.inference_mode():
        got, caches = _step(layers, cfg, prompts, decodes, first)
        assert len(calls) == 1
        seen = []
        for layer in layers:
            layer.mlp.down.register_forward_hook(lambda *a: seen.append(1))
        want, plain = _step(layers, cfg, prompts, decodes, first)
        assert len(calls) == 1 and len(seen) == n_layers
    for a, b in zip(caches[0], plain[0]):
        assert torch.equal(a, b)
    for a, b in zip(got, want):
        assert _off(a, b) < 2.0 ** (-7 if n_layers == 1 else -6)
    with torch.no_grad():                     # gradients could be asked for
        _step(layers, cfg, prompts, decodes, first)
    assert len(calls) == 1


@pytest.mark.parametrize("name", ["llama-2k", "llama-4k"])
@pytest.mark.parametrize("prompts,decodes", [
    ([], [1]), ([5], [17, 90, 3]), ([8, 9], [31] * 7), ([20, 9], [8]), ([41], []),
    ([33, 31], []), ([70, 60], []), ([100, 105, 107], [4])])
def test_rotated_products(name, prompts, decodes):
    """Keys and values that the first product of a second layer leaves in its caches:
    as above within 2^-6, elsewhere, and where a row has no slot, what was there."""
    cfg = get_config(name)
    with torch.device("cuda"):
        layers = [LlamaDecoderLayer(cfg, torch.bfloat16) for _ in range(2)]
    g = torch.Generator(device="cuda").manual_seed(1)
    for n, p in torch.nn.ModuleList(layers).named_parameters():
        p.data.normal_(1.0 if "norm" in n else 0.0, 0.02, generator=g)
    T = sum(prompts) + len(decodes)
    no_slot = (T - 1,) if T > 1 else ()
    with torch.inference_mode():
        got, caches = _step(layers, cfg, prompts, decodes, True, no_slot)
        none, before = _step(layers, cfg, prompts, decodes, True, range(T))
        layers[0].mlp.down.register_forward_hook(lambda *a: None)
        want, plain = _step(layers, cfg, prompts, decodes, True, no_slot)
    for a, b, was in zip(caches[1], plain[1], before[1]):
        new = (b != was).any(-1)                     # rows of heads
        assert int(new.sum()) == (T - len(no_slot)) * cfg.num_kv_heads
        assert torch.equal(a[~new], was[~new])
        assert _off(a[new], b[new]) < 2.0 ** -6
        off = (a[new].double() - b[new].double()).norm(dim=-1)
        assert (off < 2.0 ** -5 * b[new].double().norm(dim=-1)).all()


def test_caches_by_index():
    """A cache for every layer, found by its number: too few are refused."""
    cfg = get_config("llama-2k")
    with torch.device("cuda"):
        layers = [LlamaDecoderLayer(cfg, torch.bfloat16) for _ in range(3)]
    for p in torch.nn.ModuleList(layers).parameters():
        p.data.normal_(0.0, 0.02)
    with torch.inference_mode():
        want, _ = _step(layers, cfg, [5], [31], True)
        got, _ = _step(layers, cfg, [5], [31], True,
                       held=lambda c: dict(reversed(list(enumerate(c)))))
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        for held in (lambda c: c[:2], lambda c: tuple(c[:1]), lambda c: []):
            with pytest.raises(IndexError):
                _step(layers, cfg, [5], [31], True, held=held)


@pytest.mark.parametrize("name,value", [("scale", 0.5), ("eps", 0.25),
                                        ("mrope_sections", (16, 24, 24))])
def test_settings_of_a_layer(name, value):
    """What one layer has its own of acts on this one: results as the modules give
    them, not as all layers with the first one's settings do."""
    cfg = get_config("llama-2k")
    with torch.device("cuda"):
        layers = [LlamaDecoderLayer(cfg, torch.bfloat16) for _ in range(3)]
    g = torch.Generator(device="cuda").manual_seed(1)
    for n, p in torch.nn.ModuleList(layers).named_parameters():
        p.data.normal_(1.0 if "norm" in n else 0.0, 0.02, generator=g)
    rows = name == "mrope_sections"
    args = layers, cfg, [40, 33], [17], True
    if rows:
        for layer in layers:
            layer.attn.mrope_sections = (64, 0, 0)
    with torch.inference_mode():
        same, _ = _step(*args, mrope=rows)
        setattr(layers[1] if name == "eps" else layers[1].attn, name, value)
        got, _ = _step(*args, mrope=rows)
        for layer in layers:
            layer.mlp.down.register_forward_hook(lambda *a: None)
        want, _ = _step(*args, mrope=rows)
    assert max(_off(a, b) for a, b in zip(same, want)) > 2.0 ** -5
    for a, b in zip(got, want):
        assert _off(a, b) < 2.0 ** -6


def _exact(layers, cfg, x, residual, pos, caches, meta, cos_sin):
    """The same in 64 bits, caches included: these are replaced in `caches`."""
    T, H, G, D = x.shape[0], cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    x = x.double()
    res = None if residual is None else residual.double()
    sec = torch.zeros(D // 2, dtype=torch.long, device="cuda")
    if pos.dim() == 2:
        a, b, _ = layers[0].attn.mrope_sections
        sec[a:a + b], sec[a + b:] = 1, 2
    rows = (pos if pos.dim() == 2 else pos[None])[sec].t()      # [T, D / 2]
    at = torch.arange(D // 2, device="cuda")
    cos, sin = (cos_sin.double()[rows, at + o][:, None] for o in (0, D // 2))
    seqs, row = [], 0                            # first row, rows, keys, pages
    if meta.num_prefill_tokens:
        cu = meta.cu_q.tolist()
        for i, n in enumerate(meta.prefill_seq_lens.tolist()):
            seqs.append((cu[i], cu[i + 1] - cu[i], n,
                         meta.prefill_block_tables[i]))
        row = cu[-1]
    if meta.num_decode_tokens:
        for i, n in enumerate(meta.decode_seq_lens.tolist()):
            seqs.append((row + i, 1, n, meta.decode_block_tables[i]))
    slots = meta.slot_mapping

    def norm(z, w, eps):
        return z * torch.rsqrt(z.square().mean(-1, keepdim=True) + eps) \
            * w.double()

    def product(z, m):
        y = z @ m.weight.double().t()
        return y if m.bias is None else y + m.bias.double()

    def turn(z):
        u, w = z[..., :D // 2], z[..., D // 2:]
        return torch.cat([u * cos - w * sin, w * cos + u * sin], -1)
    for i, layer in enumerate(layers):
        res = x if res is None else res + x
        qkv = product(norm(res, layer.input_norm, layer.eps),
                      layer.attn.qkv_proj).view(T, H + 2 * G, D)
        q, k, v = turn(qkv[:, :H]), turn(qkv[:, H:H + G]), qkv[:, H + G:]
        kc, vc = (c.double() for c in caches[i])
        kc[slots // 16, :, slots % 16], vc[slots // 16, :, slots % 16] = k, v
        caches[i] = [kc, vc]
        out = torch.empty_like(q)
        for r, n, keys, pages in seqs:
            kk, vv = (c[pages.long()].transpose(1, 2).reshape(-1, G, D)[:keys]
                      .repeat_interleave(H // G, 1).transpose(0, 1)
                      .contiguous() for c in (kc, vc))
            z = torch.bmm(q[r:r + n].transpose(0, 1).contiguous(),
                          kk.transpose(1, 2).contiguous()) * layer.attn.scale
            z = z.masked_fill(torch.arange(keys, device="cuda")[None]
                              > keys - n + torch.arange(n, device="cuda")[:, None],
                              -torch.inf)
            out[r:r + n] = torch.bmm(z.softmax(-1), vv).transpose(0, 1)
        res = res + product(out.reshape(T, H * D), layer.attn.o_proj)
        gate, up = product(norm(res, layer.post_norm, layer.eps),
                           layer.mlp.gate_up).chunk(2, -1)
        x = product(torch.nn.functional.silu(gate) * up, layer.mlp.down)
    return x, res


# hidden, intermediate, heads, key heads; biases of [q | k | v] and of [gate | up];
# positions in three rows
@pytest.mark.parametrize("hidden,inter,heads,kv_heads,bias,gate_bias,mrope", [
    (512, 1024, 4, 2, True, False, True),
    (512, 1024, 4, 2, False, True, False),
    (3584, 1024, 28, 4, True, False, True),
    (3584, 2048, 28, 4, False, False, True),
    (2176, 1152, 16, 4, False, False, False),    # tiles of N no multiple of four
    (2048, 2048, 16, 4, False, False, False),
    (4096, 8192, 32, 8, True, True, False),      # more than 8192 rows of [gate | up]
])
@pytest.mark.parametrize("prompts,decodes", [
    ([], [40]), ([5], [17, 90]), ([], [31] * 24), ([33], [4] * 9), ([70, 60], [9])])
def test_layers_against_64_bits(hidden, inter, heads, kv_heads, bias, gate_bias,
                                mrope, prompts, decodes):
    """Results, and what three layers leave in their caches, are no further from 64
    bits than what the modules make. The norm of n independent errors is off by
    sqrt(1 / 2n) of itself by chance, the ratio of two by sqrt(1 / n): four of these."""
    cfg = dataclasses.replace(
        ModelConfig(), hidden_size=hidden, intermediate_size=inter,
        num_heads=heads, num_kv_heads=kv_heads, max_position=256,
        mrope_section=(16, 24, 24) if mrope else ())
    with torch.device("cuda"):
        layers = [LlamaDecoderLayer(cfg, torch.bfloat16) for _ in range(3)]
    g = torch.Generator(device="cuda").manual_seed(1)
    for layer in layers:
        for m, on in ((layer.attn.qkv_proj, bias), (layer.mlp.gate_up, gate_bias)):
            if on:
                m.bias = torch.nn.Parameter(torch.empty(
                    m.weight.shape[0], dtype=torch.bfloat16, device="cuda"))
    for n, p in torch.nn.ModuleList(layers).named_parameters():
        if "norm" in n:
            p.data.normal_(1.0, 0.2, generator=g)
        else:
            p.data.normal_(0.0, 1.0 if "bias" in n else hidden ** -0.5,
                           generator=g)
    args = layers, cfg, prompts, decodes, False
    with torch.inference_mode():
        got, caches = _step(*args, mrope=mrope)
        want, exact = _step(*args, mrope=mrope, by=_exact)
        for layer in layers:
            layer.mlp.down.register_forward_hook(lambda *a: None)
        plain, module_caches = _step(*args, mrope=mrope)
        _, before = _step(*args, range(sum(prompts) + len(decodes)), mrope=mrope)

    def no_further(a, b, w):
        more = 1.0 + 4.0 * w.numel() ** -0.5
        assert _off(a, w) <= min(2.0 ** -5, more * _off(b, w))
    for a, b, w in zip(got, plain, want):
        no_further(a, b, w)
    for a, b, w, was in zip(*(sum(map(list, c), []) for c in (
            caches, module_caches, exact, before))):
        new = (b != was).any(-1)
        assert torch.equal(a[~new], was[~new])
        no_further(a[new], b[new], w[new])


@pytest.mark.parametrize("prompts", [[90], [105], [40, 70]])
def test_layers_of_small_weights(prompts):
    """Weights of no whole kilobytes, which CUs that attention leaves idle fetch."""
    test_layers_against_64_bits(136, 40, 2, 1, False, False, False, prompts, [])


@pytest.mark.parametrize("prompts", [[90], [40, 70]])
def test_layers_of_weights_off_16_bytes(prompts, monkeypatch):
    """Weights that begin within 16 bytes, which nothing fetches by as many."""
    def layer_of(*args, make=LlamaDecoderLayer):
        layer = make(*args)
        for m in (layer.attn.qkv_proj, layer.attn.o_proj, layer.mlp.gate_up,
                  layer.mlp.down):
            room = torch.empty(m.weight.numel() + 4, dtype=torch.bfloat16)
            m.weight = torch.nn.Parameter(room[4:].view_as(m.weight))
            assert m.weight.is_contiguous() and m.weight.data_ptr() % 16 == 8
        return layer
    monkeypatch.setitem(globals(), "LlamaDecoderLayer", layer_of)
    test_layers_against_64_bits(256, 512, 2, 1, False, False, False, prompts, [])
