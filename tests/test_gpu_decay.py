"""Decayed linear attention of bf16 prompt rows at the edges of its chunks and
tiles, against the token recurrence in fp64.

The features silu(x) are rounded to bf16; inputs whose feature lies within
2^-6 of an ulp of the middle between two bf16 numbers become zero, so that
oracle and kernel round alike. What remains are 32-bit products and sums:
every output may be off by 2^-20 of the same sum over absolute values (a
weight is a product of two rounded powers; up to 2^4 roundings in a chain)."""
import pytest
import torch

from xllm_service_amd.ops import hybrid as H

pytestmark = pytest.mark.gpu
F64 = torch.float64


def features(x):
    y = x.to(F64) * torch.sigmoid(x.to(F64))
    ulp = 2.0 ** (torch.floor(torch.log2(y.abs().clamp(min=1e-30))) - 7)
    frac = (y.abs() / ulp) % 1.0
    x = torch.where((frac - 0.5).abs() < 2.0 ** -6, torch.zeros_like(x), x)
    y = x.to(F64) * torch.sigmoid(x.to(F64))
    return x, y.to(torch.bfloat16).to(F64)


def recur(q, k, v, a, S):
    """[n, H, *] features, S [H, D, V]: outputs and the state after."""
    out = []
    for t in range(q.shape[0]):
        S = a[:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    return torch.stack(out), S


def way(heads, D, V, lens):
    """How a batch goes: the way, groups of chunks that are walked, waves of outputs."""
    return "%s %d %d" % H._hyb().decay_attn_way(max(lens), sum(lens), len(lens), heads,
                                                D, V)


def run(D, V, lens, ctx, slots, decay, bound, seed):
    g = torch.Generator().manual_seed(seed)
    heads, T = len(decay), sum(lens)
    width = heads * (2 * D + V)
    rows = torch.randn(T, width + 8, generator=g).to(torch.bfloat16)
    rows[:, :width], f = features(rows[:, :width])
    cut = (0, heads * D, 2 * heads * D, width)
    a = torch.tensor(decay, dtype=torch.float32)
    state = torch.randn(max(slots) + 2, heads, D, V, generator=g)
    sd, rd = state.cuda(), rows.cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    out = torch.full((T, heads, V), 9.0, device="cuda")
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + n)
    H.decay_attn(*(rd[:, x:y] for x, y in zip(cut, cut[1:])), a.cuda(), sd,
                 torch.tensor(slots, **i32), torch.tensor(starts, **i32),
                 torch.tensor(ctx, **i32), out, max_q_len=bound)
    out, used, f, a64 = out.to(F64), set(), f.cuda(), a.cuda().to(F64)
    for s, (n, c, slot) in enumerate(zip(lens, ctx, slots)):
        x = [f[starts[s]:starts[s + 1], p:e].reshape(n, heads, -1)
             for p, e in zip(cut, cut[1:])]
        S = (state[slot] if slot >= 0 and c > 0 else torch.zeros(heads, D, V)).to(
            "cuda", F64)
        want, after = recur(*x, a64, S)
        big, top = recur(*(z.abs() for z in x), a64.abs(), S.abs())
        off = (out[starts[s]:starts[s + 1]] - want).abs() - 2.0 ** -20 * big
        assert off.max() <= 1e-30, f"sequence {s}: over by {off.max():.3g}"
        if slot >= 0:
            used.add(slot)
            off = (sd[slot].to(F64) - after).abs() - 2.0 ** -20 * top
            assert off.max() <= 1e-30, f"state {s}: over by {off.max():.3g}"
    for slot in range(state.shape[0]):
        if slot not in used:
            assert torch.equal(sd[slot].cpu(), state[slot])


@pytest.mark.parametrize("D,V", [(128, 128), (64, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("lens,bound", [
    ([1, 15, 16, 17], 17), ([31, 32, 33, 128], 128),      # one chunk each
    ([127, 128, 129, 1], 129), ([64, 65, 300, 256], 0),   # chunks and a scan
])
def test_prompt_rows(D, V, lens, bound):
    """Fresh and continued sequences, one without a slot."""
    run(D, V, lens, [0, 7, 0, 40], [3, 0, 1, -1], [0.999, 0.75, 1.0], bound,
        sum(lens) + D + V)


@pytest.mark.parametrize("D,V", [(128, 128), (64, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("lens,heads,ways", [
    # 128 x 128 | 64 x 128 | 128 x 64 | 64 x 64
    ([100, 40, 128, 3] * 23, 3, "one 0 16|one 0 16|one 0 8|two 0 4"),
    ([150, 3, 200], 32, "walk 1 16|walk 1 16|walk 1 8|walk 1 8"),
    ([300, 164, 250, 130], 32, "walk 1 4|walk 1 4|walk 1 4|walk 1 4"),
    ([130, 64, 257, 2, 65] * 20, 3, "scan 0 4|walk 1 4|walk 1 4|walk 1 4"),
    ([1500, 1, 3], 3, "scan 0 16|scan 0 16|scan 0 8|scan 0 8"),
    ([128, 256, 192], 3, "walk 2 16|walk 1 16|walk 1 8|walk 1 8")])
def test_prompt_routes(D, V, lens, heads, ways):
    """Each way from chunk to chunk, with outputs by four waves and by more; states
    carried, fresh and not kept."""
    assert way(heads, D, V, lens) == ways.split("|")[(D == 64) + 2 * (V == 64)]
    n = len(lens)
    run(D, V, lens, [5 * (i % 3 > 0) for i in range(n)],
        [i if (i + 5) % 7 else -1 for i in range(n)],
        ([0.999, 0.75, 1.0, 0.97, 0.3] * 7)[:heads], max(lens), n + D + V)


@pytest.mark.parametrize("lens,heads,groups,waves", [
    ([700, 3, 129, 384], 3, 3, 16), ([513, 1, 640, 385], 3, 3, 16),
    ([430, 130], 8, 4, 16), ([880, 881, 515], 3, 4, 16), ([880, 881, 515], 16, 2, 4),
    ([1030, 900], 16, 3, 4), ([1030], 32, 3, 4)])
def test_groups_of_chunks(lens, heads, groups, waves):
    """Sequences walked in up to four groups: whole and ragged last ones, fewer
    chunks than groups, states carried or not, one without a slot."""
    assert way(heads, 128, 128, lens) == f"walk {groups} {waves}"
    n = len(lens)
    run(128, 128, lens, [7 * (i % 3 != 1) for i in range(n)],
        [i if i != 2 else -1 for i in range(n)],
        ([0.999, 0.75, 1.0, 0.9999, 0.0, 0.3, 0.99, 0.996] * 4)[:heads], max(lens), n)


def test_many_chunks_and_hard_decays():
    """More chunks than the scan holds in flight; decays whose powers leave
    fp32's normal range within a chunk, and none at all."""
    run(128, 128, [1300, 200], [0, 9], [0, 2], [0.3, 0.0, 0.996], 1300, 4)


@pytest.mark.parametrize("long", [40, 300])         # one chunk each; a scan
def test_sequences_without_new_tokens(long):
    """A carried state stays bit for bit, a fresh one becomes zero, a sequence
    without a slot touches nothing, and the others do not notice."""
    g = torch.Generator().manual_seed(long)
    heads, D, bound = 2, 64, max(long, 17)
    a = torch.tensor([0.9, 0.99]).cuda()
    first = torch.randn(5, heads, D, D, generator=g).cuda()
    rows = torch.randn(long + 17, 3 * heads * D, generator=g).to(
        torch.bfloat16).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")

    def go(starts, ctx, slots):
        state = first.clone()
        out = torch.full((long + 17, heads, D), 9.0, device="cuda")
        H.decay_attn(*rows.chunk(3, 1), a, state, torch.tensor(slots, **i32),
                     torch.tensor(starts, **i32), torch.tensor(ctx, **i32),
                     out, max_q_len=bound)
        return out, state
    out, state = go([0, 0, long, long, long, long + 17, long + 17],
                    [5, 3, 4, 0, 0, 7], [0, 1, -1, 2, 3, 4])
    want, alone = go([0, long, long + 17], [3, 0], [1, 3])
    assert torch.equal(out, want)
    for slot in (0, 4):
        assert torch.equal(state[slot], first[slot])
    assert (state[2] == 0).all()
    for slot in (1, 3):
        assert torch.equal(state[slot], alone[slot])


def test_every_activation():
    """silu of every bf16 number below 2^100, read off as values of one-token
    sequences whose query and key meet in 2^24: those of a division, within one
    rounding to bf16, and zero where e^-x is infinite in 32 bits."""
    x = torch.arange(-2 ** 15, 2 ** 15).to(torch.int16).view(torch.bfloat16)
    x = torch.where(torch.isfinite(x) & (x.abs() < 2.0 ** 100), x,
                    torch.zeros_like(x))
    n, V = 512, 128
    q = torch.zeros(n, 64, dtype=torch.bfloat16)
    q[:, 0] = 4096.0                                 # its own activation
    i32 = dict(dtype=torch.int32, device="cuda")
    out = torch.zeros(n, 1, V, device="cuda")
    H.decay_attn(q.cuda(), q.cuda(), x.view(n, V).cuda(),
                 torch.ones(1, device="cuda"),
                 torch.zeros(1, 1, 64, V, device="cuda"),
                 torch.full((n,), -1, **i32), torch.arange(n + 1, **i32),
                 torch.zeros(n, **i32), out, max_q_len=128)   # not as short
    plain = torch.zeros_like(out)                    # decoded rows: a division
    H.decay_attn(q.cuda(), q.cuda(), x.view(n, V).cuda(),
                 torch.ones(1, device="cuda"),
                 torch.zeros(1, 1, 64, V, device="cuda"),
                 torch.full((n,), -1, **i32), None, torch.zeros(n, **i32),
                 plain)
    assert torch.equal(out, plain)
    got = out.cpu().double().flatten() / 2.0 ** 24
    x = x.double()
    want = torch.where(x < -88.7, 0.0, x * torch.sigmoid(x))
    tiny = want.abs() < 2.0 ** -126                  # not normal
    off = (got - want).abs()
    assert (off[~tiny] <= 2.0 ** -8 * want[~tiny].abs()).all()
    assert (off[tiny] <= 2.0 ** -126).all()


def test_no_less_precise_than_the_recurrence():
    """Against 64 bits, outputs and states are no further off than those of the
    kernel that walks from token to token (which rows of odd strides take)."""
    g = torch.Generator().manual_seed(11)
    heads, D, T = 4, 128, 1200
    a = torch.tensor([0.75, 0.97, 0.99, 0.996])
    x, f = features(torch.randn(T, 3 * heads * D, generator=g).to(
        torch.bfloat16))
    q, k, v = (z.reshape(T, heads, D) for z in f.chunk(3, 1))
    want, after = recur(q, k, v, a.to(F64), torch.zeros(heads, D, D,
                                                        dtype=F64))
    i32, off = dict(dtype=torch.int32, device="cuda"), []
    for pad in (0, 4):
        rows = torch.zeros(T, 3 * heads * D + pad, dtype=torch.bfloat16,
                           device="cuda")
        rows[:, :3 * heads * D] = x.cuda()
        state = torch.zeros(1, heads, D, D, device="cuda")
        out = torch.zeros(T, heads, D, device="cuda")
        H.decay_attn(*rows[:, :3 * heads * D].chunk(3, 1), a.cuda(), state,
                     torch.zeros(1, **i32), torch.tensor([0, T], **i32),
                     torch.zeros(1, **i32), out, max_q_len=T)
        off.append([float((y.cpu().to(F64) - w).norm() / w.norm())
                    for y, w in ((out, want), (state[0], after))])
    assert off[0][0] <= off[1][0] and off[0][1] <= off[1][1], off


def errors(heads, D, V, lens, ctx, decay, seed):
    """Relative errors (2-norms) of outputs and of states against 64 bits: of the kernel
    that the call takes, and of the recurrence (which rows of odd strides take)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    T, n, width = sum(lens), len(lens), heads * (2 * D + V)
    x, f = features(torch.randn(T, width, generator=g, device="cuda").to(torch.bfloat16))
    state = torch.randn(n, heads, D, V, generator=g, device="cuda")
    a = torch.tensor(decay, device="cuda")
    cut = (0, heads * D, 2 * heads * D, width)
    starts = [sum(lens[:i]) for i in range(n + 1)]
    want, after = [], []
    for i in range(n):
        rows = f[starts[i]:starts[i + 1]]
        o, S = recur(*(rows[:, p:e].reshape(lens[i], heads, -1)
                       for p, e in zip(cut, cut[1:])), a.to(F64),
                     state[i].to(F64) * (ctx > 0))
        want.append(o)
        after.append(S)
    i32, off = dict(dtype=torch.int32, device="cuda"), []
    for pad in (0, 4):
        rows = torch.zeros(T, width + pad, dtype=torch.bfloat16, device="cuda")
        rows[:, :width] = x
        got, out = state.clone(), torch.zeros(T, heads, V, device="cuda")
        H.decay_attn(*(rows[:, p:e] for p, e in zip(cut, cut[1:])), a, got,
                     torch.arange(n, **i32), torch.tensor(starts, **i32),
                     torch.full((n,), ctx, **i32), out, max_q_len=max(lens))
        off.append([float((y.to(F64) - w).norm() / w.norm())
                    for y, w in ((out, torch.cat(want)), (got, torch.stack(after)))])
    return off


@pytest.mark.parametrize("heads,D,V,n", [
    (16, 128, 128, 4), (16, 128, 128, 20), (20, 64, 128, 8), (20, 64, 128, 40),
    (20, 128, 64, 8), (20, 128, 64, 24), (20, 64, 64, 8), (20, 64, 64, 40)])
@pytest.mark.parametrize("longest", [3, 4, 5, 6, 9, 16, 24])
def test_short_prompts_no_less_precise(heads, D, V, n, longest):
    """Short sequences on both sides of the line to the recurrence, in one kernel and in
    two: errors of outputs and states are no larger than the recurrence's (half a percent
    for what a sample of 10^5 entries scatters). Where all heads decay to a half within a
    token, both are two or three roundings, and the matrix pipe cuts where the vector unit
    rounds: up to 8%."""
    lens = [longest] + [1 + (7 * i + longest) % longest for i in range(n - 1)]
    for ctx in (0, 5):
        for lo, hi, more in ((0.75, 0.996, 1.005), (0.3, 0.7, 1.08)):
            decay = [lo + (hi - lo) * h / (heads - 1) for h in range(heads)]
            here, there = errors(heads, D, V, lens, ctx, decay, longest + n)
            assert here[0] <= more * there[0] and here[1] <= more * there[1], (
                ctx, lo, here, there)


@pytest.mark.parametrize("heads,D,V,lens", [
    (16, 128, 128, [300, 256]), (16, 128, 128, [210, 130]), (16, 128, 128, [384, 200, 129]),
    (32, 128, 128, [300, 256]), (16, 64, 128, [300, 256]), (16, 64, 128, [384, 200, 129]),
    (16, 128, 64, [300, 256]), (16, 128, 64, [210, 130]), (16, 64, 64, [210, 130]),
    (32, 64, 64, [384, 200, 129])])
def test_walk_no_less_precise_than_scan(heads, D, V, lens):
    """Sequences that are walked and the same ones beside a long one, which makes the batch
    go by sums and a scan: states are no further off 64 bits (1% for what 10^5 entries
    scatter). Where all heads decay to a half within a token, half of the entries of a
    walked state are rounded twice, by sums all of them once: up to 5%."""
    assert way(heads, D, V, lens)[:4] == "walk"
    assert way(heads, D, V, lens + [4000])[:4] == "scan"
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    for lo, hi, most in ((0.3, 0.7, 1.05), (0.75, 0.996, 1.01), (0.996, 0.999, 1.01)):
        off = []
        a = torch.linspace(lo, hi, heads, device="cuda")
        x, f = features(torch.randn(sum(lens) + 4000, heads * (2 * D + V), generator=g,
                                    device="cuda").to(torch.bfloat16))
        cut = (0, heads * D, 2 * heads * D, heads * (2 * D + V))
        first = torch.randn(len(lens) + 1, heads, D, V, generator=g, device="cuda")
        after = []
        for i, n in enumerate(lens):
            rows = f[sum(lens[:i]):sum(lens[:i + 1])]
            after.append(recur(*(rows[:, p:e].reshape(n, heads, -1)
                                 for p, e in zip(cut, cut[1:])), a.to(F64),
                               first[i].to(F64))[1])
        after = torch.stack(after)
        for more in ([], [4000]):
            all_, i32 = lens + more, dict(dtype=torch.int32, device="cuda")
            state = first.clone()
            out = torch.zeros(sum(all_), heads, V, device="cuda")
            H.decay_attn(*(x[:sum(all_), p:e] for p, e in zip(cut, cut[1:])), a, state,
                         torch.arange(len(all_), **i32),
                         torch.tensor([sum(all_[:i]) for i in range(len(all_) + 1)],
                                      **i32),
                         torch.full((len(all_),), 5, **i32), out, max_q_len=max(all_))
            off.append(float((state[:len(lens)].to(F64) - after).norm() / after.norm()))
        assert off[0] <= most * off[1], (lo, off)


@pytest.mark.parametrize("heads,D,V,most", [
    (1, 128, 128, 7), (48, 64, 64, 4), (40, 128, 64, 6), (20, 64, 128, 6),
    (86, 128, 128, 3), (86, 128, 64, 4), (100, 64, 64, 3), (172, 64, 64, 2)])
def test_short_batches(heads, D, V, most):
    """Lengths on both sides of the line between the recurrence and the
    matrix-pipe form, for few and for many states."""
    for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 17, 25):
        assert (way(heads, D, V, [n] * 3)[:3] == "rec") == (n <= most)
        run(D, V, [n, max(1, n // 2), n], [0, 5, 3], [1, -1, 0],
            [0.75 + 0.24 * h / heads for h in range(heads)], n, n)


@pytest.mark.parametrize("heads,D,V,lens,kind", [
    (16, 128, 128, [128, 1, 15, 16, 17, 33, 127], "one"),    # tiles of 16 and 32 tokens
    (24, 128, 128, [63, 64, 65, 96, 97, 8] * 2, "one"),      # more than one for each CU
    (40, 64, 64, [128, 31, 5, 112, 2, 64], "one"),
    (43, 64, 64, [128, 31, 5, 112, 2, 64], "two"),
    (60, 64, 128, [32, 3, 20, 7, 16] * 2, "two"),
    (60, 64, 128, [33, 3, 20, 7, 128] * 2, "one"),
    (64, 128, 64, [33, 128, 9, 50, 16, 100, 65], "one"),
    (65, 128, 64, [33, 128, 9, 50, 16, 100, 65], "two")])
def test_one_chunk_each(heads, D, V, lens, kind):
    """States moved by the workgroups of the outputs, or after them, on both sides of the
    lines between; some states not kept, some carried."""
    assert way(heads, D, V, lens)[:3] == kind
    n = len(lens)
    run(D, V, lens, [i % 3 * 4 for i in range(n)],
        [-1 if i % 5 == 3 else i for i in range(n)],
        [0.75 + 0.249 * h / heads for h in range(heads)], max(lens), n + heads)


@pytest.mark.parametrize("tokens", [100, 200])        # a chunk; two
def test_states_of_values_that_are_not_finite(tokens):
    """One chunk or more: a value that is not finite ends up in its column alone."""
    g = torch.Generator().manual_seed(5)
    rows = torch.randn(tokens, 3 * 128, generator=g).to(torch.bfloat16)
    rows[7, 256 + 40] = float("inf")
    rows[90, 256 + 41] = float("nan")
    rows = rows.cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    state = torch.zeros(1, 1, 128, 128, device="cuda")
    out = torch.zeros(tokens, 1, 128, device="cuda")
    H.decay_attn(*rows.chunk(3, 1), torch.full((1,), 0.97, device="cuda"), state,
                 torch.zeros(1, **i32), torch.tensor([0, tokens], **i32),
                 torch.zeros(1, **i32), out, max_q_len=tokens)
    odd = ~torch.isfinite(state[0, 0]).cpu()
    assert odd[:, 40:42].all() and not odd[:, :40].any() and not odd[:, 42:].any()
