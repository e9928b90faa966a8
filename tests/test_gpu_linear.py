"""x W^T (+ bias) at the edges of its tiles, against fp64 of the bf16 inputs. Sums
are 32-bit and the result is rounded to bf16: 2^-8 of itself (half a step of 2^-7 at
a power of two) and 2^-24 times the square root of the number of terms (K up to
4096: 2^-18) of the sum of absolute products, of which twice as much is allowed."""
import pytest
import torch

from xllm_service_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 32, 33, 63, 64, 65, 100, 129, 300])
@pytest.mark.parametrize("N,K", [(8, 128), (64, 256), (72, 1152), (200, 4096),
                                 (4096, 384), (4104, 384), (2056, 2048),
                                 (3080, 4096), (8192, 2048)])
@pytest.mark.parametrize("bias,stride", [(False, 0), (True, 8)])
def test_linear(M, N, K, bias, stride):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)

    def bf(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(
            torch.bfloat16)
    x = bf(M, K + stride)[:, :K]
    w, b = bf(N, K), bf(N) if bias else None
    got = ops.linear(x, w, b)
    assert got.shape == (M, N) and got.dtype == torch.bfloat16
    want = x.double() @ w.double().t()
    big = x.double().abs() @ w.double().abs().t()
    if bias:
        want, big = want + b.double(), big + b.double().abs()
    off = (got.double() - want).abs() - 2.0 ** -8 * want.abs() \
        - 2.0 ** -17 * big
    assert off.max() <= 0, f"over by {off.max():.3g}"


@pytest.mark.parametrize("M", [8, 9, 16, 17, 24, 25, 32, 48, 49])
@pytest.mark.parametrize("N,K", [(4096, 128), (4112, 640), (6152, 1152),
                                 (8200, 256), (8200, 4096)])
def test_rows_in_steps_of_eight(M, N, K):
    """One and two row tiles of W, with and without a CU for each workgroup;
    fewer steps than waves."""
    test_linear(M, N, K, True, 8)


@pytest.mark.parametrize("M,N,K", [(64, 72, 1152), (65, 72, 1152),
                                   (129, 2056, 2048), (300, 3080, 2048)])
def test_rows_of_a_wider_tensor(M, N, K):
    """Without a bias, with which the library takes over above 64 rows."""
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = (torch.randn(r, K + 8, generator=g, device="cuda").to(torch.bfloat16)
            for r in (M, N))
    x, w = x[:, :K], w[:, :K].contiguous()
    want = x.double() @ w.double().t()
    big = x.double().abs() @ w.double().abs().t()
    off = (ops.linear(x, w).double() - want).abs() - 2.0 ** -8 * want.abs() \
        - 2.0 ** -17 * big
    assert off.max() <= 0, f"over by {off.max():.3g}"


@pytest.mark.parametrize("M,N,K,stride", [
    (65, 64, 128, 0), (97, 136, 256, 8), (128, 3080, 384, 0),    # 32 rows of x
    (200, 2056, 640, 8), (250, 3080, 1152, 0), (300, 4104, 256, 8),
    (380, 4040, 128, 0), (500, 3080, 2048, 8),                   # 128 of W
    (70, 3080, 4736, 0), (2048, 200, 384, 0), (8000, 72, 256, 8),
    (140, 4040, 4224, 0),                                        # 64, not 48, of x
    (70, 200, 128, 8), (350, 1544, 384, 0), (505, 2056, 256, 8),  # short rows
    (126, 8456, 384, 8), (300, 4872, 1024, 0), (577, 2056, 128, 8),  # square tiles
    (65, 16392, 2048, 0), (90, 8456, 1152, 8)])                  # many columns
def test_shapes_of_prompt_tiles(M, N, K, stride):
    """Every shape of a tile, with remainders of both sides and fewer steps than
    buffers; longest rows. 2^-17 covers K up to 4096, 2^-16.8 up to 4736."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = (torch.randn(r, K + stride, generator=g, device="cuda").to(
        torch.bfloat16)[:, :K] for r in (M, N))
    w = w.contiguous()
    want = x.double() @ w.double().t()
    big = x.double().abs() @ w.double().abs().t()
    off = (ops.linear(x, w).double() - want).abs() - 2.0 ** -8 * want.abs() \
        - 2.0 ** -16.8 * big
    assert off.max() <= 0, f"over by {off.max():.3g}"


@pytest.mark.parametrize("M", [1, 8, 24, 33, 64, 65, 100, 250, 500])
@pytest.mark.parametrize("N,K", [(16, 128), (48, 256), (4112, 640), (8208, 384),
                                 (3088, 2048), (4880, 1024)])
def test_gated(M, N, K):
    """Gates and their partners in one product, against fp64: 2^-8 for the result's
    rounding, and of each sum, where a caller's two products round them, 2^-8 more
    and 2^-17 as above, times the other factor (silu turns an error of the gate
    into at most 1.1 of its size)."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = (torch.randn(r, K, generator=g, device="cuda").to(torch.bfloat16)
            for r in (M, N))
    got = ops.linear_gated(x, w).double()
    assert got.shape == (M, N // 2)
    want = x.double() @ w.double().t()
    big = x.double().abs() @ w.double().abs().t()
    off = (2.0 ** -8 * want.abs() + 2.0 ** -17 * big).chunk(2, 1)
    gate, up = want.chunk(2, 1)
    y = torch.nn.functional.silu(gate) * up
    bound = 2.0 ** -8 * y.abs() + 1.1 * off[0] * up.abs() \
        + torch.nn.functional.silu(gate).abs() * off[1] + 1.1 * off[0] * off[1]
    assert ((got - y).abs() - 1.01 * bound).max() <= 0


def test_what_the_kernels_do_not_take():
    """Types, widths, gradients and shapes that go to the library."""
    for dt, M, N, K in ((torch.float32, 4, 64, 128), (torch.bfloat16, 4, 63, 128),
                        (torch.bfloat16, 4, 64, 100), (torch.bfloat16, 0, 8, 128)):
        x, w = (torch.randn(r, K, device="cuda").to(dt) for r in (M, N))
        y = ops.linear(x, w)
        assert torch.equal(y, torch.nn.functional.linear(x, w))
    x = torch.randn(2, 3, 128, device="cuda").to(torch.bfloat16)
    w = torch.randn(64, 128, device="cuda").to(torch.bfloat16)
    assert ops.linear(x, w).shape == (2, 3, 64)
    w.requires_grad_(True)
    ops.linear(x[0], w).float().sum().backward()
    assert w.grad is not None


def test_transforms_go_to_the_library():
    """vmap, forward-mode AD, autocast and a dispatch mode see the call."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    x, w = (torch.randn(r, 128, device="cuda").to(torch.bfloat16)
            for r in (6, 64))
    linear = torch.nn.functional.linear
    assert torch.equal(
        torch.vmap(lambda r: ops.linear(r, w))(x.view(3, 2, 128)),
        torch.vmap(lambda r: linear(r, w))(x.view(3, 2, 128)))
    with forward_ad.dual_level():
        y = ops.linear(forward_ad.make_dual(x, x), w)
        assert forward_ad.unpack_dual(y).tangent is not None
    with torch.autocast("cuda", torch.float16):
        assert ops.linear(x, w).dtype == torch.float16

    class Count(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.calls += 1
            return func(*args, **(kwargs or {}))
    with Count():
        ops.linear(x, w)
    assert Count.calls > 0


def test_bias_that_overrides_the_call():
    """A bias of a class with __torch_function__ is asked, like x and weight."""
    calls = []

    class Seen(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            calls.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})
    x, w = (torch.randn(r, 128, device="cuda").to(torch.bfloat16)
            for r in (6, 64))
    b = torch.randn(64, device="cuda").to(torch.bfloat16).as_subclass(Seen)
    assert isinstance(ops.linear(x, w, b), Seen)
    assert torch.nn.functional.linear in calls


def test_tuned_choices_are_kept():
    """A product that the loaded table of tuned kernels names runs on the library
    where its own kernel is the slower one; its neighbours do not."""
    import os

    import torch.cuda.tunable as tunable
    from torch.profiler import ProfilerActivity, profile
    table = os.path.join(os.path.dirname(__file__), "..", "configs",
                         "tunableop_gfx950.csv")
    x, w = (torch.randn(r, 4096, device="cuda").to(torch.bfloat16)
            for r in (128, 4096))

    def own(w):
        """Whether a kernel of linear.hip ran."""
        ops.linear(x, w)
        with profile(activities=[ProfilerActivity.CUDA]) as seen:
            ops.linear(x, w)
            torch.cuda.synchronize()
        names = [e.key for e in seen.key_averages()]
        if not any(n.startswith(("void xllm", "Cijk")) for n in names):
            pytest.skip(f"no kernel names from the profiler: {names}")
        return any("linear_tile" in n or "linear_stream" in n for n in names)
    was = tunable.is_enabled(), tunable.tuning_is_enabled()
    try:
        tunable.enable(True)
        tunable.tuning_enable(False)
        if not tunable.read_file(table):
            pytest.skip("the table is for other versions of the library")
        assert not own(w)
        assert own(w[:4064])
    finally:
        tunable.enable(was[0])
        tunable.tuning_enable(was[1])
