"""Linears of few rows in one launch: FP8 with the cast of the activation inside (bits of the two calls), and plain 16-bit ones against
64-bit sums; the edges of their ranges and what is left to the other routes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DTS = [torch.float16, torch.bfloat16]


@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("m,n,k", [(1, 32, 1280), (1, 18432, 3072), (4, 96, 3072), (8, 64, 1536), (1, 64, 12288), (3, 9216, 2304)])
def test_fp8_rows_with_the_cast_inside(dev, dt, m, n, k):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=dev).to(dt)
    x[0, 3], x[-1, k - 1] = 1e4, float("nan") if m > 1 else -1e4  # saturation; a row of NaN
    lins = []
    for i in range(2):
        w = torch.randn(n, k, generator=g, device=dev).to(torch.float8_e4m3fn).view(torch.uint8)
        lins.append((ops.repack_weight(w), torch.full((1,), 0.01 * (i + 1), device=dev), torch.full((1,), 0.02, device=dev),
                     torch.randn(n, generator=g, device=dev).to(dt) if i == 0 else None))
    want = [ops.fp8_linear(ops.fp8_scale_cast(x, sa), w, sa, sw, b, out_dtype=dt) for w, sa, sw, b in lins]
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())
    assert same(ops.fp8_linear_rows(x, lins[0]), want[0])
    got = ops.fp8_linear_rows(x, lins[0], lins[1])
    assert same(got[0], want[0]) and same(got[1], want[1])


def test_fp8_rows_leaves_the_rest_to_the_two_calls(dev):
    from lyradiff_amd import ops

    one = torch.ones(1, device=dev)
    lin = lambda n, k: (torch.zeros(n, k, dtype=torch.uint8, device=dev), one, one, None)
    x = lambda m, k: torch.zeros(m, k, dtype=torch.bfloat16, device=dev)
    for m, n, k in ((9, 64, 1280), (2, 64, 12288), (1, 64, 1024), (1, 64, 1344), (1, 32 * 1536, 1280)):
        assert ops.fp8_linear_rows(x(m, k), lin(n, k)) is None, (m, n, k)
    assert ops.fp8_linear_rows(x(0, 1280), lin(64, 1280)).shape == (0, 64)
    try:
        ops.gemm_shape_tactic("fp8", 1, 64, 1280, 3)  # a tactic stands
        assert ops.fp8_linear_rows(x(1, 1280), lin(64, 1280)) is None
    finally:
        ops.gemm_shape_tactic("fp8", 1, 64, 1280, -1)
    with ops.gemm_thread_tactic(2):
        assert ops.fp8_linear_rows(x(1, 1280), lin(64, 1280)) is None
    assert ops.fp8_linear_rows(x(1, 1280), lin(64, 1280)) is not None
    with pytest.raises(ValueError):
        ops.fp8_linear_rows(x(1, 1280), lin(64, 1536))


# one row streams the weight; 64-element pieces fewer than the eight wavefronts, a remainder of 32 rows and columns, the most rows
@pytest.mark.parametrize("dt", DTS)
@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (1, 9216, 3072), (3, 36, 576), (4, 1280, 1600), (5, 36, 64), (33, 100, 448), (154, 640, 2048), (256, 1284, 1088)])
def test_linear16(dev, dt, m, n, k):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    x, w, w2 = (torch.randn(r, k, generator=g, device=dev).to(dt) for r in (m, n, n))
    b = torch.randn(n, generator=g, device=dev).to(dt)
    half_ulp = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    for weight, bias, got in ((w, b, ops.linear16(x, w, b)), *zip((w, w2), (None, b), ops.linear16_pair(x, w, w2, None, b))):
        ref = x.double() @ weight.double().t() + (bias.double() if bias is not None else 0.0)
        terms = x.double().abs() @ weight.double().abs().t()
        bound = 1.01 * half_ulp * ref.abs() + (k // 16 + 12) * 2.0 ** -24 * terms  # one rounding to T; fp32 sums of sixteen products each
        assert bool(((got.double() - ref).abs() <= bound).all())


def test_linear16_takes_batches_and_leaves_the_rest_to_pytorch(dev):
    from lyradiff_amd import ops

    F = torch.nn.functional
    r = lambda *s, dt=torch.bfloat16: torch.randn(*s, device=dev, generator=torch.Generator(device=dev).manual_seed(sum(s))).to(dt)
    x, w = r(2, 77, 128), r(64, 128)
    assert ops.linear16_supported(x, w) and ops.linear16(x, w).shape == (2, 77, 64)
    inf = x.clone()
    inf[0, 0, 5] = float("inf")
    assert torch.equal(ops.linear16(inf, w).isfinite(), F.linear(inf, w).isfinite())
    others = [(r(257, 128), w), (r(2, 100), r(64, 100)), (r(128, 4).t(), r(64, 128)), (r(4, 128, dt=torch.float32), r(64, 128, dt=torch.float32)),
              (r(2, 128), r(66, 128)), (r(0, 128), w), (r(3 * 128 + 4)[4:].view(3, 128), w)]
    for a, b in others:
        assert not ops.linear16_supported(a, b)
        assert torch.equal(ops.linear16(a, b), F.linear(a, b)) and all(torch.equal(y, F.linear(a, b)) for y in ops.linear16_pair(a, b, b))
    leaf = r(2, 128).requires_grad_()
    ops.linear16(leaf, w).float().sum().backward()
    assert leaf.grad is not None and not ops.linear16_supported(leaf, w)
    with torch.no_grad():
        assert ops.linear16_supported(leaf, w)
    with pytest.raises(RuntimeError):
        ops.linear16(r(2, 128), r(64, 192))


def test_linear16_is_pytorchs_where_pytorch_has_to_see_it(dev):
    """Forward-mode tangents, vmap, function transforms, fake tensors, dispatch modes, tracing and autocast, through the layer that uses it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode

    from lyradiff_amd import ops, sdxl_int8

    F = torch.nn.functional
    r = lambda *s: torch.randn(*s, device=dev, generator=torch.Generator(device=dev).manual_seed(sum(s))).half()
    x, w, b = r(3, 8, 128), r(64, 128), r(64)
    lin = sdxl_int8.Linear16(w, b).forward
    with forward_ad.dual_level():
        assert ops.linear16_supported(x, w)  # a level without a tangent changes nothing
        dual = forward_ad.make_dual(x, 2 * x)
        got, want = (forward_ad.unpack_dual(f(dual)) for f in (lin, lambda t: F.linear(t, w, b)))
        assert torch.equal(got.primal, want.primal) and torch.equal(got.tangent, want.tangent)
        assert all(forward_ad.unpack_dual(y).tangent is not None for y in ops.linear16_pair(dual, w, w))
    assert torch.equal(torch.vmap(lin)(x), torch.vmap(lambda t: F.linear(t, w, b))(x))
    assert all(torch.equal(g, e) for g, e in zip(torch.func.jvp(lin, (x,), (x,)), torch.func.jvp(lambda t: F.linear(t, w, b), (x,), (x,))))
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert lin(mode.from_tensor(x)).shape == (3, 8, 64)
    with FlopCounterMode(display=False) as flops:
        lin(x)
    assert flops.get_total_flops() == 2 * x.numel() * 64
    assert torch.equal(torch.jit.trace(lin, (x[:1],))(x), F.linear(x, w, b))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert lin(x).dtype == torch.bfloat16
