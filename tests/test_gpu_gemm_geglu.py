"""The INT8 up projection with GEGLU and the next linear's codes in its epilogue against the two kernels it stands for, which
tests/test_gpu_gemm.py and tests/test_gpu_quant.py hold against the oracle: the arithmetic is the same, so every code has to be."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, outputs, k: one row, tiles of 128 and 256 rows less / exactly / more than full, the fewest and more k-tiles; at most one tile per
# workgroup (700 x 2560: 240 tiles of 128 rows) and several, where the transfers run on across tiles (1024 and 897 x 2560: 320 tiles of 128
# rows; 2049 x 2560: 360 of 256), also with k = 256, where a tile is as long as the pipeline and the next one's columns are requested in the
# first step behind an epilogue
SHAPES = [(1, 64, 256), (127, 64, 320), (128, 128, 256), (129, 192, 640), (700, 2560, 640), (1024, 5120, 1280), (2049, 2560, 640), (8192, 2560, 640),
          (1024, 2560, 640), (897, 2560, 256), (2049, 2560, 256)]


@pytest.mark.parametrize("m,inner,k", SHAPES)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_same_codes_as_gemm_then_geglu(dev, m, inner, k, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + inner + k)
    rnd = lambda *s: torch.rand(*s, generator=g, device=dev)
    codes = lambda *s: torch.randint(-128, 128, s, generator=g, device=dev, dtype=torch.int8)
    a, w = codes(m, k), ops.repack_weight(codes(2 * inner, k))
    # results of the size of a few units; a column of tiny gates, one of large ones and one of infinities leave the gate's table
    col = (0.5 + rnd(2 * inner)) * (2.0 / (73.0 * 73.0 * k ** 0.5))
    col[inner + 3], col[inner + 8], col[inner + 40] = 1e-9, 1.0, 3e38
    row, scale, pre = torch.full((1,), 1.1, device=dev), torch.full((1,), 0.03, device=dev), 0.7 + 0.6 * rnd(inner)
    bias = torch.randn(2 * inner, generator=g, device=dev).to(dt)
    bias[inner + 3] = 0.0
    for b, p in ((bias, pre), (bias, None), (None, pre)):
        want = ops.geglu_int8(ops.int8_linear(a, w, col, row, None, dt), b, p, scale)
        got = ops.int8_linear_geglu(a, w, col, row, b, p, scale, dt)
        assert torch.equal(got, want), (m, inner, k, b is None, p is None, int((got != want).sum()))
    zero = torch.zeros(1, device=dev)  # a scale without a reciprocal
    assert torch.equal(ops.int8_linear_geglu(a, w, col, row, bias, pre, zero, dt), ops.geglu_int8(ops.int8_linear(a, w, col, row, None, dt), bias, pre, zero))


def test_other_forms_keep_to_the_two_kernels(dev):
    from lyradiff_amd import ops

    a, w = torch.ones(40, 128, device=dev, dtype=torch.int8), ops.repack_weight(torch.ones(64, 128, device=dev, dtype=torch.int8))
    col, row, scale = torch.full((64,), 1e-2, device=dev), torch.ones(1, device=dev), torch.full((1,), 0.05, device=dev)
    want = ops.geglu_int8(ops.int8_linear(a, w, col, row, None, torch.float16), None, None, scale)
    assert torch.equal(ops.int8_linear_geglu(a, w, col, row, None, None, scale, torch.float16), want)
    with pytest.raises(ValueError):
        wide = ops.repack_weight(torch.ones(128, 256, device=dev, dtype=torch.int8))
        ops.int8_linear_geglu(torch.ones(4, 256, device=dev, dtype=torch.int8), wide, torch.ones(128, device=dev), row, torch.zeros(64, device=dev, dtype=torch.float16),
                              None, scale, torch.float16)


def test_tactics_of_the_up_projection_stand(dev, monkeypatch):
    from lyradiff_amd import lib, ops

    m, inner, k = 64, 128, 256
    a, w = torch.ones(m, k, device=dev, dtype=torch.int8), ops.repack_weight(torch.ones(2 * inner, k, device=dev, dtype=torch.int8))
    args = (a, w, torch.full((2 * inner,), 1e-2, device=dev), torch.ones(1, device=dev), None, None, torch.full((1,), 0.05, device=dev), torch.float16)
    want, calls = ops.int8_linear_geglu(*args), []
    plain = ops.int8_linear
    monkeypatch.setattr(ops, "int8_linear", lambda *a: (calls.append(1), plain(*a))[1])
    assert torch.equal(ops.int8_linear_geglu(*args), want) and not calls
    with ops.gemm_thread_tactic(2):
        assert torch.equal(ops.int8_linear_geglu(*args), want) and len(calls) == 1
    try:
        ops.gemm_shape_tactic("int8", m, 2 * inner, k, 3)
        assert torch.equal(ops.int8_linear_geglu(*args), want) and len(calls) == 2
    finally:
        ops.gemm_shape_tactic("int8", m, 2 * inner, k, -1)
    takes = lib.load().lq_gemm_int8_geglu_takes
    assert takes(m, inner, k) and not takes(m, inner, 192) and not takes(m, inner, 288) and not takes(m, 96, k) and not takes(-1, inner, k)


# every configuration that the rule picks (64x64, k shared, 128x128, 128x256, 256x256 tiles), full and ragged tiles.  4352x4096x1152 is 272
# whole tiles of 256x256: the plain product takes the persistent form, which declines a residual, and the sum the plain 256x256 tiles
@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (130, 96, 192), (200, 640, 2560), (1024, 1280, 1280), (4096, 640, 2560), (4100, 1280, 640), (2048, 5120, 2048), (8192, 5120, 64),
                                   (4100, 10240, 640), (4352, 4096, 1152), (4100, 3072, 1152)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_int8_linear_with_a_residual_is_the_sum(dev, m, n, k, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    codes = lambda *s: torch.randint(-128, 128, s, generator=g, device=dev, dtype=torch.int8)
    a, w = codes(m, k), ops.repack_weight(codes(n, k))
    col, row = 1e-4 * torch.rand(n, generator=g, device=dev), torch.full((1,), 0.9, device=dev)
    bias, add = torch.randn(n, generator=g, device=dev).to(dt), torch.randn(m, n, generator=g, device=dev).to(dt)
    for b in (bias, None):
        plain = ops.int8_linear(a, w, col, row, b, dt)
        if m > 1:  # the same scale given per row
            assert torch.equal(plain, ops.int8_linear(a, w, col, row.repeat(m), b, dt))
        assert torch.equal(ops.int8_linear(a, w, col, row, b, dt, addend=add), plain + add)
    strided = torch.randn(n, m, generator=g, device=dev).to(dt).t()
    assert torch.equal(ops.int8_linear(a, w, col, row, bias, dt, addend=strided), ops.int8_linear(a, w, col, row, bias, dt) + strided)


def test_a_residual_that_pytorch_has_to_see_is_added_by_pytorch(dev):
    """A sum that records a gradient, carries a tangent or runs under vmap, as it was with a sum behind the linear."""
    from torch.autograd import forward_ad

    from lyradiff_amd import ops

    a, w = torch.ones(8, 64, device=dev, dtype=torch.int8), ops.repack_weight(torch.ones(32, 64, device=dev, dtype=torch.int8))
    call = lambda r: ops.int8_linear(a, w, torch.full((32,), 1e-2, device=dev), torch.ones(1, device=dev), None, torch.float16, addend=r)
    res = torch.randn(3, 8, 32, device=dev).half()
    want = torch.stack([call(r) for r in res])
    leaf = res[0].clone().requires_grad_()
    call(leaf).backward(res[1])
    assert torch.equal(leaf.grad, res[1])
    with torch.no_grad():
        assert torch.equal(call(leaf), want[0])
    with forward_ad.dual_level():
        y, tangent = forward_ad.unpack_dual(call(forward_ad.make_dual(res[0], res[1])))
        assert torch.equal(y, want[0]) and torch.equal(tangent, res[1])
    assert torch.equal(torch.vmap(call)(res), want)
