"""FP8 and INT8 GEMMs of few tiles, whose wavefront groups share k out or whose eight wavefronts walk 128-byte k-tiles: every form at the edges of
its range (remainders of rows and columns, the smallest k, activations as rows and as k-panels) and the epilogues of the FLUX blocks, against
64-bit references."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (m, n, k): 32x32, 32x64 (k a multiple of 256), 64x128, 128x128 (a multiple of 128), and k that no form takes; eight wavefronts on 224, 256 and
# 264 tiles of 128x128, the last as 192x128
SIZES = [(1, 32, 1280), (33, 3072, 1280), (77, 3040, 1536), (65, 9216, 1152), (190, 9248, 1152), (333, 9216, 1152), (100, 12320, 2176),
         (300, 1056, 1088), (1000, 3552, 2048), (1024, 4096, 2176), (1000, 4128, 2048)]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_int8_few_tiles_exact(dev, dt):
    from lyradiff_amd import ops

    for m, n, k in SIZES:
        g = torch.Generator(device=dev).manual_seed(m + n + k)
        a, w = (torch.randint(-127, 128, (r, k), generator=g, device=dev, dtype=torch.int8) for r in (m, n))
        col, row = (1e-4 * (0.5 + torch.rand(r, generator=g, device=dev)) for r in (n, m))
        bias = torch.randn(n, generator=g, device=dev).to(dt)
        acc = (a.double() @ w.double().t()).float()  # integers below 2^24: the 32-bit sums, exactly
        want = (acc * (col[None] * row[:, None]) + bias.float()).to(dt)
        w32 = ops.repack_weight(w)
        assert torch.equal(ops.int8_linear(a, w32, col, row, bias, dt), want), (m, n, k)
        panels = a.view(m, k // 64, 64).transpose(0, 1).contiguous()
        assert torch.equal(ops.int8_linear_panels(panels, w32, col, row, bias, dt), want), (m, n, k, "panels")


def _fp8(shape, g, dev):
    return torch.randn(shape, generator=g, device=dev).clamp_(-4, 4).to(torch.float8_e4m3fn)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_fp8_few_tiles(dev, dt):
    from lyradiff_amd import ops

    half_ulp = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    for m, n, k in SIZES:
        g = torch.Generator(device=dev).manual_seed(m + n + k)
        a, w = _fp8((m, k), g, dev), _fp8((n, k), g, dev)
        sa, sw = torch.full((1,), 0.25, device=dev), torch.full((1,), 0.125, device=dev)
        bias = torch.randn(n, generator=g, device=dev).to(dt)
        acc = a.double() @ w.double().t() / 32
        ref = acc + bias.double()
        # half an ulp of T, and per matrix instruction (64 of k) 13 bits under its largest product (at most 16 here, times 1/32)
        # and 24 bits under the running sum
        terms = a.double().abs() @ w.double().abs().t() / 32
        bound = 1.01 * half_ulp * ref.abs() + (k // 64) * 64 * 0.5 * 2.0 ** -13 + (k // 64 + 4) * 2.0 ** -24 * terms
        codes, w32 = a.view(torch.uint8), ops.repack_weight(w.view(torch.uint8))
        y = ops.fp8_linear(codes, w32, sa, sw, bias, out_dtype=dt)
        assert bool(((y.double() - ref).abs() <= bound).all()), (m, n, k)
        panels = codes.view(m, k // 64, 64).transpose(0, 1).contiguous()
        top = torch.zeros(1, device=dev)
        assert torch.equal(ops.fp8_linear_panels(panels, w32, sa, sw, bias, top, dt), y), (m, n, k, "panels")
        assert float(top) == max(0.0, float(y.float().max()))
        # gate and residual: T(T(T(y) * gate) + residual) from the plain result
        gate, res = torch.randn(1, n, generator=g, device=dev).to(dt), torch.randn(m, n, generator=g, device=dev).to(dt)
        got = ops.fp8_linear_gated(codes, w32, sa, sw, bias, gate, res, m)
        assert torch.equal(got, (y * gate + res)), (m, n, k, "gated")
        # codes of the plain result, and the tanh GELU before them to one code
        s8 = torch.full((1,), 0.05, device=dev)
        got8 = ops.fp8_linear_codes(codes, w32, sa, sw, bias, s8, 0, dt)
        assert torch.equal(got8, (y.float() * (1.0 / s8)).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)), (m, n, k, "codes")


def test_a_cached_tactic_stands(dev):
    """The tactics add the k-tiles up in one sequence, where 2^-9 beside 448 * 448 is lost before that is taken off again; a form that
    shares k keeps it, in a sum of another group."""
    from lyradiff_amd import ops

    m, n, k = 64, 64, 1280
    a, w = (torch.zeros(r, k, device=dev) for r in (m, n))
    a[:, [0, 64, 256]] = torch.tensor([448.0, 2.0 ** -6, 448.0], device=dev)
    w[:, [0, 64, 256]] = torch.tensor([448.0, 2.0 ** -3, -448.0], device=dev)
    a, w = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, w))
    one, w32 = torch.ones(1, device=dev), ops.repack_weight(w)
    run = lambda: ops.fp8_linear(a, w32, one, one, None, out_dtype=torch.bfloat16)
    shared = torch.full((m, n), 2.0 ** -9, dtype=torch.bfloat16, device=dev)
    assert torch.equal(run(), shared)
    for rows in (m, 128):  # the exact entry, and that of the next power of two for 65 to 128 rows
        try:
            ops.gemm_shape_tactic("fp8", rows, n, k, 3)
            x = a if rows == m else torch.cat([a, a])[:100].contiguous()
            assert not ops.fp8_linear(x, w32, one, one, None, out_dtype=torch.bfloat16).any()
        finally:
            ops.gemm_shape_tactic("fp8", rows, n, k, -1)
    assert torch.equal(run(), shared)


# tiles of 128x128 and 192x128 in 128-byte k-tiles: one round of either, one tile less and more than a round of the former, k from where INT8
# takes them on, rows and columns that leave tiles partly filled; two rounds, which k-panels and at short k more than scales and bias leave to
# other tiles
@pytest.mark.parametrize("m,n,k", [(6000, 640, 640), (8191, 608, 768), (8192, 640, 1024), (2040, 2048, 1280), (2049, 2048, 1280), (1345, 3040, 1152),
                                   (900, 9184, 1152), (1000, 9216, 2560)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_forms_of_eight_wavefronts(dev, m, n, k, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, w = (torch.randint(-127, 128, (r, k), generator=g, device=dev, dtype=torch.int8) for r in (m, n))
    col, row = (1e-4 * (0.5 + torch.rand(r, generator=g, device=dev)) for r in (n, m))
    bias, add = torch.randn(n, generator=g, device=dev).to(dt), torch.randn(m, n, generator=g, device=dev).to(dt)
    acc = (a.double() @ w.double().t()).float()  # integers below 2^24: the 32-bit sums, exactly
    want = lambda s: (acc * (col[None] * s) + bias.float()).to(dt)
    w32, panels = ops.repack_weight(w), a.view(m, k // 64, 64).transpose(0, 1).contiguous()
    assert torch.equal(ops.int8_linear(a, w32, col, row, bias, dt), want(row[:, None]))
    assert torch.equal(ops.int8_linear_panels(panels, w32, col, row, bias, dt), want(row[:, None]))
    assert torch.equal(ops.int8_linear(a, w32, col, row[:1], bias, dt, add), want(row[:1]) + add)

    # e4m3: as above, a 13-bit sum of a matrix instruction's products and 24 bits for the running one
    a, w = _fp8((m, k), g, dev), _fp8((n, k), g, dev)
    one, w32 = torch.ones(1, device=dev), ops.repack_weight(w.view(torch.uint8))
    ref = a.double() @ w.double().t() + bias.double()
    terms = a.double().abs() @ w.double().abs().t()
    half_ulp = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    bound = 1.01 * half_ulp * ref.abs() + (k // 64) * 64 * 16.0 * 2.0 ** -13 + (k // 64 + 4) * 2.0 ** -24 * terms
    codes = a.view(torch.uint8)
    y = ops.fp8_linear(codes, w32, one, one, bias, out_dtype=dt)
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert torch.equal(ops.fp8_linear_panels(codes.view(m, k // 64, 64).transpose(0, 1).contiguous(), w32, one, one, bias, None, dt), y)
    gate, res = torch.randn(1, n, generator=g, device=dev).to(dt), torch.randn(m, n, generator=g, device=dev).to(dt)
    assert torch.equal(ops.fp8_linear_gated(codes, w32, one, one, bias, gate, res, m), y * gate + res)
