"""The FP8 GEMM of at most 32 rows against the tiled forms, which sum in the same order (an epilogue with a running maximum takes them;
tests/test_gpu_gemm_few_tiles.py holds those against 64-bit references): every bit has to agree."""
import pytest
import torch

# rows 1, 2, all but one and all of a matrix instruction (33: the tiled form itself); k gives 5, 6, 7, 12 and 48 rounds of four k-tiles,
# less than, exactly and more than the six that are requested ahead
SIZES = [(1, 32, 1280), (2, 96, 1536), (31, 3072, 1792), (32, 1056, 3072), (33, 96, 3072), (1, 18432, 3072), (17, 3072, 12288)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_fp8_few_rows(dev, m, n, k, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, w = (torch.randn(r, k, generator=g, device=dev).to(torch.float8_e4m3fn).view(torch.uint8) for r in (m, n))
    sa, sw = torch.full((1,), 0.3, device=dev), torch.full((1,), 0.01, device=dev)
    panels, w32 = a.view(m, k // 64, 64).transpose(0, 1).contiguous(), ops.repack_weight(w)
    for bias in (torch.randn(n, generator=g, device=dev).to(dt), None):
        want = ops.fp8_linear_panels(panels, w32, sa, sw, bias, torch.zeros(1, device=dev), dt)
        assert torch.equal(ops.fp8_linear_panels(panels, w32, sa, sw, bias, None, dt), want)
        assert torch.equal(ops.fp8_linear(a, w32, sa, sw, bias, out_dtype=dt), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [16, 17, 32, 33])  # rows of K bytes leave the form at 17, k-panels at 33
def test_fp8_few_rows_leave_the_form_without_a_bit_changed(dev, m):
    from lyradiff_amd import ops

    n, k = 9216, 3072
    g = torch.Generator(device=dev).manual_seed(m)
    a, w = (torch.randn(r, k, generator=g, device=dev).to(torch.float8_e4m3fn).view(torch.uint8) for r in (33, n))
    one, w32 = torch.ones(1, device=dev), ops.repack_weight(w)
    a = a[:m].contiguous()
    got = ops.fp8_linear(a, w32, one, one, None, out_dtype=torch.bfloat16)
    assert torch.equal(got, ops.fp8_linear_panels(a.view(m, k // 64, 64).transpose(0, 1).contiguous(), w32, one, one, None, None, torch.bfloat16))
    if m <= 32:  # the same sums, row by row
        assert torch.equal(got[:1], ops.fp8_linear(a[:1].contiguous(), w32, one, one, None, out_dtype=torch.bfloat16))
