"""Two FP8 linears in one launch (ops.fp8_linear_pair): every form of the rule at sizes with remainders, rows of one problem beside
columns of the other's weights, and each epilogue, against 64-bit references and the calls one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows of both, n, k: 64x64 and 128x128 tiles, the forms that share k, 256x256 tiles (plain: four wavefronts, else eight), 128x256
SIZES = [(100, 33, 64, 256), (1000, 300, 3072, 1024), (33, 65, 3072, 1280), (190, 77, 9280, 1152), (400, 100, 3072, 2176),
         (1200, 300, 3072, 1152), (4000, 300, 3072, 1152), (4096, 333, 9216, 1152), (2300, 500, 12288, 1152), (300, 20, 640, 1280)]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m1,m2,n,k", SIZES)
def test_fp8_pair(dev, dt, m1, m2, n, k):
    from lyradiff_amd import ops

    half_ulp = 2.0 ** -11 if dt == torch.float16 else 2.0 ** -8
    g = torch.Generator(device=dev).manual_seed(m1 + m2 + n + k)
    s8 = torch.full((1,), 0.05, device=dev)
    probs = []
    for i, m in enumerate((m1, m2)):
        a, w = (torch.randn(r, k, generator=g, device=dev).clamp_(-4, 4).to(torch.float8_e4m3fn) for r in (m, n))
        sa, sw = torch.full((1,), 0.25 * (i + 1), device=dev), torch.full((1,), 0.125, device=dev)
        bias = torch.randn(n, generator=g, device=dev).to(dt)
        factor = 0.25 * (i + 1) * 0.125
        ref = a.float().double() @ w.float().double().t() * factor + bias.double()
        # as in the forms of few tiles: half an ulp of T, 13 bits under a matrix instruction's largest product, 24 under the running sum
        terms = a.float().abs() @ w.float().abs().t() * factor
        bound = 1.01 * half_ulp * ref.abs() + (k // 64) * 64 * factor * 16 * 2.0 ** -13 + (k // 64 + 4) * 2.0 ** -24 * terms
        codes = a.view(torch.uint8)
        panels = codes.view(m, k // 64, 64).transpose(0, 1).contiguous()
        lin = (ops.repack_weight(w.view(torch.uint8)), sa, sw, bias)
        gate, res = torch.randn(1, n, generator=g, device=dev).to(dt), torch.randn(m, n, generator=g, device=dev).to(dt)
        probs.append((codes, panels, lin, ref, bound, gate, res, m))
    pair = lambda panels, gelu=0, **kw: ops.fp8_linear_pair(*(ops.FP8Half(p[1] if panels else p[0], *p[2], **{key: f(p) for key, f in kw.items()})
                                                              for p in probs), dt, gelu, panels)
    plain = pair(True)
    for y, r, (_, _, _, ref, bound, _, _, m) in zip(plain, pair(False), probs):
        assert bool(((y.double() - ref).abs() <= bound).all()) and torch.equal(y, r), m
    for y, got, p in zip(plain, pair(True, gate=lambda p: p[5], residual=lambda p: p[6], rows_per_gate=lambda p: p[7]), probs):
        assert torch.equal(got, y * p[5] + p[6]), p[7]  # every form of one size sums in the same order, whatever its epilogue
    cast = lambda y: (y.float() * (1.0 / s8)).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    for y, got in zip(plain, pair(False, out_fp8_scale=lambda p: s8)):
        assert torch.equal(got, cast(y))
    for dense, got in zip(pair(False, 1, out_fp8_scale=lambda p: s8), pair(True, 1, out_fp8_scale=lambda p: s8)):
        assert torch.equal(ops.fp8_panels_to_rows(got), dense)


def test_fp8_pair_with_an_empty_half_and_bad_arguments(dev):
    from lyradiff_amd import ops

    w, one = ops.repack_weight(torch.ones(64, 128, dtype=torch.uint8, device=dev)), torch.ones(1, device=dev)
    x, none = (torch.full((2, m, 64), 0x38, dtype=torch.uint8, device=dev) for m in (40, 0))
    a, b = ops.fp8_linear_pair(ops.FP8Half(x, w, one, one), ops.FP8Half(none, w, one, one), torch.bfloat16)
    assert torch.equal(a, ops.fp8_linear_panels(x, w, one, one, None)) and b.shape == (0, 64)
    with pytest.raises(TypeError):
        ops.fp8_linear_pair(ops.FP8Half(x, w, one, one), ops.FP8Half(x, w, one, one), torch.float32)
    with pytest.raises(ValueError):
        ops.fp8_linear_pair(ops.FP8Half(x, w, one, one), ops.FP8Half(x, w[:32], one, one), torch.float16)
    with pytest.raises(RuntimeError):  # outputs of two kinds
        ops.fp8_linear_pair(ops.FP8Half(x, w, one, one), ops.FP8Half(x, w, one, one, None, one), torch.float16)


# codes of full tiles (four rows a step) against those of partial ones (value by value): the same problem with one row less; 64x64, 128x128
# and 256-wide tiles, k shared between wavefront groups
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(64, 64, 128), (1024, 2048, 256), (256, 768, 2048), (4096, 3072, 1152), (4352, 3072, 1152)])
@pytest.mark.parametrize("gelu", [0, 1, 2])
def test_codes_of_full_and_of_partial_tiles_are_the_same(dev, m, n, k, dt, gelu):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k)
    a, w = (torch.randn(r, k, generator=g, device=dev).clamp_(-4, 4).to(torch.float8_e4m3fn).view(torch.uint8) for r in (m, n))
    bias = torch.randn(n, generator=g, device=dev)
    bias[5], bias[n // 2], bias[n - 3] = float("inf"), float("-inf"), float("nan")
    lin = (ops.repack_weight(w), torch.full((1,), k ** -0.5, device=dev), torch.ones(1, device=dev), bias.to(dt), torch.full((1,), 0.02, device=dev))
    codes = lambda rows: ops.fp8_panels_to_rows(ops.fp8_linear_codes_panels(a[:rows].view(rows, k // 64, 64).transpose(0, 1).contiguous(), *lin, gelu=gelu,
                                                                            round_dtype=dt))
    full, part = codes(m), codes(m - 1)
    assert torch.equal(full[:-1], part) and bool(((full[:, n - 3] & 0x7F) == 0x7F).all())


# gates of full tiles (a band's rows of the residual in registers) and of partial ones, with gates that change inside a tile and on its edge
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,rows", [(64, 64, 128, 24), (1024, 2048, 256, 100), (1024, 2048, 256, 512), (256, 768, 2048, 37), (4096, 3072, 1152, 1000), (4352, 3072, 1152, 17)])
def test_gates_that_change_inside_a_tile(dev, m, n, k, rows, dt):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(m + n + k + rows)
    a, w = (torch.randn(r, k, generator=g, device=dev).clamp_(-4, 4).to(torch.float8_e4m3fn).view(torch.uint8) for r in (m, n))
    lin = (ops.repack_weight(w), torch.full((1,), k ** -0.5, device=dev), torch.ones(1, device=dev), torch.randn(n, generator=g, device=dev).to(dt))
    gate, res = (torch.randn(r, n, generator=g, device=dev).to(dt) for r in (-(-m // rows), m))
    panels = lambda count: a[:count].view(count, k // 64, 64).transpose(0, 1).contiguous()
    for count in (m, m - 1):
        got = ops.fp8_linear_gated_panels(panels(count), *lin, gate[: -(-count // rows)], res[:count], rows_per_gate=rows)
        want = ops.fp8_linear_panels(panels(count), *lin, None, dt) * gate.repeat_interleave(rows, 0)[:count] + res[:count]
        assert torch.equal(got, want), (count, int((got != want).sum()))
    # in place: the residual is the output
    half = ops.FP8Half(panels(m), *lin, gate=gate, residual=res, rows_per_gate=rows, out=res)
    want = ops.fp8_linear_panels(panels(m), *lin, None, dt) * gate.repeat_interleave(rows, 0)[:m] + res
    empty = ops.FP8Half(panels(0), *lin, gate=gate[:0], residual=res[:0], rows_per_gate=rows)
    assert torch.equal(ops.fp8_linear_pair(half, empty, dt)[0], want)
