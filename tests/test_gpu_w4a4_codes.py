"""The W4A4 linear on codes (one e4m3 byte per 4-bit value) against the packed-nibble kernels, which tests/test_gpu_quant.py and
tests/test_gpu_gemm.py hold against the oracle: the arithmetic is the same, so every bit has to be."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, outputs, k: one row, tiles of 64 and 128 rows and columns less / exactly / more than full, one and several k-tiles; 1201 x
# 3072 is 456 tiles of 64 x 128 and 2945 x 3072 is 552 of 128 x 128, where the next larger tile takes over
SHAPES = [(1, 32, 128), (63, 96, 256), (64, 64, 384), (65, 160, 128), (129, 3072, 512), (1201, 3072, 256), (2945, 3072, 256), (4608, 9216, 128)]


def _values(words):
    """int32 words [R, K/8] -> signed values [R, K]."""
    shifts = torch.arange(0, 32, 4, device=words.device, dtype=torch.int64)
    v = (words.to(torch.int64)[..., None] >> shifts) & 15
    return torch.where(v > 7, v - 16, v).reshape(words.shape[0], -1)


def _make(dev, m, n, k, dt):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    x = rnd(m, k)
    x[0, :64] = 0.0         # a group of zeros
    x[-1, 64:128] *= 1e-41  # subnormal scale: the exact-division path
    return (x.to(dt), 0.5 + torch.rand(k, generator=g, device=dev), (0.05 * rnd(32, k)).to(dt), torch.randint(-128, 128, (n, k // 2), generator=g, device=dev, dtype=torch.int8),
            0.01 * torch.rand(n, k // 64, generator=g, device=dev), (0.05 * rnd(n, 32)).to(dt), rnd(n).to(dt), rnd)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_linear_on_codes_is_bit_identical(dev, m, n, k, dt):
    from lyradiff_amd import ops

    x, smooth, down, packed, sb, up, bias, rnd = _make(dev, m, n, k, dt)
    words, sa, act = ops.w4a4_quant_lora_down(x, smooth, down)
    codes, sa_t, act_c = ops.w4a4_quant_lora_down_codes(x, smooth, down)
    assert torch.equal(codes.view(torch.float8_e4m3fn).float(), _values(words).float())
    assert torch.equal(sa_t, sa.t()) and torch.equal(act_c, act)

    w = ops.repack_weight(packed.view(torch.uint8))
    wc = ops.w4a4_expand_weight(w)
    assert torch.equal(ops.unpack_weight(wc).view(torch.float8_e4m3fn).float(), _values(packed.view(torch.int32)).float())
    sb_t = sb.t().contiguous()
    add, res, gate = rnd(m, n).to(dt), rnd(m, n).to(dt), rnd((m + 6) // 7, n).to(dt)
    s8 = torch.tensor([0.05], device=dev)
    for epi in ({}, {"gelu": 2}, {"addend": add, "gate": gate, "residual": res, "rows_per_gate": 7}, {"gelu": 1, "out_fp8_scale": s8, "want_output": False}):
        want = ops.w4a4_linear(words, w, sa, sb, bias, dt, 64, act, up, **epi)
        got = ops.w4a4_linear_codes(codes, wc, sa_t, sb_t, bias, dt, act, up, **epi)
        assert torch.equal(got, want), (m, n, k, sorted(epi))
    assert torch.equal(ops.w4a4_linear_codes(codes, wc, sa_t, sb_t, None, dt), ops.w4a4_linear(words, w, sa, sb, None, dt))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_codes_of_nan_and_infinite_groups_are_those_of_the_packed_form(dev, dt):
    """A NaN never enters a group's maximum and becomes 0, beside finite values as beside an infinity, whose group has an infinite scale."""
    from lyradiff_amd import ops

    m, n, k = 40, 64, 256
    x, smooth, down, packed, sb, _, bias, _ = _make(dev, m, n, k, dt)
    nan, inf = float("nan"), float("inf")
    x[1, 3] = nan
    x[2, 64:72] = nan                      # all of a lane
    x[3, 128:192] = nan                    # all of a group
    x[4, 10], x[4, 11] = inf, nan
    x[5, 70] = -inf
    x[6, 200], x[6, 207], x[6, 255] = nan, 3e4, -nan
    words, sa, act = ops.w4a4_quant_lora_down(x, smooth, down)
    codes, sa_t, act_c = ops.w4a4_quant_lora_down_codes(x, smooth, down)
    assert torch.equal(codes.view(torch.float8_e4m3fn).float(), _values(words).float())
    assert torch.equal(sa_t.view(torch.int32), sa.t().contiguous().view(torch.int32))
    assert torch.equal(act_c.isnan(), act.isnan())

    w = ops.repack_weight(packed.view(torch.uint8))
    want = ops.w4a4_linear(words, w, sa, sb, bias, dt)
    got = ops.w4a4_linear_codes(codes, ops.w4a4_expand_weight(w), sa_t, sb.t().contiguous(), bias, dt)
    assert torch.isfinite(got[[1, 2, 3, 6]]).all()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


def test_linear_module_takes_either_form(dev):
    from lyradiff_amd import ops
    from lyradiff_amd.weights import W4A4Linear

    x, smooth, down, packed, sb, up, bias, _ = _make(dev, 200, 256, 384, torch.bfloat16)
    lin = W4A4Linear(ops.repack_weight(packed.view(torch.uint8)), sb, smooth, up, down, bias)
    want = lin.forward(x)  # as constructed: packed nibbles
    assert lin.weight_codes is None and lin.use_codes().weight_codes is not None
    assert torch.equal(lin.forward(x), want)


def test_linear_module_follows_its_weight_and_its_low_rank_branch(dev):
    from lyradiff_amd import ops
    from lyradiff_amd.weights import W4A4Linear

    x, smooth, down, packed, sb, up, bias, rnd = _make(dev, 96, 256, 384, torch.bfloat16)
    make = lambda: W4A4Linear(ops.repack_weight(packed.view(torch.uint8)), sb.clone(), smooth, up, down, bias)

    def scale_in_place(lin):
        lin.weight_scale.mul_(2.0)

    def other_weight(lin):
        lin.weight_rows32 = lin.weight_rows32.flip(0).contiguous()

    def weight_in_place(lin):
        lin.weight_rows32.copy_(lin.weight_rows32.flip(0))

    def no_branch(lin):
        lin.lora_up = lin.lora_down = None

    def wider_branch(lin):
        lin.lora_up, lin.lora_down = torch.cat([up, up], 1), torch.cat([down, down])

    for change in (scale_in_place, other_weight, weight_in_place, no_branch, wider_branch):
        lin, plain = make().use_codes(), make()
        before = lin.forward(x)
        change(lin), change(plain)
        want = plain.forward(x)
        assert not torch.equal(before, want) and torch.equal(lin.forward(x), want), change.__name__
        assert torch.equal(lin.use_codes().forward(x), want), change.__name__


@pytest.mark.parametrize("inference", [False, True])  # the tensors of an inference_mode block count no versions
@pytest.mark.parametrize("write", ["repack_out", "data", "in_place", "scale_data", "copy"])
def test_linear_module_sees_writes_that_autograd_does_not(dev, write, inference):
    from lyradiff_amd import ops
    from lyradiff_amd.weights import W4A4Linear

    with torch.inference_mode(inference):
        x, smooth, down, packed, sb, up, bias, _ = _make(dev, 4608, 3072, 2048, torch.bfloat16)
        make = lambda: W4A4Linear(ops.repack_weight(packed.view(torch.uint8)), sb.clone(), smooth, up, down, bias)
        other = packed.flip(0).contiguous().view(torch.uint8)
        change = {"repack_out": lambda lin: ops.repack_weight(other, out=lin.weight_rows32),  # the library's own writer
                  "data": lambda lin: lin.weight_rows32.data.bitwise_xor_(0x11),
                  "in_place": lambda lin: lin.weight_rows32.copy_(lin.weight_rows32.flip(0)),
                  "scale_data": lambda lin: lin.weight_scale.data.mul_(2.0),
                  "copy": lambda lin: lin.weight_scale.copy_(lin.weight_scale.flip(0))}[write]
        lin, plain = make().use_codes(), make()
        before = lin.forward(x)
        assert torch.equal(before, plain.forward(x))
        change(lin), change(plain)
        want = plain.forward(x)
        assert not torch.equal(before, want) and torch.equal(lin.forward(x), want)


# edges of the kernel's 32-row, 512-wide pieces: the last one with two groups, with one (k % 128 == 64), with all eight
@pytest.mark.parametrize("n,k", [(32, 64), (96, 448), (64, 512), (160, 640), (32, 1088), (3072, 3072)])
def test_weight_laid_out_for_one_call(dev, n, k):
    from lyradiff_amd import ops

    g = torch.Generator(device=dev).manual_seed(n + k)
    w = torch.randint(0, 256, (n, k // 2), generator=g, device=dev, dtype=torch.uint8)
    sb = torch.rand(n, k // 64, generator=g, device=dev)
    codes, sb_t = ops.w4a4_weight_codes(w, sb)
    assert torch.equal(codes, ops.w4a4_expand_weight(w)) and torch.equal(sb_t, sb.t())


def test_linear_module_without_smoothing_or_with_a_small_batch_takes_the_packed_weight(dev):
    from lyradiff_amd import ops
    from lyradiff_amd.weights import W4A4Linear

    x, smooth, down, packed, sb, up, bias, _ = _make(dev, 4608, 3072, 2048, torch.bfloat16)
    lin = W4A4Linear(ops.repack_weight(packed.view(torch.uint8)), sb, smooth, up, down, bias).use_codes()
    assert lin._on_codes(x) and not lin._on_codes(x[:64])
    lin.smooth = None  # the quantiser on codes needs divisors, the packed one does not
    words, sa, act = ops.w4a4_quant_lora_down(x, None, down)
    assert torch.equal(lin.forward(x), ops.w4a4_linear(words, lin.weight_rows32, sa, sb, bias, torch.bfloat16, 64, act, up))
