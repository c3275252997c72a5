"""What the Python wrappers refuse, and which route they take, before anything is enqueued (no GPU: a call that reaches the library fails
the test)."""
import ctypes as C

import pytest
import torch


class _Rules:
    """The library's functions that answer a question on the host; any other fails the test."""

    def __init__(self, lib):
        self.lib = lib

    def __getattr__(self, name):
        if not name.endswith("_takes"):
            pytest.fail(f"{name} was called")
        return getattr(self.lib, name)


@pytest.fixture
def ops(monkeypatch):
    """ops whose operands count as device tensors and whose library answers questions only."""
    from lyradiff_amd import ops as _ops

    rules = _Rules(_ops._l.load())
    monkeypatch.setattr(_ops, "_chk", lambda t, name, dtypes=None: t)
    monkeypatch.setattr(_ops._l, "load", lambda: rules)
    return _ops


@pytest.mark.parametrize("per_token", [False, True])
def test_int8_linear_refuses_a_residual_in_host_memory(ops, per_token):
    a, w = torch.zeros(4, 64, dtype=torch.int8), torch.zeros(32, 64, dtype=torch.int8)
    with pytest.raises(ValueError, match="addend must be on the device"):
        ops.int8_linear(a, w, torch.ones(32), torch.ones(4 if per_token else 1), None, torch.float16, addend=torch.zeros(4, 32, dtype=torch.float16))


def test_int8_linear_without_a_calibrated_scale_is_refused_unless_dynamic(monkeypatch):
    from lyradiff_amd import ops as _ops, weights

    lin = weights.Int8Linear(torch.zeros(32, 64, dtype=torch.int8), torch.ones(32), None, torch.ones(64))
    x, seen = torch.zeros(4, 64, dtype=torch.float16), []
    monkeypatch.setattr(_ops, "sq_quant_dynamic", lambda *a: pytest.fail("quantised per token"))
    with pytest.raises(TypeError, match="input_quant_scale"):
        lin.forward(x)
    monkeypatch.setattr(_ops, "sq_linear", lambda x, pre, scale, *a: (seen.append(scale), x)[1])
    assert lin.forward(x, dynamic=True) is x and seen == [None]


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("bad", [{1: torch.ones(0)}, {2: torch.ones(0)}, {2: torch.ones(64)}, {3: torch.zeros(32, dtype=torch.float16)}])
def test_fp8_linear_rows_refuses_short_scales_and_biases(ops, which, bad):
    x = torch.zeros(1, 1280, dtype=torch.float16)
    lin = [torch.zeros(64, 1280, dtype=torch.uint8), torch.ones(1), torch.ones(1), torch.zeros(64, dtype=torch.float16)]
    wrong = tuple(bad.get(i, t) for i, t in enumerate(lin))
    with pytest.raises(ValueError, match="one element"):
        ops.fp8_linear_rows(x, *((wrong, tuple(lin)) if which == 0 else (tuple(lin), wrong)))
    with pytest.raises(ValueError, match="one element"):
        ops.fp8_linear_rows(x, wrong)


# every linear whose kernel reads N values of a bias; m rows, n outputs, k inputs
_U8, _F = (lambda *s: torch.zeros(*s, dtype=torch.uint8)), torch.ones
LINEARS = {
    "int8_linear": lambda ops, b, m, n, k: ops.int8_linear(_U8(m, k), _U8(n, k), _F(n), _F(1), b, torch.float16),
    "int8_linear_panels": lambda ops, b, m, n, k: ops.int8_linear_panels(_U8(k // 64, m, 64), _U8(n, k), _F(n), _F(1), b, torch.float16),
    "sq_linear": lambda ops, b, m, n, k: ops.sq_linear(torch.zeros(m, k, dtype=torch.float16), _F(k), _F(1), _U8(n, k), _F(n), b),
    "fp8_linear": lambda ops, b, m, n, k: ops.fp8_linear(_U8(m, k), _U8(n, k), _F(1), _F(1), b, out_dtype=torch.float16),
    "fp8_linear_max": lambda ops, b, m, n, k: ops.fp8_linear_max(_U8(m, k), _U8(n, k), _F(1), _F(1), b, _F(1), torch.float16),
    "fp8_linear_panels": lambda ops, b, m, n, k: ops.fp8_linear_panels(_U8(k // 64, m, 64), _U8(n, k), _F(1), _F(1), b, None, torch.float16),
    "fp8_linear_gated": lambda ops, b, m, n, k: ops.fp8_linear_gated(_U8(m, k), _U8(n, k), _F(1), _F(1), b, _F(1, n), _F(m, n), max(m, 1)),
    "fp8_linear_gated_panels": lambda ops, b, m, n, k: ops.fp8_linear_gated_panels(_U8(k // 64, m, 64), _U8(n, k), _F(1), _F(1), b, _F(1, n), _F(m, n), max(m, 1)),
    "fp8_linear_codes": lambda ops, b, m, n, k: ops.fp8_linear_codes(_U8(m, k), _U8(n, k), _F(1), _F(1), b, _F(1)),
    "fp8_linear_codes_panels": lambda ops, b, m, n, k: ops.fp8_linear_codes_panels(_U8(k // 64, m, 64), _U8(n, k), _F(1), _F(1), b, _F(1)),
    "weight_only_linear": lambda ops, b, m, n, k: ops.weight_only_linear(torch.zeros(m, k, dtype=torch.float16), _U8(n, k), _F(n), b),
    "w4a4_linear": lambda ops, b, m, n, k: ops.w4a4_linear(torch.zeros(m, k // 8, dtype=torch.int32), _U8(n, k // 2), _F(m, k // 64), _F(n, k // 64), b, torch.float16),
    "w4a4_linear_codes": lambda ops, b, m, n, k: ops.w4a4_linear_codes(_U8(m, k), _U8(n, k), _F(k // 64, m), _F(k // 64, n), b, torch.float16),
}


@pytest.mark.parametrize("name", LINEARS)
def test_linears_refuse_a_bias_that_ends_before_the_outputs(ops, monkeypatch, name):
    monkeypatch.setattr(ops, "sq_quant", lambda x, pre, scale: torch.zeros(x.shape, dtype=torch.int8))
    with pytest.raises(ValueError, match="bias must have N elements"):
        LINEARS[name](ops, torch.zeros(63, dtype=torch.float16), 4, 64, 128)


def test_no_bias_is_read_for_32_bit_sums_or_no_rows(ops, monkeypatch):
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    for m, bias, dt in ((4, torch.zeros(3, dtype=torch.int32), torch.int32), (0, torch.zeros(3, dtype=torch.float16), torch.float16), (4, torch.zeros(65).half(), torch.float16)):
        with pytest.raises(pytest.fail.Exception, match="lq_gemm_int8 was called"):
            ops.int8_linear(_U8(m, 128), _U8(64, 128), _F(64), _F(1), bias, dt)


SIZES = [(m, n, k) for m in (1, 2, 4, 5, 8, 9) for n in (64, 9216, 32 * 1536) for k in (1024, 1280, 1344, 1536, 3072, 12288)]


def test_fp8_rows_rule_is_that_of_the_entry_point():
    """A misaligned weight is refused behind the rule and in front of any launch."""
    from lyradiff_amd import lib as L, ops as _ops

    lib, at, odd = L.load(), C.c_void_p(16), C.c_void_p(8)
    taken = 0
    for m, n, k in SIZES:
        takes = _ops.fp8_linear_rows_takes(m, n, k)
        assert lib.lq_linear_fp8_rows(at, None, at, L.LQ_F16, odd, None, at, None, at, None, None, None, m, n, k, None) == (-1 if takes else 1), (m, n, k)
        assert takes == (m <= 8 and m * k <= 12288 and k > 1024 and k % 256 == 0 and n < 32 * 1536), (m, n, k)
        taken += takes
        with _ops.gemm_thread_tactic(2):
            assert not _ops.fp8_linear_rows_takes(m, n, k)
    assert taken > 0


@pytest.mark.parametrize("m", [5, 8, 9])
def test_fp8_linears_of_a_few_more_rows_go_straight_to_the_two_calls(ops, monkeypatch, m):
    from lyradiff_amd import weights

    monkeypatch.setattr(torch, "empty", lambda *a, **k: pytest.fail("an output was allocated"))
    x, w, one = torch.zeros(m, 3072, dtype=torch.float16), torch.zeros(64, 3072, dtype=torch.uint8), torch.ones(1)
    lin = (w, one, one, None)
    assert ops.fp8_linear_rows(x, lin) is None and ops.fp8_linear_rows(x, lin, lin) is None
    monkeypatch.setattr(ops, "fp8_linear_rows", lambda *a: pytest.fail("the few-rows route was tried"))
    monkeypatch.setattr(ops, "fp8_scale_cast_panels", lambda x, scale: "codes")
    monkeypatch.setattr(ops, "fp8_linear_panels", lambda q, *a: torch.zeros(m, 64))
    assert weights.FP8Linear(w, one, one).forward(x).shape == (m, 64)


# rows, n, k; 1: measured ahead of the library's GEMM, 0: behind it, or a size the kernel does not take (lq_linear16.hip has the times)
@pytest.mark.parametrize("m,n,k,one", [
    (1, 640, 640, 1), (1, 18432, 3072, 1), (2, 9216, 3072, 1), (16, 18432, 3072, 1), (17, 18432, 3072, 0), (17, 9216, 3072, 0), (64, 18432, 3072, 0),
    (256, 9216, 3072, 0), (256, 640, 640, 1), (256, 3840, 1280, 1), (154, 1280, 2048, 1), (257, 640, 640, 0), (16, 1280, 5120, 0), (8, 3072, 12288, 0),
    (1, 3072, 12288, 1), (1, 3072, 15360, 0), (128, 10240, 1280, 0), (0, 640, 640, 0), (4, 642, 640, 0), (4, 640, 100, 0)])
def test_16_bit_linears_of_few_rows_are_taken_where_that_is_faster(m, n, k, one):
    from lyradiff_amd import lib as L

    assert L.load().lq_linear16_rows_takes(m, n, k) == one


# rows of both, n, k, scales and bias only; 1: measured ahead in one launch, 0: ahead one after the other (lq_gemm_fp8.hip has the times)
@pytest.mark.parametrize("m,m2,n,k,plain,one", [
    (4096, 512, 9216, 3072, 1, 1), (6400, 512, 3072, 3072, 1, 1), (6400, 512, 12288, 3072, 0, 1), (6400, 512, 3072, 12288, 0, 1), (400, 100, 3072, 12288, 0, 1),
    (5120, 512, 3072, 3072, 1, 0), (5120, 512, 3072, 12288, 0, 0), (8192, 512, 3072, 12288, 0, 0), (6144, 64, 9216, 3072, 1, 0),
    (6144, 64, 12288, 3072, 0, 0), (4096, 77, 12288, 3072, 0, 0), (2500, 200, 3072, 12288, 0, 0), (4096, 32, 3072, 3072, 1, 0)])
def test_fp8_pairs_share_a_launch_where_that_is_faster(m, m2, n, k, plain, one):
    from lyradiff_amd import lib as L, ops as _ops

    assert L.load().lq_gemm_fp8_pair_takes(m, m2, n, k, plain) == one
    with _ops.gemm_thread_tactic(2):
        assert L.load().lq_gemm_fp8_pair_takes(m, m2, n, k, plain) == 0


def test_plain_calls_are_told_from_those_that_pytorch_has_to_see():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad

    from lyradiff_amd import ops as _ops

    x, seen = torch.zeros(2, 4), []
    look = lambda t: (seen.append(_ops._plain(t)), t)[1]
    leaf = x.clone().requires_grad_()
    assert _ops._plain(x, None, torch.nn.Parameter(x, requires_grad=False)) and not _ops._plain(x, leaf) and not _ops._plain(x.to_sparse())
    with torch.no_grad():
        assert _ops._plain(leaf)
    torch.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.jit.trace(look, (x,), check_trace=False)
    with FakeTensorMode() as mode:
        look(mode.from_tensor(x))
    with forward_ad.dual_level():
        look(forward_ad.make_dual(x, x))
        assert _ops._plain(x)
    assert len(seen) >= 5 and not any(seen)
