"""What the Python wrappers refuse, and which route they take, before anything is enqueued (no GPU: a call that reaches the library fails
the test)."""
import pytest
import torch


@pytest.fixture
def ops(monkeypatch):
    """ops whose operands count as device tensors and whose library must not be called."""
    from lyradiff_amd import ops as _ops

    monkeypatch.setattr(_ops, "_chk", lambda t, name, dtypes=None: t)
    monkeypatch.setattr(_ops._l, "load", lambda: pytest.fail("the call reached the library"))
    return _ops


@pytest.mark.parametrize("per_token", [False, True])
def test_int8_linear_refuses_a_residual_in_host_memory(ops, per_token):
    a, w = torch.zeros(4, 64, dtype=torch.int8), torch.zeros(32, 64, dtype=torch.int8)
    with pytest.raises(ValueError, match="addend must be on the device"):
        ops.int8_linear(a, w, torch.ones(32), torch.ones(4 if per_token else 1), None, torch.float16, addend=torch.zeros(4, 32, dtype=torch.float16))


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
