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
