"""What the product of many rows with its activation refuses, before anything is launched (no GPU)."""
import pytest
import torch

from sharpinference_amd import ops
from sharpinference_amd.ops import lib


@pytest.fixture
def launches(monkeypatch):
    """Calls that would have reached a kernel; operands on the host pass for the GPU's."""
    calls = []
    monkeypatch.setattr(ops, "_dev", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    monkeypatch.setattr(ops, "_run", lambda name, *args: calls.append((name, args)))
    monkeypatch.setattr(ops, "dense_height", lambda *a: 128)
    return calls


@pytest.mark.parametrize("act", [0, None, -1, 4, (0, 0.0), (-1, 7.0), (3, 0.0), (3, -1.0), (3, float("nan")), 3])
def test_activations_that_are_not_known(launches, act):
    """Of half the output's columns no product without an activation may be written, and none may come back in the activation's place."""
    x, w = torch.zeros(300, 128, dtype=torch.bfloat16), ops.pack_weight(torch.zeros(64, 128, dtype=torch.bfloat16), True)
    with pytest.raises(ops.KernelError):
        ops.linear_gated(x, w, torch.bfloat16, act)
    if act is not None:                     # (None asks the product itself for the product)
        with pytest.raises(ops.KernelError):
            ops.gemm_dense(x, w, 128, act)
    assert not launches


@pytest.mark.parametrize("act,limit,relu2", [(-1, 0.0, 0), (4, 0.0, 0), (3, 0.0, 0), (3, float("nan"), 0), (1, 0.0, 1)])
def test_the_entry_refuses_them_too(act, limit, relu2):
    assert lib.load().sharpi_gemm_dense(0, 0, 0, 300, 64, 128, 128, act, limit, relu2, None) == 1001      # (SHARPI_ERR_ARG)


def test_weights_that_the_kernel_does_not_take_go_where_they_went(monkeypatch):
    """Tiles at an odd address, or not in one piece, beside rows that the library multiplies: the rule leaves them to it."""
    monkeypatch.setattr(ops, "dense_height", lambda *a: 128)
    x, w = torch.zeros(300, 128, dtype=torch.bfloat16), ops.pack_weight(torch.zeros(64, 128, dtype=torch.bfloat16), True)
    height = lambda packed: ops._dense_height_of(x, ops.PackedWeight(packed, w.rows), torch.bfloat16, True)
    odd = torch.zeros(64 * 128 + 1, dtype=torch.bfloat16)[1:].view(64, 128)
    assert height(w.packed) == 128
    assert odd.data_ptr() % 16 and height(odd) == 0
    assert height(torch.zeros(64, 256, dtype=torch.bfloat16)[:, :128]) == 0
