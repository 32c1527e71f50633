"""A request's rows of all states set to zero in one launch: those bytes and no others."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("count", [1, 7, 32, 33, 70])
def test_a_row_of_every_tensor_is_cleared_and_nothing_beside_it(count):
    from sharpinference_amd import ops

    shapes = [(3,), (3, 1), (3, 5, 7), (3, 4), (3, 16, 129), (3, 128, 1024), (3, 0)]
    types = [torch.float32, torch.bfloat16, torch.int32, torch.uint8]
    tensors = [torch.ones(shapes[i % len(shapes)], dtype=types[i % len(types)], device=DEV) for i in range(count)]
    ops.clear_row(tensors, 1)
    for t in tensors:
        assert bool((t[1] == 0).all()) and bool((t[0] == 1).all()) and bool((t[2] == 1).all())
    with pytest.raises(ops.KernelError):
        ops.clear_row(tensors, 3)
