"""The product of many rows in tiles of one height: every height at the edges of tiles and of column groups, against the product in double;
its bits are those of the grouped product with the matrix as its one group."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(M, N, K):
    from sharpinference_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, K, device=DEV, generator=g) * 0.1).bfloat16()
    return x, w, ops.pack_weight(w, True)


@pytest.mark.parametrize("height", [128, 160, 192, 224, 256])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (127, 272, 128), (257, 1040, 384), (300, 1280, 256), (641, 2304, 128), (2051, 528, 256)])
def test_rows_in_tiles(M, N, K, height):
    from sharpinference_amd import ops
    x, w, p = _case(M, N, K)
    y = ops.gemm_dense(x, p, height)
    want = x.double() @ w.double().t()
    # K float sums, each rounded by 2^-24 of the sum of magnitudes, then half a place of bfloat16
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * want.abs() + 1e-30
    assert ((y.double() - want).abs() <= bound).all()
    assert torch.equal(y, ops.linear_many_rows(x, p, torch.bfloat16))
    assert torch.equal(ops.gemm_dense(x, p, height, relu2=True), ops.activation(y, "relu2"))


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "swish_clamp"])
@pytest.mark.parametrize("M,N,K,height", [(1, 32, 128, 128), (129, 544, 256, 160), (449, 2592, 128, 224), (700, 1056, 384, 256), (385, 64, 128, 192)])
def test_gated_rows_in_tiles(M, N, K, height, act):
    from sharpinference_amd import ops
    x, _, p = _case(M, N, K)
    code = ops.gated_activation(act, 7.0 if act == "swish_clamp" else None)
    assert torch.equal(ops.gemm_dense(x, p, height, code), ops.gated_act(ops.linear_many_rows(x, p, torch.bfloat16), None, code))


def test_rows_with_infinities_stay_apart():
    from sharpinference_amd import ops
    x, _, p = _case(700, 528, 256)
    clean = ops.gemm_dense(x, p, 192)
    x[5, 3], x[300, 200] = float("inf"), float("nan")
    y = ops.gemm_dense(x, p, 192)
    keep = torch.ones(700, dtype=torch.bool, device=DEV)
    keep[[5, 300]] = False
    assert torch.equal(y[keep], clean[keep]) and not y[[5, 300]].isfinite().any()


def test_routed_calls_are_the_general_path():
    """Sizes that the rule takes, through `linear` and `linear_gated`, and from an odd address; rows that are not in one piece."""
    from sharpinference_amd import ops
    x, _, p = _case(1500, 2816, 1408)
    assert ops.dense_height(1500, 2816, 1408, True) and ops.dense_height(1500, 2816, 1408, False)
    calls = {"gated": lambda v: ops.linear_gated(v, p, torch.bfloat16, ops.ACT_SILU), "relu2": lambda v: ops.linear(v, p, torch.bfloat16, act="relu2")}
    y = ops.linear_many_rows(x, p, torch.bfloat16)
    want = {"gated": ops.gated_act(y, None, ops.ACT_SILU), "relu2": ops.activation(y, "relu2")}
    wide = torch.zeros(1500, 1408 + 8, device=DEV, dtype=torch.bfloat16)
    odd = torch.zeros(1500 * 1408 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(1500, 1408).copy_(x)
    for name, call in calls.items():
        assert torch.equal(call(x), want[name])
        assert torch.equal(call(odd), want[name])
        with pytest.raises(ops.KernelError):                    # rows that are not in one piece are refused as before
            call(wide[:, :1408])


@pytest.mark.parametrize("M", [1, 16, 32])
def test_few_rows_of_many_columns_stay_with_the_streaming_kernel(M):
    from sharpinference_amd import ops
    x, _, p = _case(M, 40960, 1408)
    want = ops.gated_act(ops.gemm_skinny(x, p, torch.bfloat16), None, ops.ACT_SILU)
    assert torch.equal(ops.linear_gated(x, p, torch.bfloat16, ops.ACT_SILU), want)


@pytest.mark.parametrize("M,N,K", [
    (300, 16384, 1408), (300, 28672, 2048), (512, 24576, 2048), (384, 20480, 3072), (400, 20480, 1408),       # fewest rows, most columns
    (8192, 2048, 1408), (8000, 2048, 3072), (5216, 2816, 2816), (2289, 2816, 1536), (1937, 3232, 1664),       # most rows, fewest columns; odd ones
    (3000, 2816, 2048), (4695, 3072, 2176), (1840, 8192, 2048), (908, 10240, 1408), (1468, 10240, 2560), (2049, 5120, 2048)])
def test_the_library_s_bits(M, N, K):
    """What the rule takes was the library's product and a kernel behind it, and keeps their bits: both are one chain of sums over k.  (A library that
    sums otherwise fails this; the results then move where the rule is entered, by a rounding of the product.)"""
    from sharpinference_amd import ops
    x, w, p = _case(M, N, K)
    assert ops.dense_height(M, N, K, True) or ops.dense_height(M, N, K, False)
    y = torch.mm(x, w.t())
    for act in (ops.ACT_SILU, ops.ACT_GELU_TANH):
        assert torch.equal(ops.linear_gated(x, p, torch.bfloat16, act), ops.gated_act(y, None, act))
    assert torch.equal(ops.linear(x, p, torch.bfloat16, act="relu2"), ops.activation(y, "relu2"))
