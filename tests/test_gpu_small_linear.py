"""Swapped Linears over few rows: the one-launch form, the small-tile products and the native host
route, against the oracle at the edges of their ranges."""

import pytest
import torch

from helpers import linear_inputs
from oracle import quant_linear as orq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64), (7, 2048, 256), (8, 24, 5120), (9, 40, 2048), (16, 4112, 2048), (17, 264, 768), (32, 16, 768),  # one launch
    (9, 40, 2112), (33, 264, 768), (17, 1280, 832), (65, 1288, 5120), (257, 520, 1344), (500, 1272, 2048),      # small tiles
    (513, 1280, 5120),                                                                                          # tiled
])
def test_dense_linear_over_few_rows_bit_exact(M, N, K):
    from samfast_amd import Int8DynamicLinear
    print(f"case small linear M={M} N={N} K={K}", flush=True)
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    if M > 1:
        x[M - 1] = 0
    lin = torch.nn.Linear(K, N, bias=M % 2 == 1, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        if lin.bias is not None:
            lin.bias.copy_(b)
    y = Int8DynamicLinear.from_float(lin).cuda()(x.cuda())  # weights quantised on the CPU, as the oracle does
    ref = orq.dynamic_int8_linear(x, w, b if lin.bias is not None else None)
    assert torch.equal(y.cpu().view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(1, 8, 256), (31, 40, 384), (33, 264, 256), (65, 1280, 5120), (500, 1288, 2048), (130, 4096, 1280)])
def test_sparse_linear_over_few_rows_bit_exact(M, N, K):
    from samfast_amd import Int8Sparse24Linear
    from samfast_amd.quant import quantize_weight_per_channel
    from samfast_amd.sparse import prune_2_of_4
    print(f"case small sparse linear M={M} N={N} K={K}", flush=True)
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    wq, sw = quantize_weight_per_channel(prune_2_of_4(w.float()))
    y = Int8Sparse24Linear.from_int8(wq.cuda(), sw.cuda(), b.float().cuda())(x.cuda())
    assert torch.equal(y.cpu().view(torch.int16), orq.sparse24_int8_linear(x, w, b).view(torch.int16))


def test_nan_and_shapes_through_the_native_route():
    """A NaN stays in its row, leading axes and dtypes survive, strided and empty inputs still work."""
    from samfast_amd import Int8DynamicLinear
    m = Int8DynamicLinear.from_float(torch.nn.Linear(256, 64, dtype=torch.bfloat16).cuda())
    x = torch.randn((2, 5, 256), device="cuda").to(torch.bfloat16)
    want = m(x.reshape(10, 256)).reshape(2, 5, 64)
    assert torch.equal(m(x), want)
    assert torch.equal(m(x.transpose(0, 1)).transpose(0, 1), want)
    assert m(x.float()).dtype == torch.float32 and torch.equal(m(x.float()), want.float())
    assert m(x[:0]).shape == (0, 5, 64)
    x[1, 2, 7] = float("nan")
    nan = torch.isnan(m(x)).all(-1)
    assert nan[1, 2] and nan.sum() == 1
