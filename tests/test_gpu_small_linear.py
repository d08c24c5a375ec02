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


def _linear(N, K, seed):
    from samfast_amd import Int8DynamicLinear
    g = torch.Generator().manual_seed(seed)
    lin = torch.nn.Linear(K, N, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(torch.randn((N, K), generator=g) * 0.02)
        lin.bias.copy_(torch.randn(N, generator=g))
    return Int8DynamicLinear.from_float(lin.cuda())


def _unfused(lin, x):
    """The same Linear as two calls on row-major codes and weights."""
    from samfast_amd import _lib, ops
    xq, sx = ops.quant_rowwise(x)
    return ops.gemm_i8_fused(xq, sx, lin.wq, lin.sw, lin.bias_f32, _lib.EPILOGUE_NONE)


@pytest.mark.parametrize("M,N,K", [
    (7, 2048, 256), (100, 3840, 1280), (33, 8, 64), (700, 520, 192),        # one launch, small tiles, fewer k tiles than stages
    (4096, 768, 768), (4000, 1288, 5120), (5000, 2304, 768), (16383, 1280, 1280),  # one tile per CU, 128 x 128 tiles, resident
    (16384, 1288, 320), (20001, 776, 1280),                                 # weights reordered on the way
])
def test_a_linear_reads_its_weights_as_they_stand(M, N, K):
    """Row-major weights beside K-block major codes: the bits of row-major both, and of weights written a moment ago."""
    print(f"case weights M={M} N={N} K={K}", flush=True)
    lin, other = _linear(N, K, 1), _linear(N, K, 2)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    assert torch.equal(lin(x), _unfused(lin, x))
    lin.wq.data.copy_(other.wq)
    lin.sw_bits.data.copy_(other.sw_bits)
    lin.bias_bits.data.copy_(other.bias_bits)
    assert torch.equal(lin(x), _unfused(other, x))


@pytest.mark.parametrize("sparse", [False, True])
def test_the_native_modules_entries_look_buffers_up_by_name(sparse):
    """Rows on the GPU: a buffer that is missing, None or of another type is declined, a missing bias is none, and a replaced buffer counts from the next call on."""
    from samfast_amd import Int8DynamicLinear, Int8Sparse24Linear, _lib
    print(f"case buffers by name sparse={sparse}", flush=True)
    make = Int8Sparse24Linear if sparse else Int8DynamicLinear
    entry = _lib.host().module_sparse_linear if sparse else _lib.host().module_linear
    gen = torch.Generator().manual_seed(11)
    floats = [torch.nn.Linear(256, 264, dtype=torch.bfloat16) for _ in range(2)]
    for f in floats:
        with torch.no_grad():
            f.weight.copy_(torch.randn((264, 256), generator=gen) * 0.02)
            f.bias.copy_(torch.randn(264, generator=gen))
    lin, other = (make.from_float(f.cuda()) for f in floats)
    x = torch.randn((9, 256), generator=gen).to(torch.bfloat16).cuda()
    y = entry(x, lin._buffers)
    assert y is not None and torch.equal(y, lin(x))
    weights = ("wc", "widx", "sw_bits") if sparse else ("wq", "sw_bits")
    for name in weights:
        without = {k: v for k, v in lin._buffers.items() if k != name}
        assert entry(x, without) is None, name
        assert entry(x, {**without, name: None}) is None, name
        assert entry(x, {**without, name: lin._buffers[name].cpu()}) is None, name
        assert entry(x, {**without, name: lin._buffers[name].float()}) is None, name
    floats[0].bias = None
    unbiased = make.from_float(floats[0])(x)
    assert not torch.equal(unbiased, y)
    without = {k: v for k, v in lin._buffers.items() if k != "bias_bits"}
    for buffers in (without, {**without, "bias_bits": None}):
        assert torch.equal(entry(x, buffers), unbiased)
    buffers = dict(lin._buffers)
    for name in weights + ("bias_bits",):
        buffers[name] = other._buffers[name]
    assert torch.equal(entry(x, buffers), other(x))
    lin.load_state_dict(other.state_dict())
    assert torch.equal(lin(x), other(x))
    for wrong in ({}, None, [], 5):
        assert entry(x, wrong) is None
    assert entry(x) is None


@pytest.mark.parametrize("M", [7, 4096, 16384])
def test_a_linears_first_call_anywhere(M):
    """Built in inference mode; first called while a graph is recorded; then called from another stream."""
    print(f"case first call M={M}", flush=True)
    x = torch.randn((M, 256), device="cuda").to(torch.bfloat16)
    with torch.inference_mode():
        lin = _linear(264, 256, 3)
        assert torch.equal(lin(x), _unfused(lin, x))
    lin = _linear(264, 256, 4)
    want = _unfused(lin, x)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        recorded = lin(x)
    assert torch.equal(lin(x), want)  # before any replay
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        there = lin(x)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(there, want)
    for _ in range(3):
        recorded.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, want)


def test_the_blocks_copy_of_a_weight_is_complete_wherever_it_is_made():
    """The K-block major copy that linear_fused keeps: first needed while a graph is recorded, then on two streams, and in
    inference mode."""
    from samfast_amd import _lib, ops
    lin = _linear(264, 256, 5)
    x = torch.randn((300, 256), device="cuda").to(torch.bfloat16)
    want = _unfused(lin, x)
    xk, sx = ops.quant_rowwise(x, _lib.LAYOUT_KB64)
    run = lambda m: m.linear_fused(xk, sx, _lib.EPILOGUE_NONE, layout=_lib.LAYOUT_KB64)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        recorded = run(lin)
    assert torch.equal(run(lin), want)  # before any replay
    for _ in range(3):
        recorded.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, want)
    fresh, side = _linear(264, 256, 5), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        there = run(fresh)
    here = run(fresh)
    torch.cuda.synchronize()
    assert torch.equal(there, want) and torch.equal(here, want)
    with torch.inference_mode():
        assert torch.equal(run(_linear(264, 256, 5)), want)


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


@pytest.mark.parametrize("M,K", [(3, 1032), (1025, 1536), (8193, 1032), (1000, 2048), (1030, 2040), (7, 2560), (9, 3072), (5, 2176), (4097, 2184),
                                 (6, 4096), (11, 3080), (5, 5120), (6145, 5120), (13, 4608), (3, 5128), (2, 8192),
                                 (2049, 4608), (4097, 5120), (4112, 5120), (2050, 6144), (2064, 6656), (2049, 7168)])
def test_quantiser_with_shared_rows_bit_exact(M, K):
    """Rows that two or four wavefronts share, in both layouts, with a NaN row and a zero row."""
    import numpy as np
    from samfast_amd import _lib, ops
    print(f"case shared rows M={M} K={K}", flush=True)
    x, _, _ = linear_inputs(M, K, 8, seed=M + K)
    x[M - 1] = 0
    q_ref, s_ref = orq.quantize_rows_absmax(x)
    xq, sx = ops.quant_rowwise(x.cuda())
    assert np.array_equal(xq.cpu().numpy(), q_ref) and np.array_equal(sx.cpu().numpy(), s_ref)
    if K % 64 == 0:
        xk, sk = ops.quant_rowwise(x.cuda(), _lib.LAYOUT_KB64)
        assert torch.equal(ops.from_kb64(xk), xq) and torch.equal(sk, sx)
    x[0, K - 1] = float("nan")
    sn = ops.quant_rowwise(x.cuda())[1]
    assert torch.isnan(sn[0]) and torch.equal(sn[1:], sx[1:])


@pytest.mark.parametrize("M,N,K,epi", [(2433, 2056, 256, 0), (2440, 2056, 1536, 0), (4000, 1288, 1344, 1), (1025, 4616, 1600, 2), (5000, 1288, 3072, 2)])
def test_middle_tile_agrees_with_the_small_one(M, N, K, epi):
    """128 x 128 tiles with two and three operand stages, ragged rows and columns: chosen by themselves,
    the bits of the 64 x 128 tiles and of integer arithmetic."""
    from samfast_amd import _lib, ops
    print(f"case middle tile M={M} N={N} K={K} epi={epi}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    xq = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    wq = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    sx, sw, bias = torch.rand(M, generator=g) * 1e-3, torch.rand(N, generator=g) * 1e-2, torch.randn(N, generator=g)
    res = torch.randn((M, N), generator=g).to(torch.bfloat16).cuda() if epi == _lib.EPILOGUE_RESIDUAL else None
    xk, wk = ops.to_kb64(xq.cuda()), ops.to_kb64(wq.cuda())
    run = lambda: ops.gemm_i8_fused(xk, sx.cuda(), wk, sw.cuda(), bias.cuda(), epi, residual=res, layout=_lib.LAYOUT_KB64)
    y = run()
    with _lib.knobs(SAMFAST_GEMM_TILE=64):
        assert torch.equal(run(), y)
    if epi == _lib.EPILOGUE_NONE:
        rows = torch.tensor([0, 1, 63, 64, 127, 128, M - 130, M - 1])
        acc = (xq[rows].double() @ wq.double().t()).float()
        assert torch.equal(y[rows.cuda()].cpu(), (acc * sx[rows, None] * sw + bias).to(torch.bfloat16))


@pytest.mark.parametrize("bm,tn,M,N,K,epi", [
    # (rows of the tile, columns / 32): whole tiles, ragged rows and columns, one tile, the shortest K loop and odd counts of k tiles
    (128, 3, 4096, 768, 768, 2), (128, 3, 130, 200, 896, 0), (128, 4, 128, 128, 1024, 1), (128, 4, 2433, 1000, 3072, 2),
    (128, 5, 4000, 1288, 1280, 2), (128, 5, 1, 8, 1408, 0), (256, 6, 257, 2304, 448, 0), (256, 6, 4096, 3072, 768, 1),
    (256, 8, 1000, 776, 384, 1), (256, 8, 255, 4096, 1024, 0), (256, 10, 3900, 5120, 1280, 1), (256, 10, 513, 328, 576, 0),
])
@pytest.mark.parametrize("layout", [0, 1])
def test_one_tile_per_cu_agrees_with_the_small_tiles(bm, tn, M, N, K, epi, layout):
    from samfast_amd import _lib, ops
    print(f"case once {bm}x{32 * tn} M={M} N={N} K={K} epi={epi} layout={layout}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    xq = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    wq = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    sx, sw, bias = torch.rand(M, generator=g) * 1e-3, torch.rand(N, generator=g) * 1e-2, torch.randn(N, generator=g)
    res = torch.randn((M, N), generator=g).to(torch.bfloat16).cuda() if epi == _lib.EPILOGUE_RESIDUAL else None
    xk, wk = xq.cuda(), wq.cuda()
    if layout == _lib.LAYOUT_KB64:
        xk, wk = ops.to_kb64(xk), ops.to_kb64(wk)
    run = lambda **kw: ops.gemm_i8_fused(xk, sx.cuda(), wk, sw.cuda(), bias.cuda() if M % 2 == 0 else None, epi, layout=layout, **kw)
    with _lib.knobs(SAMFAST_GEMM_ONCE=bm * 16 + tn, SAMFAST_GEMM_SKINNY=0):
        y = run(residual=res)
        if res is not None:  # in place, as the encoder's residual stream
            inplace = res.clone()
            assert run(residual=inplace, out=inplace) is not None and torch.equal(inplace, y)
    with _lib.knobs(SAMFAST_GEMM_TILE=64, SAMFAST_GEMM_SKINNY=0):
        assert torch.equal(run(residual=res), y)


@pytest.mark.parametrize("bm,tn,M,N,K,epi", [
    # 64-row tiles, K dealt to four groups: the shortest loop, one to three k tiles behind the last whole round of the groups, edges of rows and columns
    (64, 2, 64, 64, 1280, 0), (64, 2, 1, 8, 1344, 0), (64, 2, 633, 1288, 5120, 2), (64, 2, 130, 200, 1408, 1),
    (64, 3, 65, 96, 1472, 0), (64, 3, 1000, 776, 3072, 2), (64, 3, 63, 104, 1280, 1),
    (64, 4, 129, 128, 1280, 2), (64, 4, 1321, 1280, 4096, 0), (64, 4, 200, 136, 1600, 1),
])
@pytest.mark.parametrize("layout", [0, 1])
def test_one_tile_of_64_rows_agrees_with_the_small_tiles(bm, tn, M, N, K, epi, layout):
    test_one_tile_per_cu_agrees_with_the_small_tiles(bm, tn, M, N, K, epi, layout)


@pytest.mark.parametrize("M,N,K", [(278, 1280, 3072), (194, 1600, 3648), (39, 5120, 3776), (900, 768, 3072), (1638, 768, 4096), (1327, 1280, 4096), (2000, 1280, 4096)])
def test_linears_over_some_hundred_long_rows_against_their_codes(M, N, K):
    """Two launches through the tile that the rule takes, against the product of the quantiser's own codes in 64 bits."""
    from samfast_amd import Int8DynamicLinear, ops
    print(f"case long rows M={M} N={N} K={K}", flush=True)
    x, w, b = linear_inputs(M, K, N, seed=M)
    lin = torch.nn.Linear(K, N, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        lin.bias.copy_(b)
    lin, x = Int8DynamicLinear.from_float(lin.cuda()), x.cuda()
    y = lin(x)
    xq, sx = ops.quant_rowwise(x)
    acc = (xq.double() @ lin.wq.double().t()).float()  # (integers below 2^53: exact)
    assert torch.equal(y, (acc * sx[:, None] * lin.sw + lin.bias_f32).to(torch.bfloat16))


@pytest.mark.parametrize("sparse,M,N,K", [
    # workgroups of 8 rows and one, two, four column tiles, of 16 rows; the last calls of each, remainders of rows, columns and k steps
    (False, 63, 488, 64), (False, 64, 512, 512), (False, 65, 1000, 576), (False, 121, 1024, 1024), (False, 128, 1032, 1088), (False, 250, 1016, 1536),
    (False, 79, 760, 2048), (False, 405, 632, 704), (False, 9, 8200, 1600), (False, 31, 13000, 768), (False, 4, 8200, 512), (False, 1, 9000, 1088), (False, 5, 8200, 256),
    # long rows, several short workgroups on a CU: the last calls of the lines
    (False, 24, 1360, 5120), (False, 2041, 16, 2112), (False, 9, 4096, 4096), (False, 61, 1016, 4096), (False, 250, 256, 2112), (False, 379, 248, 1024), (False, 576, 112, 576), (False, 599, 112, 576),
    (False, 92, 1024, 320), (False, 250, 512, 512), (False, 61, 2048, 128),
    (True, 480, 520, 256), (True, 256, 1024, 2048), (True, 59, 4096, 1920), (True, 125, 1016, 3072), (True, 61, 1016, 5120), (True, 250, 256, 3200),
    (True, 1, 8, 256), (True, 63, 1000, 512), (True, 128, 1536, 1024), (True, 77, 1632, 1152), (True, 57, 1016, 2048), (True, 81, 712, 3072), (True, 4, 1288, 5120),
])
def test_one_launch_agrees_with_two(sparse, M, N, K):
    from samfast_amd import Int8DynamicLinear, Int8Sparse24Linear, _lib
    print(f"case one launch sparse={sparse} M={M} N={N} K={K}", flush=True)
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    x[M // 2] = 0
    x[M - 1, K // 3] = float("nan")
    lin = torch.nn.Linear(K, N, bias=M % 2 == 1, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        if lin.bias is not None:
            lin.bias.copy_(b)
    lin, x = (Int8Sparse24Linear if sparse else Int8DynamicLinear).from_float(lin.cuda()), x.cuda()
    layout = 2 if sparse else _lib.LAYOUT_ROWMAJOR
    assert _lib.load().samfast_linear_i8_one_launch(M, N, K, layout) == 1
    one = lin(x)
    with _lib.knobs(SAMFAST_GEMM_LINEAR_SMALL=0):
        assert _lib.load().samfast_linear_i8_one_launch(M, N, K, layout) == 0
        two = lin(x)
    assert torch.equal(one.view(torch.int16), two.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [
    # each tile at its smallest, with rows and columns moved back inside, the shortest, odd and longest K; then what the rule takes
    (32, 384, 256), (33, 392, 384), (64, 768, 256), (65, 776, 640), (127, 1528, 768), (100, 1160, 896), (200, 2304, 1024), (95, 640, 1152), (129, 1288, 1280),
    (4096, 768, 768), (2100, 2304, 768), (5300, 2304, 768), (1100, 4096, 1024), (700, 3080, 1024), (1990, 3840, 1280), (450, 1280, 1280),
])
def test_a_band_of_rows_in_one_launch_agrees_with_two(M, N, K):
    """Every tile that the shape admits and the rule's choice, weights in both layouts; rows with a NaN, an infinity, zeros and ties."""
    from samfast_amd import Int8DynamicLinear, _lib, ops
    print(f"case band M={M} N={N} K={K}", flush=True)
    lib = _lib.load()
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    x[M // 2] = 0
    x[M - 1, K // 3] = float("nan")
    x[1, K - 1] = float("inf")
    x[2] = torch.arange(K).remainder(255).sub(127).to(torch.bfloat16) / 2  # a maximum of 63.5: every second value a tie
    lin = torch.nn.Linear(K, N, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        lin.bias.copy_(b)
    lin, x = Int8DynamicLinear.from_float(lin.cuda()), x.cuda()
    stream = torch.cuda.current_stream().cuda_stream
    with _lib.knobs(SAMFAST_GEMM_LINEAR_SMALL=0):
        two = lin(x)
    assert torch.isnan(two[M - 1]).all()
    wk = ops.to_kb64(lin.wq)
    for tile in (1, 2 * 8 + 3, 4 * 8 + 3, 4 * 8 + (6 if K <= 1024 else 5)):
        rows, cols = (16 * (tile // 8), 128 * (tile % 8)) if tile > 1 else (M, N)
        if M < rows or N < cols:
            continue
        with _lib.knobs(SAMFAST_GEMM_LINEAR_BAND=tile):
            if tile > 1:  # this tile: the few-row form is off
                assert lib.samfast_linear_i8_one_launch(8, 768, 768, 0) == 0
                assert lib.samfast_linear_i8_one_launch(M, N, K, 0) == 1
            assert torch.equal(lin(x).view(torch.int16), two.view(torch.int16)), tile
            if lib.samfast_linear_i8_one_launch(M, N, K, 1):
                y = torch.empty_like(two)
                assert lib.samfast_linear_i8(x.data_ptr(), K, wk.data_ptr(), lin.sw.data_ptr(), lin.bias_f32.data_ptr(), y.data_ptr(), N, None,
                                             M, N, K, _lib.SAMFAST_BF16, _lib.LAYOUT_KB64, stream) == 0
                assert torch.equal(y.view(torch.int16), two.view(torch.int16)), tile


@pytest.mark.parametrize("M,N,K", [
    (32, 384, 256), (33, 392, 384), (64, 768, 256), (65, 776, 640), (127, 1528, 768), (200, 2304, 1024), (95, 640, 1152), (129, 1288, 1280),
    (2100, 2304, 768), (1100, 4096, 1024), (1990, 3840, 1280), (450, 1280, 1280),
])
def test_a_band_of_rows_with_sparse_weights(M, N, K):
    """2:4 weights in every tile that the shape admits and by the rule, against two launches; a row with a NaN and one of zeros."""
    from samfast_amd import Int8Sparse24Linear, _lib
    print(f"case sparse band M={M} N={N} K={K}", flush=True)
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    x[M // 2] = 0
    x[M - 1, K // 3] = float("nan")
    lin = torch.nn.Linear(K, N, bias=M % 2 == 1, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        if lin.bias is not None:
            lin.bias.copy_(b)
    lin, x = Int8Sparse24Linear.from_float(lin.cuda()), x.cuda()
    with _lib.knobs(SAMFAST_GEMM_LINEAR_SMALL=0):
        two = lin(x)
    for tile in (1, 2 * 8 + 3, 4 * 8 + 3, 4 * 8 + (6 if K <= 1024 else 5)):
        if tile > 1 and (M < 16 * (tile // 8) or N < 128 * (tile % 8)):
            continue
        with _lib.knobs(SAMFAST_GEMM_LINEAR_BAND=tile):
            if tile > 1:  # this tile: the few-row form is off
                assert _lib.load().samfast_linear_i8_one_launch(4, 768, 768, 2) == 0
                assert _lib.load().samfast_linear_i8_one_launch(M, N, K, 2) == 1
            assert torch.equal(lin(x).view(torch.int16), two.view(torch.int16)), tile


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [
    # tiles of 32 x 384, 64 x 384 and the wide one, on rows that are shorter than a lane's chunks: two k steps, three, odd counts
    (512, 1024, 256), (600, 1000, 640), (1500, 2000, 384), (700, 512, 512), (3000, 1280, 896), (4900, 1536, 256), (5000, 2304, 384), (1100, 4096, 896),
    (500, 1288, 1152), (1900, 2600, 1152),
])
def test_short_rows_by_the_bands_rule(M, N, K, layout):
    """Calls that the rule gives to the band kernel (not to the few-row form), whose rows do not fill what its lanes hold."""
    from samfast_amd import Int8DynamicLinear, Int8Sparse24Linear, _lib, ops
    print(f"case band rule M={M} N={N} K={K} layout={layout}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    assert lib.samfast_linear_i8_one_launch(M, N, K, layout) == 1
    with _lib.knobs(SAMFAST_GEMM_LINEAR_BAND=0):
        assert lib.samfast_linear_i8_one_launch(M, N, K, layout) == 0
    x, w, b = linear_inputs(M, K, N, seed=M + N + K)
    x[M // 2] = 0
    x[M - 1, K - 1] = float("nan")
    lin = torch.nn.Linear(K, N, dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(w)
        lin.bias.copy_(b)
    lin, x = (Int8Sparse24Linear if layout == 2 else Int8DynamicLinear).from_float(lin.cuda()), x.cuda()
    if layout == 1:
        wk, one = ops.to_kb64(lin.wq), torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
        assert lib.samfast_linear_i8(x.data_ptr(), K, wk.data_ptr(), lin.sw.data_ptr(), lin.bias_f32.data_ptr(), one.data_ptr(), N, None,
                                     M, N, K, _lib.SAMFAST_BF16, layout, stream) == 0
    else:
        one = lin(x)
    with _lib.knobs(SAMFAST_GEMM_LINEAR_SMALL=0):
        two = lin(x)
    assert torch.isnan(two[M - 1]).all()
    assert torch.equal(one.view(torch.int16), two.view(torch.int16))


def test_a_linear_into_its_own_rows():
    """y may be x where the caller brings the workspace: two launches, the quantiser has read every row before one is written."""
    from samfast_amd import _lib
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    for M, K in ((64, 512), (4096, 768)):
        lin = _linear(K, K, M)
        x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
        want = lin(x)
        need = lib.samfast_linear_i8_workspace(M, K, K, 0)
        assert need > 0 and lib.samfast_linear_i8_one_launch(M, K, K, 0) == 1
        work = torch.empty(need, dtype=torch.int8, device="cuda")
        assert lib.samfast_linear_i8(x.data_ptr(), K, lin.wq.data_ptr(), lin.sw.data_ptr(), lin.bias_f32.data_ptr(), x.data_ptr(), K,
                                     work.data_ptr(), M, K, K, _lib.SAMFAST_BF16, 0, stream) == 0
        assert torch.equal(x, want)


@pytest.mark.parametrize("M,K", [(1, 768), (8, 1024), (8, 5120), (16, 2048), (32, 768)])
def test_a_linear_over_a_handful_of_rows_into_those_rows(M, K):
    """The same where one launch takes scales of any alignment."""
    from samfast_amd import _lib
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    lin = _linear(K, K, M)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    want = lin(x)
    work = torch.empty(lib.samfast_linear_i8_workspace(M, K, K, 0), dtype=torch.int8, device="cuda")
    assert lib.samfast_linear_i8(x.data_ptr(), K, lin.wq.data_ptr(), lin.sw.data_ptr(), lin.bias_f32.data_ptr(), x.data_ptr(), K,
                                 work.data_ptr(), M, K, K, _lib.SAMFAST_BF16, 0, stream) == 0
    assert torch.equal(x, want)


def _into(lin, layout, x, y, work):
    """The C call on rows of x and y that may lie apart, in either layout of the weights or 2:4."""
    from samfast_amd import _lib, ops
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    (M, K), N = x.shape, y.shape[1]
    tail = (lin.sw.data_ptr(), lin.bias_f32.data_ptr(), y.data_ptr(), y.stride(0), work, M, N, K, _lib.SAMFAST_BF16)
    if layout == 2:
        return lib.samfast_linear_i8_sparse24(x.data_ptr(), x.stride(0), lin.wc.data_ptr(), lin.widx.data_ptr(), *tail, stream)
    w = ops.to_kb64(lin.wq) if layout == 1 else lin.wq
    return lib.samfast_linear_i8(x.data_ptr(), x.stride(0), w.data_ptr(), *tail, layout, stream)


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N,K,form", [(63, 488, 512, "few"), (57, 520, 1280, "few"), (600, 1000, 640, "band"), (3001, 1288, 768, "band"), (1990, 3840, 1152, "band")])
def test_rows_of_one_launch_further_apart(M, N, K, form, layout):
    """x and y as column ranges of one buffer, without a workspace: the bits of contiguous rows, and nothing beside y is written.
    Then y over x, with a workspace: the same."""
    from samfast_amd import Int8Sparse24Linear, _lib
    print(f"case strides {form} M={M} N={N} K={K} layout={layout}", flush=True)
    lib = _lib.load()
    assert lib.samfast_linear_i8_one_launch(M, N, K, layout) == 1
    with _lib.knobs(SAMFAST_GEMM_LINEAR_BAND=0):
        assert lib.samfast_linear_i8_one_launch(M, N, K, layout) == (form == "few")
    lin = _linear(N, K, M)
    if layout == 2:
        lin = Int8Sparse24Linear.from_int8(lin.wq, lin.sw, lin.bias_f32)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    want = lin(x)
    buf = torch.full((M, 8 + K + 16 + N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    for x_at, y_at in ((8, 8 + K + 16), (8 + N + 16, 8)):
        buf.fill_(7.0)
        buf[:, x_at:x_at + K] = x
        expected = buf.clone()
        expected[:, y_at:y_at + N] = want
        assert _into(lin, layout, buf[:, x_at:x_at + K], buf[:, y_at:y_at + N], None) == 0
        assert torch.equal(buf, expected)
    work = torch.empty(lib.samfast_linear_i8_workspace(M, N, K, layout), dtype=torch.int8, device="cuda")
    for shift in (0, 8):  # the same columns, and columns that overlap
        buf.fill_(7.0)
        buf[:, 8:8 + K] = x
        expected = buf.clone()
        expected[:, 8 + shift:8 + shift + N] = want
        assert _into(lin, layout, buf[:, 8:8 + K], buf[:, 8 + shift:8 + shift + N], None) == -1  # refused without it
        assert _into(lin, layout, buf[:, 8:8 + K], buf[:, 8 + shift:8 + shift + N], work.data_ptr()) == 0
        assert torch.equal(buf, expected)
