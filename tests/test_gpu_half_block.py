"""Blocks with half-type Linears: the fused route against the module composition, and its row kernels."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(1, 8), (5, 768), (7, 1280), (9, 1024), (3, 520), (4, 2056), (2, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_add_layernorm_and_gelu_rows(M, K, dtype):
    from samfast_amd import ops
    print(f"case rows M={M} K={K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    x, r = ((torch.randn((M, K), generator=g) * 3 + 1).to(dtype) for _ in range(2))
    w, b = (1 + 0.1 * torch.randn(K, generator=g)).to(dtype), (0.1 * torch.randn(K, generator=g)).to(dtype)
    total, out = ops.layernorm(x.cuda(), w.cuda(), b.cuda(), 1e-6, add=r.cuda())
    assert torch.equal(total.cpu(), x + r)
    eps = torch.finfo(dtype).eps
    for got, src in ((out, x + r), (ops.layernorm(x.cuda(), w.cuda(), b.cuda(), 1e-6), x)):
        ref = F.layer_norm(src.double(), (K,), w.double(), b.double(), 1e-6)
        assert ((got.cpu().double() - ref).abs() <= eps * ref.abs() + 2e-5).all()
    ref = F.gelu(x.double())
    got = ops.gelu_(x.cuda().clone()).cpu().double()
    assert ((got - ref).abs() <= eps * ref.abs() + 1e-6).all()


@pytest.mark.parametrize("M,N,K,epi,tile", [
    # columns / 32 of the tile (8, 10: resident, 3-5: K shared by the sides); whole and ragged edges, the shortest loop, several rounds
    (256, 256, 320, 0, 8), (700, 520, 384, 1, 8), (4096, 3840, 320, 2, 8), (20000, 1032, 320, 0, 8),
    (256, 320, 320, 1, 10), (900, 648, 448, 0, 10), (9000, 1288, 320, 1, 10),
    (256, 192, 320, 0, 192), (700, 392, 384, 1, 192), (9001, 1288, 320, 0, 192), (4096, 3072, 768, 1, 192),  # 192 columns
    (256, 96, 320, 2, 3), (700, 200, 832, 0, 3), (300, 128, 320, 1, 4), (4096, 1024, 1024, 2, 4), (256, 160, 320, 0, 5), (4000, 1288, 1280, 2, 5),
    # 320 rows by 256 columns
    (320, 256, 320, 2, 58), (700, 520, 384, 2, 58), (40900, 1016, 320, 2, 58),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_half_linear_with_its_epilogues(M, N, K, epi, tile, dtype):
    from samfast_amd import _lib, ops
    print(f"case half linear M={M} N={N} K={K} epi={epi} tile={tile} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    linear = torch.nn.Linear(K, N, bias=M % 2 == 0, device="cuda", dtype=dtype).requires_grad_(False)
    for p in linear.parameters():
        p.normal_(0.0, 0.05, generator=g)
    x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    total = torch.randn((M, N), generator=g, device="cuda").to(dtype) if epi == _lib.EPILOGUE_RESIDUAL else None
    with _lib.knobs(SAMFAST_GEMM_HALF=tile):
        outs = [ops.linear_half(x, linear, epi, residual=total, out=None) for _ in range(3)]
        if total is not None:
            inplace = total.clone()
            outs.append(ops.linear_half(x, linear, epi, residual=inplace, out=inplace))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    xd, wd, b = x.double(), linear.weight.double(), 0.0 if linear.bias is None else linear.bias.double()
    ref = xd @ wd.t() + b
    eps = torch.finfo(dtype).eps
    # one rounding to the type, and fp32 sums: at most K rounded additions of partial sums below sum |x||w|
    bound = 0.5 * eps * ref.abs() + K * 2.0 ** -24 * (xd.abs() @ wd.abs().t() + 1.0) + 2.0 ** -25
    if epi == _lib.EPILOGUE_GELU:  # slope at most 1.13, its own rounding, the fit
        ref = ref * 0.5 * torch.special.erfc(-ref * 0.5 ** 0.5)
        bound = 1.13 * bound + 0.51 * eps * ref.abs() + 2.0 ** -24
    elif total is not None:
        ref = ref + total.double()
        bound = bound * (1 + eps) + 0.5 * eps * ref.abs()
    assert ((outs[0].double() - ref).abs() <= bound * 1.0001).all()


# as few k tiles of 64 values as there are stages (tile 3: five, else four) and one to three more, both sides of the touched weights (32)
@pytest.mark.parametrize("K", [320, 384, 448, 512, 1984, 2048, 2112])
@pytest.mark.parametrize("tile", [3, 4, 5])
def test_split_half_linear_at_the_ends_of_its_loop(tile, K):
    test_half_linear_with_its_epilogues(301, 32 * tile + 40, K, 2, tile, torch.bfloat16)


@pytest.mark.parametrize("M,N,tile", [(301, 100, 3), (1500, 104, 3), (1025, 136, 4), (3000, 768, 3), (2000, 160, 5)])
def test_split_half_linear_whose_grid_touches_its_weights(M, N, tile):
    """Threads of the grid fewer and more than the lines of W, tiles no multiple of eight."""
    test_half_linear_with_its_epilogues(M, N // 8 * 8, 2048, 2, tile, torch.bfloat16)


def test_half_linear_leaves_what_it_does_not_take():
    from samfast_amd import ops
    linear = torch.nn.Linear(1024, 4096, device="cuda", dtype=torch.bfloat16).requires_grad_(False)
    x = torch.zeros((4096, 1024), device="cuda", dtype=torch.bfloat16)
    assert ops.linear_half(x, linear, 1) is not None
    assert ops.linear_half(x[:100], linear, 1) is None                       # too few rows
    assert ops.linear_half(_shifted(x), linear, 1) is None                   # off a 16-byte boundary
    assert ops.linear_half(torch.zeros((4096, 2048), device="cuda", dtype=torch.bfloat16)[:, ::2], linear, 1) is None
    linear.weight.data = linear.weight.data.t().contiguous().t()
    assert ops.linear_half(x, linear, 1) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,C,heads,window,bias", [(1, 768, 12, 14, True), (2, 320, 4, 0, True), (1, 320, 4, 11, False)])
def test_half_blocks_equal_module_composition(B, C, heads, window, bias, dtype, monkeypatch):
    from samfast_amd.modeling import image_encoder as ie
    print(f"case half block B={B} C={C} window={window} {dtype}", flush=True)
    torch.manual_seed(C + window)
    H = W = 64 if window != 11 else 25
    enc = torch.nn.Module()
    enc.blocks = torch.nn.ModuleList(
        ie.Block(C, heads, qkv_bias=bias, use_rel_pos=True, window_size=window, input_size=(H, W)) for _ in range(2))
    for p in enc.parameters():
        torch.nn.init.normal_(p, 1.0 if p.dim() == 1 and p.shape[0] == C else 0.0, 0.05)
    enc = enc.cuda().to(dtype).eval()
    x = torch.randn((B, H, W, C), device="cuda").to(dtype)
    with torch.no_grad():
        assert enc.blocks[0]._half_fused_ok(x)
        y, carry = enc.blocks[0]._forward_half_fused(x, None, enc.blocks[1].norm1)
        y = enc.blocks[1]._forward_half_fused(y, carry)[0]
        monkeypatch.setattr(ie, "FUSED_BLOCK", False)
        assert not enc.blocks[0]._half_fused_ok(x)
        ref = enc.blocks[1](enc.blocks[0](x))
    assert ((y.float() - ref.float()).norm() / ref.float().norm()).item() < 8 * torch.finfo(dtype).eps


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gelu_of_every_value(dtype):
    """No value further from x * Phi(x) than with the module it stands for, nor more of them; infinities and NaN alike."""
    from samfast_amd import ops
    print(f"case gelu {dtype}", flush=True)
    x = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dtype)
    exact = x.double() * 0.5 * torch.special.erfc(-x.double() * 0.5 ** 0.5)
    got, module = ops.gelu_(x.cuda().clone()).cpu(), F.gelu(x.cuda()).cpu()
    finite = torch.isfinite(x.float())
    assert torch.equal(got[~finite].float().nan_to_num(nan=-1.0), module[~finite].float().nan_to_num(nan=-1.0))
    assert torch.isfinite(got[finite].float()).all()
    missed = lambda y: (y[finite] != exact[finite].to(dtype)).sum().item()
    print(f"not correctly rounded: {missed(got)}, module {missed(module)}", flush=True)
    assert missed(got) <= missed(module)
    # half a unit of the type with fp32 steps in front of it, or half of fp16's smallest step; beyond |x| = 5, where Phi(-|x|)
    # is below 3e-7, the fit runs on with an error of at most 3e-12
    bound = 0.51 * torch.finfo(dtype).eps * exact[finite].abs() + (2.0 ** -25 if dtype == torch.float16 else 3e-12)
    assert ((got[finite].double() - exact[finite]).abs() <= bound).all()


def _shifted(t):
    """The same values, one element past a 16-byte boundary."""
    return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)


@pytest.mark.parametrize("what", ["eps", "norm parameters", "qkv bias", "input", "another current device"])
def test_half_block_and_layernorm2d_where_a_launch_does_not_serve(what, monkeypatch):
    """eps = 0 runs like any other; tensors off a 16-byte boundary, and a device that is not the current one, go
    through the composition."""
    from samfast_amd.modeling import image_encoder as ie
    from samfast_amd.modeling.common import LayerNorm2d
    print(f"case no launch: {what}", flush=True)
    torch.manual_seed(5)
    blk = ie.Block(128, 2, use_rel_pos=True, window_size=14, input_size=(64, 64)).cuda().to(torch.bfloat16).eval()
    norm = LayerNorm2d(128).cuda().to(torch.bfloat16)
    x = torch.randn((1, 20, 20, 128), device="cuda").to(torch.bfloat16)
    composed = what != "eps"
    with torch.no_grad():
        if what == "eps":
            blk.norm1.eps = blk.norm2.eps = norm.eps = 0.0
        elif what == "norm parameters":
            for m in (blk.norm2, norm):
                m.weight.data = _shifted(m.weight.data)
        elif what == "qkv bias":
            blk.attn.qkv.bias.data = _shifted(blk.attn.qkv.bias.data)
        elif what == "input":
            x = _shifted(x)
            assert x.data_ptr() % 16 != 0 and x.is_contiguous()
        maps = x.permute(0, 3, 1, 2)
        with monkeypatch.context() as m:
            if what == "another current device":
                m.setattr(torch.cuda, "current_device", lambda: 1)
            assert blk._half_fused_ok(x) is not composed
            assert norm._rows_ok(maps) is not (composed and what != "qkv bias")
        y, z = blk(x), norm(maps)
        monkeypatch.setattr(ie, "FUSED_BLOCK", False)
        assert ((y.float() - blk(x).float()).norm() / y.float().norm()).item() < 8 * torch.finfo(torch.bfloat16).eps
        ref = F.layer_norm(x.double(), (128,), norm.weight.double(), norm.bias.double(), norm.eps).permute(0, 3, 1, 2)
        assert ((z.double() - ref).abs() <= 8 * torch.finfo(torch.bfloat16).eps * (ref.abs() + 1)).all()


def test_hooks_and_subclasses_of_a_block_are_honoured():
    """Inside an encoder, where consecutive blocks are chained, a block with a hook is called as a module."""
    from samfast_amd.modeling import ImageEncoderViT, image_encoder as ie
    torch.manual_seed(3)
    enc = ImageEncoderViT(img_size=1024, embed_dim=128, depth=3, num_heads=2, use_rel_pos=True, window_size=14, global_attn_indexes=(1,))
    enc = enc.cuda().to(torch.bfloat16).eval()
    x = torch.randn((1, 64, 64, 128), device="cuda").to(torch.bfloat16)
    seen = []
    with torch.no_grad():
        plain = enc.forward_blocks(x)
        handles = [b.register_forward_hook(lambda m, a, out, i=i: seen.append((i, out))) for i, b in enumerate(enc.blocks)]
        watched = enc.forward_blocks(x)
        assert [i for i, _ in seen] == [0, 1, 2] and torch.equal(seen[2][1], watched)
        assert ((watched.float() - plain.float()).norm() / plain.float().norm()).item() < 8 * torch.finfo(torch.bfloat16).eps
        for h in handles:
            h.remove()
        handle = enc.blocks[2].register_forward_hook(lambda m, a, out: torch.zeros_like(out))
        assert not enc.forward_blocks(x).any()
        handle.remove()

        class Skipped(ie.Block):
            def forward(self, x):
                return x

        before = enc.blocks[:2]
        enc.blocks[2].__class__ = Skipped
        whole = enc.forward_blocks(x)
        enc.blocks = before
        assert torch.equal(whole, enc.forward_blocks(x))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,C,H,W", [(1, 256, 64, 64), (3, 256, 5, 7), (2, 8, 3, 3), (1, 264, 2, 3), (1, 512, 1, 5), (1, 520, 2, 2), (0, 256, 4, 4)])
def test_layernorm2d_over_channels_last(B, C, H, W, dtype):
    """One launch on a channels-last map; a contiguous one, and one under autograd, stay composed."""
    from samfast_amd.modeling.common import LayerNorm2d
    print(f"case layernorm2d {B}x{C}x{H}x{W} {dtype}", flush=True)
    g = torch.Generator().manual_seed(C + H)
    norm = LayerNorm2d(C)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * torch.randn(C, generator=g))
        norm.bias.copy_(0.1 * torch.randn(C, generator=g))
    norm = norm.to(dtype)
    x = (torch.randn((B, C, H, W), generator=g) * 2 + 0.5).to(dtype)
    ref = F.layer_norm(x.permute(0, 2, 3, 1).double(), (C,), norm.weight.double(), norm.bias.double(), norm.eps).permute(0, 3, 1, 2)
    gpu = norm.cuda()
    xl = x.cuda().contiguous(memory_format=torch.channels_last)
    eps = torch.finfo(dtype).eps
    with torch.no_grad():
        y = gpu(xl)
        assert y.shape == x.shape and (B == 0 or gpu._rows_ok(xl))
        # one rounding of the result, fp32 statistics
        assert ((y.cpu().double() - ref).abs() <= eps * ref.abs() + 2e-5).all()
        if B and H * W > 1:
            # the composition rounds five intermediates to the type
            assert ((gpu(x.cuda()).cpu().double() - ref).abs() <= 8 * eps * (ref.abs() + 1)).all()
    assert not gpu._rows_ok(xl)  # gradients wanted


def test_layernorm2d_stays_composed_under_transforms():
    from samfast_amd.modeling.common import LayerNorm2d
    norm = LayerNorm2d(16).to(torch.bfloat16).cuda()
    x = torch.randn((2, 3, 16, 4, 4), device="cuda").to(torch.bfloat16).flatten(0, 1).contiguous(memory_format=torch.channels_last).view(2, 3, 16, 4, 4)
    with torch.no_grad():
        want = torch.stack([norm(t) for t in x])
        assert norm._rows_ok(x[0])
        got = torch.vmap(norm)(x)
        assert (got.float() - want.float()).abs().max() <= 8 * torch.finfo(torch.bfloat16).eps * (want.float().abs().max() + 1)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x[0], torch.ones_like(x[0]))
            assert torch.autograd.forward_ad.unpack_dual(norm(dual)).tangent is not None


def test_half_block_and_layernorm2d_are_composed_where_somebody_watches(monkeypatch):
    """Autocast gives the types it gives the composition, and a dispatch mode sees its operations."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from samfast_amd.modeling import image_encoder as ie
    from samfast_amd.modeling.common import LayerNorm2d
    torch.manual_seed(6)
    blk = ie.Block(128, 2, use_rel_pos=True, window_size=14, input_size=(64, 64)).cuda().to(torch.bfloat16).eval()
    norm = LayerNorm2d(128).cuda().to(torch.bfloat16)
    x = torch.randn((1, 20, 20, 128), device="cuda").to(torch.bfloat16)
    maps = x.permute(0, 3, 1, 2)

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    def calls():
        with torch.autocast("cuda", dtype=torch.float16):
            cast = blk(x), norm(maps)
        names.clear()
        with Names():
            seen = blk(x), norm(maps)
        return cast + seen, list(names)

    names = []
    with torch.no_grad():
        assert blk._half_fused_ok(x) and norm._rows_ok(maps)
        got, got_names = calls()
        monkeypatch.setattr(ie, "FUSED_BLOCK", False)
        monkeypatch.setattr(LayerNorm2d, "_rows_ok", lambda self, x: False)
        want, want_names = calls()
    assert got_names == want_names and "gelu" in got_names
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and torch.equal(g, w)
