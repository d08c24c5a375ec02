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
