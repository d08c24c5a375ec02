"""SAM ViT image encoder with the hot path on the HIP kernels.

Class names, constructor signatures, parameter names (hence state-dict keys) and
tensor contracts follow segment_anything_fast/modeling/image_encoder.py:
ImageEncoderViT :18-117, Block :120-183, Attention :186-253, window_partition
:256-277, window_unpartition :280-302, get_rel_pos :305-335,
add_decomposed_rel_pos :338-372, PatchEmbed :375-406.

What differs is Attention.forward on a GPU in bf16: q, k and v are read by the
attention kernel straight out of the qkv Linear's (B, N, 3, nH, hd) output
through strides, the two bias factors are computed inside the kernel from
rel_pos_h / rel_pos_w, and the result is written token-major, so the head
split/merge copies (:228-230, :249) and the bias tensors (:234-242) never exist.
Any other input (CPU, fp32, shapes the kernels do not cover) follows the
reference's own composition through flash_4._attention_rel_h_rel_w.

When, in addition, the four Linears of a Block have been swapped for
quant.Int8DynamicLinear, Block.forward (:167-183) runs with no eager glue as nine kernel
launches: LayerNorm + quantise, qkv GEMM, attention, quantise, proj GEMM + residual, LayerNorm
+ quantise, lin1 GEMM, GELU + quantise, lin2 GEMM + residual.  With SAMFAST_FUSED_QUANT=1 the
three quantisers that follow a GEMM run inside that GEMM (proj + norm2 + quantise, lin1 +
quantise, lin2 + the NEXT block's norm1 + quantise: five launches per block, same bits; slower
at the measured shapes, hence not the default).  SAMFAST_FUSED_BLOCK=0 keeps the
module-by-module composition.
"""

import os
from typing import Optional, Sequence, Tuple, Type

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import _lib, flash_4, ops
from ..flash_4 import _attention_rel_h_rel_w
from .common import LayerNorm2d, MLPBlock

KB64_OPERANDS = os.environ.get("SAMFAST_KB64", "1") != "0"
WINDOWS_IN_PLACE = os.environ.get("SAMFAST_WINDOWS_IN_PLACE", "1") != "0"
# The neck on the kernels here up to this many tokens.  More are the library's convolutions, so that embeddings of large batches keep their bits: these kernels' differ by 5.4e-3
# of the norm (against 64 bits, on the tokens of five encoders, library 3.4e-3, here 3.3e-3), for little time (us with its LayerNorms, library / here: width 1280, one image 107
# / 38, four 201 / 73, ten 202 / 152, but sixteen 285 / 232 of an encoder's 58000, 32 541 / 499 of 109000)
NECK_TOKENS = 40960
# Weights that a window attention kernel reads ahead of the products behind it (read_soon): up to this many tokens, this many
# bytes a block, from this many bytes over all blocks on, and for more than half of the tokens from this many bytes a block on
SOON_TOKENS, SOON_BYTES, SOON_TOTAL, SOON_LEAST = 8192, 9 << 20, 85 << 20, 3 << 20
FUSED_BLOCK = bool(int(os.environ.get("SAMFAST_FUSED_BLOCK", 1)))


def read_soon(depth: int, tokens: int, weights: Sequence[torch.Tensor]) -> Sequence[torch.Tensor]:
    """Of `weights`, those of the products behind one of `depth` blocks' attention, what the window kernel's idle wavefront reads
    while the others multiply.  Weights that were not read lately come out of HBM, and an image's products wait for them a k tile at a
    time: proj first, then lin2, whose loop is the longest, then the next block's qkv, while they stay few enough to arrive under the attention; lin1's gains less than it
    costs there.  us a recorded pass, none / so, the middle of four recordings of each by turns, the same to 0.3 % on two machines: one image of ViT-L int8
    3262 / 3168, with 2:4 MLPs 3271 / 3116, ViT-H int8 5138 / 5065, 5011 / 4842, bf16 ViT-B 1591 / 1568, ViT-L 3661 / 3635, ViT-H 6255 / 6185 (proj alone; with
    lin2 6265 / 6309); two of ViT-B bf16 2670 / 2650, ViT-L int8 5396 / 5321, 4983 / 4921, ViT-H int8 level, bf16 11828 / 11669.
    The form that reads costs a launch of 20 us 1.7: two images of ViT-L bf16, 2 MB a block, are 6475 / 6514 (SOON_LEAST).  Encoders of other
    depths show where the weights of all blocks stay near enough without (MiB of the three Linears, times as long: width 768 int8 54 1.002, 81 0.999, 108 0.989, 135 0.985, bf16 72 1.002, 81
    1.004, 108 0.995, width 1024 int8 64 0.997, 80 0.993, 96 0.985, width 1280 75 1.001, 100 0.999): SOON_TOTAL.
    From four images on it is level (ViT-H int8 16284 / 16309)."""
    if tokens > SOON_TOKENS:
        return ()
    sizes = [w.numel() * w.element_size() for w in weights]
    if depth * sum(sizes) < SOON_TOTAL:
        return ()
    read = [w for i, w in enumerate(weights) if sum(sizes[:i + 1]) <= SOON_BYTES]
    return read if 2 * tokens <= SOON_TOKENS or sum(sizes[:len(read)]) >= SOON_LEAST else ()


def _recording(x: torch.Tensor) -> bool:
    return x.is_cuda and torch.cuda.is_current_stream_capturing()


class ImageEncoderViT(nn.Module):
    def __init__(
        self,
        img_size: int = 1024,
        patch_size: int = 16,
        in_chans: int = 3,
        embed_dim: int = 768,
        depth: int = 12,
        num_heads: int = 12,
        mlp_ratio: float = 4.0,
        out_chans: int = 256,
        qkv_bias: bool = True,
        norm_layer: Type[nn.Module] = nn.LayerNorm,
        act_layer: Type[nn.Module] = nn.GELU,
        use_abs_pos: bool = True,
        use_rel_pos: bool = False,
        rel_pos_zero_init: bool = True,
        window_size: int = 0,
        global_attn_indexes: Tuple[int, ...] = (),
    ) -> None:
        super().__init__()
        self.img_size = img_size
        grid = img_size // patch_size
        self.patch_embed = PatchEmbed(
            kernel_size=(patch_size, patch_size), stride=(patch_size, patch_size),
            in_chans=in_chans, embed_dim=embed_dim)
        self.pos_embed: Optional[nn.Parameter] = None
        if use_abs_pos:
            self.pos_embed = nn.Parameter(torch.zeros(1, grid, grid, embed_dim))
        self.blocks = nn.ModuleList([
            Block(
                dim=embed_dim, num_heads=num_heads, mlp_ratio=mlp_ratio, qkv_bias=qkv_bias,
                norm_layer=norm_layer, act_layer=act_layer, use_rel_pos=use_rel_pos,
                rel_pos_zero_init=rel_pos_zero_init,
                window_size=0 if i in global_attn_indexes else window_size,
                input_size=(grid, grid))
            for i in range(depth)
        ])
        self.neck = nn.Sequential(
            nn.Conv2d(embed_dim, out_chans, kernel_size=1, bias=False),
            LayerNorm2d(out_chans),
            nn.Conv2d(out_chans, out_chans, kernel_size=3, padding=1, bias=False),
            LayerNorm2d(out_chans),
        )

    # images per pass through the blocks; None = as many as the int8 kernels can address
    max_images_per_pass: Optional[int] = None

    def images_per_pass(self, x: torch.Tensor) -> int:
        """The int8 GEMMs and the row quantiser address an activation of M rows and K columns with
        32-bit offsets (M * K < 2^31).  The widest one is lin2's input, 4C per token: 102 images of
        64 x 64 tokens at ViT-H.  Images are independent, so a larger batch goes through the blocks
        in passes of at most that many."""
        if self.max_images_per_pass is not None:
            return max(1, int(self.max_images_per_pass))
        from ..quant import Int8LinearBase
        widest = max((m.in_features for m in self.modules() if isinstance(m, Int8LinearBase)), default=0)
        if widest == 0:
            return x.shape[0]
        return max(1, (2 ** 31 - 1) // (x.shape[1] * x.shape[2] * widest))

    def forward_blocks(self, x: torch.Tensor) -> torch.Tensor:
        """The transformer blocks on (B, H, W, C) tokens.  Consecutive blocks on the fused int8
        path are chained: a block's lin2 launch also runs the next block's norm1 and the qkv
        Linear's quantiser on the rows it has just written."""
        per_pass = self.images_per_pass(x)
        if x.shape[0] > per_pass:
            return torch.cat([self.forward_blocks(x[i:i + per_pass]) for i in range(0, x.shape[0], per_pass)])
        carry = None
        # Weights are read ahead (read_soon) in recordings.  Launches that the host issues one by one wait for it more than for the weights, and a list takes
        # it 10 us a block (us a pass, none / so: ViT-L int8 4411 / 4618, ViT-H int8 6570 / 6864, ViT-B bf16 2493 / 2570; two of ViT-L int8 5418 / 5341).
        depth = len(self.blocks) if x.shape[0] * x.shape[1] * x.shape[2] <= SOON_TOKENS and _recording(x) else 0
        for i, blk in enumerate(self.blocks):
            if not blk._int8_fused_ok(x):
                if not blk._half_fused_ok(x):
                    x, carry = blk(x), None
                    continue
                nxt = self.blocks[i + 1] if i + 1 < len(self.blocks) else None
                chained = nxt is not None and not nxt._int8_fused_ok(x) and nxt._half_fused_ok(x)
                x, carry = blk._forward_half_fused(x, carry, nxt.norm1 if chained else None, nxt.attn.qkv if chained else None, depth)
                continue
            nxt = self.blocks[i + 1] if i + 1 < len(self.blocks) else None
            next_norm = next_qkv = None
            if nxt is not None and nxt._int8_fused_ok(x) and nxt._chains_from_previous():
                next_norm, next_qkv = (nxt.norm1.weight, nxt.norm1.bias, nxt.norm1.eps), nxt.attn.qkv
            x, carry = blk._forward_int8_fused(x, carry, next_norm, next_qkv, depth)
        return x

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        x = self.patch_embed(x)
        if self.pos_embed is not None:
            x = x + self.pos_embed
        x = self.forward_blocks(x)
        if self._neck_launchable(x):
            conv1, norm1, conv3, norm2 = self.neck
            rows = lambda norm: lambda y: ops.layernorm(y, norm.weight, norm.bias, norm.eps)
            return rows(norm2)(ops.neck_convs(x, conv1.weight, rows(norm1), conv3.weight)).permute(0, 3, 1, 2)
        return self.neck(x.permute(0, 3, 1, 2))

    def _neck_launchable(self, x: torch.Tensor) -> bool:
        """Whether the neck is what the constructor builds and nothing else (no hook, subclass or other convolution), over few
        enough tokens for the kernels here, with nobody watching."""
        if not (FUSED_BLOCK and x.is_cuda and x.dim() == 4 and x.dtype in (torch.bfloat16, torch.float16) and not torch.is_grad_enabled()
                and x.shape[0] * x.shape[1] * x.shape[2] <= NECK_TOKENS and ops.unwatched(x)):
            return False
        kinds = (nn.Conv2d, LayerNorm2d, nn.Conv2d, LayerNorm2d)
        if type(self.neck) is not nn.Sequential or len(self.neck) != 4 or tuple(type(m) for m in self.neck) != kinds:
            return False
        if any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ for m in (self.neck, *self.neck)):
            return False
        if nn.modules.module._global_forward_hooks or nn.modules.module._global_forward_pre_hooks:
            return False
        conv1, norm1, conv3, norm2 = self.neck
        for m, size in ((conv1, 1), (conv3, 3)):
            if not (m.kernel_size == (size, size) and m.padding == (size // 2, size // 2) and m.stride == m.dilation == (1, 1)
                    and m.groups == 1 and m.bias is None and m.padding_mode == "zeros"
                    and m.weight.shape == (m.out_channels, m.in_channels, size, size)
                    and m.in_channels % 64 == 0 and m.out_channels % 64 == 0 and m.in_channels <= 4096 and m.out_channels <= 4096):
                return False
        tensors = (x, conv1.weight, norm1.weight, norm1.bias, conv3.weight, norm2.weight, norm2.bias)
        return (all(type(t) in (torch.Tensor, nn.Parameter) and t.dtype == x.dtype for t in tensors) and ops.rows_launchable(*tensors)
                and conv1.in_channels == x.shape[3] and conv1.out_channels == conv3.in_channels and conv3.in_channels * 18 <= 96 * 1024
                and norm1.weight.numel() == norm1.bias.numel() == conv1.out_channels
                and norm2.weight.numel() == norm2.bias.numel() == conv3.out_channels
                and norm1.eps >= 0 and norm2.eps >= 0)


class Block(nn.Module):
    """Pre-norm transformer block; window_size > 0 runs attention inside
    non-overlapping windows, 0 runs it over the whole grid."""

    def __init__(
        self,
        dim: int,
        num_heads: int,
        mlp_ratio: float = 4.0,
        qkv_bias: bool = True,
        norm_layer: Type[nn.Module] = nn.LayerNorm,
        act_layer: Type[nn.Module] = nn.GELU,
        use_rel_pos: bool = False,
        rel_pos_zero_init: bool = True,
        window_size: int = 0,
        input_size: Optional[Tuple[int, int]] = None,
    ) -> None:
        super().__init__()
        self.norm1 = norm_layer(dim)
        self.attn = Attention(
            dim, num_heads=num_heads, qkv_bias=qkv_bias, use_rel_pos=use_rel_pos,
            rel_pos_zero_init=rel_pos_zero_init,
            input_size=input_size if window_size == 0 else (window_size, window_size))
        self.norm2 = norm_layer(dim)
        self.mlp = MLPBlock(embedding_dim=dim, mlp_dim=int(dim * mlp_ratio), act=act_layer)
        self.window_size = window_size

    def _int8_fused_ok(self, x: torch.Tensor) -> bool:
        from ..quant import Int8LinearBase
        attn, mlp = self.attn, self.mlp
        if not (FUSED_BLOCK and flash_4.USE_CUSTOM_KERNEL and x.is_cuda
                and x.dtype == torch.bfloat16 and x.dim() == 4 and attn.use_rel_pos):
            return False
        if not all(isinstance(m, Int8LinearBase) for m in (attn.qkv, attn.proj, mlp.lin1, mlp.lin2)):
            return False
        if self.window_size > 0 and not attn.proj.supports_row_scatter:
            return False
        if not (isinstance(self.norm1, nn.LayerNorm) and isinstance(self.norm2, nn.LayerNorm)
                and self.norm1.elementwise_affine and self.norm2.elementwise_affine
                and self.norm1.bias is not None and self.norm2.bias is not None
                and self.norm1.weight.dtype == torch.bfloat16
                and attn.rel_pos_h.dtype == torch.bfloat16 and attn.rel_pos_w.dtype == torch.bfloat16
                and isinstance(mlp.act, nn.GELU) and getattr(mlp.act, "approximate", "none") == "none"):
            return False
        B, H, W, C = x.shape
        g = self.window_size if self.window_size > 0 else None
        gh, gw = (g, g) if g else (H, W)
        return (attn.rel_pos_h.shape[0] == 2 * gh - 1 and attn.rel_pos_w.shape[0] == 2 * gw - 1
                and ops.attn_supported(gh * gw, (gh, gw), C // attn.num_heads, x.dtype))

    def _pad_rows(self, nH: int, hd: int, device):
        """(nH, hd) bf16 k and v rows of a zero-padded token: the qkv bias, rounded as the
        Linear's epilogue rounds it."""
        from ..quant import kept_copy
        qkv, C = self.attn.qkv, nH * hd

        def rows():
            bias = qkv.bias_f32
            if bias is None:
                return (torch.zeros((nH, hd), dtype=torch.bfloat16, device=device),) * 2
            return tuple(bias[i * C:(i + 1) * C].to(torch.bfloat16).view(nH, hd).contiguous() for i in (1, 2))

        return kept_copy(self, "_pad_kv", qkv.sw_bits if qkv.bias_bits is None else qkv.bias_bits, rows)

    def _chains_from_previous(self) -> bool:
        """Whether this block's norm1 + quantiser can run in the previous block's lin2 launch:
        its rows must be the image-ordered tokens (no window gather in front of qkv)."""
        return self.window_size == 0 or WINDOWS_IN_PLACE

    def _forward_int8_fused(self, x: torch.Tensor, carry=None, next_norm=None, next_qkv=None, depth=0):
        """image_encoder.py:167-183 with every step on the HIP kernels.

        `carry` = (xq, sx): this block's norm1 output, already quantised by the previous block's
        lin2 launch.  `next_norm` = (gamma, beta, eps) of the next block's norm1: lin2 then
        also returns that block's carry; `next_qkv`: that block's first Linear; `depth`: of how many
        blocks this is one whose weights may be read ahead (0: of none).  Returns (tokens (B, H, W, C), carry for the next block)."""
        from .. import quant
        B, H, W, C = x.shape
        attn, mlp = self.attn, self.mlp
        nH = attn.num_heads
        hd = C // nH
        tokens = x.contiguous().view(B * H * W, C)
        # int8 activations travel K-block major between the quantisers and the GEMMs
        L = _lib.LAYOUT_KB64 if (C % 64 == 0 and KB64_OPERANDS) else _lib.LAYOUT_ROWMAJOR
        ws = self.window_size
        norm2 = (self.norm2.weight, self.norm2.bias, self.norm2.eps)
        if ws > 0 and not WINDOWS_IN_PLACE:
            # windows materialised: the partition is a row gather in the LayerNorm+quant kernel,
            # the unpartition a row scatter in the proj epilogue
            row_map, _ = ops.window_row_maps(B, H, W, ws, x.device)
            N = ws * ws
            xq, sx = ops.layernorm_quant(tokens, self.norm1.weight, self.norm1.bias, self.norm1.eps, row_map, layout=L)
            Bw = sx.shape[0] // N
            qkv = attn.qkv.linear_fused(xq, sx, _lib.EPILOGUE_NONE, layout=L).view(Bw, N, 3, nH, hd)
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
            o = ops.attn_relpos(q, k, v, attn.rel_pos_h, attn.rel_pos_w, (ws, ws), attn.scale)
            oq, so = ops.quant_rowwise(o.permute(0, 2, 1, 3).reshape(Bw * N, C), layout=L)
            tokens = attn.proj.linear_fused(oq, so, _lib.EPILOGUE_RESIDUAL, residual=tokens, dst_row=row_map, layout=L)
            hq, sh = ops.layernorm_quant(tokens, *norm2, layout=L)
        else:
            # norm1 + qkv's activation quantiser (unless the previous block's lin2 launch has done
            # it), qkv GEMM on the image-ordered tokens
            if carry is not None:
                xq, sx = carry
            else:
                xq, sx = ops.layernorm_quant(tokens, self.norm1.weight, self.norm1.bias, self.norm1.eps, layout=L)
            qkv = attn.qkv.linear_fused(xq, sx, _lib.EPILOGUE_NONE, layout=L).view(B, H * W, 3, nH, hd)
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
            if ws > 0:
                # the attention kernel cuts the windows itself; the reference's zero-padded tokens
                # enter as keys / values with the rows a zero input gives the qkv Linear: its bias
                pad_k, pad_v = self._pad_rows(nH, hd, x.device)
                soon = () if depth == 0 else read_soon(depth, B * H * W, [t for m in (attn.proj, mlp.lin2, next_qkv) if m is not None for t in m.weight_operands(L)])
                o = ops.attn_relpos_windowed(q, k, v, attn.rel_pos_h, attn.rel_pos_w, pad_k, pad_v,
                                             (H, W), ws, attn.scale, soon).view(B * H * W, C)
            else:
                o = ops.attn_relpos(q, k, v, attn.rel_pos_h, attn.rel_pos_w, (H, W), attn.scale)
                o = o.permute(0, 2, 1, 3).reshape(B * H * W, C)
            # proj's quantiser, proj + `shortcut + x`, norm2 + lin1's quantiser: one launch for few tokens
            one = None
            if type(attn.proj) is quant.Int8DynamicLinear and L == _lib.LAYOUT_KB64 and not quant.FUSED_QUANT:
                one = ops.proj_block(o, attn.proj._weight_for(L), attn.proj.sw, attn.proj.bias_f32, tokens, norm2)
            if one is not None:
                tokens, hq, sh = one
            else:
                oq, so = ops.quant_rowwise(o, layout=L)
                tokens, hq, sh = attn.proj.linear_fused_quant(oq, so, _lib.EPILOGUE_RESIDUAL, residual=tokens,
                                                              layout=L, ln=norm2, out_layout=L)
        # lin1, GELU, lin2's quantiser, lin2 + `x + mlp(...)` (+ the next block's norm1 and quantiser).  GELU runs in the
        # quantiser, which waits for memory, except where an image's lin1 is short (lin1 + quantiser, us, GELU in lin1 / in the quantiser:
        # 8192 x 768 45.9 / 42.7, 12288 x 768 66.6 / 57.8, 4096 x 1024 34.9 / 31.4, 4096 x 1280 51.7 / 47.4, 65536 x 1280 661 / 601, 65536 x
        # 768 335 / 313, 4096 x 768 29.1 / 28.1; all twelve blocks of a ViT-B, one image 1404 / 1412, two 2261 / 2222, five 4897 / 4722)
        if quant.FUSED_QUANT or (C < 1024 and tokens.shape[0] < 8192):
            _, gq, sg = mlp.lin1.linear_fused_quant(hq, sh, _lib.EPILOGUE_GELU, layout=L, out_layout=L)
        else:
            gq, sg = ops.quant_rowwise(mlp.lin1.linear_fused(hq, sh, _lib.EPILOGUE_NONE, layout=L), layout=L, gelu=True)
        if next_norm is not None:
            tokens, nq, sn = mlp.lin2.linear_fused_quant(gq, sg, _lib.EPILOGUE_RESIDUAL, residual=tokens,
                                                         out=tokens, layout=L, ln=next_norm, out_layout=L)
            return tokens.view(B, H, W, C), (nq, sn)
        tokens = mlp.lin2.linear_fused(gq, sg, _lib.EPILOGUE_RESIDUAL, residual=tokens, out=tokens, layout=L)
        return tokens.view(B, H, W, C), None

    def _as_built(self) -> bool:
        """Whether calling this block is what its constructor wrote and nothing else: no subclass, hook or
        forward of an instance's own on it or on the modules inside, and no hook on every module."""
        attn, mlp = self.attn, self.mlp
        built = ((self, Block), (self.norm1, nn.LayerNorm), (attn, Attention), (self.norm2, nn.LayerNorm),
                 (mlp, MLPBlock), (mlp.act, nn.GELU),
                 *((m, nn.Linear) for m in (attn.qkv, attn.proj, mlp.lin1, mlp.lin2)))
        return (all(type(m) is cls and not m._forward_hooks and not m._forward_pre_hooks and "forward" not in m.__dict__
                    for m, cls in built)
                and not nn.modules.module._global_forward_hooks and not nn.modules.module._global_forward_pre_hooks)

    def _half_fused_ok(self, x: torch.Tensor) -> bool:
        """Whether this block, its Linears left in the half type, can run through _forward_half_fused:
        inference on a GPU in bf16 / fp16 at a shape the attention kernels cover, with nobody's hook or
        class in the way."""
        attn, mlp = self.attn, self.mlp
        if not (FUSED_BLOCK and flash_4.USE_CUSTOM_KERNEL and x.is_cuda and x.dim() == 4
                and x.dtype in (torch.bfloat16, torch.float16) and attn.use_rel_pos and not torch.is_grad_enabled()):
            return False
        if not ops.unwatched(x) or not self._as_built() or mlp.act.approximate != "none":
            return False
        B, H, W, C = x.shape
        for n in (self.norm1, self.norm2):
            if n.weight is None or n.bias is None or n.weight.dtype != x.dtype or n.normalized_shape != (C,) or not n.eps >= 0:
                return False
        # what the row kernels read as it is (the qkv bias: the window kernel's padding rows)
        rows = [self.norm1.weight, self.norm1.bias, self.norm2.weight, self.norm2.bias]
        if attn.qkv.bias is not None:
            rows.append(attn.qkv.bias)
        if not ops.rows_launchable(*rows) or x.device != rows[0].device or x.data_ptr() % 16 != 0:
            return False
        ws = self.window_size
        gh, gw = (ws, ws) if ws > 0 else (H, W)
        return (attn.qkv.weight.dtype == x.dtype and C % 8 == 0 and C <= 4096 and mlp.lin1.out_features % 8 == 0
                and attn.rel_pos_h.dtype == x.dtype and attn.rel_pos_w.dtype == x.dtype
                and attn.rel_pos_h.shape[0] == 2 * gh - 1 and attn.rel_pos_w.shape[0] == 2 * gw - 1
                and ops.attn_supported(gh * gw, (gh, gw), C // attn.num_heads, x.dtype)
                and (ws == 0 or ws * ws <= 208))

    def _forward_half_fused(self, x: torch.Tensor, carry=None, next_norm=None, next_qkv=None, depth=0):
        """image_encoder.py:167-183 with half-type Linears: four products, those that pay on this library's kernels with
        GELU or the residual add in them (ops.linear_half), and two or three launches around them.  The
        attention kernel cuts the windows out of the image-ordered tokens, so the products run on the image's tokens only
        (the zero-padded windows have a fifth more) and nothing is partitioned, padded or copied; a residual
        add that is in no product runs with the norm that follows it.
        `carry`: norm1's output, where the previous block has made it; `next_norm`, `next_qkv`, `depth`: as above.
        Returns (tokens, carry for the next block)."""
        B, H, W, C = x.shape
        attn, mlp, ws = self.attn, self.mlp, self.window_size
        nH = attn.num_heads
        hd = C // nH
        tokens = x.contiguous().view(B * H * W, C)
        h = carry if carry is not None else ops.layernorm(tokens, self.norm1.weight, self.norm1.bias, self.norm1.eps)
        qkv = ops.linear_half(h, attn.qkv)
        qkv = (attn.qkv(h) if qkv is None else qkv).view(B, H * W, 3, nH, hd)
        q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
        if ws > 0:
            # a zero-padded token's k and v rows: the qkv bias
            pads = (torch.zeros((2, nH, hd), dtype=x.dtype, device=x.device) if attn.qkv.bias is None
                    else attn.qkv.bias[C:].view(2, nH, hd))
            soon = () if depth == 0 else read_soon(depth, B * H * W, [m.weight for m in (attn.proj, mlp.lin2, next_qkv) if m is not None])
            o = ops.attn_relpos_windowed(q, k, v, attn.rel_pos_h, attn.rel_pos_w, pads[0], pads[1], (H, W), ws, attn.scale, soon)
        else:
            o = ops.attn_relpos(q, k, v, attn.rel_pos_h, attn.rel_pos_w, (H, W), attn.scale).permute(0, 2, 1, 3)
        o = o.reshape(B * H * W, C)

        def add(rows, linear, total, norm):
            """(total + linear(rows), norm of that)"""
            summed = ops.linear_half(rows, linear, _lib.EPILOGUE_RESIDUAL, residual=total)
            if summed is None and norm is not None:
                return ops.layernorm(total, norm.weight, norm.bias, norm.eps, add=linear(rows))
            if summed is None:
                return total + linear(rows), None
            return summed, None if norm is None else ops.layernorm(summed, norm.weight, norm.bias, norm.eps)

        tokens, h = add(o, attn.proj, tokens, self.norm2)
        m = ops.linear_half(h, mlp.lin1, _lib.EPILOGUE_GELU)
        tokens, h = add(ops.gelu_(mlp.lin1(h)) if m is None else m, mlp.lin2, tokens, next_norm)
        return tokens.view(B, H, W, C), h

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self._int8_fused_ok(x):
            return self._forward_int8_fused(x)[0]
        if self._half_fused_ok(x):
            return self._forward_half_fused(x)[0]
        shortcut = x
        x = self.norm1(x)
        if self.window_size > 0:
            H, W = x.shape[1], x.shape[2]
            x, pad_hw = window_partition(x, self.window_size)
        x = self.attn(x)
        if self.window_size > 0:
            x = window_unpartition(x, self.window_size, pad_hw, (H, W))
        x = shortcut + x
        return x + self.mlp(self.norm2(x))


class Attention(nn.Module):
    """Multi-head attention over a (B, H, W, C) token grid with decomposed
    relative-position bias."""

    def __init__(
        self,
        dim: int,
        num_heads: int = 8,
        qkv_bias: bool = True,
        use_rel_pos: bool = False,
        rel_pos_zero_init: bool = True,
        input_size: Optional[Tuple[int, int]] = None,
    ) -> None:
        super().__init__()
        self.num_heads = num_heads
        head_dim = dim // num_heads
        self.scale = head_dim ** -0.5
        self.qkv = nn.Linear(dim, dim * 3, bias=qkv_bias)
        self.proj = nn.Linear(dim, dim)
        self.use_rel_pos = use_rel_pos
        if self.use_rel_pos:
            assert input_size is not None, \
                "Input size must be provided if using relative positional encoding."
            self.rel_pos_h = nn.Parameter(torch.zeros(2 * input_size[0] - 1, head_dim))
            self.rel_pos_w = nn.Parameter(torch.zeros(2 * input_size[1] - 1, head_dim))

    def _fused_ok(self, qkv: torch.Tensor, H: int, W: int, hd: int) -> bool:
        return (self.use_rel_pos and flash_4.USE_CUSTOM_KERNEL and qkv.is_cuda
                and self.rel_pos_h.shape[0] == 2 * H - 1 and self.rel_pos_w.shape[0] == 2 * W - 1
                and ops.attn_supported(H * W, (H, W), hd, qkv.dtype))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        B, H, W, C = x.shape
        nH = self.num_heads
        hd = C // nH
        qkv = self.qkv(x).reshape(B, H * W, 3, nH, hd)
        if self._fused_ok(qkv, H, W, hd):
            # strided (B, nH, N, hd) views of the token-major qkv buffer: no copies
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
            out = ops.attn_relpos(q, k, v, self.rel_pos_h, self.rel_pos_w, (H, W), self.scale)
            x = out.permute(0, 2, 1, 3).reshape(B, H, W, C)  # already token-major: a view
            return self.proj(x)

        q, k, v = qkv.permute(2, 0, 3, 1, 4).reshape(3, B * nH, H * W, hd).unbind(0)
        if self.use_rel_pos:
            rel_h, rel_w = add_decomposed_rel_pos(q, self.rel_pos_h, self.rel_pos_w, (H, W), (H, W))
            rel_h = rel_h.view(B, nH, H * W, H, 1)
            rel_w = rel_w.view(B, nH, H * W, 1, W)
        q, k, v = (t.view(B, nH, H * W, hd) for t in (q, k, v))
        if self.use_rel_pos:
            x = _attention_rel_h_rel_w(q, k, v, rel_h, rel_w)
        else:
            x = F.scaled_dot_product_attention(q, k, v)
        x = x.view(B, nH, H, W, hd).permute(0, 2, 3, 1, 4).reshape(B, H, W, C)
        return self.proj(x)


def window_partition(x: torch.Tensor, window_size: int) -> Tuple[torch.Tensor, Tuple[int, int]]:
    """(B, H, W, C) -> ((B * nWindows, ws, ws, C), (Hp, Wp)), zero padding the
    bottom and right edges up to a multiple of the window."""
    B, H, W, C = x.shape
    pad_h = (-H) % window_size
    pad_w = (-W) % window_size
    if pad_h or pad_w:
        x = F.pad(x, (0, 0, 0, pad_w, 0, pad_h))
    Hp, Wp = H + pad_h, W + pad_w
    x = x.reshape(B, Hp // window_size, window_size, Wp // window_size, window_size, C)
    windows = x.transpose(2, 3).reshape(-1, window_size, window_size, C)
    return windows, (Hp, Wp)


def window_unpartition(windows: torch.Tensor, window_size: int, pad_hw: Tuple[int, int],
                       hw: Tuple[int, int]) -> torch.Tensor:
    """Inverse of window_partition: back to (B, H, W, C) without the padding."""
    Hp, Wp = pad_hw
    H, W = hw
    per_image = (Hp // window_size) * (Wp // window_size)
    B = windows.shape[0] // per_image
    x = windows.view(B, Hp // window_size, Wp // window_size, window_size, window_size, -1)
    x = x.transpose(2, 3).reshape(B, Hp, Wp, -1)
    if Hp > H or Wp > W:
        x = x[:, :H, :W, :].contiguous()
    return x


def get_rel_pos(q_size: int, k_size: int, rel_pos: torch.Tensor) -> torch.Tensor:
    """(q_size, k_size, C) relative-position embeddings gathered from an (L, C)
    table, resizing the table linearly when L != 2*max(q_size, k_size) - 1."""
    span = int(2 * max(q_size, k_size) - 1)
    table = rel_pos
    if table.shape[0] != span:
        table = F.interpolate(table.t()[None], size=span, mode="linear")[0].t()
    q_pos = torch.arange(q_size, device=rel_pos.device)[:, None] * max(k_size / q_size, 1.0)
    k_pos = torch.arange(k_size, device=rel_pos.device)[None, :] * max(q_size / k_size, 1.0)
    rel = (q_pos - k_pos) + (k_size - 1) * max(q_size / k_size, 1.0)
    return table[rel.long()]


def add_decomposed_rel_pos(
    q: torch.Tensor,
    rel_pos_h: torch.Tensor,
    rel_pos_w: torch.Tensor,
    q_size: Tuple[int, int],
    k_size: Tuple[int, int],
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Bias factors for q (Bh, q_h*q_w, C): rel_h (Bh, q_h*q_w, k_h, 1) and
    rel_w (Bh, q_h*q_w, 1, k_w)."""
    q_h, q_w = q_size
    k_h, k_w = k_size
    Rh = get_rel_pos(q_h, k_h, rel_pos_h)
    Rw = get_rel_pos(q_w, k_w, rel_pos_w)
    Bh, _, dim = q.shape
    grid = q.reshape(Bh, q_h, q_w, dim)
    rel_h = torch.einsum("byxc,ykc->byxk", grid, Rh)
    rel_w = torch.einsum("byxc,xkc->byxk", grid, Rw)
    return (rel_h.reshape(Bh, q_h * q_w, k_h, 1), rel_w.reshape(Bh, q_h * q_w, 1, k_w))


class PatchEmbed(nn.Module):
    """Image to patch embedding: strided convolution, output (B, H, W, C)."""

    def __init__(
        self,
        kernel_size: Tuple[int, int] = (16, 16),
        stride: Tuple[int, int] = (16, 16),
        padding: Tuple[int, int] = (0, 0),
        in_chans: int = 3,
        embed_dim: int = 768,
    ) -> None:
        super().__init__()
        self.proj = nn.Conv2d(in_chans, embed_dim, kernel_size=kernel_size, stride=stride,
                              padding=padding)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        p = self.proj
        kh, kw = p.kernel_size
        if (x.is_cuda and p.stride == p.kernel_size and p.padding == (0, 0) and p.dilation == (1, 1)
                and p.groups == 1 and x.shape[2] % kh == 0 and x.shape[3] % kw == 0):
            # non-overlapping patches: the convolution is one GEMM over (channel, dy, dx) whose
            # output is already (B, H, W, C)
            B, C, H, W = x.shape
            gh, gw = H // kh, W // kw
            cols = ops.patch_rows(x) if FUSED_BLOCK and kh == kw == 16 else None
            if cols is None:
                cols = x.reshape(B, C, gh, kh, gw, kw).permute(0, 2, 4, 1, 3, 5).reshape(B * gh * gw, C * kh * kw)
            y = F.linear(cols, p.weight.reshape(p.out_channels, C * kh * kw), p.bias)
            return y.view(B, gh, gw, p.out_channels)
        return self.proj(x).permute(0, 2, 3, 1)
