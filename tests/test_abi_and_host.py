"""CPU-side checks of the boundary: the C-ABI library loads and exports every symbol
include/samfast.h declares (no compute calls without a GPU); the Python mirror keeps the
reference's names and signatures; the product refuses to run without its kernels."""

import ctypes
import inspect
import re
import threading
import time
from pathlib import Path
from types import SimpleNamespace

import pytest
import torch
import torch.nn as nn

ROOT = Path(__file__).resolve().parents[1]


def _header_functions(header="samfast.h"):
    text = (ROOT / "include" / header).read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(samfast_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    """include/samfast.h is the path's boundary; include/samfast_bench.h holds the measurement
    aids.  The library exports exactly what the two declare and the Python binding mirrors both."""
    from samfast_amd import _lib
    names = _header_functions()
    assert len(names) >= 8
    assert not [n for n in names if n.startswith("samfast_bench_")]
    bench = _header_functions("samfast_bench.h")
    assert bench and all(n.startswith("samfast_bench_") for n in bench)
    lib = ctypes.CDLL(str(_lib.lib_path()))
    for n in names + bench:
        assert hasattr(lib, n), n
    assert sorted(_lib.EXPORTED_SYMBOLS) == names
    assert sorted(_lib.BENCH_SYMBOLS) == bench
    loaded = _lib.load()
    assert loaded.samfast_version() == 1
    assert loaded.samfast_arch() == b"gfx950"


def test_knobs_are_named_and_bounded_without_gpu():
    """The variant knobs take the documented names only; the bare matrix-instruction loops refuse
    launches that would hold the GPU for more than about a second (checked before any launch)."""
    from samfast_amd import _lib
    lib = _lib.load()
    assert lib.samfast_bench_set_knob(b"SAMFAST_GEMM_PERSIST", 1, 0) == 0
    assert lib.samfast_bench_set_knob(b"SAMFAST_GEMM_PERSIST", 0, 1) == 0
    assert lib.samfast_bench_set_knob(b"SAMFAST_NO_SUCH_KNOB", 1, 0) == -1
    assert b"unknown knob" in lib.samfast_last_error()
    # every knob the bench header and the internal enumeration name is known to the library, and they
    # name the same set
    import re
    root = Path(__file__).resolve().parents[1]
    documented = set(re.findall(r"SAMFAST_(?:GEMM|ATTN|SPARSE)_[A-Z0-9_]+", (root / "include" / "samfast_bench.h").read_text()))
    internal = set(re.findall(r"// (SAMFAST_[A-Z0-9_]+):", (root / "segment-anything-fast_amd" / "csrc" / "samfast_internal.hpp").read_text()))
    assert documented == internal and len(documented) >= 11, documented ^ internal
    for name in sorted(documented):
        assert lib.samfast_bench_set_knob(name.encode(), 0, 1) == 0, name
    buf = ctypes.create_string_buffer(65536)
    p = ctypes.addressof(buf)
    p += (-p) % 16
    assert lib.samfast_bench_mfma_ceiling(0, p, 1 << 20, 1 << 24, None, p, None) == -1
    assert b"2^27" in lib.samfast_last_error()
    assert lib.samfast_bench_mfma_valu_overlap(0, p, 1 << 12, 1 << 20, 0, p, None) == -1
    assert b"2^27" in lib.samfast_last_error()


def test_the_half_product_knob_names_built_tiles_only():
    """A tile that is not built is left to the framework's product, whatever number the knob holds."""
    from samfast_amd import _lib
    lib = _lib.load()
    built = {_lib.EPILOGUE_NONE: {3, 4, 5, 8, 10}, _lib.EPILOGUE_GELU: {3, 4, 5, 8, 10}, _lib.EPILOGUE_RESIDUAL: {3, 4, 5, 8, 58}}
    for value in (-1, 0, *range(3, 80)):
        with _lib.knobs(SAMFAST_GEMM_HALF=value):
            for epilogue, tiles in built.items():
                assert lib.samfast_linear_half_pays(4096, 4096, 1280, epilogue) == (value in tiles), (value, epilogue)


def test_the_half_products_lines():
    """Both sides of each line between the library's kernels and the framework's: (M, N, K, epilogue, paid)."""
    from samfast_amd import _lib
    lib = _lib.load()
    none, gelu, residual = _lib.EPILOGUE_NONE, _lib.EPILOGUE_GELU, _lib.EPILOGUE_RESIDUAL
    for *call, paid in ((4096, 2304, 768, none, 0), (4096, 3072, 768, none, 1), (57344, 2304, 768, none, 1), (65536, 2304, 768, none, 0),
                        (65536, 3072, 1024, none, 1), (4096, 2304, 768, gelu, 1), (2048, 2304, 768, gelu, 0),
                        (8192, 1024, 1024, residual, 0), (12288, 768, 768, residual, 1), (65536, 1280, 1280, residual, 0),
                        (57344, 1280, 1280, residual, 1), (8192, 1280, 5120, residual, 0), (12288, 1280, 5120, residual, 1)):
        assert lib.samfast_linear_half_pays(*call) == paid, call


def test_fused_quant_gemm_refuses_outputs_its_quantiser_cannot_address():
    """lin1-shaped call with M * N >= 2^31: the in-kernel quantiser's 32-bit offsets would wrap, so
    the entry point (and its allocation-free form) refuses before anything is launched."""
    from samfast_amd import _lib
    lib = _lib.load()
    M, N, K = 900000, 5120, 1280  # M * K < 2^31 <= M * N
    args = [None, None, None, None, None, None, N, M, N, K, 0, 1, None, 0, 1, None, None, 0.0, None, None, 1]
    assert lib.samfast_gemm_i8_fused_quant(*args, None, None) == -1
    assert b"2^31" in lib.samfast_last_error()
    assert lib.samfast_gemm_i8_fused_quant_noalloc(*args, None) == -1
    assert b"2^31" in lib.samfast_last_error()


def test_empty_calls_are_no_ops_without_gpu():
    """No rows / no images: every entry point validates the shape, launches nothing and returns 0,
    also with null row buffers (what an empty tensor hands over); a negative count is an error."""
    from samfast_amd import _lib
    lib = _lib.load()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    p += (-p) % 16
    assert lib.samfast_quant_rowwise_i8(None, 256, None, None, 0, 256, 0, 0, None) == 0
    assert lib.samfast_quant_rowwise_i8(None, 256, None, None, 0, 256, 0, 1, None) == 0
    assert lib.samfast_layernorm_quant_i8(None, 256, p, p, 1e-6, None, None, None, 0, 256, 0, 0, None) == 0
    assert lib.samfast_gemm_i8_i32(None, p, None, 0, 64, 256, None) == 0
    assert lib.samfast_gemm_i8_scale_bias(None, None, p, p, None, None, 64, 0, 64, 256, 0, None) == 0
    assert lib.samfast_gemm_i8_fused(None, None, p, p, p, None, 64, 0, 64, 256, 0, 2, None, 64, None, 1, None) == 0
    assert lib.samfast_gemm_i8_sparse24_i32(None, p, p, None, 0, 64, 256, None) == 0
    assert lib.samfast_gemm_i8_sparse24_fused(None, None, p, p, p, None, None, 64, 0, 64, 256, 0, 1, None, 0, 0, None) == 0
    strides = [64] * 12
    assert lib.samfast_attn_relpos_fwd(None, None, None, None, None, None, 0, 12, 64, 64, 64,
                                       *strides, 0, 0.125, None) == 0
    assert lib.samfast_attn_relpos_bias_fwd(None, None, None, None, None, None, 0, 12, 14, 14, 80,
                                            *([80] * 12), *([16] * 6), 0, 0.1, None) == 0
    # the shape is still checked
    assert lib.samfast_quant_rowwise_i8(None, 256, None, None, -1, 256, 0, 0, None) == -1
    assert lib.samfast_gemm_i8_i32(None, p, None, 0, 64, 100, None) == -1
    assert lib.samfast_attn_relpos_fwd(None, None, None, None, None, None, 0, 12, 64, 64, 48,
                                       *strides, 0, 0.125, None) == -2
    assert lib.samfast_attn_relpos_fwd(None, None, None, None, None, None, -1, 12, 64, 64, 64,
                                       *strides, 0, 0.125, None) == -1


def test_lists_of_buffers_read_soon():
    """The C entry takes up to eight buffers and refuses others before any launch; an encoder asks for what a window kernel can bring
    in time, and for nothing where the cache holds its weights, for many tokens and outside an encoder."""
    from samfast_amd import _lib
    from samfast_amd.modeling.image_encoder import read_soon
    lib = _lib.load()

    def call(pointers, sizes, n):
        ptrs = None if pointers is None else (ctypes.c_void_p * len(pointers))(*pointers)
        return lib.samfast_attn_relpos_windowed_soon_fwd(
            *([None] * 8), 0, 12, 64, 64, 14, 80, *([64] * 12), 0, 0.125, ptrs, None if sizes is None else (ctypes.c_int64 * len(sizes))(*sizes), n, None)

    buf = ctypes.create_string_buffer(64)
    p = ctypes.addressof(buf)
    assert call([p] * 8, [64] * 8, 8) == call([None], [0], 1) == -1 and b"padding rows" in lib.samfast_last_error()  # (further on)
    for bad in (([p] * 9, [1] * 9, 9), ([p], [-1], 1), ([None], [4], 1), (None, [4], 1), ([p], None, 1), ([p], [4], -1)):
        assert call(*bad) == -1 and b"read soon" in lib.samfast_last_error(), bad
    weights = lambda C, size: [torch.empty((n, C * size), dtype=torch.int8, device="meta") for n in (C, 4 * C, 3 * C)]
    asked = lambda depth, tokens, C, size: len(read_soon(depth, tokens, weights(C, size)))
    assert asked(24, 4096, 1024, 1) == 3 and asked(32, 4096, 1280, 1) == 2 and asked(32, 4096, 1280, 2) == 1
    assert asked(12, 4096, 768, 1) == asked(24, 8193, 1024, 1) == asked(0, 4096, 1024, 1) == 0 and asked(24, 8192, 1024, 1) == 3
    assert len(read_soon(24, 4096, [])) == 0


def test_two_images_weights_are_read_ahead_where_they_repay_it():
    """A block's 2 MB do not, 3.3 MB do; one image's do either way: (depth, tokens, width, bytes a value, buffers named)."""
    from samfast_amd.modeling.image_encoder import read_soon
    for depth, tokens, C, size, want in ((24, 4096, 1024, 2, 1), (24, 4097, 1024, 2, 0), (24, 8192, 1024, 2, 0), (32, 8192, 1280, 2, 1), (12, 8192, 768, 2, 3), (24, 8192, 1024, 1, 3),
                                         (32, 8192, 1280, 1, 2)):
        assert len(read_soon(depth, tokens, [torch.empty((n, C * size), dtype=torch.int8, device="meta") for n in (C, 4 * C, 3 * C)])) == want, (depth, tokens, C, size)


@pytest.mark.parametrize("kind", ["int8", "half"])
def test_weights_are_looked_up_to_be_read_ahead_in_recordings_of_few_tokens(monkeypatch, kind):
    """Nothing is asked of a Linear, and no list is made, where the host issues the launches or the tokens are many: a block is told it is one of none."""
    from samfast_amd import ops
    from samfast_amd.modeling import ImageEncoderViT, image_encoder
    enc = ImageEncoderViT(img_size=64, embed_dim=64, depth=3, num_heads=1, use_rel_pos=True, window_size=2).to(torch.bfloat16)
    told, lists = [], []
    monkeypatch.setattr(image_encoder.Block, "_int8_fused_ok", lambda self, x: kind == "int8")
    monkeypatch.setattr(image_encoder.Block, "_half_fused_ok", lambda self, x: True)
    name = f"_forward_{kind}_fused"
    monkeypatch.setattr(image_encoder.Block, name, lambda self, x, carry=None, norm=None, qkv=None, depth=0: (told.append(depth), (x, None))[1])
    x = torch.zeros((2, 4, 4, 64), dtype=torch.bfloat16)
    for recorded, most, want in ((False, 32, 0), (True, 32, 3), (True, 31, 0)):
        monkeypatch.setattr(image_encoder, "_recording", lambda x: recorded, raising=False)
        monkeypatch.setattr(image_encoder, "SOON_TOKENS", most)
        enc.forward_blocks(x)
        assert told == [want] * 3, (recorded, most)
        told.clear()
    monkeypatch.undo()
    # a block of none, as far as its attention
    class Reached(Exception):
        pass

    def attention(*args):
        raise Reached(args[-1])

    monkeypatch.setattr(image_encoder, "read_soon", lambda *args: lists.append(args) or ())
    monkeypatch.setattr(ops, "layernorm", lambda x, *args, **kwargs: x)
    monkeypatch.setattr(ops, "layernorm_quant", lambda x, *args, **kwargs: (x, None))
    monkeypatch.setattr(ops, "linear_half", lambda x, linear, *args, **kwargs: linear(x))
    monkeypatch.setattr(ops, "attn_relpos_windowed", attention)
    block = enc.blocks[0]
    if kind == "int8":
        block.attn.qkv.linear_fused = lambda x, *args, **kwargs: block.attn.qkv(x)
        block._pad_rows = lambda *args: (None, None)
        block.attn.proj.weight_operands = block.mlp.lin2.weight_operands = lambda layout: lists.append(layout) or ()
    for depth in (0, 3):
        with torch.no_grad(), pytest.raises(Reached) as reached:
            getattr(block, name)(x, depth=depth)
        assert reached.value.args == ((),) and bool(lists) == (depth > 0)


def test_a_weight_that_is_read_ahead_is_the_one_that_the_product_reads():
    """A K-block-major copy is named while it is current, and not once its weight was written to, moved or replaced: the next product
    makes another, and the memory of the old one is given back, whoever still holds its address."""
    from samfast_amd import _lib, quant
    from samfast_amd.sparse import Int8Sparse24Linear
    linear = quant.Int8DynamicLinear.from_float(torch.nn.Linear(128, 64))
    copy = lambda: quant.kept_copy(linear, "_kb64", linear.wq, lambda: linear.wq.clone())
    kb, row = _lib.LAYOUT_KB64, _lib.LAYOUT_ROWMAJOR
    named = lambda: linear.weight_operands(kb)
    assert named() == () and linear.weight_operands(row)[0] is linear.wq
    first = copy()
    assert copy() is first and len(named()) == 1 and named()[0] is first
    linear.wq.copy_(linear.wq.flip(0))  # (in place, as load_state_dict does)
    assert named() == () and linear.weight_operands(row)[0] is linear.wq
    second = copy()
    assert second is not first and named()[0] is second
    linear.wq = linear.wq.clone()
    assert named() == ()
    third = copy()
    assert named()[0] is third
    linear.wq.data = linear.wq.data.clone()  # (elsewhere: the module's .to())
    assert named() == ()
    with torch.inference_mode():
        linear.wq = linear.wq.clone()
    copy()
    assert named() == ()  # (writes to it leave no trace: none is kept)
    packed = Int8Sparse24Linear(128, 64, torch.zeros((2, 64, 32), dtype=torch.int8), torch.zeros((2, 64, 2), dtype=torch.int32), torch.ones(64), None)
    assert [t is b for t, b in zip(packed.weight_operands(kb), (packed.wc, packed.widx))] == [True, True]


def test_empty_calls_of_block_neck_and_image_are_no_ops_without_gpu():
    """The same for the half-type Linear, the int8 block's middle, the neck's convolutions and the image's preparation."""
    from samfast_amd import _lib
    lib = _lib.load()
    for epilogue in (0, 1, 2):
        assert lib.samfast_linear_half(None, 768, None, None, None, 3072, 0, 3072, 768, 0, epilogue, None, 3072, None) == 0
        assert lib.samfast_linear_half(None, 768, None, None, None, 3072, -1, 3072, 768, 0, epilogue, None, 3072, None) == -1
    proj = lambda M: lib.samfast_proj_block_i8(None, 768, None, None, None, None, None, None, None, 1e-6, None, None, M, 768, 0, None)
    assert proj(0) == 0 and proj(-1) == -1
    for taps in (1, 9):
        conv = lambda B, channels=768: lib.samfast_neck_conv(None, None, None, B, 64, 64, channels, 256, taps, 0, None, None, 0, 0, None)
        assert conv(0) == 0 and conv(-1) == -1 and conv(0, 100) == -1
    image = lambda B, size=1024: lib.samfast_preprocess(None, 1, None, None, None, B, 700, 1024, size, 0, None)
    assert image(0) == 0 and image(-1) == -1 and image(0, 1001) == -1


def test_patch_rows_refused_or_empty_without_gpu():
    from samfast_amd import _lib
    patches = lambda B, H=1024, W=1024, C=3: _lib.load().samfast_patch_rows(None, None, B, C, H, W, None)
    assert patches(0) == 0 and patches(-1) == patches(0, 1000) == patches(0, 1024, 8) == patches(0, 1024, 0) == patches(0, C=0) == patches(1) == -1


@pytest.mark.parametrize("C,H,W,images", [(3, 1024, 1024, 21845), (1, 16, 16, (1 << 26) - 4), (3, 65536, 16, 5461), (2, 16, 80, 1 << 24)])
def test_patches_beyond_one_launch_are_left_to_the_permutation(monkeypatch, C, H, W, images):
    """The C entry refuses what a launch of under 2^32 threads does not cover, before it looks at a pointer, and the operator declines it."""
    from samfast_amd import _lib, ops
    most = _lib.PATCH_ROWS_MAX // (C * (H // 16) * ((W + 63) // 64))
    assert abs(images - most) <= 1
    for B, large in ((most, False), (most + 1, True)):
        assert _lib.load().samfast_patch_rows(None, None, B, C, H, W, None) == -1
        assert (b"too large" in _lib.load().samfast_last_error()) == large
    monkeypatch.setattr(ops, "unwatched", lambda x: True)
    monkeypatch.setattr(ops, "rows_launchable", lambda *tensors: True)
    monkeypatch.setattr(torch, "empty", lambda *args, **kwargs: pytest.fail("not declined"))
    x = SimpleNamespace(is_cuda=True, dim=lambda: 4, dtype=torch.bfloat16, numel=lambda: 1, shape=(most + 1, C, H, W), device=None)
    with torch.no_grad():
        assert ops.patch_rows(x) is None
        x.shape = (most, C, H, W)
        with pytest.raises(pytest.fail.Exception, match="not declined"):
            ops.patch_rows(x)


def test_argument_validation_without_gpu():
    """Validation runs on the host before any launch, so error codes are testable here."""
    from samfast_amd import _lib
    lib = _lib.load()
    rc = lib.samfast_gemm_i8_i32(None, None, None, 16, 16, 64, None)
    assert rc == -1 and b"null pointer" in lib.samfast_last_error()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    p += (-p) % 16
    rc = lib.samfast_gemm_i8_i32(p, p, p, 16, 16, 100, None)
    assert rc == -1 and b"multiple of 64" in lib.samfast_last_error()
    rc = lib.samfast_quant_rowwise_i8(p, 12, p, p, 4, 12, 0, 0, None)
    assert rc == -1 and b"multiple of 8" in lib.samfast_last_error()
    rc = lib.samfast_quant_rowwise_i8(p, 96, p, p, 4, 96, 0, 1, None)  # K-block major needs K % 64 == 0
    assert rc == -1 and b"K-block major" in lib.samfast_last_error()
    rc = lib.samfast_gemm_i8_fused(p, p, p, p, None, p, 64, 4, 64, 256, 0, 0, None, 0, None, 7, None)
    assert rc == -1 and b"layout" in lib.samfast_last_error()
    strides = [0] * 12
    rc = lib.samfast_attn_relpos_fwd(p, p, p, p, p, p, 1, 1, 10, 10, 48, *strides, 0, 0.125, None)
    assert rc == -2 and b"head_dim" in lib.samfast_last_error()
    rc = lib.samfast_attn_relpos_fwd(p, p, p, p, p, p, 1, 1, 20, 20, 64, *([64] * 12), 0, 0.125, None)
    assert rc == -2 and b"neither" in lib.samfast_last_error()
    rc = lib.samfast_attn_relpos_fwd(p, p, p, p, p, p, 1, 1, 14, 14, 64, *([64] * 12), 2, 0.125, None)
    assert rc == -2 and b"element type" in lib.samfast_last_error()  # neither SAMFAST_BF16 nor SAMFAST_F16
    rc = lib.samfast_quant_rowwise_i8(p, 64, p, p, 4, 64, 1, 0, None)
    assert rc == -2  # the linears are bf16 only


def test_ops_refuse_cpu_tensors():
    from samfast_amd import ops
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.quant_rowwise(x)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.gemm_i8_i32(torch.zeros(4, 64, dtype=torch.int8), torch.zeros(8, 64, dtype=torch.int8))


def test_registry_surface():
    import samfast_amd
    for reg in (samfast_amd.sam_model_registry, samfast_amd.sam_model_fast_registry):
        assert set(reg) == {"default", "vit_h", "vit_l", "vit_b"}
    sig = inspect.signature(samfast_amd.build_sam_fast_vit_h)
    assert list(sig.parameters) == ["checkpoint", "compile_mode", "dtype"]
    assert sig.parameters["compile_mode"].default == "max-autotune"
    assert sig.parameters["dtype"].default == torch.bfloat16
    sam = samfast_amd.sam_model_fast_registry["vit_b"]()
    assert next(sam.image_encoder.parameters()).dtype == torch.bfloat16 and not sam.image_encoder.training
    pred = samfast_amd.SamPredictor(sam)
    assert pred.is_image_set is False
    img = torch.zeros(1, 3, 512, 1024)
    assert sam.preprocess(img).shape == (1, 3, 1024, 1024)


def test_fast_registry_wraps_the_encoder_for_graph_replay():
    """compile_mode of the fast builders (build_sam.py:67-71 of the reference compiles the encoder
    with it): any mode wraps the encoder for HIP-graph replay, None leaves it bare.  The wrapper
    forwards attributes, keeps the reference's post-compile state-dict prefix and drops its
    recordings whenever weights or modules are replaced."""
    import samfast_amd
    from samfast_amd import tools
    from samfast_amd.graphs import ReplayedEncoder
    from samfast_amd.modeling import ImageEncoderViT
    sam = samfast_amd.sam_model_fast_registry["vit_b"]()
    enc = sam.image_encoder
    assert isinstance(enc, ReplayedEncoder) and enc.compile_mode == "max-autotune"
    assert enc.img_size == 1024 and len(enc.blocks) == 12 and isinstance(enc._orig_mod, ImageEncoderViT)
    assert all(k.startswith("_orig_mod.") for k in enc.state_dict())
    bare = samfast_amd.sam_model_fast_registry["vit_b"](compile_mode=None).image_encoder
    assert isinstance(bare, ImageEncoderViT)
    assert not enc.replays(torch.zeros(1, 3, 1024, 1024))  # CPU tensors run eagerly
    for mutate in (lambda: tools.replace_with_custom_fn_if_matches_filter(enc, lambda m: m, lambda m, f: False),
                   lambda: enc.load_state_dict(enc.state_dict()),
                   lambda: samfast_amd.apply_fake_sparsity(sam, lambda m, f: False),
                   lambda: enc.float()):
        enc._graphs["stale"] = object()
        mutate()
        assert not enc._graphs


def test_module_signatures_follow_reference():
    from samfast_amd.modeling import Attention, Block, ImageEncoderViT, MLPBlock
    assert list(inspect.signature(Attention.__init__).parameters)[1:] == [
        "dim", "num_heads", "qkv_bias", "use_rel_pos", "rel_pos_zero_init", "input_size"]
    assert list(inspect.signature(MLPBlock.__init__).parameters)[1:] == ["embedding_dim", "mlp_dim", "act"]
    assert list(inspect.signature(Block.__init__).parameters)[1:] == [
        "dim", "num_heads", "mlp_ratio", "qkv_bias", "norm_layer", "act_layer", "use_rel_pos",
        "rel_pos_zero_init", "window_size", "input_size"]
    att = Attention(64, 2, use_rel_pos=True, input_size=(14, 14))
    assert {n for n, _ in att.named_parameters()} == {
        "qkv.weight", "qkv.bias", "proj.weight", "proj.bias", "rel_pos_h", "rel_pos_w"}
    assert att.rel_pos_h.shape == (27, 32)
    enc_sig = inspect.signature(ImageEncoderViT.__init__)
    assert enc_sig.parameters["window_size"].default == 0 and enc_sig.parameters["embed_dim"].default == 768


def test_swap_helpers():
    from samfast_amd import Int8DynamicLinear, apply_dynamic_quant
    from samfast_amd.tools import replace_with_custom_fn_if_matches_filter
    from samfast_amd.modeling import Block
    blk = Block(64, 2, use_rel_pos=True, window_size=3, input_size=(8, 8))
    seen = []
    replace_with_custom_fn_if_matches_filter(
        blk, lambda m: m, lambda m, fqn: (seen.append(fqn) or False))
    assert {"norm1", "attn", "attn.qkv", "attn.proj", "norm2", "mlp", "mlp.lin1", "mlp.lin2", "mlp.act"} <= set(seen)
    w = blk.mlp.lin1.weight.detach().clone()
    apply_dynamic_quant(blk, lambda m, fqn: fqn.startswith("mlp."))
    assert isinstance(blk.mlp.lin1, Int8DynamicLinear) and isinstance(blk.mlp.lin2, Int8DynamicLinear)
    assert isinstance(blk.attn.qkv, nn.Linear)
    assert blk.mlp.lin1.wq.dtype == torch.int8 and blk.mlp.lin1.sw.dtype == torch.float32
    assert (blk.mlp.lin1.weight - w).abs().max() <= blk.mlp.lin1.sw.max() * 0.5001
    blk = blk.to(torch.bfloat16)  # scales and integer weights survive a dtype cast untouched
    assert blk.mlp.lin1.sw.dtype == torch.float32 and blk.mlp.lin1.wq.dtype == torch.int8
    with pytest.raises(RuntimeError, match="GPU"):
        blk.mlp(torch.zeros(1, 8, 8, 64, dtype=torch.bfloat16))  # no CPU route for the int8 path


def test_composite_cpu_route_is_the_reference_fallback():
    """fp32 / CPU inputs take the eager SDPA route exactly as flash_4.py:368-370."""
    from samfast_amd.flash_4 import _attention_rel_h_rel_w
    from oracle import relpos_attention as ora
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(1, 2, 196, 64, generator=g) for _ in range(3))
    rel_h, rel_w = torch.randn(1, 2, 196, 14, 1, generator=g), torch.randn(1, 2, 196, 1, 14, generator=g)
    got = _attention_rel_h_rel_w(q, k, v, rel_h, rel_w)
    assert torch.allclose(got, ora.attention_rel_h_rel_w(q, k, v, rel_h, rel_w), atol=1e-5)
    assert hasattr(torch.ops.customflash, "custom_flash_aligned")


def test_checkpoint_with_reference_key_names_loads(tmp_path):
    """A checkpoint in the layout the released SAM files have (key names follow the module
    tree of the reference, modeling/image_encoder.py:15-120 and modeling/sam.py:18-58; prompt
    encoder and mask decoder entries present) loads through the registry, and the quantised
    modules are then built from the loaded weights."""
    import samfast_amd
    from samfast_amd import Int8DynamicLinear, apply_dynamic_quant
    donor = samfast_amd.sam_model_registry["vit_b"]()
    g = torch.Generator().manual_seed(11)
    sd = {}
    for k, v in donor.state_dict().items():
        sd[k] = (torch.randn(v.shape, generator=g) * 0.02).to(torch.float16) if v.is_floating_point() else v
    # what the module tree of the reference's encoder gives, written out by rule
    expect = {"image_encoder.pos_embed", "image_encoder.patch_embed.proj.weight", "image_encoder.patch_embed.proj.bias",
              "image_encoder.neck.0.weight", "image_encoder.neck.1.weight", "image_encoder.neck.1.bias",
              "image_encoder.neck.2.weight", "image_encoder.neck.3.weight", "image_encoder.neck.3.bias"}
    for i in range(12):
        for leaf in ("norm1.weight", "norm1.bias", "attn.rel_pos_h", "attn.rel_pos_w", "attn.qkv.weight",
                     "attn.qkv.bias", "attn.proj.weight", "attn.proj.bias", "norm2.weight", "norm2.bias",
                     "mlp.lin1.weight", "mlp.lin1.bias", "mlp.lin2.weight", "mlp.lin2.bias"):
            expect.add(f"image_encoder.blocks.{i}.{leaf}")
    assert {k for k in sd if k.startswith("image_encoder.")} == expect
    # entries of the parts that are not built here
    sd["prompt_encoder.pe_layer.positional_encoding_gaussian_matrix"] = torch.zeros(2, 128)
    sd["mask_decoder.iou_token.weight"] = torch.zeros(1, 256)
    path = tmp_path / "sam_vit_b.pth"
    torch.save(sd, path)
    sam = samfast_amd.sam_model_registry["vit_b"](checkpoint=str(path))
    w = sam.image_encoder.blocks[3].mlp.lin1.weight
    assert torch.equal(w, sd["image_encoder.blocks.3.mlp.lin1.weight"].float())
    assert sam.image_encoder.blocks[0].attn.rel_pos_h.shape == (27, 64)     # windowed block: 2*14-1
    assert sam.image_encoder.blocks[2].attn.rel_pos_h.shape == (127, 64)    # global block: 2*64-1
    apply_dynamic_quant(sam.image_encoder.blocks[3])
    q = sam.image_encoder.blocks[3].mlp.lin1
    assert isinstance(q, Int8DynamicLinear)
    assert (q.weight - w).abs().max() <= q.sw.max() * 0.5001


def test_attention_wrappers_reject_mismatched_shapes_before_any_launch():
    """The library is only told the grid; it would walk gh*gw tokens of every (batch, head) slice
    whatever the tensors hold.  The wrappers therefore pin every shape on the host - these raise
    on CPU tensors, i.e. before the device check and before anything could be launched."""
    from samfast_amd import flash_4, ops
    bf = torch.bfloat16
    q = torch.zeros(1, 2, 2048, 64, dtype=bf)
    tabs = torch.zeros(127, 64, dtype=bf)
    with pytest.raises(RuntimeError, match="must be"):            # 2048 tokens on a 64x64 grid
        ops.attn_relpos(q, q, q, tabs, tabs, (64, 64))
    q4 = torch.zeros(1, 2, 4096, 64, dtype=bf)
    with pytest.raises(RuntimeError, match="shape of q"):
        ops.attn_relpos(q4, q4[:, :, :2048], q4, tabs, tabs, (64, 64))
    with pytest.raises(RuntimeError, match="dtype of q"):
        ops.attn_relpos(q4, q4.float(), q4, tabs, tabs, (64, 64))
    with pytest.raises(RuntimeError, match="out must"):
        ops.attn_relpos(q4, q4, q4, tabs, tabs, (64, 64), out=torch.zeros(1, 2, 2048, 64, dtype=bf))
    rel_h = torch.zeros(1, 2, 2048, 64, dtype=bf)
    with pytest.raises(RuntimeError, match="must be"):            # bias says 64x64 keys, q has 2048 tokens
        ops.attn_relpos_bias(q, q, q, rel_h, rel_h)
    with pytest.raises(RuntimeError, match="bias factors"):       # bias rows do not match q's tokens
        ops.attn_relpos_bias(q4, q4, q4, rel_h, torch.zeros(1, 2, 4096, 64, dtype=bf))
    with pytest.raises(RuntimeError, match="must be"):
        ops.attn_relpos_windowed(q, q, q, torch.zeros(27, 64, dtype=bf), torch.zeros(27, 64, dtype=bf),
                                 torch.zeros(2, 64, dtype=bf), torch.zeros(2, 64, dtype=bf), (64, 64), 14, 0.125)
    # the registered operator derives the key grid from the token count: 64-wide rows only
    with pytest.raises(RuntimeError, match="64-wide key grid"):
        flash_4._custom_flash_aligned_gpu(q[:, :, :2000], q[:, :, :2000], q[:, :, :2000],
                                          torch.zeros(1, 2, 2000, 128, dtype=bf), 0.125)
    # a consistent call gets as far as the device check
    with pytest.raises(RuntimeError, match="GPU"):
        ops.attn_relpos(q4, q4, q4, tabs, tabs, (64, 64))


def test_weight_quantiser_conventions_closed_form():
    """The default per-channel convention (absmax / 127, clamp +-127) and torchao's
    (absmax / 127.5 clamped at float32 eps, clamp -128..127, arithmetic in the weight's dtype),
    on values whose quotients are exact."""
    from samfast_amd.quant import quantize_weight_per_channel
    w = torch.tensor([[127.0, -63.5, 1.0, 0.0], [-255.0, 255.0, 2.0, -1.0], [0.0, 0.0, 0.0, 0.0]])
    q, s = quantize_weight_per_channel(w)
    assert torch.equal(s, torch.tensor([1.0, 255.0 / 127.0, 1e-5 / 127.0]))
    assert q.tolist() == [[127, -64, 1, 0], [-127, 127, 1, 0], [0, 0, 0, 0]]   # -63.5 -> -64: half to even
    q, s = quantize_weight_per_channel(w, "torchao")
    eps = torch.finfo(torch.float32).eps
    assert torch.equal(s, torch.tensor([127.0 / 127.5, 2.0, eps]))
    # row 1: +-255 / 2 = +-127.5 -> +-128 (half to even) -> clamped to 127 on the positive side only
    assert q[1].tolist() == [-128, 127, 1, 0]
    assert q[0].tolist() == [127, -64, 1, 0] and q[2].tolist() == [0, 0, 0, 0]   # 127.5 -> 128 -> 127; -63.75 -> -64
    # bf16 weights: the scale is rounded to bf16 and the division runs in bf16, as torch would
    wb = torch.tensor([[3.0, -1.0, 0.5, 0.25]], dtype=torch.bfloat16)
    q, s = quantize_weight_per_channel(wb, "torchao")
    sb = (torch.tensor(3.0) / 127.5).to(torch.bfloat16)
    assert s.dtype == torch.float32 and torch.equal(s, sb.float()[None])
    assert torch.equal(q, torch.round(wb / sb).clamp(-128, 127).to(torch.int8))
    with pytest.raises(ValueError):
        quantize_weight_per_channel(w, "other")


def test_int8_linear_keeps_one_bias():
    """The fp32 bias lives in one buffer; `bias` is a view of it, and loading a float `bias`
    entry (what an nn.Linear state dict carries) lands in that buffer."""
    from samfast_amd import Int8DynamicLinear
    lin = nn.Linear(64, 16)
    q = Int8DynamicLinear.from_float(lin, "torchao")
    assert {k for k in q.state_dict()} == {"sw_bits", "bias_bits", "wq"}
    assert torch.equal(q.bias, lin.bias.detach()) and q.bias.data_ptr() == q.bias_bits.data_ptr()
    sd = q.state_dict()
    del sd["bias_bits"]
    sd["bias"] = torch.full((16,), 0.25, dtype=torch.bfloat16)
    q.load_state_dict(sd)
    assert torch.equal(q.bias_f32, torch.full((16,), 0.25))
    q = q.to(torch.bfloat16)
    assert q.bias.dtype == torch.float32
    assert Int8DynamicLinear.from_float(nn.Linear(64, 16, bias=False)).bias is None


def test_a_block_counts_as_built_only_without_hooks_and_overrides():
    """Only such a block may leave its modules uncalled (the fused half-type route)."""
    from samfast_amd.modeling import Block
    blk = Block(64, 2, use_rel_pos=True, window_size=3, input_size=(8, 8))
    assert blk._as_built()
    nothing = lambda *args: None
    inside = (blk, blk.norm1, blk.attn, blk.attn.qkv, blk.attn.proj, blk.norm2, blk.mlp, blk.mlp.lin1, blk.mlp.act, blk.mlp.lin2)
    for m in inside:
        for register in (m.register_forward_hook, m.register_forward_pre_hook):
            handle = register(nothing)
            assert not blk._as_built()
            handle.remove()
        m.forward = nothing
        assert not blk._as_built()
        del m.forward
    for register in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook):
        handle = register(nothing)
        assert not blk._as_built()
        handle.remove()
    assert blk._as_built()
    blk.mlp.act = nn.ReLU()
    assert not blk._as_built()

    class Other(Block):
        def forward(self, x):
            return x

    assert not Other(64, 2, use_rel_pos=True, window_size=3, input_size=(8, 8))._as_built()


def test_native_calls_decline_where_somebody_watches():
    """The host module launches on raw pointers; under a tracer, a functional transform, a dispatch or function mode,
    and for tensors that are more than their memory, the call has to go through torch's dispatcher."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from samfast_amd import _lib
    plain = _lib.host().plain
    x = torch.randn(2, 3)
    assert plain(x) and plain(nn.Parameter(x)) and plain(x.t()) and plain(x[:0])
    with torch.no_grad():
        assert plain(x)
    with torch.inference_mode():
        assert plain(x) and plain(torch.zeros(2))
    assert plain(torch.ones(2, requires_grad=True) * 2)
    with torch.device("cpu"):  # a function mode, but one for factory functions
        assert plain(x)
    answers = []

    def watched(t):
        answers.append((plain(t), plain(x)))
        return t * 2

    torch.jit.trace(watched, x, check_trace=False)
    torch.vmap(watched)(x)
    torch.func.grad(lambda t: watched(t).sum())(x)
    torch.func.functionalize(watched)(x)

    class Through(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Pass(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Through, Pass):
        with mode():
            watched(x)
    with torch.device("cpu"), Pass():
        watched(x)
    assert len(answers) == 7 and not any(any(a) for a in answers), answers
    with torch.autograd.forward_ad.dual_level():
        assert not plain(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))

    class Sub(torch.Tensor):
        pass

    assert not plain(x.as_subclass(Sub)) and not plain(torch._neg_view(x)) and not plain(x.to_sparse())
    assert plain(x)


def test_no_inline_assembly_writes_m0_itself():
    """m0 cannot be listed as clobbered; a statement that needs a value in it takes it as an operand there."""
    for src in sorted((ROOT / "segment-anything-fast_amd" / "csrc").glob("*.h*")):
        for statement in re.findall(r"\basm\b[^;]*;", re.sub(r"//[^\n]*", "", src.read_text())):
            assert not re.search(r'[a-z_0-9]+ m0\s*,', statement), (src.name, statement)


def test_copies_derived_from_a_buffer_are_kept_only_while_they_hold():
    from samfast_amd.quant import kept_copy
    holder, made = nn.Module(), []

    def copy_of(t):
        def make():
            made.append(t.clone())
            return made[-1]
        return kept_copy(holder, "_copy", t, make)

    a = torch.arange(4.0)
    assert copy_of(a) is copy_of(a) and len(made) == 1
    a += 1
    assert torch.equal(copy_of(a), a) and len(made) == 2
    b = a.clone()
    assert copy_of(b) is not copy_of(a) and len(made) == 4
    a.data = b.clone() + 1  # the same tensor object, elsewhere
    assert torch.equal(copy_of(a), a) and len(made) == 5
    with torch.inference_mode():
        c = torch.zeros(3)
        copy_of(c)
        c += 1
        assert torch.equal(copy_of(c), c) and len(made) == 7
    assert copy_of(a) is made[4]


def test_proj_block_pays_on_one_range_of_rows():
    from samfast_amd import _lib
    lib = _lib.load()
    for width, first in ((768, 0), (1024, 1665)):
        assert [m for m in range(9000) if lib.samfast_proj_block_pays(m, width)] == list(range(first, 8193))
    assert not any(lib.samfast_proj_block_pays(m, 1280) for m in (1, 4096))


class _Recording:
    """A GraphedEncoder's buffer and replay, without a GPU: the embedding is what the buffer holds."""

    def __init__(self, shape):
        self._in = SimpleNamespace(is_cuda=True, shape=shape, dim=lambda: 4, value=None, dtype=torch.bfloat16, device=torch.device("cuda", 0))

    def follow(self):
        pass

    def __call__(self, x):
        if x is not self._in:
            self._in.value = x.value
        time.sleep(1e-3)
        value = self._in.value
        return SimpleNamespace(clone=lambda: value)


@pytest.fixture
def predictor(monkeypatch):
    """A predictor over an encoder with such a recording of one image; an image of value v gives the embedding v."""
    from samfast_amd import SamPredictor, ops
    from samfast_amd.graphs import ReplayedEncoder
    from samfast_amd.modeling import Sam
    inner = torch.nn.Linear(1, 1, dtype=torch.bfloat16)
    inner.img_size, inner.forward = 64, lambda x: x.value
    encoder, recording = ReplayedEncoder(inner).eval(), _Recording((1, 3, 64, 64))
    encoder._graphs[((1, 3, 64, 64), torch.bfloat16, torch.device("cuda", 0))] = recording

    def preprocess(image, mean, std, size, dtype, out):
        out = _Recording((1, 3, size, size))._in if out is None else out
        out.value = image.value
        written.append(out)
        return out

    written = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops, "preprocess", preprocess)
    predictor = SamPredictor(Sam(encoder))
    predictor.encode = lambda value: predictor._encoded(SimpleNamespace(shape=(1, 3, 40, 64), device=torch.device("cuda", 0), value=value), 64, torch.bfloat16)
    predictor.written, predictor.buffer = written, recording._in
    return predictor


@pytest.mark.parametrize("who", ["nobody", "hook", "pre-hook", "global hook", "global pre-hook", "own forward", "subclass", "capture", "eager"])
def test_a_recording_s_input_buffer_is_written_only_where_nobody_is_handed_it(who, predictor, monkeypatch):
    """A predictor writes the image straight into the buffer that a recorded encoder reads; whoever else would see that
    tensor, overwritten by the next image, makes it a tensor of its own."""
    from torch.nn.modules import module
    encoder = predictor.model.image_encoder
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: who == "capture")
    handle = {"hook": encoder.register_forward_hook, "pre-hook": encoder.register_forward_pre_hook,
              "global hook": module.register_module_forward_hook,
              "global pre-hook": module.register_module_forward_pre_hook}.get(who, lambda f: None)(lambda *a: None)
    if who == "own forward":
        encoder.forward = lambda x: x.value
    elif who == "subclass":
        encoder.__class__ = type("Mine", (type(encoder),), {})
    elif who == "eager":
        encoder.compile_mode = None
    try:
        with torch.no_grad():
            assert predictor.encode(7) == 7
    finally:
        if handle is not None:
            handle.remove()
    assert [w is predictor.buffer for w in predictor.written] == [who == "nobody"]


def test_threads_that_share_a_recorded_encoder_get_their_own_embeddings(predictor):
    wrong = []

    def work(value):
        with torch.no_grad():
            wrong.extend(i for i in range(20) if predictor.encode((value, i)) != (value, i))

    threads = [threading.Thread(target=work, args=(v,)) for v in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []


class _Recorder:
    """A library whose entry points launch nothing: the names called, in order."""

    def __init__(self):
        self.called = []

    def __getattr__(self, name):
        def call(*args):
            self.called.append(name)
            return 1 if name.endswith("_pays") else 0
        return call

    def launches(self):
        return [n for n in self.called if not n.endswith("_pays")]


@pytest.fixture
def recorder(monkeypatch):
    """ops on CPU tensors, up to the call into the library."""
    from samfast_amd import _lib, ops
    lib = _Recorder()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "check", lambda code, what: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_require_gpu", lambda *tensors: None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    return lib


def test_half_linear_launches_nothing_on_other_shapes(recorder):
    """What the kernel would read past its end never reaches it: a weight or bias of another shape is the framework's
    product's to refuse, a residual or output of another shape, type or stride an error."""
    from samfast_amd import _lib, ops
    half = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    make = lambda w, b: SimpleNamespace(weight=w, bias=b)
    x, linear = half(256, 320), make(half(96, 320), half(96))
    assert ops.linear_half(x, linear).shape == (256, 96) and recorder.launches() == ["samfast_linear_half"]
    recorder.called.clear()
    for other in (make(half(96, 256), half(96)), make(half(96, 384), None), make(half(96, 320), half(95)), make(half(96, 320), half(1)),
                  make(half(320), None)):
        assert ops.linear_half(x, other) is None
    for bad in (half(255, 96), half(256, 104), half(96), half(256, 96).float(), half(96, 256).t()):
        with pytest.raises(RuntimeError):
            ops.linear_half(x, linear, _lib.EPILOGUE_RESIDUAL, residual=bad)
        with pytest.raises(RuntimeError):
            ops.linear_half(x, linear, _lib.EPILOGUE_RESIDUAL, residual=half(256, 96), out=bad)
    assert recorder.launches() == []


def test_proj_block_launches_nothing_on_other_shapes(recorder):
    """Scales, bias or norm parameters of another length or type are left to the checks of the separate launches."""
    from samfast_amd import ops
    C, M = 768, 32
    x, res = (torch.zeros((M, C), dtype=torch.bfloat16) for _ in range(2))
    wq, sw, bias = torch.zeros((C // 64, C, 64), dtype=torch.int8), torch.ones(C), torch.zeros(C)
    norm = torch.ones(C, dtype=torch.bfloat16)
    assert ops.proj_block(x, wq, sw, bias, res, (norm, norm, 1e-6)) is not None and recorder.launches() == ["samfast_proj_block_i8"]
    recorder.called.clear()
    short = norm[:C - 8].clone()
    for args in ((wq, sw, bias, res, (short, norm, 1e-6)), (wq, sw, bias, res, (norm, short, 1e-6)), (wq, sw[:8].clone(), bias, res, (norm, norm, 1e-6)),
                 (wq, sw, bias[:8].clone(), res, (norm, norm, 1e-6)), (wq, sw.bfloat16(), bias, res, (norm, norm, 1e-6)),
                 (wq, sw, bias.bfloat16(), res, (norm, norm, 1e-6)), (wq[1:].clone(), sw, bias, res, (norm, norm, 1e-6))):
        assert ops.proj_block(x, *args) is None
    assert recorder.launches() == []


def test_neck_launches_nothing_on_other_shapes(recorder):
    from samfast_amd import ops
    half = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    x, w1, w3 = half(1, 4, 4, 128), half(64, 128, 1, 1), half(64, 64, 3, 3)
    assert ops.neck_convs(x, w1, lambda y: y, w3).shape == (1, 4, 4, 64) and recorder.launches() == ["samfast_neck_conv"] * 2
    recorder.called.clear()
    for args in ((x, half(64, 64, 1, 1), w3), (x, half(64, 128, 3, 3), w3), (x, w1, half(64, 128, 3, 3)), (x, w1, half(64, 64, 1, 1)),
                 (x, w1.float(), w3), (x.transpose(1, 2), w1, w3), (x, w1, w3.to(memory_format=torch.channels_last))):
        with pytest.raises(RuntimeError):
            ops.neck_convs(args[0], args[1], lambda y: y, args[2])
    assert recorder.launches() == []
    with pytest.raises(RuntimeError):
        ops.neck_convs(x, w1, lambda y: y[:, :2], w3)
    assert recorder.launches() == ["samfast_neck_conv"]


def test_a_recording_follows_the_stream_of_its_last_call(monkeypatch):
    """Another stream waits for the last one's work, and the input buffer is known to the allocator as used there."""
    from samfast_amd.graphs import GraphedEncoder

    class Stream:
        def wait_stream(self, other):
            seen.append(("waits for", self, other))

    seen, streams = [], [Stream(), Stream()]
    recording = GraphedEncoder.__new__(GraphedEncoder)
    nn.Module.__init__(recording)
    recording._in, recording._stream = SimpleNamespace(record_stream=lambda s: seen.append(("used on", s))), streams[0]
    for i in (0, 1, 1, 0):
        monkeypatch.setattr(torch.cuda, "current_stream", lambda: streams[i])
        recording.follow()
    assert seen == [("waits for", streams[1], streams[0]), ("used on", streams[1]),
                    ("waits for", streams[0], streams[1]), ("used on", streams[0])]


def _linear_route(M, N, K, x_at, ldx, y_at, ldy, sparse=False):
    """Which launches a call without a workspace would be: "one", or "two" (refused then).  The type is one that no kernel
    takes, so that nothing is launched: the one launch refuses it, the two ask for their workspace first."""
    from samfast_amd import _lib
    lib = _lib.load()
    base = 1 << 40  # elements are 2 bytes; weights, scales and bias lie elsewhere
    weights = (base - (1 << 30),) + ((base - (1 << 29),) if sparse else ())
    args = (base + 2 * x_at, ldx) + weights + (base - (1 << 28), base - (1 << 27), base + 2 * y_at, ldy, None, M, N, K, _lib.SAMFAST_F16)
    code = lib.samfast_linear_i8_sparse24(*args, None) if sparse else lib.samfast_linear_i8(*args, 0, None)
    error = lib.samfast_last_error()
    assert (code == -2 and b"only bf16" in error) or (code == -1 and b"workspace must be" in error), (code, error)
    return "one" if code == -2 else "two"


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("M,N,K", [(40, 384, 256), (600, 640, 256), (64, 64, 256)])  # few rows, a band of rows, N under K
def test_a_linear_is_one_launch_unless_its_rows_share_memory(M, N, K, sparse):
    """x and y as column ranges of one buffer do not; one element in common does.  Against a count of the elements."""
    import random
    rng = random.Random(M + N)
    assert _linear_route(M, N, K, 0, K, 0, N, sparse) == "two"  # y over x
    ld = K + N
    assert _linear_route(M, N, K, 0, ld, K, ld, sparse) == "one"
    assert _linear_route(M, N, K, N, ld, 0, ld, sparse) == "one"
    assert _linear_route(M, N, K, 0, ld, K - 8, ld, sparse) == "two"
    assert _linear_route(M, N, K, N - 8, ld, 0, ld, sparse) == "two"
    assert _linear_route(M, N, K, 0, ld, K + M * ld, ld, sparse) == "one"  # behind one another
    for _ in range(40):
        ldx, ldy = K + 8 * rng.randint(0, 90), N + 8 * rng.randint(0, 90)
        ldy = ldx if rng.random() < 0.5 and ldx >= N else ldy
        x_at, y_at = 0, 8 * rng.randint(0, (M * ldx) // 8)
        if rng.random() < 0.5:
            x_at, y_at = y_at, x_at
        taken = {e for i in range(M) for e in range((x_at + i * ldx) // 8, (x_at + i * ldx + K) // 8)}
        shared = any(e in taken for i in range(M) for e in range((y_at + i * ldy) // 8, (y_at + i * ldy + N) // 8))
        assert _linear_route(M, N, K, x_at, ldx, y_at, ldy, sparse) == ("two" if shared else "one"), (x_at, ldx, y_at, ldy)


@pytest.mark.parametrize("M,K", [(1, 256), (8, 1024), (8, 5120), (9, 2048), (16, 2048), (17, 768), (32, 768)])
def test_a_linear_over_a_handful_of_rows_into_those_rows_takes_a_workspace(M, K):
    """The sizes at which scales of any alignment are taken: one launch reads rows of x in every workgroup while others write y, so
    that y over x is two launches there too, refused without a workspace, and the size of one is told."""
    from samfast_amd import _lib
    lib = _lib.load()
    assert lib.samfast_linear_i8_one_launch(M, K, K, 0) == 1
    assert lib.samfast_linear_i8_workspace(M, K, K, 0) >= M * K + 4 * M
    assert _linear_route(M, K, K, 0, K, 0, K) == "two"
    assert _linear_route(M, K, K, 0, 2 * K, K, 2 * K) == "one"


@pytest.mark.parametrize("M,N,K,layout", [(0, 768, 768, 0), (-1, 768, 768, 0), (8, 0, 768, 1), (8, -8, 768, 2), (8, 768, 0, 0), (8, 768, -64, 2), (8, 768, 768, 3),
                                          (8, 768, 768, -1), (4096, 768, 768, 7)])
def test_questions_about_no_linear_are_refused(M, N, K, layout):
    from samfast_amd import _lib
    lib = _lib.load()
    for name in ("samfast_linear_i8_workspace", "samfast_linear_i8_one_launch"):
        assert getattr(lib, name)(M, N, K, layout) == -1, name
        assert name[8:].encode() in lib.samfast_last_error()


def test_the_sparse_products_lines():
    """Both sides of each line between the 128-token kernel and the tiles by turns: (M, N, K, epilogue, channels of the tile)."""
    from samfast_amd import _lib
    lib = _lib.load()
    none, gelu, residual = _lib.EPILOGUE_NONE, _lib.EPILOGUE_GELU, _lib.EPILOGUE_RESIDUAL
    turns = lambda M, N, K, epilogue, stride=None: lib.samfast_bench_sparse24_turns(M, N, K, epilogue, stride or N)
    for *call, channels in ((4096, 4096, 1024, none, 0), (4200, 4096, 1024, none, 320), (16384, 1024, 1280, none, 0), (4096, 5120, 1280, none, 320),
                            (36149, 4096, 768, none, 256), (27377, 3840, 768, none, 0), (16384, 3072, 2560, none, 256), (16453, 3840, 2560, none, 0),
                            (14612, 5120, 3072, none, 320), (23968, 3840, 1280, none, 0), (4261, 4096, 768, none, 320), (4096, 3072, 768, none, 0),
                            (30232, 5120, 640, none, 320), (4096, 5120, 512, none, 0), (65536, 5120, 1280, none, 320), (65536, 5120, 1280, gelu, 0),
                            (131072, 1024, 4096, residual, 256), (57344, 768, 2048, residual, 0), (40960, 3072, 3072, residual, 0),
                            (8192, 2304, 1024, residual, 320), (11654, 1536, 640, residual, 0), (13632, 1280, 896, residual, 320),
                            (10317, 3840, 2048, residual, 320), (16338, 2304, 1280, residual, 0), (40960, 1280, 5120, residual, 320),
                            (69627, 1280, 640, residual, 0), (40504, 5120, 4096, residual, 320), (40960, 2560, 2560, residual, 0)):
        assert turns(*call) == channels, call
    # rows that are no whole cache lines, at sizes that are otherwise taken
    for M, N, K, epilogue in ((32288, 4904, 640, none), (38665, 1992, 640, none), (20496, 5096, 640, residual), (24576, 1288, 5120, residual)):
        assert turns(M, N, K, epilogue) == 0
    assert turns(65536, 5120, 1280, none, 5128) == 0 and turns(65536, 5120, 1280, none, 5184) == 320
    assert turns(0, 5120, 1280, none) == -1 and turns(65536, 5120, 1280, none, 5112) == -1


def test_the_half_type_products_lines_between_widths():
    """Tiles of 192 columns among the wider ones by the price of their rounds, with GELU a little dearer: (M, N, K, epilogue, 1000 * rows + columns)."""
    from samfast_amd import _lib
    none, gelu, residual = _lib.EPILOGUE_NONE, _lib.EPILOGUE_GELU, _lib.EPILOGUE_RESIDUAL
    for *call, tile in ((4096, 3072, 768, gelu, 256192), (8192, 3072, 768, gelu, 256192), (4096, 3072, 1024, none, 256192), (28672, 3072, 1024, none, 256192), (12288, 3072, 1024, none, 256192),
                        (23243, 1408, 5120, none, 256192), (23243, 1408, 5120, gelu, 256320), (27762, 1280, 768, gelu, 256320), (17289, 4096, 1280, gelu, 256256), (28072, 3072, 1024, gelu, 256192),
                        (4096, 5120, 1280, gelu, 256320), (4096, 1280, 5120, residual, 128160), (20480, 1024, 4096, residual, 320256), (4096, 2304, 768, none, 0)):
        assert _lib.load().samfast_bench_linear_half(*call) == tile, call
        assert _lib.load().samfast_linear_half_pays(*call) == (tile != 0), call


def test_the_dense_products_lines_between_widths():
    """Tiles of 192, 256 and 320 columns by the price of their rounds, 0 for the smaller members: (M, N, K, columns)."""
    from samfast_amd import _lib
    for M, N, K, columns in ((4096, 3072, 1024, 192), (4096, 2304, 768, 0), (8192, 3072, 768, 192), (8192, 2304, 768, 320), (12288, 3072, 1024, 192), (12288, 2304, 768, 256),
                             (28672, 3072, 768, 256), (6144, 3840, 1280, 192), (16384, 3840, 1280, 320), (65536, 3840, 1280, 256)):
        assert _lib.load().samfast_bench_gemm_i8_turns(M, N, K, _lib.EPILOGUE_NONE, N) == columns, (M, N, K)
    for M, N, K, columns in ((12288, 768, 3072, 192), (10700, 768, 3200, 0), (16384, 1280, 5120, 192), (24576, 768, 3072, 256), (32768, 768, 3072, 256), (32768, 768, 768, 0)):
        assert _lib.load().samfast_bench_gemm_i8_turns(M, N, K, _lib.EPILOGUE_RESIDUAL, N) == columns, (M, N, K)


def test_the_lines_of_the_workgroups_of_a_linear_over_few_rows():
    """One column tile each on up to 768 workgroups, nine k steps on up to 512; 2:4 up to 1024, 256 values on up to 768 where the band
    kernel takes the others: (M, N, K, layout, 1000 * rows + columns)."""
    from samfast_amd import _lib
    tile = _lib.load().samfast_bench_linear_i8_few_rows
    for *call, want in ((576, 112, 576, 0, 8016), (599, 112, 576, 0, 8064), (66, 1280, 576, 0, 8064), (91, 776, 576, 1, 8064), (66, 1280, 512, 0, 8016), (66, 1280, 640, 0, 8016), (829, 104, 640, 0, 8016),
                        (45, 2304, 576, 0, 8064), (13, 3840, 4096, 0, 8032), (24, 1280, 5120, 0, 8016), (32, 1280, 5120, 0, 0), (64, 1024, 5120, 2, 8032),
                        (472, 408, 256, 2, 8032), (480, 408, 256, 2, 0), (480, 520, 256, 2, 0), (480, 512, 256, 2, 8032), (480, 520, 384, 2, 8032), (60, 4096, 256, 2, 8032), (31, 6152, 256, 2, 8032), (1276, 144, 256, 2, 8032)):
        assert tile(*call) == want, call
    assert tile(0, 1024, 576, 0) == -1 and tile(8, 1024, 576, 3) == -1


def test_the_lines_of_the_products_of_few_rows():
    """64 x 32 tiles end at 2304 values, but not where row-major weights of an odd multiple of 64 meet K-block-major codes: (M, N, K, codes' and weights'
    layout, 1000 * rows + columns)."""
    from samfast_amd import _lib
    row, kb, tile = _lib.LAYOUT_ROWMAJOR, _lib.LAYOUT_KB64, _lib.load().samfast_bench_gemm_i8_few_rows
    for *call, want in ((194, 1600, 2240, kb, row, 64032), (194, 1600, 2304, kb, row, 0), (194, 1600, 3648, kb, row, 64032), (39, 5120, 3776, kb, row, 64032), (39, 5120, 3840, kb, row, 0),
                        (194, 1600, 3648, row, row, 0), (194, 1600, 3648, kb, kb, 0), (331, 1280, 5056, kb, row, 64032), (600, 1280, 5056, kb, row, 0), (64, 4096, 4096, kb, row, 32032)):
        assert tile(*call) == want, call
    assert tile(0, 1600, 2240, kb, row) == -1


def test_a_linear_reorders_no_weights_for_products_by_turns():
    """From 16384 rows on, the workspace holds reordered weights for the products that read them, and none for those by turns, whose tiles of 192
    columns are among them."""
    from samfast_amd import _lib
    lib, seen = _lib.load(), set()
    for M in (16384, 16404, 20000, 28042, 40000, 65536):
        for K in (576, 640, 768, 1280, 2048, 5120):
            for N in (128, 400, 496, 768, 1280, 2304, 3840):
                turns = lib.samfast_bench_gemm_i8_turns(M, N, K, _lib.EPILOGUE_NONE, N)
                spare = lib.samfast_linear_i8_workspace(M, N, K, 0) - M * K - 4 * M
                assert spare < 32 if turns else N * K <= spare < N * K + 32, (M, N, K, turns)
                seen.add(turns)
    assert seen == {0, 192, 256, 320}
    assert lib.samfast_linear_i8_workspace(16383, 400, 2048, 0) < 16383 * 2052 + 32


def test_the_dense_products_lines_within_one_round_of_192_columns():
    """From two thirds of the CUs' time on where the loop is longer than 768, half of it from 2048 on: (M, N, K, columns)."""
    from samfast_amd import _lib
    for M, N, K, columns in ((4096, 2304, 896, 192), (2437, 3584, 1024, 192), (2200, 3904, 5120, 192), (12973, 696, 1280, 192), (8192, 1024, 1024, 0), (4604, 1792, 1152, 0), (6262, 1024, 4096, 192),
                             (5618, 1408, 2048, 192), (4025, 1728, 1280, 0), (1401, 3584, 4096, 0),
                             (4096, 2304, 640, 0), (4096, 2304, 960, 0), (16385, 768, 1024, 0)):
        assert _lib.load().samfast_bench_gemm_i8_turns(M, N, K, _lib.EPILOGUE_NONE, N) == columns, (M, N, K)


def test_the_dense_residual_products_lines_where_rows_are_no_whole_lines():
    """Loops under 1280 beyond two rounds are left to the smaller tiles there, others by turns as on whole lines: (M, N, K, columns)."""
    from samfast_amd import _lib
    turns = lambda M, N, K, epilogue, stride=None: _lib.load().samfast_bench_gemm_i8_turns(M, N, K, epilogue, stride or N)
    residual = _lib.EPILOGUE_RESIDUAL
    for *call, columns in ((28672, 1992, 640, 0), (14563, 4904, 640, 0), (40960, 4904, 1024, 0), (16384, 1992, 640, 256), (7556, 1992, 1024, 256),
                           (28672, 1992, 1280, 256)):
        assert turns(*call, residual) == columns, call
    assert turns(28672, 1992, 640, residual, 2048) == 256 and turns(28672, 1024, 1024, residual) == 256  # whole lines
    assert turns(65536, 3840, 1280, _lib.EPILOGUE_NONE) in (256, 320) and turns(65536, 3840, 1280, _lib.EPILOGUE_GELU) == 0
    assert turns(-1, 3840, 1280, residual) == -1


def test_the_lines_of_a_linear_in_one_launch_on_wide_tiles():
    """Both sides of each line of the band's widest tiles: (M, N, K, layout, one launch)."""
    from samfast_amd import _lib
    one = _lib.load().samfast_linear_i8_one_launch
    for *call, taken in ((200, 32000, 1024, 0, 0), (200, 32000, 1024, 2, 0), (64, 139008, 1024, 0, 1), (1024, 8192, 1024, 2, 0), (1100, 8192, 1024, 2, 1),
                         (2256, 3072, 1024, 0, 1), (2980, 2048, 512, 2, 1), (1497, 4096, 1024, 0, 0), (1650, 4096, 1024, 0, 1), (1540, 4096, 1024, 2, 0),
                         (761, 10880, 512, 0, 0), (1451, 5120, 256, 0, 0), (1651, 5120, 256, 0, 1), (3490, 2048, 256, 0, 1), (1500, 5120, 768, 2, 1), (1300, 5120, 768, 2, 0), (351, 16384, 1280, 0, 0), (480, 16384, 1280, 0, 1),
                         (1600, 3840, 1280, 0, 1), (492, 16384, 1280, 2, 0), (520, 16384, 1280, 2, 1), (331, 20680, 1152, 2, 0),
                         (1900, 3456, 1152, 2, 1), (4630, 1280, 1152, 2, 1), (4096, 3072, 768, 0, 1)):
        assert one(*call) == taken, call


def test_the_lines_of_a_linear_in_one_launch_over_few_rows():
    """Both sides of each line of long rows (shorter ones may be the band's): (M, N, K, layout, one launch)."""
    from samfast_amd import _lib
    one = _lib.load().samfast_linear_i8_one_launch
    for *call, taken in ((24, 1280, 5120, 0, 1), (32, 1280, 5120, 0, 0), (64, 1024, 4096, 0, 1), (65, 1024, 4096, 0, 0), (64, 1024, 4160, 0, 0), (128, 512, 2112, 1, 1), (129, 512, 2112, 1, 0),
                         (256, 1024, 2048, 2, 1), (257, 1024, 2048, 2, 0), (128, 1024, 3072, 2, 1), (129, 1024, 3072, 2, 0), (64, 1024, 5120, 2, 1), (65, 1024, 5120, 2, 0)):
        assert one(*call) == taken, call


@pytest.mark.parametrize("M,N,K", [(8, 1024, 1024), (64, 1024, 1024), (4096, 3072, 768), (5000, 1280, 5120)])  # few rows, more, a band, two launches
def test_a_linear_of_another_type_is_unsupported_in_every_form(M, N, K):
    from samfast_amd import _lib
    lib, p = _lib.load(), [1 << 40 + i for i in range(7)]  # (refused before anything is launched)
    assert lib.samfast_linear_i8(p[0], K, p[1], p[2], p[3], p[4], N, p[5], M, N, K, _lib.SAMFAST_F16, 0, None) == -2
    assert lib.samfast_linear_i8_sparse24(p[0], K, p[1], p[2], p[3], p[4], p[5], N, p[6], M, N, K, _lib.SAMFAST_F16, None) == -2


def test_the_native_modules_entries_decline_rows_on_the_cpu():
    """Such a call, or one without a module's buffers, is left to the Python route."""
    from samfast_amd import _lib
    from samfast_amd.quant import Int8DynamicLinear
    host = _lib.host()
    lin = Int8DynamicLinear.from_float(torch.nn.Linear(256, 16))
    x = torch.randn(3, 256).to(torch.bfloat16)
    for entry in (host.module_linear, host.module_sparse_linear):
        assert entry(x, lin._buffers) is None
        assert entry(x, {}) is None
        assert entry(x, None) is None
        assert entry(x) is None
    with pytest.raises(RuntimeError):
        lin(x)
