"""Global attention with caller-computed factors: every form of the kernel against the oracle."""

import math

import pytest
import torch

from helpers import bias_inputs
from oracle import relpos_attention as ora

pytestmark = pytest.mark.gpu

FORMS = {"eight wavefronts": dict(SAMFAST_ATTN_WAVES=8), "four": dict(SAMFAST_ATTN_WAVES=4), "key split": dict(SAMFAST_ATTN_SPLIT=2)}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("B,nH,gh,hd,ramp,dtype", [
    (1, 3, 64, 64, 0.0, torch.bfloat16),
    (2, 1, 64, 80, 0.0, torch.float16),
    (1, 1, 2, 80, 0.0, torch.bfloat16),     # the shortest grid: two key rows
    (2, 2, 34, 64, 0.0, torch.float16),     # rel_h renewed for two rows only, its rows not 16-byte aligned
    (1, 2, 36, 80, 30.0, torch.bfloat16),   # logits that rise along the keys: the reference moves again and again
    (1, 2, 64, 64, 30.0, torch.float16),
])
def test_bias_kernels_vs_oracle(form, B, nH, gh, hd, ramp, dtype):
    from samfast_amd import _lib, ops
    print(f"case {form} B={B} nH={nH} gh={gh} hd={hd} {dtype}", flush=True)
    q, k, v, rel_h, rel_w = bias_inputs(B, nH, gh, 64, hd, seed=gh + hd, dtype=dtype)
    if ramp:
        u = torch.full((hd,), 1 / math.sqrt(hd))
        steps = torch.arange(gh * 64) / (gh * 64)
        q = (q.float() + 4.0 * u).to(dtype)
        k = (k.float() + ramp * steps[None, None, :, None] * u).to(dtype)
    ref = ora.attention_rel_h_rel_w(q, k, v, rel_h, rel_w, compute_dtype=torch.float32)
    with _lib.knobs(**FORMS[form]):
        out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), rel_h.squeeze(-1).cuda(), rel_w.squeeze(-2).cuda())
    diff = (out.float().cpu() - ref.float()).abs()
    print(f"max-abs {diff.max().item():.2e} mean-abs {diff.mean().item():.2e}", flush=True)
    assert diff.max().item() <= 2e-2 and diff.mean().item() <= 1e-3


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_denominator_sums_unrounded_probabilities(form, dtype):
    """One key of probability one (a power of two) against 4095 of one smaller probability, whose rounding - the same for all
    of them - stays out of the denominator at head_dim 64."""
    from samfast_amd import _lib, ops
    print(f"case denominator {form} {dtype}", flush=True)
    N, hd = 4096, 64
    q, k, v = torch.zeros((1, 1, N, hd)), torch.zeros((1, 1, N, hd)), torch.zeros((1, 1, N, hd))
    q[..., 0] = torch.linspace(2.0, 7.0, N)
    k[0, 0, 0, 0], v[0, 0, 0] = 8.0, 1.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    zeros = torch.zeros((1, 1, N, 64), dtype=dtype)
    ref = (q.double() @ k.double().transpose(-1, -2) * hd ** -0.5).softmax(-1) @ v.double()
    with _lib.knobs(**FORMS[form]):
        out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), zeros.cuda(), zeros.cuda())
    # the result's own rounding, half an eps, and a sixteenth for exponentials and sums in fp32
    assert ((out.cpu().double() - ref).abs() / ref).max() <= (0.5 + 0.0625) * torch.finfo(dtype).eps


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("where", [0, 31, 40, 2000, 4095])
def test_fp16_probabilities_far_below_the_maximum(form, hd, where):
    """One key 2^12 to 2^14 above 4095 equal ones, which carry half of the sum: their probabilities keep the type's bits."""
    from samfast_amd import _lib, ops
    print(f"case tail {form} hd={hd} key {where}", flush=True)
    N = 4096
    q, k, v = torch.zeros((1, 1, N, hd)), torch.zeros((1, 1, N, hd)), torch.ones((1, 1, N, hd))
    q[..., 0] = torch.linspace(12.0, 13.9, N) * math.log(2) * math.sqrt(hd)
    k[0, 0, where, 0], v[0, 0, where] = 1.0, 0.0
    q, k, v = (t.to(torch.float16) for t in (q, k, v))
    zeros = torch.zeros((1, 1, N, 64), dtype=torch.float16)
    ref = (q.double() @ k.double().transpose(-1, -2) * hd ** -0.5).softmax(-1) @ v.double()
    with _lib.knobs(**FORMS[form]):
        out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), zeros.cuda(), zeros.cuda())
    # a normal fp16 probability and the result, rounded once each (2^-11); 2^-13 for exponentials and sums in fp32
    assert ((out.cpu().double() - ref).abs() / ref).max() <= 2.0 ** -10 + 2.0 ** -13


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("gh", [2, 34, 64])
def test_every_other_sixteen_queries_move_their_reference(gh, which, dtype):
    """A lane of the split form has two queries, 16 apart: the logits of one rise along the keys, the other's do not."""
    from samfast_amd import ops
    print(f"case two queries gh={gh} which={which} {dtype}", flush=True)
    q, k, v, rel_h, rel_w = bias_inputs(1, 2, gh, 64, 64, seed=gh + which, dtype=dtype)
    n = torch.arange(gh * 64)
    q = (q.float() + 0.5 * (n // 16 % 2 == which)[None, None, :, None]).to(dtype)
    k = (k.float() + 3.75 * (n / (gh * 64))[None, None, :, None]).to(dtype)
    out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), rel_h.squeeze(-1).cuda(), rel_w.squeeze(-2).cuda()).double().cpu()
    qd, kd, vd = q.double(), k.double(), v.double()
    scores = qd @ kd.transpose(-1, -2) * 0.125 + (rel_h.double().reshape(1, 2, gh * 64, gh, 1) + rel_w.double().reshape(1, 2, gh * 64, 1, 64)).reshape(1, 2, gh * 64, gh * 64)
    p = torch.softmax(scores, -1)
    ref, weight = p @ vd, p @ vd.abs()
    eps = torch.finfo(dtype).eps
    # probabilities and output rounded to the type, scores and sums in fp32; fp16 probabilities below 2^-14 to 2^-25, the denominator being at least one
    floor = gh * 64 * 2.0 ** -25 * vd.abs().amax() if dtype == torch.float16 else 0.0
    assert ((out - ref).abs() <= 0.51 * eps * (weight + ref.abs()) + 1e-4 * weight + floor + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("gh,form", [(2, "four"), (32, "four"), (34, "four"), (36, "eight wavefronts"), (64, "eight wavefronts")])
def test_unsplit_keys_of_80_channels_near_64_bits(gh, form, which, dtype):
    """The same where keys are not split, at 80 channels (whose last sixteen are a k step of their own): one query of a lane moves its reference, the
    other does not, and rel_h is renewed at key row 32.  Larger values in the last channels, so that each of them counts."""
    from samfast_amd import _lib, ops
    print(f"case 80 channels gh={gh} {form} which={which} {dtype}", flush=True)
    q, k, v, rel_h, rel_w = bias_inputs(1, 2, gh, 64, 80, seed=gh + which, dtype=dtype)
    n = torch.arange(gh * 64)
    last = 1.0 + (torch.arange(80) >= 64) * 1.0
    q = (q.float() * last + 0.4 * (n // 16 % 2 == which)[None, None, :, None]).to(dtype)
    k = (k.float() * last + 3.5 * (n / (gh * 64))[None, None, :, None]).to(dtype)
    with _lib.knobs(**FORMS[form]):
        out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), rel_h.squeeze(-1).cuda(), rel_w.squeeze(-2).cuda()).double().cpu()
    qd, kd, vd = q.double(), k.double(), v.double()
    bias = (rel_h.double().reshape(1, 2, gh * 64, gh, 1) + rel_w.double().reshape(1, 2, gh * 64, 1, 64)).reshape(1, 2, gh * 64, gh * 64)
    p = torch.softmax(qd @ kd.transpose(-1, -2) * 80 ** -0.5 + bias, -1)
    ref, weight = p @ vd, p @ vd.abs()
    eps = torch.finfo(dtype).eps
    # as above; the denominator sums rounded probabilities, half an eps more
    floor = gh * 64 * 2.0 ** -25 * vd.abs().amax() if dtype == torch.float16 else 0.0
    assert ((out - ref).abs() <= 0.51 * eps * (weight + 2 * ref.abs()) + 1e-4 * weight + floor + 1e-6).all()


@pytest.mark.parametrize("hd,dtype", [(64, torch.bfloat16), (64, torch.float16), (80, torch.float16)])
@pytest.mark.parametrize("gh", [64, 16, 6])  # hd 64: up to 256 workgroups of 64 queries and more, two orders of one kernel's instructions
def test_a_slice_has_the_same_bits_in_any_batch(hd, dtype, gh):
    from samfast_amd import ops
    print(f"case batch hd={hd} {dtype} gh={gh}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(hd + gh)
    N = gh * 64
    q, k, v = ((torch.randn((4, 16, N, hd), generator=g, device="cuda") * 0.5).to(dtype) for _ in range(3))
    rh = (torch.randn((4, 16, N, gh), generator=g, device="cuda") * 0.5).to(dtype)
    rw = (torch.randn((4, 16, N, 64), generator=g, device="cuda") * 0.5).to(dtype)
    whole = ops.attn_relpos_bias(q, k, v, rh, rw)
    for b, h in ((1, 8), (1, 12), (2, 9), (3, 12)):
        assert torch.equal(ops.attn_relpos_bias(*(t[:b, :h] for t in (q, k, v, rh, rw))), whole[:b, :h]), (b, h)


def test_bias_kernels_read_strided_factors():
    """The factors as slices of one (B, nH, N, 128) tensor, q / k / v of a token-major buffer: same bits as contiguous."""
    from samfast_amd import ops
    B, nH, N, hd = 1, 2, 4096, 64
    g = torch.Generator(device="cuda").manual_seed(1)
    qkv = torch.randn((B, N, 3, nH, hd), generator=g, device="cuda").to(torch.bfloat16)
    both = (torch.randn((B, nH, N, 128), generator=g, device="cuda") * 0.5).to(torch.bfloat16)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    a = ops.attn_relpos_bias(q, k, v, both[..., :64], both[..., 64:])
    b = ops.attn_relpos_bias(q.contiguous(), k.contiguous(), v.contiguous(), both[..., :64].contiguous(), both[..., 64:].contiguous())
    assert torch.equal(a, b)


def test_the_operator_is_there_for_those_who_watch():
    """A trace and a compiled graph record it, vmap loops over it, a dispatch mode sees it - and nobody gets another result."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from samfast_amd.flash_4 import _attention_rel_h_rel_w as attention
    args = [t.cuda() for t in bias_inputs(1, 2, 64, 64, 64, seed=1)]
    other = [t.cuda() for t in bias_inputs(1, 2, 64, 64, 64, seed=2)]
    want, want_other = attention(*args), attention(*other)
    traced = torch.jit.trace(attention, args, check_trace=False)
    assert "customflash::custom_flash_aligned" in str(traced.graph)
    assert torch.equal(traced(*other), want_other)
    both = torch.vmap(attention)(*(torch.stack(pair) for pair in zip(args, other)))
    assert torch.equal(both[0], want) and torch.equal(both[1], want_other)

    graphs = []

    def keep(graph_module, example_inputs):
        graphs.append(graph_module.code)
        return graph_module.forward

    assert torch.equal(torch.compile(attention, backend=keep, fullgraph=True)(*args), want)
    assert "custom_flash_aligned" in graphs[0]

    class Names(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    with Names():
        got = attention(*args)
    assert torch.equal(got, want) and any("custom_flash_aligned" in n for n in Names.names)


MASKS = {
    "first half of every row": lambda gh: (None, slice(0, 32)),
    "second half of every row": lambda gh: (None, slice(32, 64)),
    "all columns but one": lambda gh: (None, slice(0, 63)),
    "first rows": lambda gh: (slice(0, 3), None),
    "all rows but the last": lambda gh: (slice(0, gh - 1), None),
    "first rows and first half": lambda gh: (slice(0, 2), slice(0, 32)),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("hd,dtype,values", [
    (64, torch.bfloat16, (-math.inf, torch.finfo(torch.bfloat16).min, -1e30, -1e9, -1e4)),
    (80, torch.bfloat16, (-math.inf, torch.finfo(torch.bfloat16).min, -1e30, -1e9, -1e4)),
    (64, torch.float16, (-math.inf, torch.finfo(torch.float16).min, -1e3)),
    (80, torch.float16, (-math.inf, torch.finfo(torch.float16).min, -1e3)),
])
def test_bias_kernels_with_masked_keys(form, mask, hd, dtype, values):
    """Factors that take keys away - for every query, and for every second one - against the softmax in 64 bits."""
    from samfast_amd import _lib, ops
    B, nH, gh = 1, 2, 4
    q, k, v, rel_h, rel_w = bias_inputs(B, nH, gh, 64, hd, seed=gh + hd, dtype=dtype)
    rows, cols = MASKS[mask](gh)
    for value in values:
        for step in (1, 2):
            print(f"case masked {form}, {mask}, hd={hd} {dtype} {value} every {step}", flush=True)
            rh, rw = rel_h.squeeze(-1).clone(), rel_w.squeeze(-2).clone()
            if rows is not None:
                rh[:, :, ::step, rows] = value
            if cols is not None:
                rw[:, :, ::step, cols] = value
            s = q.double() @ k.double().transpose(-1, -2) * hd ** -0.5 + (rh.double()[..., None] + rw.double()[..., None, :]).flatten(-2)
            ref = s.softmax(-1) @ v.double()
            with _lib.knobs(**FORMS[form]):
                out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), rh.cuda(), rw.cuda())
            # probabilities and result in the half type: half an ulp each, and one for the sums between
            assert (out.cpu().double() - ref).abs().max() <= 4 * torch.finfo(dtype).eps * v.abs().max().item()


@pytest.mark.parametrize("layout", ["tokens", "rows"])
@pytest.mark.parametrize("gh,gw", [(14, 14), (13, 14), (14, 5), (6, 8), (7, 13)])
@pytest.mark.parametrize("hd,dtype,values", [
    (64, torch.bfloat16, (-math.inf, torch.finfo(torch.bfloat16).min, -1e30, -1e9, -1e4)),
    (80, torch.bfloat16, (-math.inf, -1e9)),
    (64, torch.float16, (-math.inf, torch.finfo(torch.float16).min, -1e3)),
    (80, torch.float16, (-math.inf, -1e3)),
])
def test_window_kernels_with_masked_keys(layout, gh, gw, hd, dtype, values):
    """As on the grid: rows and columns taken away, the first key tiles of 32 whole among them, for every and every second query."""
    from samfast_amd import _lib, ops
    q, k, v, rel_h, rel_w = bias_inputs(3, 2, gh, gw, hd, seed=gh + gw, dtype=dtype)
    for rows, cols in ((slice(0, gh - 1), None), (None, slice(0, gw - 1)), (slice(0, 3), slice(0, 2)), (slice(1, gh), None), (slice(3, 5), slice(2, 4))):
        for value in values:
            for step in (1, 2):
                print(f"case masked window {layout} {gh}x{gw} hd={hd} {dtype} {rows} {cols} {value} every {step}", flush=True)
                rh, rw = rel_h.squeeze(-1).clone(), rel_w.squeeze(-2).clone()
                if rows is not None:
                    rh[:, :, ::step, rows] = value
                if cols is not None:
                    rw[:, :, ::step, cols] = value
                s = q.double() @ k.double().transpose(-1, -2) * hd ** -0.5 + (rh.double()[..., None] + rw.double()[..., None, :]).flatten(-2)
                ref = s.softmax(-1) @ v.double()
                with _lib.knobs(SAMFAST_ATTN_WINDOW_ROWS=int(layout == "rows")):
                    out = ops.attn_relpos_bias(q.cuda(), k.cuda(), v.cuda(), rh.cuda(), rw.cuda())
                assert (out.cpu().double() - ref).abs().max() <= 4 * torch.finfo(dtype).eps * v.abs().max().item()


@pytest.mark.parametrize("gh,gw", [(14, 14), (2, 2), (13, 14), (14, 5), (6, 8), (1, 16), (15, 13)])
@pytest.mark.parametrize("hd,dtype", [(64, torch.bfloat16), (80, torch.float16)])
def test_window_factors_read_in_pairs_or_one_by_one(gh, gw, hd, dtype):
    """Factor rows of even length are read as pairs where they start on 4 bytes; a view that starts on
    2 takes single reads, with the same bits, and both follow the softmax in 64 bits."""
    from samfast_amd.flash_4 import _attention_rel_h_rel_w
    print(f"case window factors {gh}x{gw} hd={hd} {dtype}", flush=True)
    g = torch.Generator().manual_seed(gh * 100 + gw + hd)
    N = gh * gw
    q, k, v = (torch.randn((3, 2, N, hd), generator=g).mul(0.5).to(dtype) for _ in range(3))
    rh, rw = torch.randn((3, 2, N, gh, 1), generator=g).mul(0.5).to(dtype), torch.randn((3, 2, N, 1, gw), generator=g).mul(0.5).to(dtype)

    def shifted(t):  # the same values one element into a longer buffer
        return torch.cat([torch.zeros(1, dtype=dtype), t.flatten()]).cuda()[1:].view(t.shape)

    args = [t.cuda() for t in (q, k, v)]
    y = _attention_rel_h_rel_w(*args, rh.cuda(), rw.cuda())
    assert torch.equal(y, _attention_rel_h_rel_w(*args, shifted(rh), shifted(rw)))
    s = q.double() @ k.double().transpose(-1, -2) * hd ** -0.5 + (rh.double() + rw.double()).flatten(-2)
    ref = s.softmax(-1) @ v.double()
    # probabilities and result in the half type, as the operator's other tests
    eps = torch.finfo(dtype).eps
    assert (y.cpu().double() - ref).abs().max() <= 4 * eps * v.abs().max().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("gh,gw", [(1, 1), (5, 5), (2, 16), (3, 11), (8, 8), (5, 13), (6, 16), (7, 14), (9, 13), (8, 16), (10, 13)])
def test_small_windows_same_bits_in_any_batch(gh, gw, hd, dtype):
    """Workgroups sized to the window (many windows), of four wavefronts (some) and of eight (few) at the edges of 32-token tiles,
    strided operands; the few against the oracle."""
    from samfast_amd import ops
    print(f"case small windows {gh}x{gw} hd={hd} {dtype}", flush=True)
    nH, N = 4, gh * gw
    g = torch.Generator(device="cuda").manual_seed(N + hd)
    qkv = (torch.randn((140, N, 3, nH, hd), generator=g, device="cuda") * 0.5).to(dtype)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    rel_h, rel_w = ((torch.randn((140, nH, N, n), generator=g, device="cuda") * 0.5).to(dtype) for n in (gh, gw))
    rel_h[1, :, :, 0] = float("-inf") if gh > 1 else 0
    run = lambda b: ops.attn_relpos_bias(q[b], k[b], v[b], rel_h[b], rel_w[b])
    many, some, few = run(slice(0, 140)), run(slice(0, 60)), run(slice(0, 3))  # 560, 240 and 12 items
    assert torch.equal(many[:60], some) and torch.equal(some[:3], few)
    last = run(slice(130, 140))
    assert torch.equal(many[130:], last)
    ref = ora.attention_rel_h_rel_w(*(t[:3].cpu() for t in (q, k, v)), rel_h[:3, ..., None].cpu(), rel_w[:3, :, :, None].cpu(), compute_dtype=torch.float32)
    diff = (few.float().cpu() - ref.float()).abs()
    assert diff.max().item() <= 2e-2 and diff.mean().item() <= 1e-3
