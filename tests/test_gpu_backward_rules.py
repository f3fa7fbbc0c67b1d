"""The backward kernels (and the generic tri-mul prologue) on both sides of the
rules that choose between their forms: the same results either way.  An empty batch has zero gradients."""
import pytest
import torch

from genie_tk.pair_transform import PairTransition
from tests import helpers as H
from tests.gpu_common import ext, trimul_module, triattn_module

pytestmark = pytest.mark.gpu


def _inputs(B, N, dt, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(1, N, N, 128, generator=gen, device="cuda").to(dt)
    dy = torch.randn(1, N, N, 128, generator=gen, device="cuda").to(dt)
    m = torch.ones(1, N, N, device="cuda")
    m[:, N - 5:] = 0
    m[:, :, N - 5:] = 0
    return (t.expand(B, *t.shape[1:]).contiguous() for t in (x, dy, m))


@pytest.mark.parametrize("outgoing", [True, False])
@pytest.mark.parametrize("B,N", [(1, 33), (2, 50), (1, 150), (1, 301)])
def test_contraction_backward_on_64_tiles(monkeypatch, outgoing, B, N):
    """Planes of an odd multiple of 64: operands read transposed give the bits
    of planes transposed first (the same products in the same order)."""
    mod = trimul_module(H.draw_params(H.tri_mul_shapes(128, 128), seed=N, bias_random=True), outgoing,
                        torch.bfloat16)
    x, dy, m = _inputs(B, N, torch.bfloat16, N)
    x.requires_grad_()
    runs = []
    for force in ("0", "1"):
        monkeypatch.setenv("GENIE_TK_TRANSPOSE_PLANES", force)
        runs.append(torch.autograd.grad(mod(x, m), [x, *mod.parameters()], dy))
    for a, b in zip(*runs):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("starting", [True, False])
def test_attention_backward_split_tiles(starting):
    """fp32, N = 72: 216 row tiles take the prologue backward that four waves
    share, 8 copies (1728 tiles) the one of a wave a tile, 9 copies (1944, two
    whole rounds of the chip) also the projections of a wave a tile.  Each copy's
    dx is the single call's up to the order of four partial sums of 32-bit values."""
    mod = triattn_module(H.draw_params(H.tri_attn_shapes(128, 32, 4), seed=9, bias_random=True), starting, 4,
                         torch.float32)
    dx = []
    for B in (1, 8, 9):
        x, dy, m = _inputs(B, 72, torch.float32, 72)
        x.requires_grad_()
        dx.append(torch.autograd.grad(mod(x, m), x, dy)[0])
    one, *many = dx
    for d in many:
        for k in range(d.shape[0]):
            err = (d[k] - one[0]).norm() / one[0].norm()
            assert err < 1e-6, err


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_attention_backward_entries_agree(dt):
    """_C.tri_attn_backward (gtk_tri_attn_backward: four heads of 32) and
    _C.tri_attn_backward_heads (every head shape) are one pass: the same bits."""
    mod = triattn_module(H.draw_params(H.tri_attn_shapes(64, 128, 4), seed=5, bias_random=True), True, 4, dt)
    x, dy, m = _inputs(1, 45, dt, 45)
    x, dy = x[..., :64].contiguous(), dy[..., :64].contiguous()
    params = [p.detach() for p in mod._param_list()]
    C = ext()
    one = C.tri_attn_backward(x, m, dy, params, 64, 128, 4, True)
    every = C.tri_attn_backward_heads(x, m, dy, params, 64, 128, 4, True)
    for a, b in zip(one[:-1], every[:-1]):  # (the last is the buffer that holds them, with its gaps)
        assert torch.isfinite(a).all() and torch.equal(a, b)
    narrow = triattn_module(H.draw_params(H.tri_attn_shapes(64, 32, 4), seed=5), True, 4, dt)
    with pytest.raises(RuntimeError, match="unsupported"):
        C.tri_attn_backward(x, m, dy, [p.detach() for p in narrow._param_list()], 64, 32, 4, True)


@pytest.mark.parametrize("c", [32, 64, 128])
def test_trimul_prologue_parts(c):
    """fp32, N = 30: 128 prologue tiles a copy, dealt to 2 c / 32 waves each; 12
    copies (1536 tiles) to fewer, 15 (1920, two whole rounds of the chip) to one
    at c <= 64.  The same products in every form: the same bits."""
    mod = trimul_module(H.draw_params(H.tri_mul_shapes(c, c), seed=c, bias_random=True), True, torch.float32)
    x, _, m = _inputs(1, 30, torch.float32, 30)
    x = x[..., :c].contiguous()
    with torch.no_grad():
        one = mod(x, m)
        for B in (12, 15):
            many = mod(x.expand(B, -1, -1, -1).contiguous(), m.expand(B, -1, -1).contiguous())
            for k in range(B):
                assert torch.equal(many[k], one[0])


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,N", [(0, 8), (2, 0)])
def test_empty_batch_has_zero_gradients(dt, B, N):
    """As autograd of the PyTorch path gives them."""
    mods = [trimul_module(H.draw_params(H.tri_mul_shapes(128, 128), seed=1), True, dt),
            triattn_module(H.draw_params(H.tri_attn_shapes(128, 32, 4), seed=2), True, 4, dt),
            triattn_module(H.draw_params(H.tri_attn_shapes(128, 128, 4), seed=3), False, 4, dt),
            PairTransition(128, 4).to("cuda", dt)]
    for mod in mods:
        x = torch.zeros(B, N, N, 128, device="cuda", dtype=dt, requires_grad=True)
        y = mod(x, torch.ones(B, N, N, device="cuda"))
        assert y.shape == x.shape
        junk = [torch.full((1 << 17,), float("nan"), device="cuda") for _ in range(8)]
        del junk  # what a gradient buffer might hold
        grads = torch.autograd.grad(y, [x, *mod.parameters()], torch.zeros_like(y))
        for g, p in zip(grads, [x, *mod.parameters()]):
            assert g.shape == p.shape and g.dtype == p.dtype and not g.any()
