"""Narrow heads in fp32 (four heads of at most 8 channels, the reference layer's
default) at the sizes where their kernels can go wrong: one tile, a ragged tile,
one position past a 128- and a 256-key LDS segment, several segments; heads
narrower than 8; every c_in; masked, fractional and fully masked rows; masks
whose bias overflows; row chunks, bit-identical to the whole.  Against the float64 oracle with the fp32
tolerance (a fully masked row is uniform there, as its fp32 scores are)."""
import numpy as np
import pytest
import torch

from oracle import pair_ops
from tests import helpers as H
from tests.gpu_common import check_fp32, log, to_np, triattn_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("starting", [True, False])
@pytest.mark.parametrize("N,cin,ch", [(20, 32, 32), (64, 128, 16), (129, 64, 32), (257, 128, 32), (520, 32, 32)])
def test_narrow_heads_fp32(starting, N, cin, ch):
    log(f"narrow heads fp32 N={N} c_in={cin} c_h={ch} starting={starting}")
    P = H.draw_params(H.tri_attn_shapes(cin, ch, 4), seed=N, ln_random=True, bias_random=True)
    x = H.pair_input(1, N, cin, seed=N + 1)
    rng = np.random.default_rng(N + 2)
    m = (rng.random((1, N, N)) >= 0.1).astype(np.float32)
    m[0, 3, :] = 0.0
    m[0, :, 5] = 0.0
    mod = triattn_module(P, starting, 4, torch.float32)
    xd, md = torch.from_numpy(x).to("cuda"), torch.from_numpy(m).to("cuda")
    with torch.no_grad():
        y = mod(xd, md)
        y_res = mod.forward_residual(xd, md)
        y_chunk = mod(xd, md, chunk_size=48)
        y_nm = mod(xd)
    torch.cuda.synchronize()
    assert torch.equal(y, y_chunk), "row chunks differ from the unchunked output"
    rows = sorted({0, 3, 5, 17, N // 2, N - 1})
    sel = (lambda a: a[:, rows]) if starting else (lambda a: a[:, :, rows])
    ref = pair_ops.tri_attn(x, m, P, starting, 4, dtype=np.float64, rows=rows)
    check_fp32(to_np(sel(y)), ref, f"narrow heads N={N}")
    check_fp32(to_np(sel(y_res)), ref + sel(x), f"narrow heads residual N={N}")
    ref = pair_ops.tri_attn(x, None, P, starting, 4, dtype=np.float64, rows=rows)
    check_fp32(to_np(sel(y_nm)), ref, f"narrow heads, no mask, N={N}")


@pytest.mark.parametrize("starting", [True, False])
@pytest.mark.parametrize("value", [float("-inf"), float(np.finfo(np.float32).min)])
@pytest.mark.parametrize("N,lead", [(70, 32), (129, 40), (300, 290)])
def test_narrow_heads_mask_bias_of_minus_infinity(starting, value, N, lead):
    """The first `lead` keys of every row (a whole tile, more than one, more
    than a whole LDS segment) take the bias -inf: no weight, whatever comes
    first.  The PyTorch path gives the same."""
    log(f"narrow heads, mask {value} over {lead} of {N} keys, starting={starting}")
    P = H.draw_params(H.tri_attn_shapes(64, 32, 4), seed=N, ln_random=True, bias_random=True)
    x = H.pair_input(1, N, 64, seed=N + 1)
    m = np.ones((1, N, N), dtype=np.float32)
    if starting:
        m[:, :, :lead] = value
    else:
        m[:, :lead, :] = value
    mod = triattn_module(P, starting, 4, torch.float32)
    xd, md = torch.from_numpy(x).to("cuda"), torch.from_numpy(m).to("cuda")
    with torch.no_grad():
        y = mod(xd, md)
        y_chunk = mod(xd, md, chunk_size=48)
        pt = mod._forward_pytorch(xd, md)
    torch.cuda.synchronize()
    assert torch.equal(y, y_chunk), "row chunks differ from the unchunked output"
    rows = sorted({0, 5, N // 2, N - 1})
    sel = (lambda a: a[:, rows]) if starting else (lambda a: a[:, :, rows])
    keep = np.where(m == 1, 1.0, 0.0).astype(np.float32)  # weight 0 either way
    ref = pair_ops.tri_attn(x, keep, P, starting, 4, dtype=np.float64, rows=rows)
    check_fp32(to_np(sel(y)), ref, f"mask {value}, N={N}")
    check_fp32(to_np(y), to_np(pt), f"mask {value}, N={N}, PyTorch path")


@pytest.mark.parametrize("starting", [True, False])
@pytest.mark.parametrize("N", [60, 200])
def test_narrow_heads_fractional_mask(starting, N):
    """inf = 10: a mask value m takes the score bias 10 (m - 1), which fractional
    values and zeros both leave in the softmax's range."""
    log(f"narrow heads, fractional mask, N={N} starting={starting}")
    P = H.draw_params(H.tri_attn_shapes(128, 32, 4), seed=N, ln_random=True, bias_random=True)
    x = H.pair_input(1, N, 128, seed=N + 1)
    rng = np.random.default_rng(N + 2)
    m = rng.choice(np.float32([0.0, 0.25, 0.5, 0.75, 1.0]), size=(1, N, N)).astype(np.float32)
    mod = triattn_module(P, starting, 4, torch.float32)
    mod.inf = 10.0
    with torch.no_grad():
        y = mod(torch.from_numpy(x).to("cuda"), torch.from_numpy(m).to("cuda"))
    rows = sorted({0, 5, N // 2, N - 1})
    sel = (lambda a: a[:, rows]) if starting else (lambda a: a[:, :, rows])
    ref = pair_ops.tri_attn(x, m, P, starting, 4, inf=10.0, dtype=np.float64, rows=rows)
    check_fp32(to_np(sel(y)), ref, f"fractional mask, N={N}")
