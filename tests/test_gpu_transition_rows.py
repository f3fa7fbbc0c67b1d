"""The bf16 PairTransition backward at the row counts where its two kernels can
go wrong: one row, a ragged last tile, one split of the weight gradients and
several of unequal length, more tiles than waves in flight.  Against the
gradient oracle, with the ReLU's pass pattern of the hidden values as bf16
forms them and dy = 0 in rows where one of them is nearly zero (see
test_gpu_pair_block.test_pair_transition_backward; 1e-3 here, since with many
rows some x_hat round the other way, which moves h by up to 2^-9 |x_hat w|).

And the closing sums of the fp32 backwards, which add their partials in pairs."""
import numpy as np
import pytest
import torch

from genie_tk.pair_transform import PairTransition
from oracle import grads
from tests import helpers as H
from tests.gpu_common import log, to_np
from tests.test_gpu_grads import _check_grad
from tests.test_gpu_pair_block import _hidden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("rows", [1, 31, 33, 161, 4 * 32 * 9 + 5, 70001])
def test_transition_backward_rows(c, rows):
    log(f"transition backward rows={rows} c={c}")
    P = H.bf16_params(H.draw_params(H.pair_transition_shapes(c), rows + c, ln_random=True, bias_random=True))
    rng = np.random.default_rng(rows)
    p = H.bf16_round(rng.standard_normal((rows, c)).astype(np.float32))
    dy = H.bf16_round(rng.standard_normal((rows, c)).astype(np.float32))
    h = _hidden(p, P, True)
    dy[(np.abs(h) < 1e-3).any(axis=-1)] = 0.0
    mod = PairTransition(c, 4)
    mod.load_state_dict(H.to_state_dict(P))
    mod = mod.to("cuda", torch.bfloat16)
    pk = torch.from_numpy(p).to("cuda", torch.bfloat16).requires_grad_(True)
    g = torch.autograd.grad(mod(pk), [pk, *mod.parameters()], torch.from_numpy(dy).to("cuda", torch.bfloat16))
    dp_ref, g_ref = grads.pair_transition_grad(p, P, dy, gate=h > 0)
    _check_grad(to_np(g[0]), dp_ref, "bf16", "dp")
    for (name, _), gk in zip(mod.named_parameters(), g[1:]):
        _check_grad(to_np(gk), g_ref[name], "bf16", name)


def test_closing_sums_add_in_pairs():
    """fp32, 512 rows: the gradient of linear_2's bias is the sum of dy over eight
    segments of 64 rows.  Their sums 2^24, 1, 0, 1, 0, ... add up exactly in
    pairs; one after the other, each 1 is lost to the rounding of 2^24 + 1."""
    log("closing sums in pairs")
    mod = PairTransition(128, 4)
    mod.load_state_dict(H.to_state_dict(H.draw_params(H.pair_transition_shapes(128), 3)))
    mod = mod.to("cuda")
    p = torch.randn(512, 128, generator=torch.Generator().manual_seed(4)).to("cuda").requires_grad_()
    dy = torch.zeros(512, 128, device="cuda")
    dy[5] = 2.0 ** 24
    dy[64 + 9] = 1.0
    dy[3 * 64 + 11] = 1.0
    g = torch.autograd.grad(mod(p), mod.linear_2.bias, dy)[0]
    assert torch.equal(g, torch.full_like(g, 2.0 ** 24 + 2))
