"""The bf16 PairTransition backward at the row counts where its two kernels can
go wrong: one row, a ragged last tile, one split of the weight gradients and
several of unequal length, more tiles than waves in flight.  Against the
gradient oracle, with the ReLU's pass pattern of the hidden values as bf16
forms them and dy = 0 in rows where one of them is nearly zero (see
test_gpu_pair_block.test_pair_transition_backward; 1e-3 here, since with many
rows some x_hat round the other way, which moves h by up to 2^-9 |x_hat w|)."""
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
