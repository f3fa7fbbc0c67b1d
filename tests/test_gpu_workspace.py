"""No result depends on a workspace value that the same call did not write: with
every uninitialised byte 0xff (NaN in bf16 and fp32) the results are those of
any other call.  The sizes cover each form of the kernels: resident and streamed
forward, the (row, head) backward up to 512 and 1024 and the one beyond, narrow
and full heads, ragged tiles of every operator."""
import pytest
import torch

from genie_tk.pair_transform import PairTransition
from tests import helpers as H
from tests.gpu_common import trimul_module, triattn_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dname", ["bf16", "fp32"])
@pytest.mark.parametrize("op,N", [("tri_attn", 7), ("tri_attn", 33), ("tri_attn", 77), ("tri_attn", 264),
                                  ("tri_attn", 520), ("tri_attn", 1030), ("tri_attn_wide", 77),
                                  ("tri_attn_wide", 520), ("tri_mul", 33), ("tri_mul", 77), ("tri_mul", 301),
                                  ("transition", 1), ("transition", 33)])
def test_results_do_not_depend_on_workspace_contents(dname, op, N):
    dt = torch.bfloat16 if dname == "bf16" else torch.float32
    if op in ("tri_attn", "tri_attn_wide"):
        c_h = 32 if op == "tri_attn" else 128
        mod = triattn_module(H.draw_params(H.tri_attn_shapes(128, c_h, 4), seed=3, bias_random=True), True, 4, dt)
    elif op == "transition":
        mod = PairTransition(128, 4)
        mod.load_state_dict(H.to_state_dict(H.draw_params(H.pair_transition_shapes(128), seed=3, bias_random=True)))
        mod = mod.to("cuda", dt)
    else:
        mod = trimul_module(H.draw_params(H.tri_mul_shapes(128, 128), seed=3, bias_random=True), True, dt)
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(1, N, N, 128, generator=gen, device="cuda").to(dt).requires_grad_()
    dy = torch.randn(1, N, N, 128, generator=gen, device="cuda").to(dt)
    m = torch.ones(1, N, N, device="cuda")
    m[:, N - 3:] = 0
    m[:, :, N - 3:] = 0

    def run():
        y = mod(x, m)
        return [y, *torch.autograd.grad(y, [x, *mod.parameters()], dy)]

    plain = run()
    was = torch.utils.deterministic.fill_uninitialized_memory
    torch.use_deterministic_algorithms(True, warn_only=True)
    torch.utils.deterministic.fill_uninitialized_memory = True
    try:
        filled = run()
    finally:
        torch.use_deterministic_algorithms(False)
        torch.utils.deterministic.fill_uninitialized_memory = was
    for a, b in zip(filled, plain):
        assert torch.isfinite(a).all()
        assert torch.equal(a, b)
