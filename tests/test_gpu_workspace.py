"""The kernels read no workspace value that the same call did not write: with
every uninitialised byte 0xff (NaN in bf16 and fp32) the results are those of
any other call."""
import pytest
import torch

from tests import helpers as H
from tests.gpu_common import trimul_module, triattn_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dname", ["bf16", "fp32"])
@pytest.mark.parametrize("op,N", [("tri_attn", 7), ("tri_attn", 33), ("tri_attn", 77), ("tri_attn", 264),
                                  ("tri_mul", 33), ("tri_mul", 77)])
def test_results_do_not_depend_on_workspace_contents(dname, op, N):
    dt = torch.bfloat16 if dname == "bf16" else torch.float32
    if op == "tri_attn":
        mod = triattn_module(H.draw_params(H.tri_attn_shapes(128, 32, 4), seed=3, bias_random=True), True, 4, dt)
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
