"""The experts that a Mixtral block's forward pass runs are those that its gradients go through."""

import pytest
import torch

from petals_amd.ops.fused_moe import MixtralFastPath

BF16 = torch.bfloat16


def router(device, width=4096, experts=8, top=2, tokens=4096):
    gen = torch.Generator().manual_seed(0)
    fast = MixtralFastPath.__new__(MixtralFastPath)
    fast.top_k, fast.num_experts, fast.hip = top, experts, None
    fast.w_router = (torch.randn(experts, width, generator=gen) * 0.02).to(BF16).to(device)
    fast.w_router_t = fast.w_router.t()
    return fast, torch.randn(tokens, width, generator=gen).to(BF16).to(device)


def test_router_keeps_32_bits():
    fast, x = router("cpu")
    weights, chosen = fast._route(x)
    logits = x.double() @ fast.w_router.double().t()
    best, want = torch.topk(logits, 2, dim=-1)
    assert torch.equal(chosen, want)
    assert (weights.double() - torch.softmax(best, -1)).abs().max() < 1e-5  # 32-bit sums of 4096 terms


def test_router_gradients():
    fast, x = router("cpu", width=64, experts=5, top=3, tokens=7)
    x, g = x.float().requires_grad_(True), torch.randn(7, 3, generator=torch.Generator().manual_seed(1))
    (got,) = torch.autograd.grad(fast._route(x)[0], x, g)
    z = x.detach().double().requires_grad_(True)
    share = torch.topk(torch.softmax(z @ fast.w_router.double().t(), -1), 3, dim=-1)[0]
    (want,) = torch.autograd.grad(share / share.sum(-1, keepdim=True), z, g.double())
    assert (got - want).norm() <= 1e-5 * want.norm()


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs MI355X")
@pytest.mark.parametrize("dtype", [BF16, torch.float32])
def test_training_chooses_as_inference(dtype):
    from petals_amd import ops

    fast, x = router("cuda")
    fast.hip = ops._load_hip_ops()
    x = x.to(dtype)
    x[::2] = (x[::2].float() * (1 + 2.0**-9)).to(dtype)
    # experts in pairs that differ in one weight's last place: near-ties, decided by order of summation
    fast.w_router[1::2] = fast.w_router[::2]
    fast.w_router[1::2, 5] *= 1 + 2.0**-7
    weights, chosen = fast._route_rows(x)
    trained, want = fast._route(x.requires_grad_(True))
    assert torch.equal(chosen.long(), want)
    assert (weights - trained.detach()).abs().max() < 1e-5
