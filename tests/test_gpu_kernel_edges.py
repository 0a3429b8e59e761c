"""HIP kernels at the sizes where their tiles, splits and rules of dispatch change,
against plain 32-bit or 64-bit references."""

import pytest
import torch

pytestmark = pytest.mark.gpu

requires_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs MI355X")
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def hip():
    from petals_amd import ops

    mod = ops._load_hip_ops()
    assert mod is not None, f"HIP extension must load on a GPU box: {ops._hip_import_error!r}"
    return mod


@requires_gpu
@pytest.mark.parametrize("n", [1, 7, 2047, 2048, 2049, 600 * 14336])
def test_swiglu_writes_every_value(hip, n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    gate, up = (torch.randn(n, device="cuda", generator=gen).to(BF16) for _ in range(2))
    ref = torch.nn.functional.silu(gate.float()) * up.float()
    err = (hip.swiglu(gate, up).float() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-6).all())  # one rounding to bf16
