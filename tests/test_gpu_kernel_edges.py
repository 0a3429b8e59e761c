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


@requires_gpu
@pytest.mark.parametrize("quant", ["none", "nf4"])
@pytest.mark.parametrize(
    "counts,k_in,n_out",
    [
        ([1], 64, 128),  # one row, half a tile of columns
        ([0, 32, 33, 0, 5], 128, 384),  # empty experts; a whole tile and one row more
        ([128, 129, 127, 31], 192, 256),  # around a group of 128 rows
        ([300, 0, 1, 256], 64, 640),  # several groups of one expert
        ([3] * 70, 64, 128),  # more tiles than lanes of a wave
        ([2050, 40], 64, 128),  # a run of one expert longer than a wave's lanes
    ],
)
def test_expert_gemm_group_edges(hip, quant, counts, k_in, n_out):
    from petals_amd.ops.fused_moe import _StackedExperts, sort_pairs_by_expert

    gen = torch.Generator(device="cuda").manual_seed(sum(counts) + n_out)
    experts = len(counts)
    weights = [
        (torch.randn(k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16) for _ in range(experts)
    ]
    st = _StackedExperts(weights, hip, quant)
    sel = torch.cat([torch.full((n,), e, device="cuda") for e, n in enumerate(counts)])
    sel = sel[torch.randperm(len(sel), device="cuda", generator=gen)].view(-1, 1)
    x = torch.randn(len(sel), k_in, device="cuda", generator=gen).to(BF16)
    order, tiles = sort_pairs_by_expert(sel, experts)
    out = st.moe_gemm(x, order, tiles, 1, len(sel)).double()
    for e in range(experts):
        rows = torch.where(sel[:, 0] == e)[0]
        if len(rows):
            xe, we = x[rows].double(), st.dense(e).double()
            ref = xe @ we
            # 32-bit sums of exact products of bf16, rounded once
            bound = 2.0**-8 * ref.abs() + k_in * 2.0**-24 * (xe.abs() @ we.abs())
            assert bool(((out[rows] - ref).abs() <= bound).all()), e
