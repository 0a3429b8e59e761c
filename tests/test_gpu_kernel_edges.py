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


NF4_LEVELS = torch.tensor([
    -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
    -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
    0.24611230194568634, 0.33791524171829224, 0.4407098293304443, 0.5626170039176941, 0.7229568362236023, 1.0,
])  # fmt: skip


def nf4_weights(hip, k_in, n_out, gen):
    """(tiles, scales), the weights that they hold in 64 bits [in, out], scales [in, out]"""
    w = (torch.randn(k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16)
    packed, absmax = hip.nf4_quantize(w)
    codes = torch.stack([packed & 15, packed >> 4], dim=-1).view(k_in, n_out).long()
    scale = absmax.double().repeat_interleave(64, dim=1)
    return hip.nf4_tile(packed, absmax), NF4_LEVELS.cuda().double()[codes] * scale, scale


@requires_gpu
@pytest.mark.parametrize("batch", range(1, 9))
@pytest.mark.parametrize(
    "k_in,n_out", [(1, 64), (64, 64), (127, 192), (129, 64), (513, 128), (1030, 64), (2048, 64), (4544, 192), (8192, 8192)]
)
def test_nf4_tiles_against_64_bits(hip, k_in, n_out, batch):
    gen = torch.Generator(device="cuda").manual_seed(k_in * 8 + batch)
    (tiles, scales), w, scale = nf4_weights(hip, k_in, n_out, gen)
    assert torch.equal(hip.nf4_untile(tiles, scales, k_in), w.to(torch.float32).to(BF16))
    x = torch.randn(batch, k_in, device="cuda", generator=gen)
    x[:, :: max(1, k_in // 5)] *= 50.0  # loud channels
    x[batch // 2] *= 1e-30
    if batch > 2:
        x[1] = 0.0
        x[2] *= 1e30
    y = hip.gemv_nf4_tiles(tiles, scales, k_in, x, torch.empty(0, device="cuda"), None, 0).double()
    xd = x.double()
    # levels are off by 2.4e-8 at most, inputs by 2^-31 of the largest (but not by less than
    # 2^-127), and 2^3 roundings follow
    bound = (xd.abs() @ scale) * 2.4e-8 + 2.0**-21 * (xd.abs() @ w.abs())
    bound += k_in * (2.0**-31 * xd.abs().amax(1, keepdim=True) * scale.amax() + 2.0**-127)
    assert bool(((y - xd @ w).abs() <= bound + 1e-38).all())


@requires_gpu
@pytest.mark.parametrize("batch", [1, 3, 8])
def test_nf4_tiles_infinities(hip, batch):
    gen = torch.Generator(device="cuda").manual_seed(batch)
    (tiles, scales), w, _ = nf4_weights(hip, 1100, 64, gen)
    x = torch.randn(batch, 1100, device="cuda", generator=gen)
    x[0, 700], x[batch - 1, 3], x[batch // 2, 1099] = float("inf"), float("-inf"), float("nan")
    y = hip.gemv_nf4_tiles(tiles, scales, 1100, x, torch.empty(0, device="cuda"), None, 0).cpu()
    ref = torch.stack([(row[:, None] * w.float()).sum(0) for row in x]).cpu()  # products of zeros too
    odd = ~torch.isfinite(ref)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(y[odd & ~torch.isnan(ref)], ref[odd & ~torch.isnan(ref)])
    assert torch.allclose(y[~odd], ref[~odd], atol=1e-4, rtol=1e-4)


@requires_gpu
@pytest.mark.parametrize("experts,tokens,top,k_in,n_out", [(8, 1, 2, 256, 128), (3, 5, 3, 1100, 64), (8, 8, 2, 4096, 4096)])
def test_nf4_tiles_of_experts(hip, experts, tokens, top, k_in, n_out):
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    made = [nf4_weights(hip, k_in, n_out, gen) for _ in range(experts)]
    tiles, scales = (torch.stack([m[0][i] for m in made]) for i in range(2))
    sel = torch.randint(0, experts, (tokens * top,), device="cuda", generator=gen, dtype=torch.int32)
    x = torch.randn(tokens, k_in, device="cuda", generator=gen)
    y = hip.gemv_nf4_tiles_moe(tiles, scales, k_in, x, sel, top, torch.empty(0, device="cuda"), 0).double()
    for r, e in enumerate(sel.tolist()):
        xd, w, scale = x[r // top].double(), made[e][1], made[e][2]
        bound = (xd.abs() @ scale) * 2.4e-8 + 2.0**-21 * (xd.abs() @ w.abs())
        assert bool(((y[r] - xd @ w).abs() <= bound + k_in * 2.0**-31 * xd.abs().max() * scale.amax()).all())


def sum_bound(xd, w):
    """Sums of exact products in 32 bits: three for each of 32 inputs, and a few at the end."""
    return (3 * (xd.shape[-1] // 32 + 1) + 16) * 2.0**-24 * (xd.abs() @ w.abs())


@requires_gpu
@pytest.mark.parametrize("batch", [1, 2, 5, 8])
@pytest.mark.parametrize(
    "k_in,n_out",
    [(1, 8), (7, 128), (32, 120), (33, 136), (127, 1000), (130, 129), (512, 8), (513, 264), (2048, 2560), (4544, 65024), (300, 12)],
)
def test_gemv_against_64_bits(hip, k_in, n_out, batch):
    gen = torch.Generator(device="cuda").manual_seed(k_in * 8 + batch)
    w = torch.randn(k_in, n_out, device="cuda", generator=gen).to(BF16)
    x = torch.randn(batch, k_in, device="cuda", generator=gen)
    x[:, :: max(1, k_in // 5)] *= 50.0
    x[batch // 2] *= 1e-20
    y = hip.gemv_bf16(w, x, torch.empty(0, device="cuda"), None, 0)
    assert bool(((y.double() - x.double() @ w.double()).abs() <= sum_bound(x.double(), w.double())).all())
    parts = hip.gemv_bf16(w, x, torch.empty(0, device="cuda"), None, -1)
    assert bool(((parts.double().sum(0) - x.double() @ w.double()).abs() <= sum_bound(x.double(), w.double())).all())


@requires_gpu
def test_gemv_infinities(hip):
    gen = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randn(200, 136, device="cuda", generator=gen).to(BF16)
    w[w.abs() < 0.05] = 0.0
    x = torch.randn(3, 200, device="cuda", generator=gen)
    x[0, 100], x[1, 5] = float("inf"), float("nan")
    y = hip.gemv_bf16(w, x, torch.empty(0, device="cuda"), None, 0).cpu()
    ref = torch.stack([(row[:, None] * w.float()).sum(0) for row in x]).cpu()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.isfinite(y[2]).all()
    odd = torch.isinf(ref)
    assert odd.any() and torch.equal(y[odd], ref[odd])


@requires_gpu
@pytest.mark.parametrize("tokens,top,k_in,n_out", [(1, 2, 96, 136), (8, 2, 2048, 4096), (16, 4, 40, 24), (2, 1, 64, 12)])
def test_gemv_of_experts(hip, tokens, top, k_in, n_out):
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    w = torch.randn(5, k_in, n_out, device="cuda", generator=gen).to(BF16)
    sel = torch.randint(0, 5, (tokens * top,), device="cuda", generator=gen, dtype=torch.int32)
    x = torch.randn(tokens, k_in, device="cuda", generator=gen)
    y = hip.gemv_bf16_moe(w, x, sel, top, torch.empty(0, device="cuda"), 0).double()
    for r, e in enumerate(sel.tolist()):
        xd, wd = x[r // top].double(), w[e].double()
        assert bool(((y[r] - xd @ wd).abs() <= sum_bound(xd, wd)).all())
