"""HIP kernels at the sizes where their tiles, splits and rules of dispatch change,
against plain 32-bit or 64-bit references."""

import dataclasses

import pytest
import torch

from expert_pairs import sort_pairs_by_expert

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
        ([1100, 40], 192, 2304),  # more groups than share a run of columns, several runs
    ],
)
def test_expert_gemm_group_edges(hip, quant, counts, k_in, n_out):
    from petals_amd.ops.fused_moe import MOE_GEMM_MT, _StackedExperts

    gen = torch.Generator(device="cuda").manual_seed(sum(counts) + n_out)
    experts = len(counts)
    weights = [
        (torch.randn(k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16) for _ in range(experts)
    ]
    st = _StackedExperts(weights, hip, quant)
    sel = torch.cat([torch.full((n,), e, device="cuda") for e, n in enumerate(counts)])
    sel = sel[torch.randperm(len(sel), device="cuda", generator=gen)].view(-1, 1)
    x = torch.randn(len(sel), k_in, device="cuda", generator=gen).to(BF16)
    order, tiles = sort_pairs_by_expert(sel, experts, MOE_GEMM_MT)
    out = st.moe_gemm(x, order, tiles, 1, len(sel))
    # by the kernel that prompts use, which leaves fewer unused tiles
    order, tiles = hip.moe_group(sel.view(-1).to(torch.int32), experts, MOE_GEMM_MT)
    assert torch.equal(st.moe_gemm(x, order, tiles, 1, len(sel)), out)
    out = out.double()
    for e in range(experts):
        rows = torch.where(sel[:, 0] == e)[0]
        if len(rows):
            xe, we = x[rows].double(), st.dense(e).double()
            ref = xe @ we
            # 32-bit sums of exact products of bf16, rounded once
            bound = 2.0**-8 * ref.abs() + k_in * 2.0**-24 * (xe.abs() @ we.abs())
            assert bool(((out[rows] - ref).abs() <= bound).all()), e


@requires_gpu
@pytest.mark.parametrize(
    "counts,k_in,n_out",
    [
        ([1, 33, 65, 97, 129, 161, 193, 225], 64, 384),  # groups of 1 to 8 tiles, of one row more than the tile before
        ([256, 257, 0, 480, 512, 513], 128, 256),  # around one and two full groups, an empty expert between
        ([290] * 8, 192, 4096),  # smaller groups, as few columns are
        ([40, 0, 700, 31] * 20, 64, 2176),  # runs that end in another chunk of tiles than they start in
        ([3000], 256, 128),  # a run of one expert longer than a wave's lanes
        ([5, 40, 96, 128, 0, 1], 128, 640),  # few rows and columns: runs of 128 columns, groups of 1 to 4 tiles
        ([200, 3, 3, 3], 64, 128),  # the same, one expert with more rows than a group
    ],
)
def test_expert_gemm_equal_groups(hip, counts, k_in, n_out):
    """Rows of an expert in groups that are as equal as tiles of 32 allow, two rows a token."""
    from petals_amd.ops.fused_moe import MOE_GEMM_MT

    gen = torch.Generator(device="cuda").manual_seed(len(counts) + n_out)
    w = (torch.randn(len(counts), k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16)
    pairs = torch.cat([torch.full((n,), e, device="cuda", dtype=torch.int32) for e, n in enumerate(counts)])
    pairs = pairs[torch.randperm(len(pairs), device="cuda", generator=gen)]
    x = torch.randn((len(pairs) + 1) // 2, k_in, device="cuda", generator=gen).to(BF16)
    order, tiles = hip.moe_group(pairs, len(counts), MOE_GEMM_MT)
    out = hip.moe_gemm(w, None, None, x, order, tiles, 2, len(pairs)).double()
    rows = x.double().repeat_interleave(2, 0)[: len(pairs)]
    for e in range(len(counts)):
        mine, we = pairs == e, w[e].double()
        ref = rows[mine] @ we
        # 32-bit sums of exact products of bf16, rounded once
        loose = k_in * 2.0**-24 * (rows[mine].abs() @ we.abs())
        assert bool(((out[mine] - ref).abs() <= 2.0**-8 * ref.abs() + loose).all()), e


@requires_gpu
@pytest.mark.parametrize(
    "counts,k_in,n_out",
    [([1], 64, 128), ([0, 32, 33, 0, 5], 128, 384), ([128, 129, 127, 31], 192, 256), ([2050, 40], 64, 128), ([1100, 40], 192, 2304)],
)
def test_expert_gemm_without_limits(hip, counts, k_in, n_out):
    """The kernel that experts beyond offsets of 32 bits have, which no test is large enough for."""
    from petals_amd.ops.fused_moe import MOE_GEMM_MT

    gen = torch.Generator(device="cuda").manual_seed(sum(counts))
    w = (torch.randn(len(counts), k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16)
    pairs = torch.cat([torch.full((n,), e, device="cuda", dtype=torch.int32) for e, n in enumerate(counts)])
    pairs = pairs[torch.randperm(len(pairs), device="cuda", generator=gen)]
    x = torch.randn(len(pairs), k_in, device="cuda", generator=gen).to(BF16)
    order, tiles = hip.moe_group(pairs, len(counts), MOE_GEMM_MT)
    out = hip.moe_gemm(w, None, None, x, order, tiles, 1, len(pairs), general=True).double()
    for e in range(len(counts)):
        mine, we = pairs == e, w[e].double()
        ref = x[mine].double() @ we
        # 32-bit sums of exact products of bf16, rounded once
        loose = k_in * 2.0**-24 * (x[mine].double().abs() @ we.abs())
        assert bool(((out[mine] - ref).abs() <= 2.0**-8 * ref.abs() + loose).all()), e


@requires_gpu
def test_gelu_over_all_of_bf16(hip):
    """GELU of every finite bf16 number, infinities and NaN, beside 64 bits."""
    x = torch.arange(1 << 16, device="cuda", dtype=torch.int32).to(torch.int16).view(BF16)
    y = x.clone().view(-1, 1024)
    hip.bias_gelu_rows(y, None)
    y, xd = y.flatten().double(), x.double()
    u = (2 / torch.pi) ** 0.5 * (xd + 0.044715 * xd**3)
    want = torch.where(xd > 0, xd / (1 + torch.exp(-2 * u)), xd * torch.exp(2 * u) / (1 + torch.exp(2 * u)))
    small = xd.abs() <= 2.0**20
    # one rounding to bf16, whose 8 bits are good to 2^-8; 32-bit: 2u has an error of 2^-22 of itself, which is that of a small exponential, flushed below 2^-126
    slack = want.abs() * (2.0**-8 + 2.0**-22 * (2 + 2 * u.abs())) + 2.0**-125 * xd.abs().clamp(min=1.0)
    assert bool(((y - want).abs() <= slack)[small].all())
    large = xd.isfinite() & ~small
    assert torch.equal(y[large & (xd > 0)], xd[large & (xd > 0)]) and not y[large & (xd < 0)].any()
    assert y[xd == float("inf")].isposinf().all()
    assert y[xd.isnan() | (xd == float("-inf"))].isnan().all()  # 0 times infinity


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
    assert bool(((y - xd @ w).abs() <= nf4_bound(xd, w, scale)).all())


def nf4_bound(xd, w, scale):
    """Scaled inputs are rounded to 2^-20 of their run's mean, large ones clipped, or finer (but not
    below 2^-126), levels are off by 9.4e-8 of themselves, and 2^3 roundings follow."""
    return 2.0**-21 * (xd.abs() @ scale) + 2.0**-20 * (xd.abs() @ w.abs()) + xd.shape[-1] * 2.0**-126


@requires_gpu
@pytest.mark.parametrize("batch", range(1, 9))
@pytest.mark.parametrize("loud", [[30.0], [1e4], [1e10], [1e20], [1e3, 1e6, 1e9], [1e2, 1e15, 1e30]])
def test_nf4_tiles_of_a_wide_range(hip, batch, loud):
    """A few inputs that dwarf the rest cost it nothing where they meet a weight of zero."""
    k_in, n_out = 1030, 128
    gen = torch.Generator(device="cuda").manual_seed(batch)
    w = (torch.randn(k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16)
    at = torch.tensor([0, 127, 128, 300, 400, 500, 511, 512, 600, 700, 1029], device="cuda")
    w[at, ::2] = 0.0
    packed, absmax = hip.nf4_quantize(w)
    codes = torch.stack([packed & 15, packed >> 4], dim=-1).view(k_in, n_out).long()
    scale = absmax.double().repeat_interleave(64, dim=1)
    held = NF4_LEVELS.cuda().double()[codes] * scale
    assert not held[at, ::2].any()
    x = torch.randn(batch, k_in, device="cuda", generator=gen)
    for b in range(batch):
        for i, k in enumerate(at.tolist()):
            if (i + b) % 4 or b == batch // 2:  # all of one row
                x[b, k] = loud[i % len(loud)]
    if batch > 3:
        x[0, ::2] = 0.0
        x[3, 5:-5] = 0.0
    y = hip.gemv_nf4_tiles(*hip.nf4_tile(packed, absmax), k_in, x, torch.empty(0, device="cuda"), None, 0).double()
    xd, quiet = x.double(), x.double()
    quiet[:, at] = 0.0
    error = (y - xd @ held).abs()
    assert bool((error[:, ::2] <= nf4_bound(quiet, held, scale)[:, ::2]).all())
    assert bool((error <= nf4_bound(xd, held, scale)).all())


@requires_gpu
@pytest.mark.parametrize("batch", range(5, 9))
@pytest.mark.parametrize(
    "k_in,n_out,parts",
    [
        (4440, 18176, 3),  # two steps of 256 inputs; the last run has 3 of 4 tiles, the three after it none
        (4440, 29184, 2),  # four steps; the last run's second one is half there
        (4097, 32768, 2),  # four steps; one input in the last run
    ],
)
@pytest.mark.parametrize("loud", [[50.0], [1e4, 1e9]])
def test_nf4_tiles_of_long_runs(hip, batch, k_in, n_out, parts, loud):
    """Runs of several steps, which end within one: loud inputs in each step cost the quiet ones nothing
    where they meet a weight of zero."""
    gen = torch.Generator(device="cuda").manual_seed(k_in + n_out + batch)
    w = (torch.randn(k_in, 192, device="cuda", generator=gen) * 0.05).to(BF16)
    at = torch.tensor([*range(17, k_in, 251), k_in - 1], device="cuda")
    w[at, ::2] = 0.0
    packed, absmax = hip.nf4_quantize(w)
    scale = absmax.double().repeat_interleave(64, dim=1)
    held = NF4_LEVELS.cuda().double()[torch.stack([packed & 15, packed >> 4], dim=-1).view(k_in, 192).long()] * scale
    which = torch.randint(0, 3, (n_out // 64,), device="cuda", generator=gen)  # each run of 64 columns one of three
    tiles, scales = (t[which].contiguous() for t in hip.nf4_tile(packed, absmax))
    x = torch.randn(batch, k_in, device="cuda", generator=gen)
    for i, k in enumerate(at.tolist()):
        x[i % batch, k] = loud[i % len(loud)]
    empty = torch.empty(0, device="cuda")
    assert hip.gemv_nf4_tiles(tiles, scales, k_in, x, empty, None, -1).shape[0] == parts
    y = hip.gemv_nf4_tiles(tiles, scales, k_in, x, empty, None, 0).double().view(batch, -1, 64)
    xd, quiet = x.double(), x.double()
    quiet[:, at] = 0.0
    want, bound, still = ((v.view(batch, 3, 64)[:, which]) for v in (xd @ held, nf4_bound(xd, held, scale), nf4_bound(quiet, held, scale)))
    error = (y - want).abs()
    assert bool((error <= bound).all())
    if loud[0] > 100:  # beyond what digits hold; 50 times the mean is not, and takes the others' last places
        assert bool((error[..., ::2] <= still[..., ::2]).all())


@requires_gpu
@pytest.mark.parametrize("batch", [1, 5])
def test_nf4_tiles_of_many_inputs(hip, batch):
    """2^30 bytes of codes for a run of columns and more: inputs at both ends and around 2^29 and 2^30 bytes count."""
    n_kb = (1 << 18) + 5
    k_in = n_kb * 128 - 84
    gen = torch.Generator(device="cuda").manual_seed(batch)
    tiles = torch.zeros(1, n_kb, 4, 64, 16, device="cuda", dtype=torch.uint8)
    scales = torch.zeros(1, n_kb * 128, device="cuda", dtype=BF16)
    x = torch.zeros(batch, k_in, device="cuda")
    want = bound = 0.0
    for at in (0, (1 << 17) - 2, (1 << 18) - 2, n_kb - 2):
        size = min(512, k_in - at * 128)
        (t, s), w, scale = nf4_weights(hip, size, 64, gen)
        tiles[:, at : at + t.shape[1]], scales[:, at * 128 : at * 128 + s.shape[1]] = t, s
        x[:, at * 128 : at * 128 + size] = torch.randn(batch, size, device="cuda", generator=gen)
        xd = x[:, at * 128 : at * 128 + size].double()
        want, bound = want + xd @ w, bound + nf4_bound(xd, w, scale)
    y = hip.gemv_nf4_tiles(tiles, scales, k_in, x, torch.empty(0, device="cuda"), None, 0).double()
    assert bool(((y - want).abs() <= bound).all()) and bool((want.abs() > 100 * bound).any())


@requires_gpu
@pytest.mark.parametrize("batch", [1, 5])
def test_nf4_tiles_of_the_largest_numbers(hip, batch):
    """An input that overflows with its block's scale is multiplied by its weight, which may be zero."""
    gen = torch.Generator(device="cuda").manual_seed(batch)
    w = torch.randn(300, 64, device="cuda", generator=gen).to(BF16)
    w[7] = torch.tensor([0.0, 0.08 * 64, 64.0, 0.0] * 16, device="cuda").to(BF16)
    packed, absmax = hip.nf4_quantize(w)
    held = NF4_LEVELS.cuda().double()[torch.stack([packed & 15, packed >> 4], dim=-1).view(300, 64).long()]
    held = held * absmax.double().repeat_interleave(64, dim=1)
    x = torch.randn(batch, 300, device="cuda", generator=gen)
    x[0, 7] = 2e37  # times 64, beyond 32-bit floats; times 5, not
    y = hip.gemv_nf4_tiles(*hip.nf4_tile(packed, absmax), 300, x, torch.empty(0, device="cuda"), None, 0)
    ref = x.double() @ held
    assert bool(torch.isinf(y[0, 2::4]).all())
    y[0, 2::4] = ref[0, 2::4] = 0.0
    quiet = x.double()
    quiet[0, 7] = 0.0
    bound = nf4_bound(quiet, held, absmax.double().repeat_interleave(64, dim=1)) + 2.0**-20 * (x.double() * 64).abs().amax(1, keepdim=True) * (held[7] != 0)
    assert bool(((y.double() - ref).abs() <= bound).all())


@requires_gpu
@pytest.mark.parametrize("batch", [4, 8])
def test_nf4_tiles_round_inputs(hip, batch):
    """Errors of a sum of like terms cancel: scaled inputs are rounded, not cut off."""
    k_in = 8192
    gen = torch.Generator(device="cuda").manual_seed(batch)
    w = torch.ones(k_in, 64, device="cuda", dtype=BF16)
    w[::256, ::2] = 0.0
    x = torch.rand(batch, k_in, device="cuda", generator=gen) + 1.0
    x[:, ::256] = 1e6  # in every run: the others are then held to 2^-21 or 2^-20
    made = hip.nf4_tile(*hip.nf4_quantize(w))
    y = hip.gemv_nf4_tiles(*made, k_in, x, torch.empty(0, device="cuda"), None, 0).double()
    error = (y - x.double() @ w.double())[:, ::2]  # without the large ones
    # cut off, 2^-22 an input or more; rounded, the 32-bit sums' errors of 2^-11 now and then
    assert abs(float(error.mean())) <= 0.5 * k_in * 2.0**-22


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
        assert bool(((y[r] - xd @ w).abs() <= nf4_bound(xd, w, scale)).all())


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
@pytest.mark.parametrize("splits", [1, 3, 8])
def test_gemv_in_as_many_parts_as_asked_for(hip, splits):
    gen = torch.Generator(device="cuda").manual_seed(splits)
    k_in, n_out = 768, 256
    w = torch.randn(2, k_in, n_out, device="cuda", generator=gen).to(BF16)
    x = torch.randn(3, k_in, device="cuda", generator=gen)
    empty, sel = torch.empty(0, device="cuda"), torch.tensor([1, 0, 1], dtype=torch.int32, device="cuda")
    parts = hip.gemv_bf16(w[0], x, empty, None, -1, splits)
    assert parts.shape == (splits, 3, n_out)
    ref = x.double() @ w[0].double()
    bound = k_in * 2.0**-24 * (x.double().abs() @ w[0].double().abs())  # 32-bit sums in any order
    assert bool(((parts.double().sum(0) - ref).abs() <= bound).all())
    # experts' parts have 256 inputs or more
    assert hip.gemv_bf16_moe(w, x, sel, 1, empty, -1, splits).shape == (min(splits, 3), 3, n_out)


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


def attention_64(q, k, v, offset, scale, causal, slopes):
    """(result, weights @ |v|) of [B, H, S, hd] over [B, G, L, hd], 64 bits"""
    group = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double().repeat_interleave(group, 1), v.double().repeat_interleave(group, 1)
    at = torch.arange(k.shape[2], device="cuda")
    score = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    if slopes is not None:
        score = score + slopes.double()[:, None, None] * at
    if causal:
        score = score.masked_fill(at > torch.arange(offset, offset + q.shape[2], device="cuda")[:, None], float("-inf"))
    p = torch.softmax(score, dim=-1)
    return torch.matmul(p, v), torch.matmul(p, v.abs())


@requires_gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize(
    "b,qh,kh,s,offset,causal,alibi",
    [
        (1, 1, 1, 1, 0, True, False), (1, 2, 1, 15, 0, True, True), (2, 4, 2, 64, 0, True, False),
        (1, 8, 8, 65, 7, True, True), (3, 6, 1, 130, 63, True, False), (1, 4, 4, 17, 200, True, False),
        (2, 3, 3, 33, 31, False, True), (4, 128, 8, 129, 0, True, False), (2, 71, 1, 300, 100, True, False),
        (8, 64, 64, 127, 1, False, True),
    ],
)  # fmt: skip
def test_prompt_attention_edges(hip, hd, b, qh, kh, s, offset, causal, alibi):
    gen = torch.Generator(device="cuda").manual_seed(qh * s + hd)

    def made(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(BF16)

    length = offset + s
    k, v = (made(b + 1, kh, length + 5, hd) for _ in range(2))
    slopes = torch.rand(qh, device="cuda", generator=gen) * 0.1 if alibi else None
    rows = made(b, s, qh + 2, hd)  # queries among other columns
    q = rows.transpose(1, 2)[:, 1 : 1 + qh]
    ref, bound = attention_64(q, k[:b, :, :length], v[:b, :, :length], offset, hd**-0.5, causal, slopes)
    bound = 2.0**-7 * bound + 1e-5  # weights and results are rounded to bf16, by up to 2^-8 each
    out = hip.attn_prefill_rows(q, k[:b], v[:b], length, offset, hd**-0.5, causal, slopes)
    assert out.shape == (b, s, qh * hd)
    assert bool(((out.view(b, s, qh, hd).transpose(1, 2).double() - ref).abs() <= bound).all())
    fused = hip.attn_prefill_fused(
        q.contiguous(), k[:b].contiguous(), v[:b].contiguous(), length, offset, hd**-0.5, causal, slopes
    )
    assert torch.equal(fused.transpose(1, 2).reshape(b, s, qh * hd), out)


@requires_gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("length", [63, 64, 65])
@pytest.mark.parametrize("step", ["0", "8", "half", "wide"])
def test_prompt_attention_strides(hip, hd, length, step):
    """Keys and values whose rows overlap, are one row or lie far apart are read like their copies."""
    gen = torch.Generator(device="cuda").manual_seed(hd + length)
    row = {"0": 0, "8": 8, "half": hd // 2, "wide": 1 << 17}[step]
    store = torch.randn(2 * (row * length + hd), device="cuda", generator=gen).to(BF16)
    k = store.as_strided((1, 2, length, hd), (store.numel(), store.numel() // 2, row, 1))
    v = store.flip(0).as_strided(k.shape, k.stride())
    q = torch.randn(1, 4, length, hd, device="cuda", generator=gen).to(BF16)
    out = hip.attn_prefill_rows(q, k, v, length, 0, hd**-0.5, True, None)
    k, v = (t.clone(memory_format=torch.contiguous_format) for t in (k, v))
    assert torch.equal(out, hip.attn_prefill_rows(q, k, v, length, 0, hd**-0.5, True, None))


@requires_gpu
@pytest.mark.parametrize("hd,qh,kh,s,start", [(64, 3, 1, 1, 0), (128, 4, 2, 33, 5), (64, 2, 2, 70, 130)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("turns", [False, True])
@pytest.mark.parametrize("cached", [False, True])
def test_qkv_rows(hip, hd, qh, kh, s, start, bias, turns, cached):
    from petals_amd.ops import reference

    gen = torch.Generator(device="cuda").manual_seed(s)
    b, width = 2, (qh + 2 * kh) * hd
    qkv = torch.randn(b, s, width, device="cuda", generator=gen).to(BF16)
    c = torch.randn(width, device="cuda", generator=gen).to(BF16) if bias else None
    cos, sin = (t.cuda() for t in reference.build_rope_cache(hd, start + s))
    ref = (qkv.float() + (0.0 if c is None else c.float())).view(b, s, -1, hd).transpose(1, 2)
    if turns:
        pos = torch.arange(start, start + s, device="cuda")
        q, k = reference.apply_rope(ref[:, :qh], ref[:, qh : qh + kh], cos, sin, pos)
        ref = torch.cat([q, k, ref[:, qh + kh :]], dim=1)
    ref = ref.to(BF16)
    caches = [torch.zeros(b + 1, kh, start + s + 3, hd, device="cuda", dtype=BF16) for _ in range(2)]
    args = caches if cached else (None, None)
    hip.qkv_rows(qkv, c, *((cos, sin) if turns else (None, None)), *args, start, qh, kh, hd)
    got = qkv.view(b, s, -1, hd).transpose(1, 2)

    def same(a, r):  # products and sums may be contracted: one unit in the last place
        assert bool(((a.float() - r.float()).abs() <= 2.0**-7 * r.float().abs() + 1e-6).all())

    same(got[:, :qh], ref[:, :qh])
    if cached:
        for t, lo in zip(caches, (qh, qh + kh)):
            same(t[:b, :, start : start + s], ref[:, lo : lo + kh])
            assert not t[b].any() and not t[:, :, :start].any() and not t[:, :, start + s :].any()
    else:
        same(got, ref)


@requires_gpu
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 2048), (5, 2056), (130, 4544), (2, 16384)])
def test_rows_between_products(hip, rows, width):
    gen = torch.Generator(device="cuda").manual_seed(width)
    x, y, z = (torch.randn(rows, width, device="cuda", generator=gen).to(BF16) for _ in range(3))
    c, w, b = (torch.randn(width, device="cuda", generator=gen).to(BF16) for _ in range(3))
    fn = torch.nn.functional

    def close(a, r):
        assert bool(((a.double() - r).abs() <= 2.0**-8 * r.abs() + 1e-4).all())

    close(hip.add_rows(x, y), x.double() + y.double())
    close(hip.add_rows(x, y, z, c), x.double() + y.double() + z.double() + c.double())
    for bias, layer in ((None, False), (c, False), (c, True)):
        h, n = hip.add_norm_rows(x, y, bias, w, b if layer else None, 1e-5)
        close(h, x.double() + y.double() + (0.0 if bias is None else c.double()))
        hd = h.double()
        if layer:
            close(n, fn.layer_norm(hd, (width,), w.double(), b.double(), 1e-5))
        else:
            close(n, hd * torch.rsqrt(hd.square().mean(-1, keepdim=True) + 1e-5) * w.double())
    both = torch.cat([x, y], dim=-1)
    close(hip.swiglu_rows(both), fn.silu(x.double()) * y.double())
    for bias in (None, c):
        t = x.clone()
        hip.bias_gelu_rows(t, bias)
        close(t, fn.gelu(x.double() + (0.0 if bias is None else c.double()), approximate="tanh"))


@requires_gpu
@pytest.mark.parametrize("width", [20, 4100, 16384, 16392])
@pytest.mark.parametrize("biased", [False, True])
def test_rows_of_any_width(hip, width, biased):
    """Shards of uneven sizes, and rows that are too long for a norm's registers."""
    from petals_amd.ops.fused_decode import add_norm, bias_gelu

    gen = torch.Generator(device="cuda").manual_seed(width)
    x, y = (torch.randn(3, width, device="cuda", generator=gen).to(BF16) for _ in range(2))
    c, w, b = (torch.randn(width, device="cuda", generator=gen).to(BF16) for _ in range(3))
    fn, c = torch.nn.functional, c if biased else None
    total = y.double() + (0.0 if c is None else c.double())
    got = bias_gelu(hip, y.clone(), c)
    want = fn.gelu(total, approximate="tanh")
    # a sum and a result rounded to bf16; the function's slope is 1.13 at most
    assert bool(((got.double() - want).abs() <= 2.0**-8 * (want.abs() + 1.2 * total.abs()) + 1e-4).all())
    for layer in (None, b):
        h, n = add_norm(hip, x, y, c, w, layer, 1e-5)
        assert bool(((h.double() - x.double() - total).abs() <= 2.0**-8 * (h.double().abs() + total.abs())).all())
        hd = h.double()
        if layer is None:
            want = hd * torch.rsqrt(hd.square().mean(-1, keepdim=True) + 1e-5) * w.double()
        else:
            want = fn.layer_norm(hd, (width,), w.double(), b.double(), 1e-5)
        assert bool(((n.double() - want).abs() <= 2.0**-8 * want.abs() + 1e-4).all())


@requires_gpu
@pytest.mark.parametrize("tokens,limit", [(37, 1 << 28), (300, 1 << 18), (300, 1)])
def test_prompt_chunks_are_one_prompt(hip, tokens, limit):
    """However a prompt is cut, its outputs and its cache are the same."""
    from petals_amd.models.config_base import load_model_config
    from petals_amd.server.backend import TransformerBackend
    from petals_amd.server.from_pretrained import load_pretrained_block

    config = load_model_config("test-llama-hd128")
    block = load_pretrained_block("test-llama-hd128", config, 0, torch_dtype=BF16, device=torch.device("cuda"))
    backend = TransformerBackend("b", block, config=config, memory_cache=None, dtype=BF16, max_chunk_size_bytes=limit)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(2, tokens, config.hidden_size, device="cuda", generator=gen).to(BF16)
    n = backend._estimate_max_chunk_length(x, 0)
    widest = 2 * config.intermediate_size
    assert n == max(1, limit // (config.num_attention_heads * 2 * 4 * tokens), limit // (2 * 2 * widest))
    caches = [[torch.zeros(2, 2, tokens, 128, device="cuda", dtype=BF16) for _ in "kv"] for _ in "ab"]
    with torch.inference_mode():
        whole = block(x, kv_cache=caches[0], prefix_length=0)
        parts = [block(x[:, i : i + n], kv_cache=caches[1], prefix_length=i) for i in range(0, tokens, n)]
    tol = dict(atol=0.03, rtol=0.03)  # dense products of other row counts are summed in other orders
    assert torch.allclose(torch.cat(parts, 1).float(), whole.float(), **tol)
    for a, b in zip(*caches):
        assert torch.allclose(a.float(), b.float(), **tol)


def off_by_one_value(t):
    """The same values, contiguous, on an address that is no multiple of 16 bytes."""
    moved = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:].view(t.shape)
    assert moved.is_contiguous() and moved.data_ptr() % 16
    return moved.copy_(t)


@requires_gpu
@pytest.mark.parametrize("preset", ["test-llama-hd128", "test-bloom-hd64", "test-falcon-hd64"])
def test_prompts_at_any_address(hip, preset):
    from petals_amd.models.config_base import load_model_config
    from petals_amd.server.from_pretrained import build_empty_block, init_random_block_, load_pretrained_block

    config = load_model_config(preset)
    block = load_pretrained_block(preset, config, 0, torch_dtype=BF16, device=torch.device("cuda"))
    assert block._fast is not None
    moved = build_empty_block(config, 0, torch.device("cuda"), BF16)
    init_random_block_(moved, config, 0)
    for p in moved.parameters():
        p.data = off_by_one_value(p.data)
    moved = moved.eval().optimize_for_inference()
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(2, 19, config.hidden_size, device="cuda", generator=gen).to(BF16)
    empty = [torch.zeros(shape, device="cuda", dtype=BF16) for shape in block.kv_cache_shape(2, 32)]
    with torch.inference_mode():
        assert torch.equal(block(off_by_one_value(x)), block(x))
        want = [t.clone() for t in empty]
        out = block(x, kv_cache=want, prefix_length=3)
        for caches in ([t.clone() for t in empty], [off_by_one_value(t) for t in empty]):
            assert torch.equal(block(off_by_one_value(x), kv_cache=caches, prefix_length=3), out)
            assert all(torch.equal(a, b) for a, b in zip(caches, want))
        assert torch.isfinite(moved(x).float()).all()
    moved(x.requires_grad_(True)).sum().backward()
    assert torch.isfinite(x.grad.float()).all()


@requires_gpu
@pytest.mark.parametrize("preset", ["test-llama-hd128", "test-bloom-hd64", "test-falcon-hd64"])
def test_prompts_with_sums_over_ranks(hip, preset, monkeypatch):
    """A shard that holds everything, whose sums over ranks have one term, is the block."""
    from petals_amd.models.config_base import load_model_config
    from petals_amd.server.from_pretrained import load_pretrained_block

    config = load_model_config(preset)
    block = load_pretrained_block(preset, config, 0, torch_dtype=BF16, device=torch.device("cuda"))
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(2, 19, config.hidden_size, device="cuda", generator=gen).to(BF16)
    caches = [[torch.zeros(shape, device="cuda", dtype=BF16) for shape in block.kv_cache_shape(2, 32)] for _ in "ab"]
    with torch.inference_mode():
        want = block(x, kv_cache=caches[0], prefix_length=3)
        monkeypatch.setattr(type(block._fast), "_tp_reduce", lambda self, t: t)
        block._fast.tp_world = 2
        got = block(x, kv_cache=caches[1], prefix_length=3)
    # sums are rounded to bf16 once or twice more on the way
    assert (got.double() - want.double()).norm() <= 2.0**-6 * want.double().norm()
    assert all(torch.equal(a, b) for a, b in zip(*caches))


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, BF16])
@pytest.mark.parametrize("tokens,dim,experts,top", [(1, 8, 1, 1), (3, 64, 4, 2), (5, 4096, 8, 2), (2, 520, 64, 16), (7, 128, 65, 3), (1, 2048, 256, 8)])
def test_router(hip, dtype, tokens, dim, experts, top):
    gen = torch.Generator(device="cuda").manual_seed(experts)
    x = torch.randn(tokens, dim, device="cuda", generator=gen).to(dtype)
    w = torch.randn(experts, dim, device="cuda", generator=gen).to(BF16)
    weights, sel = hip.moe_route(x, w, top)
    logits = x.double() @ w.double().t()
    best, chosen = torch.topk(logits, top, dim=-1)
    assert torch.equal(sel.long(), chosen)  # no ties among random values
    # 32-bit logits: sums of dim terms; exponentials and a division
    err = 2.0**-24 * (dim / 64 + 16) * (x.double().abs() @ w.double().abs().t()).amax() + 2.0**-20
    assert bool(((weights.double() - torch.softmax(best, -1)).abs() <= err).all())


@requires_gpu
@pytest.mark.parametrize("dtype", [torch.float32, BF16])
def test_router_of_infinities(hip, dtype):
    """Weights that a softmax has no numbers for are NaNs, and experts are always some."""
    gen = torch.Generator(device="cuda").manual_seed(0)
    w = torch.randn(70, 64, device="cuda", generator=gen).to(BF16)
    x = torch.randn(6, 64, device="cuda", generator=gen).to(dtype)
    x[1, 3], x[2, 5], x[3, 7] = float("nan"), float("inf"), float("-inf")
    x[4, 9], w[:, 9] = float("inf"), -w[:, 9].abs()  # all logits below every number
    for spoilt in (False, True):
        if spoilt:
            w[66, 0] = float("nan")  # one expert's logits
        weights, sel = (t.cpu() for t in hip.moe_route(x, w, 3))
        logits = (x.double() @ w.double().t()).cpu()
        best, chosen = torch.topk(torch.softmax(logits, -1), 3, dim=-1)
        want = best / best.sum(-1, keepdim=True)
        assert torch.equal(torch.isnan(weights), torch.isnan(want))
        assert bool(((sel >= 0) & (sel < 70)).all()) and all(len(set(row.tolist())) == 3 for row in sel)
        fine = ~torch.isnan(want)
        assert torch.allclose(weights[fine].double(), want[fine], atol=1e-3)
        assert torch.equal(sel[fine].long(), chosen[fine])
        assert fine.any() != spoilt


@requires_gpu
@pytest.mark.parametrize("tokens,top,splits,width", [(1, 1, 1, 8), (3, 2, 5, 72), (2, 3, 7, 4096), (130, 2, 1, 128)])
def test_expert_sums(hip, tokens, top, splits, width):
    gen = torch.Generator(device="cuda").manual_seed(width)
    parts = torch.randn(splits, tokens * top, width, device="cuda", generator=gen)
    weights = torch.rand(tokens, top, device="cuda", generator=gen)
    residual = torch.randn(tokens, width, device="cuda", generator=gen).to(BF16)

    def check(y, rows):
        ref = residual.double() + (rows.view(tokens, top, width) * weights.double()[..., None]).sum(1)
        assert bool(((y.double() - ref).abs() <= 2.0**-8 * ref.abs() + 1e-4).all())

    check(hip.moe_combine(parts, weights, residual), parts.double().sum(0))
    rows = parts[0].to(BF16)
    check(hip.moe_combine(rows, weights, residual), rows.double())


# ------------------------------------------------- gradients of a prompt's rows


def _bf16_leaf(gen, *shape, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=gen) * scale).to(BF16).requires_grad_(True)


def _gradients(outputs, inputs, grads, **kw):
    return torch.autograd.grad(outputs, inputs, grads, **kw)


@requires_gpu
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 2048), (5, 2056), (7, 16384)])
def test_norm_gradients(hip, rows, dim):
    from petals_amd.ops import prompt_grad

    gen = torch.Generator(device="cuda").manual_seed(dim)
    x, y = _bf16_leaf(gen, rows, dim), _bf16_leaf(gen, rows, dim)
    w = torch.randn(dim, device="cuda", generator=gen).to(BF16)
    gh, gn = (torch.randn(rows, dim, device="cuda", generator=gen).to(BF16) for _ in range(2))
    h, n = prompt_grad.add_norm(x, y, w, 1e-5, hip)
    got = _gradients([h, n], [x, y], [gh, gn])
    s = h.detach().double().requires_grad_(True)
    normed = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    (want,) = _gradients([s, normed], [s], [gh.double(), gn.double()])
    # one rounding to bf16 of a sum in 32 bits; terms of the sum may cancel
    inv = torch.rsqrt(s.detach().pow(2).mean(-1, keepdim=True) + 1e-5)
    terms = gh.double().abs() + inv * (gn.double() * w.double()).abs() * 2 + want.abs()
    for t in got:
        assert bool(((t.double() - want).abs() <= 2.0**-8 * want.abs() + 2.0**-18 * (terms + terms.mean(-1, keepdim=True))).all())
    only = _gradients([prompt_grad.norm(x, w, 1e-5, hip)], [x], [gn])[0]
    z = x.detach().double().requires_grad_(True)
    (want,) = _gradients([z * torch.rsqrt(z.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()], [z], [gn.double()])
    inv = torch.rsqrt(z.detach().pow(2).mean(-1, keepdim=True) + 1e-5)
    terms = inv * (gn.double() * w.double()).abs() * 2 + want.abs()
    assert bool(((only.double() - want).abs() <= 2.0**-8 * want.abs() + 2.0**-18 * (terms + terms.mean(-1, keepdim=True))).all())


@requires_gpu
@pytest.mark.parametrize("rows,inner", [(1, 8), (3, 72), (130, 2048)])
def test_swiglu_gradients(hip, rows, inner):
    from petals_amd.ops import prompt_grad

    gen = torch.Generator(device="cuda").manual_seed(inner)
    gu = _bf16_leaf(gen, rows, 2 * inner, scale=3.0)
    g = torch.randn(rows, inner, device="cuda", generator=gen).to(BF16)
    (got,) = _gradients([prompt_grad.swiglu(gu, hip)], [gu], [g])
    z = gu.detach().double().requires_grad_(True)
    (want,) = _gradients([torch.nn.functional.silu(z[:, :inner]) * z[:, inner:]], [z], [g.double()])
    # a rounding to bf16; 1 + a (1 - gate) may cancel, with terms up to |a|
    size = (g.double() * gu.detach().double()[:, inner:]).abs() * (1 + gu.detach().double()[:, :inner].abs())
    slack = torch.cat([size, (g.double() * gu.detach().double()[:, :inner]).abs()], dim=-1)
    assert bool(((got.double() - want).abs() <= 2.0**-8 * want.abs() + 2.0**-20 * slack).all())


@requires_gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize(
    "b,s,qh,kh,start",
    [
        (1, 1, 1, 1, 0),  # a row that sees itself
        (2, 63, 2, 2, 0),  # a tile, not filled
        (1, 65, 4, 1, 3),  # one row more than a tile; heads that share keys
        (3, 128, 6, 2, 0),
        (1, 200, 8, 8, 11),  # several tiles; heads a multiple of the chiplets
    ],
)
def test_prompt_attention_gradients(hip, hd, b, s, qh, kh, start):
    from petals_amd.ops import prompt_grad, reference

    gen = torch.Generator(device="cuda").manual_seed(s + hd)
    cos, sin = (t.to("cuda") for t in reference.build_rope_cache(hd, start + s + 2))
    qkv = _bf16_leaf(gen, b, s, (qh + 2 * kh) * hd)
    g = torch.randn(b, s, qh * hd, device="cuda", generator=gen).to(BF16)
    out = prompt_grad.attention(qkv, cos, sin, start, qh, kh, hd, hd**-0.5, hip)
    (got,) = _gradients([out], [qkv], [g])

    z = qkv.detach().cpu().double().requires_grad_(True)
    want_out = prompt_grad.torch_attention(z.float(), cos.cpu(), sin.cpu(), start, qh, kh, hd)
    heads = z.view(b, s, qh + 2 * kh, hd).transpose(1, 2)
    c, n = (t.cpu().double()[start : start + s] for t in (cos, sin))

    def turn(t):
        return t * c + torch.cat([-t[..., hd // 2 :], t[..., : hd // 2]], -1) * n

    q, k, v = turn(heads[:, :qh]), turn(heads[:, qh : qh + kh]), heads[:, qh + kh :]
    k, v = (t.repeat_interleave(qh // kh, 1) for t in (k, v))
    scores = (q @ k.transpose(-1, -2) * hd**-0.5).masked_fill(torch.ones(s, s).triu(1).bool(), float("-inf"))
    exact = (torch.softmax(scores, -1) @ v).transpose(1, 2).reshape(b, s, qh * hd)
    (want,) = _gradients([exact], [z], [g.cpu().double()])
    assert bool((want_out.double() - exact).abs().max() < 1e-3)  # the composition is the same function
    # Turned queries and keys are rounded to bf16, 2^-9 each: scores off by delta at most, weights
    # by a factor of exp(2 delta). Results, weights and rows enter products rounded, four times at
    # most. Errors of a sum are bounded by its terms' sizes, of which turning back adds two.
    with torch.no_grad():
        go = g.cpu().double().view(b, s, qh, hd).transpose(1, 2)
        delta = hd**-0.5 * (q.abs() @ k.abs().transpose(-1, -2)).max() * 2.0**-8
        share = torch.expm1(2 * delta) + 2.0**-7
        weights = torch.softmax(scores, -1)
        dots = (go.abs() * (weights @ v).abs()).sum(-1, keepdim=True)
        ds = weights * ((go @ v.transpose(-1, -2)).abs() + dots) * hd**-0.5
        parts = [ds @ k.abs(), ds.transpose(-1, -2) @ q.abs(), weights.transpose(-1, -2) @ go.abs()]
        parts[:2] = [t + t.roll(hd // 2, -1) for t in parts[:2]]
        parts[1:] = [t.view(b, kh, qh // kh, s, hd).sum(2) for t in parts[1:]]
        terms = torch.cat(parts, 1)
    err = (got.cpu().double() - want).view(b, s, -1, hd).transpose(1, 2)
    assert bool((err.abs() <= share * terms).all())
    assert bool(err.norm() <= 2.0**-7 * want.norm())  # and roundings don't all add up


def cancelling_gradient(hip, hd, s, spread):
    """Gradients of queries whose keys are all alike, so that nothing is left of them, beside what
    they are sums of: [b, qh, s] sums of p (|dP| + |dot|), of p |dP - dot|, and of the gradient."""
    from petals_amd.ops import prompt_grad

    gen = torch.Generator(device="cuda").manual_seed(s + hd)
    b, qh, kh = 2, 4, 2
    cos, sin = torch.ones(s, hd, device="cuda"), torch.zeros(s, hd, device="cuda")
    heads = torch.randn(b, s, qh + 2 * kh, hd, device="cuda", generator=gen)
    heads[:, :, qh : qh + kh] = heads[:, :1, qh : qh + kh]
    heads[:, :, qh + kh :] = heads[:, :1, qh + kh :] + spread * heads[:, :, qh + kh :]
    qkv = heads.view(b, s, -1).to(BF16).requires_grad_(True)
    g = torch.randn(b, s, qh * hd, device="cuda", generator=gen).to(BF16)
    (got,) = _gradients([prompt_grad.attention(qkv, cos, sin, 0, qh, kh, hd, hd**-0.5, hip)], [qkv], [g])
    heads = qkv.detach().double().view(b, s, -1, hd).transpose(1, 2)
    k, v = (t.repeat_interleave(qh // kh, 1) for t in (heads[:, qh : qh + kh], heads[:, qh + kh :]))
    dp = torch.matmul(g.double().view(b, s, qh, hd).transpose(1, 2), v.transpose(2, 3).contiguous())
    p = torch.ones(s, s, device="cuda", dtype=torch.float64).tril()
    p = p / p.sum(-1, keepdim=True)  # scores are alike, too
    dot = (p * dp).sum(-1, keepdim=True)
    left = got.double().view(b, s, -1, hd)[:, :, :qh].transpose(1, 2) / k * hd**0.5
    return (p * (dp.abs() + dot.abs())).sum(-1), left.abs().amax(-1)


@requires_gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("s", [8, 70, 200])
def test_score_gradients_add_up_to_nothing(hip, hd, s):
    """With values far from zero: the mean that is taken off is that of the same 32-bit terms."""
    sums, left = cancelling_gradient(hip, hd, s, 0.01)
    assert bool((left <= 2.0**-18 * sums).all())


@requires_gpu
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("s", [8, 70, 200])
def test_score_gradients_keep_32_bits(hip, hd, s):
    sums, left = cancelling_gradient(hip, hd, s, 1.0)
    assert bool((left <= 2.0**-21 * sums).all())


def near(got, want, rel):
    assert (got.double() - want.double()).norm() <= rel * want.double().norm()


@requires_gpu
@pytest.mark.parametrize("which", ["norm", "add_norm", "swiglu", "attention"])
def test_prompt_gradients_have_gradients(hip, which):
    """First gradients with create_graph are the kernels', second ones those of the function."""
    from petals_amd.ops import prompt_grad, reference

    gen = torch.Generator(device="cuda").manual_seed(0)
    cos, sin = (t.to("cuda") for t in reference.build_rope_cache(64, 8))
    w = torch.rand(64, device="cuda", generator=gen).to(BF16) + 0.5
    a = (torch.randn(64, 64, device="cuda", generator=gen) * 0.125).to(BF16)

    def composed(t):  # 32-bit
        if which == "norm":
            return reference.rms_norm(t, w, 1e-5)
        if which == "add_norm":
            return reference.rms_norm(t + t @ a.float(), w, 1e-5)
        if which == "swiglu":
            return reference.swiglu(*t.chunk(2, dim=-1))
        return prompt_grad.torch_attention(t, cos, sin, 0, 1, 1, 64)

    kernels = {
        "norm": lambda t: prompt_grad.norm(t, w, 1e-5, hip),
        "add_norm": lambda t: prompt_grad.add_norm(t, t @ a, w, 1e-5, hip)[1],
        "swiglu": lambda t: prompt_grad.swiglu(t, hip),
        "attention": lambda t: prompt_grad.attention(t, cos, sin, 0, 1, 1, 64, 0.125, hip),
    }[which]
    x = _bf16_leaf(gen, 2, 5, 192 if which == "attention" else 64)
    z = x.detach().float().requires_grad_(True)
    (plain,) = _gradients([kernels(x).float().pow(3).sum()], [x], [None])
    found = []
    for function, leaf in ((kernels, x), (composed, z)):
        (g,) = _gradients([function(leaf).float().pow(3).sum()], [leaf], [None], create_graph=True)
        found.append((g.detach(), *_gradients([g.float().square().sum()], [leaf], [None])))
    # a dozen roundings to bf16 of 2^-9 on the way, of which a gradient's gradient has twice as many
    near(found[0][0], plain, 12 * 2.0**-9)
    near(found[0][0], found[1][0], 12 * 2.0**-9)
    near(found[0][1], found[1][1], 24 * 2.0**-9)


@requires_gpu
def test_prompt_gradients_by_transforms(hip):
    from petals_amd.ops import prompt_grad

    x = torch.randn(2, 64, device="cuda").to(BF16)
    assert prompt_grad.fused_training(x)
    seen = []
    torch.func.vmap(lambda t: (seen.append(prompt_grad.fused_training(t)), t)[1])(x)
    with torch.autograd.forward_ad.dual_level():
        seen.append(prompt_grad.fused_training(x))
    assert seen == [False, False]


@requires_gpu
@pytest.mark.parametrize("shape", [(0, 5), (2, 0)])
def test_gradients_of_no_rows(hip, shape):
    from petals_amd.models.config_base import load_model_config
    from petals_amd.server.from_pretrained import load_pretrained_block

    config = load_model_config("test-llama-hd128")
    block = load_pretrained_block("test-llama-hd128", config, 0, torch_dtype=BF16, device=torch.device("cuda"))
    x = torch.zeros(*shape, config.hidden_size, device="cuda", dtype=BF16, requires_grad=True)
    block(x).sum().backward()
    assert x.grad.shape == x.shape


@requires_gpu
def test_block_gradients_by_transforms(hip):
    """What traces or transforms a block's training pass gets the gradients that the kernels give."""
    from petals_amd.models.config_base import load_model_config
    from petals_amd.ops import prompt_grad
    from petals_amd.server.from_pretrained import load_pretrained_block
    from torch.fx.experimental.proxy_tensor import make_fx

    config = load_model_config("test-llama-hd128")
    block = load_pretrained_block("test-llama-hd128", config, 0, torch_dtype=BF16, device=torch.device("cuda"))
    gen = torch.Generator(device="cuda").manual_seed(0)
    x, other = (_bf16_leaf(gen, 2, 9, config.hidden_size) for _ in range(2))
    grads = torch.randn(3, 2, 9, config.hidden_size, device="cuda", generator=gen).to(BF16)
    assert prompt_grad.fused_training(x)

    def pull(t, g, **kw):
        t = t.detach().requires_grad_(True)
        return _gradients([block(t)], [t], [g], **kw)[0]

    want = [pull(x, g) for g in grads]
    rel = 24 * 2.0**-9  # roundings to bf16 of rows between products, at most so many on the way and back
    near(pull(x, grads[0], create_graph=True).detach(), want[0], rel)
    near(pull(x, grads, is_grads_batched=True), torch.stack(want), rel)
    near(make_fx(lambda t, g: pull(t, g))(other.detach(), grads[1])(x.detach(), grads[0]), want[0], rel)
    out = block(x)
    back = make_fx(lambda g: _gradients([out], [x], [g], retain_graph=True)[0])(grads[1])
    near(back(grads[0]), want[0], rel)
    assert torch.equal(_gradients([out], [x], [grads[0]])[0], want[0])


# ------------------------------------------------------ decode attention


@requires_gpu
@pytest.mark.parametrize("hd,gq,kv,alibi", [(128, 1, 3, True), (128, 8, 2, False), (64, 16, 1, True), (64, 71, 1, False), (128, 32, 1, False)])
@pytest.mark.parametrize(
    "kv_len,lmax",
    [
        (1, 64),
        (31, 32),
        (33, 200),  # a tile and one key more
        (161, 384),  # one part, second round of the first wave
        (3, 4096),  # parts without keys
        (385, 385),  # parts that end within a tile
        (4000, 8300),  # more parts than a wave has lanes, of few heads
    ],
)
def test_decode_attention_edges(hip, hd, gq, kv, alibi, kv_len, lmax):
    b = 2
    gen = torch.Generator(device="cuda").manual_seed(kv_len + gq)
    q = torch.randn(b, kv * gq * hd, device="cuda", generator=gen)
    k, v = (torch.full((b, kv, lmax, hd), float("nan"), device="cuda", dtype=BF16) for _ in range(2))
    for t in (k, v):  # nothing from kv_len on is used
        t[:, :, :kv_len] = torch.randn(b, kv, kv_len, hd, device="cuda", generator=gen).to(BF16)
    slopes = torch.rand(kv * gq, device="cuda", generator=gen) * 0.1 if alibi else None
    empty = torch.empty(0, device="cuda")
    length = torch.tensor([kv_len], dtype=torch.int32, device="cuda")
    got = hip.attn_decode_fused(q, k, v, length, gq, 0, empty, empty, hd**-0.5, slopes).view(b, kv, gq, hd).double()
    qd, kd, vd = q.view(b, kv, gq, hd).double(), k[:, :, :kv_len].double(), v[:, :, :kv_len].double()
    scores = qd @ kd.transpose(-1, -2) * hd**-0.5
    if alibi:
        scores = scores + slopes.double().view(kv, gq, 1) * torch.arange(kv_len, device="cuda")
    weights = torch.softmax(scores, -1)
    # scaled queries are rounded to bf16 (2^-9 each), weights too (2^-9), scores with slopes to 24 bits
    delta = (qd.abs() @ kd.abs().transpose(-1, -2) * hd**-0.5).max() * 2.0**-9 + scores.abs().max() * 2.0**-22
    bound = (torch.expm1(2 * delta) + 2.0**-8) * (weights @ vd.abs())
    assert bool(((got - weights @ vd).abs() <= bound).all())


@requires_gpu
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("tile", [0, 1, 2, 3, -1])
@pytest.mark.parametrize(
    "m,k,n",
    [
        (1, 64, 64),  # one step, fewer columns than a tile
        (33, 128, 320),  # fewer steps than buffers; a row and 64 columns beyond a tile
        (127, 256, 576),  # as many steps as buffers
        (129, 704, 256),  # a row beyond two tiles, steps that end in the middle of the buffers
        (300, 4160, 192),  # parts along K, the last one shorter
        (640, 1024, 3328),  # the lowest tile: a whole wave and some left over, in parts
        (640, 1024, 13312),  # the same for all tiles: 256, 512 or 1024 and 4, 8 or 16
        (640, 448, 13312),  # and left over, but not in parts
        (512, 192, 16384),  # whole waves and none left over
    ],
)
def test_prompt_product_edges(hip, m, k, n, tile, transposed):
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(BF16)

    x, w, residual, bias = normal(m, k), normal(k, n) * 0.125, normal(m, n), normal(n)
    given = w.t().contiguous() if transposed else w
    ref = x.double() @ w.double()
    # one rounding to bf16, and sums of k terms in 32 bits
    loose = (x.double().abs() @ w.double().abs()) * k * 2.0**-24

    def check(y, want, slack):
        assert y.shape == want.shape and bool(torch.isfinite(y).all())
        assert bool(((y.double() - want).abs() <= 2.0**-8 * want.abs() + slack + 1e-6).all())

    check(hip.gemm_rows(x, given, transposed, 0, None, None, tile), ref, loose)
    check(hip.gemm_rows(x, given, transposed, 1, residual, bias, tile), ref + residual.double() + bias.double(), loose)
    gelu = torch.nn.functional.gelu(ref + bias.double(), approximate="tanh")
    check(hip.gemm_rows(x, given, transposed, 2, None, bias, tile), gelu, 1.2 * loose)  # its slope is at most 1.13
    (g, u), (lg, lu) = ref.chunk(2, dim=-1), loose.chunk(2, dim=-1)
    # silu's slope is at most 1.1; its exponential is good to 2^-20
    silu = torch.nn.functional.silu(g)
    slack = 1.1 * lg * u.abs() + silu.abs() * lu + (silu * u).abs() * 2.0**-20
    check(hip.gemm_rows(x, given, transposed, 3, None, None, tile), silu * u, slack)


@requires_gpu
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("tile", [0, 4, 5, 6, 7, 8])  # 128 (eight waves), 256, 192, 160 and 96 rows; 128 and 192 columns
@pytest.mark.parametrize(
    "m,k,n",
    [
        (1, 64, 16),  # one step, two groups of columns
        (95, 128, 272),  # a row less than a tile, two steps; 16 columns beyond a tile
        (193, 192, 528),  # a row beyond, as many steps as stages
        (257, 2112, 304),  # parts along K, the last one shorter, of two tiles of columns
        (2049, 256, 1040),  # bands of rows, the last one shorter
        (4100, 64, 4112),  # the same with whole turns of workgroups and some left over
        (1030, 1088, 4624),  # left over, in parts
    ],
)
def test_prompt_products_of_four_waves(hip, m, k, n, tile, transposed):
    if tile < 8:
        return test_prompt_product_edges(hip, m, k, n, tile, transposed)
    with pytest.raises(RuntimeError, match="no such tile"):  # for gates and ups, which come last
        test_prompt_product_edges(hip, m, k, n, tile, transposed)


@requires_gpu
@pytest.mark.parametrize(
    "m,k,n,tile,own",
    [
        (17, 4096, 4096, 3, True), (64, 4096, 6144, 2, False), (100, 4096, 4096, 1, True), (150, 6144, 8192, 0, False),
        (200, 4096, 6144, 0, False), (283, 4096, 6144, 2, False),  # `own`: others have that tile too
    ],
)
def test_products_ahead_of_a_router(hip, m, k, n, tile, own):
    """Their sums are cut along K as the tiles of eight waves cut them, to the bit."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    x, w = (torch.randn(*s, device="cuda", generator=gen).to(BF16) for s in ((m, k), (k, n)))
    steady = hip.gemm_rows(x, w, steady=True)
    assert torch.equal(steady, hip.gemm_rows(x, w, tile=tile))
    assert torch.equal(steady, hip.gemm_rows(x, w)) == own


@requires_gpu
@pytest.mark.parametrize("model,routed", [("test-mixtral", True), ("tinyllama-1.1b", False)])
def test_blocks_with_a_router_ask_for_steady_products(hip, monkeypatch, model, routed):
    from petals_amd.models.config_base import load_model_config
    from petals_amd.server.from_pretrained import build_empty_block, init_random_block_

    config = load_model_config(model)
    if routed:  # heads that the kernels take
        config = dataclasses.replace(config, hidden_size=256, intermediate_size=256)
    block = build_empty_block(config, 0, torch.device("cuda"), BF16)
    init_random_block_(block, config, 0)
    block = block.eval().optimize_for_inference()
    asked, gemm_rows = set(), hip.gemm_rows

    def watched(x, w, transposed=False, epilogue=0, residual=None, bias=None, tile=-1, steady=False):
        asked.add((transposed, steady))
        return gemm_rows(x, w, transposed, epilogue, residual, bias, tile, steady)

    monkeypatch.setattr(hip, "gemm_rows", watched)
    x = torch.randn(2, 20, config.hidden_size, device="cuda").to(BF16)
    with torch.inference_mode():
        block(x)
    assert asked == {(False, routed)}
    leaf = x.clone().requires_grad_(True)
    block(leaf).sum().backward()
    assert asked == {(False, routed), (True, False)}  # no router reads gradients


@requires_gpu
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,k,n", [(40, 128, 128), (70, 1024, 320)])  # whole sums, and in parts
def test_prompt_products_of_extreme_values(hip, m, k, n, transposed):
    """Infinities, NaNs and large values stay in their rows and columns, and activations and
    residuals have them as the library's product and the kernels after it do."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    x, residual = (torch.randn(m, c, device="cuda", generator=gen).to(BF16) for c in (k, n))
    w = (torch.randn(k, n, device="cuda", generator=gen) * 0.125).to(BF16)
    bias = torch.randn(n, device="cuda", generator=gen).to(BF16)
    inf, nan = float("inf"), float("nan")
    x[1, 3], x[2, k - 1], x[5, 0], x[6, 7], x[m - 1, 9] = inf, nan, -inf, 3e38, -3e38
    w[11, 5], w[12, n // 2 + 5], w[k - 1, n - 1] = inf, nan, -inf
    residual[3, 2], residual[4, 3], residual[7, 4] = inf, nan, -inf
    bias[17], bias[18], bias[n - 2] = inf, nan, -inf
    given = w.t().contiguous() if transposed else w
    y = torch.matmul(x, w)
    gelu = y.clone()
    hip.bias_gelu_rows(gelu, bias)
    want = [
        (y, hip.gemm_rows(x, given, transposed, 0)),
        (hip.add_rows(residual, y, None, bias), hip.gemm_rows(x, given, transposed, 1, residual, bias)),
        (gelu, hip.gemm_rows(x, given, transposed, 2, None, bias)),
        (hip.swiglu_rows(y), hip.gemm_rows(x, given, transposed, 3)),
    ]
    for ref, got in want:
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
        assert torch.equal(got[got.isinf()], ref[ref.isinf()])
        finite = got.isfinite()
        assert 0.5 < finite.float().mean() < 1
        a, b = got[finite].double(), ref[finite].double()
        # the reference rounds its product to bf16 (2^-9 of it) before the activation or residual
        size = y.double().abs().clamp(max=1e30)[:, : got.shape[1]][finite] + 4
        if got is want[3][1]:
            size = size * y.double().abs().clamp(max=1e30)[:, n // 2 :][finite] + 4
        assert bool(((a - b).abs() <= 2.0**-7 * b.abs() + 2.0**-8 * size).all())


@requires_gpu
@pytest.mark.parametrize("family,rows", [("llama", 40), ("bloom", 40), ("falcon", 40), ("llama", 700)])
def test_prompt_products_match_the_library(hip, monkeypatch, family, rows):
    """A block's prompt with and without csrc/gemm.hip, and its gradients where they go through it."""
    from petals_amd.models.config_base import load_model_config
    from petals_amd.ops import prompt_grad
    from petals_amd.server.from_pretrained import build_empty_block, init_random_block_

    config = load_model_config({"llama": "tinyllama-1.1b", "bloom": "bloom-7b1", "falcon": "falcon-7b"}[family])
    block = build_empty_block(config, 0, torch.device("cuda"), BF16)
    init_random_block_(block, config, 0)
    block = block.eval().optimize_for_inference()
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x, g = (torch.randn(2, rows // 2, config.hidden_size, device="cuda", generator=gen).to(BF16) for _ in range(2))
    calls, gemm_rows = set(), hip.gemm_rows

    def watched(x, w, transposed=False, epilogue=0, *rest):
        calls.add((transposed, epilogue))
        return gemm_rows(x, w, transposed, epilogue, *rest)

    def run():
        with torch.inference_mode():
            y = block(x)
        by_prompt = frozenset(calls)
        calls.clear()
        if family != "llama":  # their gradients are torch's
            return by_prompt, y
        leaf = x.clone().requires_grad_(True)
        (dx,) = torch.autograd.grad(block(leaf), leaf, g)
        return by_prompt, y, dx

    monkeypatch.setattr(hip, "gemm_rows", watched)
    prompts, *got = run()
    plain, residual, gelu, swiglu = ((False, epilogue) for epilogue in range(4))
    assert prompts == {
        ("llama", 40): {plain, swiglu, residual}, ("llama", 700): {residual},
        ("bloom", 40): {plain, gelu, residual}, ("falcon", 40): {plain, gelu},
    }[family, rows]
    assert calls == ({plain, (True, 0)} if family == "llama" else set())
    calls.clear()
    monkeypatch.setattr(prompt_grad, "takes_gemm", lambda *args, **kwargs: False)
    prompts, *want = run()
    assert not prompts and not calls
    for a, b in zip(got, want):
        # both round every product to bf16: errors of 2^-9 each, over a block's half a dozen
        assert (a.double() - b.double()).norm() <= 2.0**-6 * b.double().norm()


@requires_gpu
@pytest.mark.parametrize("kind", [torch.float16, BF16])
def test_prompt_product_under_autocast(hip, kind):
    """In the type that autocast gives torch's product, whichever kernel would have it."""
    from petals_amd.ops.fused_decode import _FastWeight, prompt_product

    gen = torch.Generator(device="cuda").manual_seed(1)
    x, w = (torch.randn(*s, device="cuda", generator=gen).to(BF16) for s in ((40, 4096), (4096, 4096)))
    with torch.inference_mode(), torch.autocast("cuda", kind):
        y = prompt_product(hip, x, _FastWeight(w, hip, "none"))
        want = torch.matmul(x, w)
    assert y.dtype == want.dtype == kind
    if kind != BF16:
        assert torch.equal(y, want)


@requires_gpu
def test_modes_see_prompt_products(hip):
    from torch.utils.flop_counter import FlopCounterMode

    from petals_amd.ops.fused_decode import _FastWeight, prompt_product

    x, w = (torch.ones(*s, device="cuda", dtype=BF16) for s in ((40, 256), (256, 512)))
    weight = _FastWeight(w, hip, "none")
    with torch.inference_mode():
        with FlopCounterMode(display=False) as counter:
            seen = prompt_product(hip, x, weight)
        assert torch.equal(seen, prompt_product(hip, x, weight))
    assert counter.get_total_flops() == 2 * 40 * 256 * 512


@requires_gpu
@pytest.mark.parametrize("shape", [(2, 3, 128), (4, 32)])
def test_prompt_product_refuses_rows_that_do_not_fit(hip, shape):
    from petals_amd.ops.fused_decode import _FastWeight, prompt_product

    weight = _FastWeight(torch.ones(64, 128, device="cuda", dtype=BF16), hip, "none")
    assert prompt_product(hip, torch.ones(2, 3, 64, device="cuda", dtype=BF16), weight).shape == (2, 3, 128)
    with pytest.raises(RuntimeError, match="mat"):
        prompt_product(hip, torch.ones(shape, device="cuda", dtype=BF16), weight)


@requires_gpu
@pytest.mark.parametrize("batch", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("k_in,n_out", [(8, 128), (136, 192), (1088, 64), (2056, 264), (4544, 2560), (8192, 1024)])
def test_products_of_a_norm(hip, k_in, n_out, batch):
    """The norm within the product, with its sums of squares given or not, against 64 bits."""
    gen = torch.Generator(device="cuda").manual_seed(k_in + batch)
    w = (torch.randn(k_in, n_out, device="cuda", generator=gen) * 0.05).to(BF16)
    h = torch.randn(batch, k_in, device="cuda", generator=gen).to(BF16)
    h[:, :: max(1, k_in // 5)] *= 300.0  # loud channels
    if batch > 1:  # next to which eps is large, so that it says nothing about the sum of squares
        h[batch // 2] *= 1e-10
    weight = (1 + 0.1 * torch.randn(k_in, device="cuda", generator=gen)).to(BF16)
    hd = h.double()
    x = hd * torch.rsqrt(hd.square().mean(-1, keepdim=True) + 1e-5) * weight.double()
    # and the factor: some dozen roundings
    bound = sum_bound(x, w.double()) + 16 * 2.0**-24 * (x @ w.double()).abs()
    parts = torch.stack([c.float().square().sum(-1) for c in h.split(64, dim=-1)], dim=1)
    for sumsq in (None, parts):
        y = hip.gemv_bf16_normed(w, h, weight, sumsq, 1e-5, torch.empty(0, device="cuda"), 0)
        assert bool(((y.double() - x @ w.double()).abs() <= bound).all())


@requires_gpu
@pytest.mark.parametrize("batch", [1, 2, 6])
@pytest.mark.parametrize("k_in,width,inner", [(64, 128, 64), (192, 1024, 136), (136, 1152, 72), (128, 2176, 128), (2048, 4096, 512)])
def test_products_of_a_norm_of_a_sum(hip, k_in, width, inner, batch):
    """As a decoding step has them: a product added to the stream leaves sums of squares, and gate and up
    take the norm with them, in 1, 8, 9, 17 and, wider, 32 parts."""
    gen = torch.Generator(device="cuda").manual_seed(width + batch)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(BF16)

    wo, both, weight = normal(k_in, width) * 0.05, normal(width, 2 * inner) * 0.05, 1 + 0.1 * normal(width)
    x, h = torch.randn(batch, k_in, device="cuda", generator=gen), normal(batch, width) * 3
    h[:, :: width // 5] *= 100.0  # loud channels
    sums = torch.full((batch, width // 64), float("nan"), device="cuda")
    ws = torch.empty(64 * batch * max(width, 2 * inner), device="cuda")
    h2 = hip.gemv_bf16(wo, x, ws, h, 2, 0, None, sums)
    hd = h2.double()
    squares = hd.square().view(batch, -1, 64).sum(-1)
    assert bool(((sums.double() - squares).abs() <= 2.0**-20 * squares).all())
    act = hip.gemv_bf16_normed(both, h2, weight, sums, 1e-5, ws, 3)
    # and with sums of squares that every workgroup takes
    alone = hip.gemv_bf16_normed(both, h2, weight, None, 1e-5, torch.empty(0, device="cuda"), 3)
    n = hd * torch.rsqrt(hd.square().mean(-1, keepdim=True) + 1e-5) * weight.double()
    gu = n @ both.double()
    bound = sum_bound(n, both.double()) + 16 * 2.0**-24 * gu.abs()
    (g, u), (bg, bu) = gu.chunk(2, dim=-1), bound.chunk(2, dim=-1)
    silu = torch.nn.functional.silu(g)
    # silu's slope is at most 1.1; its exponential is good to 2^-20
    bound = 1.1 * bg * (u.abs() + bu) + silu.abs() * bu + (silu * u).abs() * 2.0**-20 + 1e-12
    for y in (act, alone):
        assert bool(((y.double() - silu * u).abs() <= bound).all())


@requires_gpu
@pytest.mark.parametrize("k_in", [136, 4096])
def test_products_of_a_norm_of_extreme_rows(hip, k_in):
    """Infinities, NaNs and values whose squares overflow, as the norm kernel has them."""
    gen = torch.Generator(device="cuda").manual_seed(k_in)
    w = (torch.randn(k_in, 192, device="cuda", generator=gen) * 0.05).to(BF16)
    h = torch.randn(8, k_in, device="cuda", generator=gen).to(BF16)
    weight = (2 + 0.1 * torch.randn(k_in, device="cuda", generator=gen)).to(BF16)
    h[1, 3] = float("inf")
    h[2, 5] = float("nan")
    h[3] = (h[3].float() * 1e38).clamp(-3e38, 3e38).to(BF16)  # twice these are infinite
    h[4, 7] = 3e38
    h[5, ::2] = 2.0**63.5  # no square is infinite, their sum is
    h[6, 1], h[6, 2] = -3e38, float("-inf")
    h[7, 7] = 2.0**63
    empty = torch.empty(0, device="cuda")
    want = hip.gemv_bf16(w, hip.rms_norm_f32out(h, weight, 1e-5), empty, None, 0)
    assert want.isnan().all(-1).tolist() == [False, True, True, False, False, False, True, False]
    assert not bool(want[3:6].any())
    parts = torch.stack([c.float().square().sum(-1) for c in h.split(64, dim=-1)], dim=1)
    for sumsq in (None, parts):
        got = hip.gemv_bf16_normed(w, h, weight, sumsq, 1e-5, empty, 0)
        assert torch.equal(got.isnan(), want.isnan())
        kept = ~want.isnan()
        torch.testing.assert_close(got[kept], want[kept], rtol=1e-4, atol=1e-4)


@requires_gpu
def test_position_of_a_decoding_step():
    from petals_amd.ops.fused_decode import DecodeContext

    ctx = DecodeContext(torch.device("cuda"))
    for p in (0, 1, 7900, (1 << 31) - 3):
        ctx.set_position(p)
        assert (ctx.pos.tolist(), ctx.kv_len.tolist()) == ([p], [p + 1])
        ctx.advance()
        assert (ctx.pos.tolist(), ctx.kv_len.tolist()) == ([p + 1], [p + 2])
    assert ctx.pos.dtype == ctx.kv_len.dtype == torch.int32


@requires_gpu
def test_rounding_to_bf16(hip):
    """Ties, subnormal numbers, overflow, infinities and NaNs: sums of two bf16 values, rounded once, are torch's to the bit."""
    bits = torch.arange(1 << 16, device="cuda", dtype=torch.int32)
    x = bits.to(torch.int16).view(BF16).view(256, 256)  # every bf16 value
    gen = torch.Generator(device="cuda").manual_seed(0)
    near = torch.randint(-9, 10, (1 << 16,), device="cuda", generator=gen) * 128  # exponents up to nine apart
    others = [x.flip(0), (bits ^ 1).to(torch.int16).view(BF16).view_as(x), (bits + near).to(torch.int16).view(BF16).view_as(x)]
    for apart in range(1, 9):  # y's last digits make up half of a place of x: ties wherever the sum's place is x's
        digits = torch.randint(0, 128, (1 << 16,), device="cuda", generator=gen) >> apart << apart | 1 << (apart - 1)
        exponent = ((bits >> 7 & 255) - apart).clamp(min=1)
        y = (bits & 0x8000 | exponent << 7 | digits & 127).to(torch.int16).view(BF16).view_as(x)
        ties = (x.float() + y.float()).view(torch.int32) & 0xFFFF == 0x8000  # of two bf16 values so close, exact in 32 bits
        assert ties.float().mean() > 0.2
        others.append(y)
    for y in others:
        got, want = hip.add_rows(x.contiguous(), y.contiguous()), x + y
        assert torch.equal(got.isnan(), want.isnan())
        kept = ~want.isnan()
        assert torch.equal(got[kept].view(torch.int16), want[kept].view(torch.int16))


@requires_gpu
@pytest.mark.parametrize("tile", [-1, 0, 1, 2])
@pytest.mark.parametrize(
    "m,k,n",
    [
        (1, 128, 64),  # one tile of codes, fewer columns than a wave pair's
        (31, 256, 192), (32, 384, 256), (33, 640, 320),  # edges of 32 rows; fewer tiles of codes than are fetched ahead, odd numbers
        (65, 1152, 704), (129, 1280, 4160),  # edges of 64 and 128 rows; parts along K, the last one shorter
        (640, 1024, 3328), (513, 512, 13312),  # whole waves of tiles and some left over
    ],
)
def test_nf4_prompt_product_edges(hip, m, k, n, tile):
    gen = torch.Generator(device="cuda").manual_seed(m + k + n)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(BF16)

    x, residual, bias = normal(m, k), normal(m, n), normal(n)
    tiles, scales = hip.nf4_tile(*hip.nf4_quantize(normal(k, n) * 0.125))
    w = hip.nf4_untile(tiles, scales, k)  # the copy in bf16 whose products these are
    ref = x.double() @ w.double()
    # one rounding to bf16, and sums of k terms in 32 bits
    loose = (x.double().abs() @ w.double().abs()) * k * 2.0**-24

    def check(y, want, slack):
        assert y.shape == want.shape and bool(torch.isfinite(y).all())
        assert bool(((y.double() - want).abs() <= 2.0**-8 * want.abs() + slack + 1e-6).all())

    def product(*args):
        return hip.gemm_nf4_rows(x, tiles, scales, *args, tile=tile)

    check(product(0), ref, loose)
    check(product(1, residual, bias), ref + residual.double() + bias.double(), loose)
    gelu = torch.nn.functional.gelu(ref + bias.double(), approximate="tanh")
    check(product(2, None, bias), gelu, 1.2 * loose)  # its slope is at most 1.13
    (g, u), (lg, lu) = ref.chunk(2, dim=-1), loose.chunk(2, dim=-1)
    # silu's slope is at most 1.1; its exponential is good to 2^-20
    silu = torch.nn.functional.silu(g)
    check(product(3), silu * u, 1.1 * lg * u.abs() + silu.abs() * lu + (silu * u).abs() * 2.0**-20)


@requires_gpu
@pytest.mark.parametrize("m", [5, 70])
def test_nf4_prompt_products_of_extreme_values(hip, m):
    """Infinities, NaNs and large values stay in their rows, those of scales in their blocks; blocks of zeros are zeros."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, 256, device="cuda", generator=gen).to(BF16)
    w = (torch.randn(256, 192, device="cuda", generator=gen) * 0.125).to(BF16)
    w[7, :64] = 0.0
    inf, nan = float("inf"), float("nan")
    x[0, 3], x[1, 255], x[2, 0], x[4, 9] = inf, nan, -inf, 3e38
    tiles, scales = hip.nf4_tile(*hip.nf4_quantize(w))
    for scale in (None, inf, nan):
        if scale is not None:
            scales[1, 11] = scale
        dense = hip.nf4_untile(tiles, scales, 256)
        want, got = x.double() @ dense.double(), hip.gemm_nf4_rows(x, tiles, scales)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        finite = want.isfinite()
        assert torch.equal(got[got.isinf()].double(), want[want.isinf()]) and 0.2 < finite.float().mean() < 1
        # one rounding to bf16, and sums of 256 terms in 32 bits
        loose = (x.double().abs() @ dense.double().abs())[finite] * 2.0**-16
        assert bool(((got[finite].double() - want[finite]).abs() <= 2.0**-8 * want[finite].abs() + loose).all())


@requires_gpu
def test_nf4_prompts_read_codes(hip, monkeypatch):
    """Rows that the rule gives to csrc/nf4_gemm.hip make no copy of the matrix, others do; both are the same product.
    Rows of other lengths and codes of other sizes are refused."""
    from petals_amd.ops import fused_decode, prompt_grad
    from petals_amd.ops.fused_decode import _FastWeight, prompt_product

    assert prompt_grad.takes_nf4_gemm(32, 4096, 6144) and not prompt_grad.takes_nf4_gemm(33, 4096, 6144)
    assert prompt_grad.takes_nf4_gemm(128, 8192, 8192) and not prompt_grad.takes_nf4_gemm(129, 8192, 8192)
    # few columns: 2 us slower from codes beyond 64 rows
    assert prompt_grad.takes_nf4_gemm(64, 16384, 4096) and not prompt_grad.takes_nf4_gemm(65, 16384, 4096)
    assert not prompt_grad.takes_nf4_gemm(128, 16384, 4608) and prompt_grad.takes_nf4_gemm(128, 18176, 4544)
    assert not prompt_grad.takes_nf4_gemm(0, 8192, 8192) and not prompt_grad.takes_nf4_gemm(8, 8192 + 64, 8192)
    gen = torch.Generator(device="cuda").manual_seed(0)
    weight = _FastWeight((torch.randn(512, 320, device="cuda", generator=gen) * 0.125).to(BF16), hip, "nf4")
    x = torch.randn(2, 9, 513, device="cuda", generator=gen).to(BF16)[..., 1:]  # not aligned, not contiguous
    residual = torch.randn(2, 9, 320, device="cuda", generator=gen).to(BF16)
    made = []
    monkeypatch.setattr(fused_decode, "_dequant_cached", lambda w, make: made.append(w) or make())
    got = []
    for takes in (True, False):
        monkeypatch.setattr(prompt_grad, "takes_nf4_gemm", lambda *sizes: takes)
        got.append((prompt_product(hip, x, weight), prompt_product(hip, x, weight, 1, residual), prompt_product(hip, x, weight, 3)))
        assert len(made) == (0 if takes else 3)
    for a, b in zip(*got):
        assert a.shape == b.shape and (a.double() - b.double()).norm() <= 2.0**-7 * b.double().norm()
    for bad in (x[0, :, :448].contiguous(), x[0].float().contiguous(), x.contiguous()):
        with pytest.raises(RuntimeError):
            hip.gemm_nf4_rows(bad, weight.tiles, weight.scales)
    with pytest.raises(RuntimeError):
        hip.gemm_nf4_rows(x[0].contiguous(), weight.tiles, weight.scales[:, :256].contiguous())
    with pytest.raises(RuntimeError):
        hip.gemm_nf4_rows(x[0].contiguous(), weight.tiles, weight.scales, 1)  # a residual is missing
