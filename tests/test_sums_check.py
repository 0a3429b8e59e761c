"""What the build looks for in the kernels whose matrix instructions are in asm, on listings with one mistake each."""

import os

import pytest

from petals_amd.ops import build, sums_check

HEAD = ["v_accvgpr_write_b32 a0, 0", "s_barrier"]
LOOP = [
    "ds_read_b128 v[2:5], v80", "s_waitcnt lgkmcnt(0)", "v_mfma_f32_16x16x32_bf16 a[0:3], v[2:5], v[6:9], a[0:3]",
    "v_add_u32_e32 v80, s1, v81", "v_mfma_f32_16x16x32_bf16 v[10:13], v[6:9], v[2:5], v[10:13]",
]
TAIL = ["s_nop 15", "s_nop 15", "v_accvgpr_read_b32 v20, a3", "v_mov_b32_e32 v21, v10", "s_endpgm"]


def listing(head=HEAD, loop=LOOP, tail=TAIL):
    ops = [*head, *loop, f"s_cbranch_scc0 {65536 - len(loop) - 1}", *tail]
    return "0 <gemm_wide_kernel>:\n" + "\n".join(f"\t{op:<50} // {4 * i:012X}: 00000000" for i, op in enumerate(ops))


def test_listing_without_faults():
    assert sums_check.faults(listing()) == []


@pytest.mark.parametrize(
    "changed,fault",
    [
        (dict(loop=[*LOOP, "v_accvgpr_read_b32 v30, a2"]), "moved in a loop"),
        (dict(loop=["scratch_store_dwordx4 off, v[10:13], off", *LOOP]), "moved in a loop"),
        (dict(loop=["v_accvgpr_mov_b32 a1, a9", *LOOP]), "moved in a loop"),  # over the branch
        (dict(tail=["s_nop 14", "v_mov_b32_e32 v21, v10"]), "too early"),  # 16 slots with the branch
        (dict(tail=["v_mov_b32_e32 v21, v13", *TAIL]), "too early"),
        (dict(loop=[*LOOP[:3], "v_mov_b32_e32 v7, v90", *LOOP[4:]]), "too late"),
        (dict(loop=[*LOOP[:3], "v_pk_mov_b32 v[4:5], v[90:91], v[92:93]", "s_nop 0", *LOOP[4:]]), "too late"),
        (dict(loop=[op for op in LOOP if "mfma" not in op]), "0 loops"),
    ],
)
def test_faults_are_found(changed, fault):
    assert any(fault in found for found in sums_check.faults(listing(**changed)))


def test_operands_that_are_in_time():
    late = [*LOOP[:3], "v_mov_b32_e32 v7, v90", "s_nop 1", *LOOP[4:]]
    assert sums_check.faults(listing(loop=late)) == []


@pytest.mark.skipif(not os.path.exists(os.path.join(build.PKG_DIR, "_build", "gemm_hip.cuda.o")), reason="not built here")
def test_built_kernels():
    assert sums_check.check(os.path.join(build.PKG_DIR, "_build")) == 12
