"""Differentiable pieces of a prompt's pass: what stands between its dense products, by
the HIP kernels in either direction (csrc/prefill_rows.hip, csrc/attn_grad.hip).

As torch operations, a llama block's forward and backward was 133 launches besides its
products, 1.1 of its 2.0 ms at 2 x 379 tokens, width 4096; now it is 11, 0.15 ms. Kept for the backward: rows, and
one number per attention row, where torch kept several [heads, rows, rows] matrices.

Ordinary reverse mode only (`fused_training`): the kernels read and write memory by its address,
which what traces, transforms or counts torch operations does not see. Under any of these, and
for gradients of gradients and batches of gradients, the operations of `ops.reference` are run.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from petals_amd.ops import reference


def watched(*tensors) -> bool:
    """Whether something stands between torch operations and memory: a trace, a transform or a
    mode, in force or wrapped around one of these tensors."""
    wrapped = torch._C._functorch
    return (
        getattr(forward_ad, "_current_level", -1) >= 0
        or wrapped.peek_interpreter_stack() is not None
        or torch._C._len_torch_dispatch_stack() > 0
        or torch.jit.is_tracing()
        or torch.compiler.is_compiling()
        or any(
            type(t) not in (torch.Tensor, torch.nn.Parameter)
            or wrapped.is_functorch_wrapped_tensor(t)
            or wrapped.is_legacy_batchedtensor(t)
            for t in tensors
        )
    )


def fused_training(*rows: torch.Tensor) -> bool:
    """Whether these bf16 rows go through the kernels."""
    return all(t.is_cuda and t.dtype == torch.bfloat16 and t.shape[-1] % 8 == 0 for t in rows) and not watched(*rows)


def aligned(t: torch.Tensor) -> torch.Tensor:
    """Contiguous rows that 16-byte loads can read."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


def recast(rows: torch.Tensor) -> bool:
    """Whether autocast has torch's products of these rows, which are on a GPU, in another type than bf16."""
    kind = rows.device.type
    return torch.is_autocast_enabled(kind) and torch.get_autocast_dtype(kind) != torch.bfloat16


def gemm_matrix(w: torch.Tensor) -> bool:
    """A matrix [K, N] that ops/csrc/gemm.hip takes, from either side."""
    return (
        w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous() and w.data_ptr() % 16 == 0
        and w.shape[0] % 64 == 0 and w.shape[1] % 64 == 0 and 0 < w.numel() < 1 << 31
    )


def takes_gemm(m: int, k: int, n: int, transposed: bool = False, fused: bool = False, added: bool = False) -> bool:
    """Whether m rows of k times a matrix with n columns are faster by ops/csrc/gemm.hip than by the
    library. `fused`: an activation follows, `added`: a residual, which would be a launch of its own.

    Up to 128 rows weights are what a product reads, and up to half as many tiles of 128 x 256 as there are
    compute units the library leaves most of these idle: it takes 1.3 times as long in the mean (16384 x
    4096: 139 beside 38 us at 128 rows, 156 beside 121 at 900). A call of the library also takes the
    host 18 us and the kernel's 8, so that a product alone is the kernel's where it is up to 10 us the
    slower of the two (2048 x 2560, 2 rows: both 11 us, alone 35 and 21): a small model's launches are
    what bounds its prompts and gradients. Where it was slower by more, the library has the product: see
    below, us on MI355X by the library (with what follows) and by the kernel, and
    profiles/prompt_products.csv for all that was measured."""
    if m <= 0 or m * k >= 1 << 31:
        return False
    weights, tiles = k * n, -(-m // 128) * -(-n // 256)
    # three rows of tiles, nearly full, fit the library; the kernel's 96 tiles in two parts each leave a
    # quarter of the compute units idle. 28672 x 8192: 283 rows 237, 193; 384 rows 200, 210.
    # 57344 to 8192: 283 rows 331, 391
    if n >= 8192 and weights >= 1 << 27 and (256 if weights > 1 << 28 else 320) < m <= 384:
        return False
    if transposed:
        # 16384 to 16384: 16 rows 97, 140; 128 rows 137, 153. 18432 to 16384: 128 rows 140, 130
        if weights >= 1 << 28 and 8 * k < 9 * n:
            return False
        # 32768 to 8192: 16 rows 100, 132; 64 rows 152, 136. 57344 to 14336: 40 rows 286, 312; 128 rows 411, 335
        if weights >= 1 << 28 and m <= 40 and 2 * n <= k <= 4 * n:
            return False
        if weights > 1 << 29 and m > 128:  # 106496 to 16384: 128 rows 632, 601; 129 rows 666, 1079
            return False
        # 12288 to 4096: 256 rows 51, 41; 758 rows 89, 93. 22016 to 4096: 758 rows 231, 160
        return tiles <= 64 and k >= n or tiles <= 128 and k >= 4 * n
    # 2048 x 2560, where prompts are long enough for the host: 384 rows 14.0, 19.9; 1024 rows 26, 18
    if 1 << 22 <= weights < 1 << 23 and m > 256 and tiles < 70 and n < 3 * k and not (fused or added and k >= 2 * n):
        return False
    # 8192 x 14336: 256 rows 98, 99; 384 rows 109, 135; 512 rows 135, 124
    if fused and tiles > 128 and 256 < m <= 384 and weights >= 96 << 20:
        return False
    if n >= 4 * k and weights > 1 << 29 and m <= 16:  # 16384 x 106496: 16 rows 597, 635; 64 rows 766, 644
        return False
    # 8192 x 10240: 128 rows 76, 44; 384 rows 95, 84; 512 rows 108, 109. 4096 x 28672: 256 rows 79, 73; 283 rows 80, 100
    return m <= 128 or tiles <= (256 if fused else 128)


def takes_wide_gemm(m: int, k: int, n: int, transposed: bool = False, followed: bool = False, gelu: bool = False) -> bool:
    """Whether m rows of k times a large matrix with n columns, which `takes_gemm` leaves to the library, are
    faster by the large tiles of ops/csrc/gemm.hip. `followed`: by a residual or a SwiGLU, which would be launches of
    their own; `gelu`: by that, which is a shorter one.

    These are products that the GPU is waited for. Matrices of fewer columns than rows leave the library's tiles of 256 x 256
    without work for all compute units up to some 1500 rows, and it takes 1.2 times as long in the mean; the more columns
    there are, the sooner they fill the chip, and beyond that it is slower only by what follows. Sizes that are no multiples
    of 128 it has no good kernel for, but where columns are so many that rows don't matter. us on MI355X by the library (with what follows) and
    by the kernel: 758 rows of 28672 x 8192 with a residual 314, 298, of 4096 x
    22016 with SwiGLU 144, 124; 4096 x 28672 with SwiGLU, 4096 rows 797, 735; plain, 1024 rows 195, 211; 4096 x 12288, 512 rows
    57.5, 58.7, 1024 rows 88, 100; 18176 x 4544, 2048 rows 368, 284. Transposed: 22016 to 4096, 758 rows 231, 117;
    8192 to 8192, 512 rows 74, 71, 1024 rows 110, 115; 4096 to 11008, 256 rows 48, 39, 512 rows 52, 54.

    The library's tiles are 256 x 256 mostly and never cut along K: where some are left over after one or two turns of all
    compute units, these cost it another turn, whatever the matrix (measured from 4096 x 4096 on). 258 tiles: 758 rows of 4096 x 22016 134, 128, 1400 of
    4096 x 11008 234, 128; 272: 4200 rows of 4096 x 4096 176, 131; 518: 1700 rows of 3584 x 18944 212, 219; 36 such
    products took 0.5 to 1.04 of the library's time, 0.8 in the mean. Where it has no good kernel either, it is so as long as less
    than four fifths of these turns have work, and from the fourth turn on: 4544 x 18176, 1024 rows (284 tiles) 229, 154, 2048 rows (568)
    317, 299, 4096 rows 648, 542, transposed, 1200 rows (355) 257, 184; but 758 rows (213) 104, 111, 1500 rows (426) 205, 227.

    All that was measured, the median of three runs on three cards, is in profiles/prompt_products_wide.csv: what is taken
    takes 0.88 of the library's time in the mean, and 1.07 at most."""
    weights = k * n
    if not 128 < m < (1 << 31) // k or weights > 1 << 29:
        return False
    tiles = -(-m // 256) * -(-n // 256)
    if weights >= 1 << 24 and 256 < tiles < 768 and 0 < tiles % 256 <= 20:
        return True
    odd, small = k % 128 > 0 or n % 128 > 0, weights <= 3 << 23
    # smaller ones gain little (4096 x 6144, 758 rows: 55, 54), but for sizes that the library does not like
    if small and not (odd and weights >= 1 << 24):
        return False
    if odd and n >= 3 * k and tiles > 256 and (tiles > 768 or 5 * tiles < 4 * 256 * -(-tiles // 256)):
        return True
    if transposed:
        if small:
            return m <= 960
        if k > n:
            return m <= (1536 if n < 8192 else 1024) or odd
        return m <= 640 if k == n else m <= 320 and (n < 3 * k or odd)
    if followed:
        return True
    if odd:
        return gelu or n < 3 * k or m <= 512
    most = 768 if n <= 3 * k else 320 if n <= 6 * k else 128
    return m <= (1536 if gelu or n < 2 * k or k >= 5120 else most)


def takes_nf4_gemm(m: int, k: int, n: int) -> bool:
    """Whether m rows of k times an NF4 matrix with n columns are faster by ops/csrc/nf4_gemm.hip, which reads
    the codes, than by a product with a copy of it in bf16 that is there already.

    Codes are a quarter of the bytes, but each is looked up and rounded: large matrices gain up to 128 rows, beyond which
    the matrix cores bound both; smaller ones gain as long as reading a copy takes longer than the
    launches. Matrices of few columns have few tiles, which are cut into more parts along K that have to be added up. us on
    MI355X, with a copy and from codes (profiles/nf4_prompt_products.csv has all that was measured): 2048 x 11264, 32 rows
    17.1, 16.0, 64 rows 19.4, 20.8; 11008 x 4096, 64 rows 28.9, 27.7, 128 rows 29.4, 33.3; 16384 x 4096, 128 rows
    37.7, 39.4; 18176 x 4544, 128 rows 42.9, 43.2; 8192 x 57344, 128 rows 178, 150, 192 rows 204, 282.

    Where there is no copy, making one comes on top (33 us for 8192 x 8192, 230 for 8192 x 57344): in the first prompt, and in
    every prompt of a span whose copies together are more than the cache of them holds. So 8192 x 8192, and other
    matrices of 64 << 20 to 76 << 20 weights that are not narrow, are read as codes up to 128 rows, though with a copy
    they would take up to 4 us less (112 rows 36.2, 40.1; 5120 x 13824, 96 rows 38.9, 41.2). From 129 rows on it is not
    looked at whether there is one: 8192 x 57344 with 192 rows would take less from codes in such a span."""
    if m <= 0 or k % 128:
        return False
    weights = k * n
    if m <= 64:
        return weights >= (20 << 20 if m <= 32 else 40 << 20)
    return m <= 128 and weights >= (64 << 20 if n > 4608 else 76 << 20)


def _by_torch(*grads) -> bool:
    """Whether these gradients are taken through torch operations: those that are to have gradients
    themselves, and those that are watched, which the forward pass need not have been."""
    return torch.is_grad_enabled() or watched(*(g for g in grads if g is not None))


def _through_torch(function, inputs, grads, needed=(True,)):
    """Gradients by torch operations. They are taken at aliases of the inputs: one input may
    depend on another, and that path is the caller's graph's to follow."""
    create_graph = torch.is_grad_enabled()
    with torch.enable_grad():
        inputs = tuple(t.view_as(t) for t in inputs)
        outputs = function(*inputs)
        outputs = outputs if isinstance(outputs, tuple) else (outputs,)
        kept = [(o, g) for o, g in zip(outputs, grads) if g is not None]
        wanted = [t for t, need in zip(inputs, needed) if need]
        found = iter(
            torch.autograd.grad(
                [o for o, _ in kept], wanted, [g for _, g in kept], create_graph=create_graph, allow_unused=True
            )
        )
        return tuple(next(found) if need else None for need in needed)


class _Norm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, eps, hip):
        ctx.save_for_backward(x)
        ctx.w, ctx.eps, ctx.hip = w, eps, hip
        return hip.rms_norm(aligned(x), w, eps)

    @staticmethod
    def backward(ctx, g):
        (x,), w = ctx.saved_tensors, ctx.w
        if _by_torch(g):
            return (*_through_torch(lambda t: reference.rms_norm(t, w, ctx.eps), (x,), (g,)), None, None, None)
        return ctx.hip.norm_rows_grad(aligned(x), w, aligned(g), None, ctx.eps), None, None, None


class _AddNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, y, w, eps, hip):
        h, n = hip.add_norm_rows(aligned(x), aligned(y), None, w, None, eps)
        ctx.save_for_backward(x, y, h)
        ctx.set_materialize_grads(False)
        ctx.w, ctx.eps, ctx.hip = w, eps, hip
        return h, n

    @staticmethod
    def backward(ctx, gh, gn):
        (x, y, h), w = ctx.saved_tensors, ctx.w
        if gh is None and gn is None:
            return None, None, None, None, None
        if _by_torch(gh, gn):

            def composed(a, b):
                s = a + b
                return s, reference.rms_norm(s, w, ctx.eps)

            return (*_through_torch(composed, (x, y), (gh, gn), ctx.needs_input_grad[:2]), None, None, None)
        if gn is not None:
            gh = ctx.hip.norm_rows_grad(aligned(h), w, aligned(gn), None if gh is None else aligned(gh), ctx.eps)
        return gh, gh, None, None, None


class _SwiGLU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gateup, hip):
        ctx.save_for_backward(gateup)
        ctx.hip = hip
        return hip.swiglu_rows(aligned(gateup))

    @staticmethod
    def backward(ctx, g):
        (gateup,) = ctx.saved_tensors
        if _by_torch(g):
            return (*_through_torch(lambda t: reference.swiglu(*t.chunk(2, dim=-1)), (gateup,), (g,)), None)
        return ctx.hip.swiglu_rows_grad(aligned(gateup), aligned(g)), None


def torch_attention(qkv, cos, sin, start, qh, kh, hd):
    """Causal attention of a fused projection [B, S, (qh + 2 kh) * hd], by torch operations."""
    B, S, _ = qkv.shape
    heads = qkv.view(B, S, qh + 2 * kh, hd).transpose(1, 2)
    pos = torch.arange(start, start + S, device=qkv.device)
    q, k = reference.apply_rope(heads[:, :qh], heads[:, qh : qh + kh], cos, sin, pos)
    attn = reference.attention(q, k, heads[:, qh + kh :], causal=True)
    return attn.transpose(1, 2).reshape(B, S, qh * hd)


class _Attention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qkv, cos, sin, start, qh, kh, hd, scale, hip):
        rows = hip.rotate_rows(aligned(qkv), cos, sin, start, qh, kh, hd)
        heads = rows.view(*rows.shape[:2], qh + 2 * kh, hd).transpose(1, 2)
        out, sums = hip.attn_prefill_sums(heads[:, :qh], heads[:, qh : qh + kh], heads[:, qh + kh :], scale)
        ctx.save_for_backward(qkv, rows, sums)
        ctx.tables = cos, sin  # constants, maybe made in inference mode: such tensors can't be saved
        ctx.shape, ctx.scale, ctx.hip = (start, qh, kh, hd), scale, hip
        return out

    @staticmethod
    def backward(ctx, g):
        (qkv, rows, sums), (cos, sin) = ctx.saved_tensors, ctx.tables
        none = (None,) * 8
        # the kernels address a tile's rows by 32 bits
        if _by_torch(g) or qkv.shape[-1] >= 1 << 24:
            return (*_through_torch(lambda t: torch_attention(t, cos, sin, *ctx.shape), (qkv,), (g,)), *none)
        return (ctx.hip.attn_prompt_grad(aligned(rows), aligned(g), sums, cos, sin, *ctx.shape, ctx.scale), *none)


class _Product(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, hip, steady=False):
        # saved as torch's product saves it: hooks see it, and a change before the backward pass is
        # an error. What was made in inference mode can't be saved
        ctx.w = w if w.is_inference() else None
        if ctx.w is None:
            ctx.save_for_backward(w)
        ctx.hip = hip
        return rows_product(x, w, hip, steady=steady)

    @staticmethod
    def backward(ctx, g):
        w = ctx.saved_tensors[0] if ctx.w is None else ctx.w
        if _by_torch(g, w):
            return torch.matmul(g, w.t()), None, None, None
        return rows_product(g, aligned(w), ctx.hip, transposed=True), None, None, None


def rows_product(x, w, hip, transposed=False, steady=False):
    """x [..., K] times w [K, N], or [..., N] times its transpose: by ops/csrc/gemm.hip where that is
    the faster one, else the library's. `steady`: a router reads the result, see there."""
    k, n = w.shape if not transposed else w.shape[::-1]
    if k and x.shape[-1] == k:  # torch refuses rows of other lengths
        m = x.numel() // k
        if takes_gemm(m, k, n, transposed) or not steady and takes_wide_gemm(m, k, n, transposed):
            rest = (0, None, None, -1, True) if steady else ()
            return hip.gemm_rows(aligned(x).view(-1, k), w, transposed, *rest).view(*x.shape[:-1], n)
    return torch.matmul(x, w.t() if transposed else w)


def norm(x, w, eps, hip):
    return _Norm.apply(x, w, eps, hip)


def product(x, w, hip, steady=False):
    """x [..., K] times a frozen matrix [K, N]"""
    if w.requires_grad or not (fused_training(x) and gemm_matrix(w)) or recast(x):
        return torch.matmul(x, w)
    return _Product.apply(x, w, hip, steady)


def add_norm(x, y, w, eps, hip):
    """(x + y, its RMS norm)"""
    return _AddNorm.apply(x, y, w, eps, hip)


def swiglu(gateup, hip):
    """[..., gate | up] -> silu(gate) * up"""
    return _SwiGLU.apply(gateup, hip)


def attention(qkv, cos, sin, start, qh, kh, hd, scale, hip):
    return _Attention.apply(qkv, cos, sin, start, qh, kh, hd, scale, hip)
