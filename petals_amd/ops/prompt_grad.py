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


def gemm_matrix(w: torch.Tensor) -> bool:
    """A matrix [K, N] that ops/csrc/gemm.hip takes, from either side."""
    return (
        w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous() and w.data_ptr() % 16 == 0
        and w.shape[0] % 64 == 0 and w.shape[1] % 64 == 0 and 0 < w.numel() < 1 << 31
    )


def takes_gemm(m: int, k: int, n: int, transposed: bool = False, fused: bool = False) -> bool:
    """Whether m rows of k times a matrix with n columns are faster by ops/csrc/gemm.hip than by the
    library. `fused`: an activation follows, which would be a launch of its own.

    Up to 128 rows weights are what a product reads, and up to half as many tiles of 128 x 256 as there are
    compute units the library leaves most of these idle: it takes 1.0 to 3.6 times as long (16384 x
    4096: 139 beside 38 us at 128 rows, 156 beside 121 at 900). With 192 to 512 tiles it takes 0.76 to 1.0 times
    as long (4096 x 28672: 77 beside 98 us at 283 rows). With a transposed matrix it does as well, but
    where the sum is long beside the columns (22016 to 4096: 232 beside 162 us at 758 rows)."""
    if m <= 0 or m * k >= 1 << 31:
        return False
    tiles = -(-m // 128) * -(-n // 256)
    if transposed:
        return tiles <= 64 and k >= n or tiles <= 128 and k >= 4 * n
    return m <= 128 or tiles <= (256 if fused else 128)


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
        if _by_torch(g):
            return (*_through_torch(lambda t: torch_attention(t, cos, sin, *ctx.shape), (qkv,), (g,)), *none)
        return (ctx.hip.attn_prompt_grad(aligned(rows), aligned(g), sums, cos, sin, *ctx.shape, ctx.scale), *none)


class _Product(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, hip):
        # saved as torch's product saves it: hooks see it, and a change before the backward pass is
        # an error. What was made in inference mode can't be saved
        ctx.w = w if w.is_inference() else None
        if ctx.w is None:
            ctx.save_for_backward(w)
        ctx.hip = hip
        return rows_product(x, w, hip)

    @staticmethod
    def backward(ctx, g):
        w = ctx.saved_tensors[0] if ctx.w is None else ctx.w
        if _by_torch(g, w):
            return torch.matmul(g, w.t()), None, None
        return rows_product(g, aligned(w), ctx.hip, transposed=True), None, None


def rows_product(x, w, hip, transposed=False):
    """x [..., K] times w [K, N], or [..., N] times its transpose: by ops/csrc/gemm.hip where that is
    the faster one, else the library's."""
    k, n = w.shape if not transposed else w.shape[::-1]
    if takes_gemm(x.numel() // k, k, n, transposed):
        return hip.gemm_rows(aligned(x).view(-1, k), w, transposed).view(*x.shape[:-1], n)
    return torch.matmul(x, w.t() if transposed else w)


def norm(x, w, eps, hip):
    return _Norm.apply(x, w, eps, hip)


def product(x, w, hip):
    """x [..., K] times a frozen matrix [K, N]. Autocast may have torch's product in another type."""
    if w.requires_grad or torch.is_autocast_enabled(x.device.type) or not (fused_training(x) and gemm_matrix(w)):
        return torch.matmul(x, w)
    return _Product.apply(x, w, hip)


def add_norm(x, y, w, eps, hip):
    """(x + y, its RMS norm)"""
    return _AddNorm.apply(x, y, w, eps, hip)


def swiglu(gateup, hip):
    """[..., gate | up] -> silu(gate) * up"""
    return _SwiGLU.apply(gateup, hip)


def attention(qkv, cos, sin, start, qh, kh, hd, scale, hip):
    return _Attention.apply(qkv, cos, sin, start, qh, kh, hd, scale, hip)
