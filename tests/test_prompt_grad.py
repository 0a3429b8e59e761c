"""Gradients of what stands between a prompt's products (ops/prompt_grad.py), without a GPU:
the kernels are stood for by torch operations that autograd does not see."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import _disable_current_modes
from torch.utils.flop_counter import FlopCounterMode

from petals_amd.ops import prompt_grad, reference

QH, KH, HD, START = 2, 1, 8, 3
COS, SIN = reference.build_rope_cache(HD, 16)


class Kernels:
    """The kernels' results on plain tensors; like them, it reads memory by its address, and no
    mode sees what it does."""

    def __getattribute__(self, name):
        found = object.__getattribute__(self, name)
        if name.startswith("_") or not callable(found):
            return found

        def unseen(*args):
            with _disable_current_modes():
                return found(*args)

        return unseen

    @staticmethod
    def _plain(*tensors):
        for t in tensors:
            assert t.data_ptr() % 16 == 0 and t.is_contiguous()
        return [t.detach().clone() for t in tensors]

    def _pull(self, function, t, g):
        t, g = self._plain(t, g)
        with torch.enable_grad():
            t.requires_grad_(True)
            return torch.autograd.grad(function(t), t, g)[0]

    def rms_norm(self, x, w, eps):
        return reference.rms_norm(*self._plain(x), w, eps)

    def add_norm_rows(self, x, y, y_bias, w, b, eps):
        x, y = self._plain(x, y)
        return x + y, reference.rms_norm(x + y, w, eps)

    def norm_rows_grad(self, x, w, g, residual, eps):
        d = self._pull(lambda t: reference.rms_norm(t, w, eps), x, g)
        return d if residual is None else d + self._plain(residual)[0]

    def swiglu_rows(self, gateup):
        return reference.swiglu(*self._plain(gateup)[0].chunk(2, dim=-1))

    def swiglu_rows_grad(self, gateup, g):
        return self._pull(lambda t: reference.swiglu(*t.chunk(2, dim=-1)), gateup, g)

    def gemm_rows(self, x, w, transposed=False):
        x, w = self._plain(x, w)
        return x @ (w.t() if transposed else w)

    def rotate_rows(self, qkv, cos, sin, start, qh, kh, hd):
        (qkv,) = self._plain(qkv)
        self.projection = qkv  # what attn_prompt_grad turns its rows back to
        return qkv.clone()

    def attn_prefill_sums(self, q, k, v, scale):
        shape = (START, QH, KH, HD)
        return prompt_grad.torch_attention(self.projection, COS, SIN, *shape).detach(), torch.zeros(1)

    def attn_prompt_grad(self, rows, g, sums, cos, sin, start, qh, kh, hd, scale):
        return self._pull(lambda t: prompt_grad.torch_attention(t, cos, sin, start, qh, kh, hd), rows, g)


HIP = Kernels()
W = torch.rand(16, generator=torch.Generator().manual_seed(0)) + 0.5


def through_kernels(x, a, b, c, d):
    """A llama block without its quantization: what `forward_autograd` composes."""
    n = prompt_grad.norm(x, W, 1e-5, HIP)
    attn = prompt_grad.attention(n @ a, COS, SIN, START, QH, KH, HD, HD**-0.5, HIP)
    h, n = prompt_grad.add_norm(x, attn @ b, W, 1e-5, HIP)
    return h + prompt_grad.swiglu(n @ c, HIP) @ d


def through_torch(x, a, b, c, d):
    attn = prompt_grad.torch_attention(reference.rms_norm(x, W, 1e-5) @ a, COS, SIN, START, QH, KH, HD)
    h = x + attn @ b
    return h + reference.swiglu(*(reference.rms_norm(h, W, 1e-5) @ c).chunk(2, dim=-1)) @ d


def kernel_add_norm(x, y):
    return prompt_grad.add_norm(x, y, W, 1e-5, HIP)


def torch_add_norm(x, y):
    return x + y, reference.rms_norm(x + y, W, 1e-5)


def drawn(*shapes):
    gen = torch.Generator().manual_seed(1)
    return [torch.randn(s, generator=gen) * 0.3 for s in shapes]


def block_inputs():
    x, *weights = drawn((2, 5, 16), (16, (QH + 2 * KH) * HD), (QH * HD, 16), (16, 24), (12, 16))
    return x.requires_grad_(True), weights


def close(got, want):
    assert (got - want).norm() <= 1e-5 * want.norm()  # 32-bit sums


@pytest.mark.parametrize("create_graph", [False, True])
def test_block_gradients(create_graph):
    """Gradients that will have gradients themselves are the same as those that will not."""
    x, weights = block_inputs()
    (want,) = torch.autograd.grad(through_torch(x, *weights).pow(3).sum(), x, create_graph=create_graph)
    (got,) = torch.autograd.grad(through_kernels(x, *weights).pow(3).sum(), x, create_graph=create_graph)
    close(got, want)
    if create_graph:
        close(*(torch.autograd.grad(g.square().sum(), x)[0] for g in (got, want)))


@pytest.mark.parametrize("same", [False, True])
def test_sum_and_norm_of_dependent_rows(same):
    """The second operand is made of the first, or is the first."""
    x, a = drawn((3, 16), (16, 16))
    x.requires_grad_(True)
    got, want = (
        torch.autograd.grad(h.square().sum() + n.pow(3).sum(), x, create_graph=True)[0]
        for h, n in (function(x, x if same else x @ a) for function in (kernel_add_norm, torch_add_norm))
    )
    close(got, want)
    close(*(torch.autograd.grad(g.square().sum(), x)[0] for g in (got, want)))


@pytest.mark.parametrize("first", [False, True])
def test_one_operand_needs_gradients(first):
    """Rows that are frozen beside rows that an adapter, say, has had a part in."""
    x, y = drawn((3, 16), (3, 16))
    leaf = (x if first else y).requires_grad_(True)
    got, want = (
        torch.autograd.grad(sum(t.pow(3).sum() for t in function(x, y)), leaf, create_graph=True)[0]
        for function in (kernel_add_norm, torch_add_norm)
    )
    close(got, want)
    close(*(torch.autograd.grad(g.square().sum(), leaf)[0] for g in (got, want)))


def test_batched_gradients():
    """Several gradients of the result at once (is_grads_batched), as they are one by one."""
    x, weights = block_inputs()
    (grads,) = drawn((3, *x.shape))
    (got,) = torch.autograd.grad(through_kernels(x, *weights), x, grads, is_grads_batched=True)
    (want,) = torch.autograd.grad(through_torch(x, *weights), x, grads, is_grads_batched=True)
    close(got, want)
    by_one = [torch.autograd.grad(through_kernels(x, *weights), x, g)[0] for g in grads]
    close(got, torch.stack(by_one))


def test_traced_gradients():
    """A trace of the backward pass holds operations, not what the kernels once returned."""
    x, weights = block_inputs()
    first, second = drawn((2, *x.shape))[0]
    out = through_kernels(x, *weights)

    def pull(g):
        return torch.autograd.grad(out, x, g, retain_graph=True)[0]

    close(make_fx(pull)(first)(second), pull(second))


def test_what_watches_torch_operations():
    assert not prompt_grad.watched()
    seen = []

    def look(t):
        seen.append(prompt_grad.watched())
        return t * 2

    t = torch.ones(2, 3)
    make_fx(look)(t)
    with FlopCounterMode(display=False):
        look(t)
    torch.func.vmap(look)(t)
    torch.func.grad(lambda u: look(u).sum())(t)
    torch.jit.trace(look, t, check_trace=False)
    with torch.autograd.forward_ad.dual_level():
        look(t)
    assert seen == [True] * 6 and not prompt_grad.watched()
    with FakeTensorMode() as mode:
        fake = mode.from_tensor(t)
    assert prompt_grad.watched(fake) and not prompt_grad.watched(t, torch.nn.Parameter(t))


def test_gradients_of_dual_numbers():
    """The backward pass is linear in the result's gradient: so are the tangents it carries. (That
    of silu has none in torch.)"""
    x, (a, b, _, _) = block_inputs()
    g, tangent = drawn((2, *x.shape))[0]
    attn = prompt_grad.attention(prompt_grad.norm(x, W, 1e-5, HIP) @ a, COS, SIN, START, QH, KH, HD, HD**-0.5, HIP)
    out = prompt_grad.add_norm(x, attn @ b, W, 1e-5, HIP)[1]
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(g, tangent)
        (got,) = torch.autograd.grad(out, x, dual, retain_graph=True)
        value, moved = torch.autograd.forward_ad.unpack_dual(got)
    close(value, torch.autograd.grad(out, x, g, retain_graph=True)[0])
    close(moved, torch.autograd.grad(out, x, tangent)[0])


def test_saved_tensors_from_hooks():
    """Hooks may give back what they were given at another address, as copies from a buffer do."""

    def unpack(t):
        moved = torch.empty(t.numel() + 1, dtype=t.dtype)[1:].view(t.shape)
        return moved.copy_(t)

    x, weights = block_inputs()
    (want,) = torch.autograd.grad(through_kernels(x, *weights).sum(), x)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = through_kernels(x, *weights)
    close(torch.autograd.grad(out.sum(), x)[0], want)


def test_products_with_a_frozen_matrix(monkeypatch):
    """Rows, their gradients, gradients of these and batches of them, whichever kernel multiplies."""
    w = torch.randn(64, 128, generator=torch.Generator().manual_seed(1), dtype=torch.float64)
    x, v, u = (torch.randn(2, 3, n, dtype=torch.float64) for n in (64, 128, 64))
    for takes in (False, True):
        monkeypatch.setattr(prompt_grad, "takes_gemm", lambda *sizes: takes)

        def product(t):
            return prompt_grad._Product.apply(t, w, HIP)

        leaf = x.clone().requires_grad_(True)
        y = product(leaf)
        torch.testing.assert_close(y, x @ w)
        (g,) = torch.autograd.grad(y, leaf, v, retain_graph=True)
        torch.testing.assert_close(g, v @ w.t())
        cut = v.clone().requires_grad_(True)
        (g,) = torch.autograd.grad(y, leaf, cut, retain_graph=True, create_graph=True)
        torch.testing.assert_close(torch.autograd.grad(g, cut, u)[0], u @ w)
        many = torch.stack([v, 2 * v])
        (g,) = torch.autograd.grad(y, leaf, many, is_grads_batched=True)
        torch.testing.assert_close(g, many @ w.t())


@pytest.mark.parametrize("takes", [False, True])
def test_frozen_matrix_is_saved(monkeypatch, takes):
    """As by torch's product: hooks pack and unpack it, maybe to another address, and changing it
    before the backward pass is an error."""
    monkeypatch.setattr(prompt_grad, "takes_gemm", lambda *sizes: takes)
    w = torch.randn(64, 128, dtype=torch.float64)
    x, v = (torch.randn(3, n, dtype=torch.float64) for n in (64, 128))
    x.requires_grad_(True)

    def unpack(t):
        moved = torch.empty(t.numel() + 1, dtype=t.dtype)[1:].view(t.shape)
        return moved.copy_(t)

    for product in (torch.matmul, lambda a, b: prompt_grad._Product.apply(a, b, HIP)):
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, unpack):
            y = product(x, w)
        assert any(t.data_ptr() == w.data_ptr() for t in packed)
        torch.testing.assert_close(torch.autograd.grad(y, x, v)[0], v @ w.t())
        y = product(x, w)
        w.mul_(2)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(y, x, v)
    with torch.inference_mode():
        constant = w.clone()
    y = prompt_grad._Product.apply(x, constant, HIP)
    torch.testing.assert_close(torch.autograd.grad(y, x, v)[0], v @ w.t())


def test_products_of_rows_that_do_not_fit(monkeypatch):
    """Rows of another length are refused, also where there are whole ones of the matrix's in all."""
    monkeypatch.setattr(prompt_grad, "takes_gemm", lambda *sizes, **kinds: True)
    w = torch.randn(64, 128, dtype=torch.float64)
    for rows in (torch.randn(2, 3, 128, dtype=torch.float64), torch.randn(4, 32, dtype=torch.float64)):
        with pytest.raises(RuntimeError, match="mat"):
            prompt_grad._Product.apply(rows, w, HIP)
    y = prompt_grad._Product.apply(torch.randn(4, 64, dtype=torch.float64, requires_grad=True), w, HIP)
    assert y.shape == (4, 128)


@pytest.mark.parametrize("takes", [False, True])
def test_products_ahead_of_a_router(monkeypatch, takes):
    """Their sums keep their order, and tiles that have another one are not asked; gradients have the fastest ones."""
    monkeypatch.setattr(prompt_grad, "takes_gemm", lambda *sizes: takes)
    monkeypatch.setattr(prompt_grad, "takes_wide_gemm", lambda *sizes: True)
    asked = []

    class Watched(Kernels):
        def gemm_rows(self, x, w, transposed=False, epilogue=0, residual=None, bias=None, tile=-1, steady=False):
            asked.append((transposed, steady))
            return x @ (w.t() if transposed else w)

    w = torch.randn(64, 128, dtype=torch.float64)
    x = torch.randn(3, 64, dtype=torch.float64, requires_grad=True)
    y = prompt_grad._Product.apply(x, w, Watched(), True)
    torch.testing.assert_close(y, x @ w)
    torch.testing.assert_close(torch.autograd.grad(y, x, y)[0], y @ w.t())
    assert asked == [(False, True)] * takes + [(True, False)]


def test_attention_gradients_of_the_widest_rows():
    """Rows of 2^24 numbers, which the kernels' offsets don't reach, have the gradients of torch operations."""
    hd, kh = 64, 1 << 16
    qh, tables = 2 * kh, (torch.ones(1, hd), torch.zeros(1, hd))

    class Narrow(Kernels):
        def attn_prefill_sums(self, q, k, v, scale):
            return v.repeat_interleave(2, 1).transpose(1, 2).flatten(2), torch.zeros(1)  # one key has all the weight

        def attn_prompt_grad(self, rows, g, *rest):
            raise RuntimeError("too many rows at once")

    qkv = torch.randn(1, 1, (qh + 2 * kh) * hd, generator=torch.Generator().manual_seed(1)).requires_grad_(True)
    out = prompt_grad.attention(qkv, *tables, 0, qh, kh, hd, hd**-0.5, Narrow())
    (got,) = torch.autograd.grad(out, qkv, torch.ones_like(out))
    want = torch.zeros(qkv.shape)
    want[..., -kh * hd :] = 2
    assert torch.equal(got, want)


def test_products_with_a_matrix_without_rows():
    """Sums of nothing are zeros, as by torch's product; rows of some length don't fit."""
    from types import SimpleNamespace

    from petals_amd.ops.fused_decode import prompt_product

    w = torch.ones(0, 128, dtype=torch.float64)
    weight = SimpleNamespace(shape=w.shape, tiles=None, dense=lambda: w)
    for product in (lambda x: prompt_product(HIP, x, weight), lambda x: prompt_grad._Product.apply(x, w, HIP)):
        assert torch.equal(product(torch.ones(2, 3, 0, dtype=torch.float64)), torch.zeros(2, 3, 128, dtype=torch.float64))
        with pytest.raises(RuntimeError, match="mat"):
            product(torch.ones(3, 64, dtype=torch.float64))


def test_products_under_autocast(monkeypatch):
    """They come in the type that autocast gives torch's products, with gradients. Devices that have
    no autocast are not asked for it."""
    shapes = (torch.ones(*s, device="meta", dtype=torch.bfloat16) for s in ((3, 64), (64, 128)))
    assert prompt_grad.product(*shapes, HIP).shape == (3, 128)
    for rule in ("fused_training", "gemm_matrix"):
        monkeypatch.setattr(prompt_grad, rule, lambda *tensors: True)
    w = torch.randn(64, 128).bfloat16()
    x = torch.randn(2, 3, 64).bfloat16().requires_grad_(True)
    for kind in (torch.float16, torch.bfloat16):
        with torch.autocast("cpu", kind):
            y = prompt_grad.product(x, w, HIP)
            want = torch.matmul(x, w)
        assert y.dtype == want.dtype == kind and torch.equal(y, want)
        g = torch.randn(y.shape).to(kind)
        assert torch.equal(*(torch.autograd.grad(t, x, g)[0] for t in (y, want)))


@pytest.mark.parametrize("rows", [1, 128, 129, 758, 1024, 1025])
def test_rule_of_products(rows):
    # many rows of a wide matrix are the library's, few rows and sums that are long are the kernel's
    assert prompt_grad.takes_gemm(rows, 16384, 4096) == (rows <= 1024)
    assert prompt_grad.takes_gemm(rows, 4096, 28672) == (rows <= 128)
    assert prompt_grad.takes_gemm(rows, 22016, 4096, transposed=True) == (rows <= 1024)
    assert prompt_grad.takes_gemm(rows, 4096, 11008, transposed=True) is False
    assert not prompt_grad.takes_gemm(0, 64, 64)
