"""MI355X fast path for Mixtral blocks: fused Llama-style attention decode +
device-routed expert GEMVs.

Decode routing runs entirely ON the GPU (router gemm -> softmax -> top-k ->
int32 expert ids in a device tensor) and the expert GEMVs read their expert's
stacked weights through that tensor (ops/csrc/moe.hip), so there is no host
sync per step and the whole span is hipGraph-capturable (graph_safe) for the
bf16 and NF4 quantizations. Each selected expert's weights are read exactly
once per token — the decode-time degenerate case of a grouped GEMM.

(The reference runs Mixtral experts densely inside one server's HF block with
host-side routing: reference models/mixtral/block.py:73-81.)

int8 expert weights keep the host-routed per-expert GEMV path
(graph_safe = False).
"""

from __future__ import annotations

from typing import List, Optional

import torch
import torch.nn.functional as F

from petals_amd.ops import prompt_grad
from petals_amd.ops.fused_decode import (
    _EPI_PLAIN_F32,
    _EPI_RAW,
    _EPI_SWIGLU_F32,
    LlamaFastPath,
    _FastWeight,
    _dequant_cached,
    _vector,
)


MOE_GEMM_MT = 32  # rows of a tile of one expert (ops/csrc/moe.hip MOE_MT)


class _CacheKey:
    """Weakref-able identity key for the dequant LRU (plain object() cannot
    carry weak references, which _dequant_cached uses for eviction)."""

    __slots__ = ("__weakref__",)


class _StackedExperts:
    """All experts' transposed [in, out] weights stacked on a leading expert
    axis, in the exact layout the moe.hip kernels stream."""

    def __init__(self, t_list: List[torch.Tensor], hip, quant: str):
        self.hip = hip
        self.quant = quant
        self.in_dim, self.out_dim = t_list[0].shape
        if quant == "nf4":
            tiles, scales = zip(*(hip.nf4_tile(*hip.nf4_quantize(t.contiguous())) for t in t_list))
            self.tiles_all, self.scales_all = torch.stack(tiles), torch.stack(scales)
        else:
            assert quant == "none"
            self.wt_all = torch.stack([t.contiguous() for t in t_list]).contiguous()
        # per-expert identity keys for the dequant LRU (fused_decode._dequant_cached
        # keys by object id): multi-chunk prefills reuse each expert's dense form
        self._cache_keys = [_CacheKey() for _ in t_list]

    def moe_gemv(self, x: torch.Tensor, sel: torch.Tensor, k_per_tok: int, ws: torch.Tensor,
                 epilogue: int) -> torch.Tensor:
        if self.quant == "nf4":
            return self.hip.gemv_nf4_tiles_moe(
                self.tiles_all, self.scales_all, self.in_dim, x, sel, k_per_tok, ws, epilogue
            )
        return self.hip.gemv_bf16_moe(self.wt_all, x, sel, k_per_tok, ws, epilogue)

    def moe_gemm(self, x: torch.Tensor, sorted_pairs: torch.Tensor, tile_expert: torch.Tensor,
                 k_per_tok: int, n_rows: int) -> torch.Tensor:
        """Grouped MFMA GEMM (prefill): C[pair] = x[pair // k] @ W[expert(pair)]."""
        if self.quant == "nf4":
            return self.hip.moe_gemm(None, self.tiles_all, self.scales_all, x,
                                     sorted_pairs, tile_expert, k_per_tok, n_rows)
        return self.hip.moe_gemm(self.wt_all, None, None, x, sorted_pairs, tile_expert,
                                 k_per_tok, n_rows)

    @property
    def gemm_ok(self) -> bool:
        return self.out_dim % 128 == 0 and self.in_dim % 64 == 0

    def dense(self, e: int) -> torch.Tensor:
        """Expert e as a dense bf16 [in, out] (prefill/training matmuls),
        LRU-cached so chunked prefills pay the dequant once per expert."""
        if self.quant == "nf4":
            return _dequant_cached(
                self._cache_keys[e],
                lambda: self.hip.nf4_untile(self.tiles_all[e], self.scales_all[e], self.in_dim),
            )
        return self.wt_all[e]


class MixtralFastPath(LlamaFastPath):
    # the router consumes the true ln2-weighted normed activations (softmax is
    # not scale-invariant), so the MLP norm cannot fold into expert weights
    supports_fold_norm = False
    dense_mlp = False

    def _init_mlp_weights(self, block, hip_ops, quant):
        def t(w):
            return w.detach().to(torch.bfloat16).t().contiguous()

        moe = block.block_sparse_moe
        self.top_k = moe.top_k
        self.num_experts = moe.num_experts
        self.w_router = _vector(moe.gate.weight)  # [E, H]
        self.w_router_t = self.w_router.t()
        self.stacked_gu: Optional[_StackedExperts] = None
        self.stacked_down: Optional[_StackedExperts] = None
        self.wgateup_e: List[_FastWeight] = []
        self.wdown_e: List[_FastWeight] = []
        if quant in ("none", "nf4"):
            gu_list = [torch.cat([t(e.w1.weight), t(e.w3.weight)], dim=1) for e in moe.experts]
            down_list = [t(e.w2.weight) for e in moe.experts]
            self.stacked_gu = _StackedExperts(gu_list, hip_ops, quant)
            self.stacked_down = _StackedExperts(down_list, hip_ops, quant)
            self.graph_safe = True  # device-routed decode: capturable
        else:
            for expert in moe.experts:
                self.wgateup_e.append(
                    _FastWeight(torch.cat([t(expert.w1.weight), t(expert.w3.weight)], dim=1), hip_ops, quant)
                )
                self.wdown_e.append(_FastWeight(t(expert.w2.weight), hip_ops, quant))
            self.graph_safe = False  # host-routed fallback
        for expert in moe.experts:
            for lin in (expert.w1, expert.w2, expert.w3):
                lin.weight.data = self._empty_bf16
        moe.gate.weight.data = self._empty_bf16

    def _max_gemv_out(self) -> int:
        gu_out = self.stacked_gu.out_dim if self.stacked_gu is not None else self.wgateup_e[0].shape[1]
        return max(gu_out, self.wqkv_t.shape[1], self.wo_t.shape[1])

    def widest_row(self) -> int:
        return self.top_k * self._max_gemv_out()  # a row per chosen expert

    def _takes_router(self, x: torch.Tensor) -> bool:
        """Rows and experts that the router's kernel takes."""
        return x.is_cuda and x.shape[1] % 8 == 0 and self.num_experts <= 256 and self.top_k <= 16

    def _route(self, xn2: torch.Tensor):
        """Router on [tokens, H] f32/bf16 -> (weights [t, k] f32, experts [t, k]), differentiable.
        Logits in 32 bits as in the kernel, and the kernel's choice where it can be asked, so that
        gradients go through the experts that the forward pass runs.
        All-device: safe inside hipGraph capture."""
        selected = None
        if self._takes_router(xn2) and not prompt_grad.watched(xn2):
            weights, selected = self._route_rows(xn2.detach())
            selected = selected.long()
            if not (torch.is_grad_enabled() and xn2.requires_grad):
                return weights, selected
        logits = xn2.float() @ self.w_router_t.float()
        if selected is None:
            selected = torch.topk(logits, self.top_k, dim=-1)[1]
        # a softmax over all, renormalized over the chosen
        return F.softmax(logits.gather(1, selected), dim=-1), selected

    def _route_rows(self, x: torch.Tensor):
        """Router on [tokens, H]: (weights [t, k] f32, experts [t, k] int32), one launch
        for as many experts as the kernel takes."""
        if self._takes_router(x):
            return self.hip.moe_route(prompt_grad.aligned(x), self.w_router, self.top_k)
        weights, selected = self._route(x)
        return weights.contiguous(), selected.to(torch.int32).contiguous()

    def _mlp_decode(self, xn2, h2, ws, adapter):
        """xn2 f32 [B, H]; returns h3 bf16 [B, H]."""
        B = xn2.shape[0]
        if self.stacked_gu is not None:
            weights, sel = self._route_rows(xn2.contiguous())
            sel = sel.view(-1)  # [B*k]
            act = self.stacked_gu.moe_gemv(xn2.contiguous(), sel, self.top_k, ws, _EPI_SWIGLU_F32)
            parts = self.stacked_down.moe_gemv(act, sel, 1, ws, _EPI_RAW)
            return self.hip.moe_combine(parts, weights, h2)
        weights, selected = self._route(xn2)

        # int8: host-synced routing (~10 us, amortized against MBs of expert reads)
        sel_l = selected.tolist()
        w_l = weights.tolist()
        moe_out = torch.zeros_like(xn2)  # f32 [B, H]
        for b in range(B):
            xb = xn2[b : b + 1].contiguous()
            for j in range(self.top_k):
                e = sel_l[b][j]
                act = self.wgateup_e[e].gemv(xb, ws, None, _EPI_SWIGLU_F32)  # [1, I] f32
                down = self.wdown_e[e].gemv(act, ws, None, _EPI_PLAIN_F32)  # [1, H] f32
                moe_out[b] += down[0] * w_l[b][j]
        return (h2.float() + moe_out).to(torch.bfloat16)

    def _expert_dense(self, e: int) -> torch.Tensor:
        return self.stacked_gu.dense(e) if self.stacked_gu is not None else self.wgateup_e[e].dense()

    def _expert_down_dense(self, e: int) -> torch.Tensor:
        return self.stacked_down.dense(e) if self.stacked_down is not None else self.wdown_e[e].dense()

    def _mlp_prompt(self, h2, xn2, adapter, x_delta):
        """Prompts run the grouped MFMA GEMM (ops/csrc/moe.hip moe_gemm: NF4 dequant fused
        into the staging, so packed weights are what crosses HBM)."""
        stacked = self.stacked_gu is not None and self.stacked_gu.gemm_ok and self.stacked_down.gemm_ok
        if not stacked or xn2.device.type != "cuda" or self.tp_world > 1:
            return super()._mlp_prompt(h2, xn2, adapter, x_delta)
        x = xn2.reshape(-1, xn2.shape[-1]).contiguous()
        weights, sel = self._route_rows(x)
        order, tile_expert = self.hip.moe_group(sel.view(-1), self.num_experts, MOE_GEMM_MT)
        gateup = self.stacked_gu.moe_gemm(x, order, tile_expert, self.top_k, sel.numel())
        down = self.stacked_down.moe_gemm(self.hip.swiglu_rows(gateup), order, tile_expert, 1, sel.numel())
        return self.hip.moe_combine(down, weights, h2.reshape(x.shape[0], -1)).view(h2.shape)

    def _mlp_dense(self, xn2, adapter, autograd: bool, x_delta=None):
        """MLP over the routed experts by token-grouped dense matmuls: training, CPU, and
        geometries or quantizations that the grouped GEMM does not take."""
        shape = xn2.shape
        x = xn2.reshape(-1, shape[-1])
        weights, selected = self._route(x)
        out_dim = self.stacked_down.out_dim if self.stacked_down is not None else self.wdown_e[0].shape[1]
        out = torch.zeros(x.shape[0], out_dim, dtype=torch.float32, device=x.device)
        expert_mask = F.one_hot(selected, num_classes=self.num_experts).permute(2, 1, 0)
        for e in range(self.num_experts):
            k_idx, tok_idx = torch.where(expert_mask[e])
            if tok_idx.numel() == 0:
                continue
            xe = x[tok_idx].to(torch.bfloat16)
            gateup = xe @ self._expert_dense(e)
            inter = gateup.shape[-1] // 2
            act = F.silu(gateup[..., :inter].float()) * gateup[..., inter:].float()
            down = act.to(torch.bfloat16) @ self._expert_down_dense(e)
            out.index_add_(0, tok_idx, down.float() * weights[tok_idx, k_idx, None])
        return out.reshape(*shape[:-1], -1).to(xn2.dtype)
