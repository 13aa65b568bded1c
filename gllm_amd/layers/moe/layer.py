"""Fused MoE layer (reference: layers/moe/fused_moe_triton/layer.py).

Round-1 compute path: expert-loop gather/scatter over hipBLASLt GEMMs —
correct on CPU and GPU, TP-sharded intermediate dim. The CDNA4 grouped
MFMA GEMM kernel (sorted token ids, block-aligned, tuned per (E, N))
replaces the loop in the optimization pass. EP: contiguous expert shards
with a trailing EP all-reduce (reference layer.py:686-735 — the
reference's EP comm is allgather+allreduce, not all-to-all).
"""

from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from gllm_amd import ops
from gllm_amd.parallel import (get_ep_rank, get_ep_size, get_tp_rank,
                               get_tp_size, tensor_parallel_all_reduce)


class FusedMoE(nn.Module):
    def __init__(self, num_experts: int, top_k: int, hidden_size: int,
                 intermediate_size: int, renormalize: bool = True,
                 use_ep: bool = False, params_dtype=None,
                 activation: str = "silu_glu",
                 fp32_routing_weights: bool = False,
                 act_limit: float = 0.0, act_alpha: float = 1.702):
        """``activation``: "silu_glu" — gated experts, w13 holds gate
        and up rows, act = silu(gate) * up; "relu2" — ungated experts,
        w13 holds the up rows only, act = max(z, 0)^2; "swiglu_clamp" —
        gated experts with clamped pre-activations: g = min(gate,
        act_limit), u = clamp(up, +-act_limit), act = g * sigmoid(
        act_alpha g) * (u + 1).
        ``fp32_routing_weights``: keep the routing weights in fp32 up to
        the weighted sum in the segment loop too, instead of rounding them
        to the model dtype (the grouped GEMMs always take them in fp32)."""
        super().__init__()
        assert activation in ("silu_glu", "relu2", "swiglu_clamp")
        self.activation = activation
        self.act_args = (float(act_limit), float(act_alpha)) \
            if activation == "swiglu_clamp" else ()
        self.gated = activation != "relu2"
        self.fp32_routing_weights = fp32_routing_weights
        dtype = params_dtype or torch.get_default_dtype()
        self.num_experts = num_experts
        self.top_k = top_k
        self.hidden_size = hidden_size
        self.renormalize = renormalize
        self.use_ep = use_ep

        if use_ep:
            ep_rank, ep_size = get_ep_rank(), get_ep_size()
            base, rem = divmod(num_experts, ep_size)
            counts = [base + (1 if r < rem else 0) for r in range(ep_size)]
            self.expert_start = sum(counts[:ep_rank])
            self.num_local_experts = counts[ep_rank]
            self.intermediate_per_rank = intermediate_size
        else:
            self.expert_start = 0
            self.num_local_experts = num_experts
            tp = get_tp_size()
            assert intermediate_size % tp == 0
            self.intermediate_per_rank = intermediate_size // tp

        I = self.intermediate_per_rank
        self.w13_weight = nn.Parameter(
            torch.empty(self.num_local_experts,
                        (2 if self.gated else 1) * I, hidden_size,
                        dtype=dtype), requires_grad=False)
        self.w2_weight = nn.Parameter(
            torch.empty(self.num_local_experts, hidden_size, I, dtype=dtype),
            requires_grad=False)
        self.w13_weight.weight_loader = self._load_w13
        self.w2_weight.weight_loader = self._load_w2
        # set by quantization/ converters (convert_moe_to_{fp8,int4}
        # / convert_moe_to_int4_packed)
        self.fp8_block = None
        self.int4_cfg = None
        self.int4_packed = None
        self._dq_cache = None

    # ---- loading: per-expert pulls with EP ownership / TP sharding ----
    def _local_expert(self, expert_id: int) -> Optional[int]:
        lid = expert_id - self.expert_start
        if 0 <= lid < self.num_local_experts:
            return lid
        return None

    def _load_w13(self, param, loaded, expert_id: int, shard_id: int):
        """shard_id: 0 = gate (w1), 1 = up (w3); ungated experts have
        the up rows only (shard 0)."""
        assert self.gated or shard_id == 0
        lid = self._local_expert(expert_id)
        if lid is None:
            return
        I = self.intermediate_per_rank
        if self.use_ep:
            shard = loaded
        else:
            shard = loaded.narrow(0, get_tp_rank() * I, I)
        param.data[lid].narrow(0, shard_id * I, I).copy_(shard)

    def _load_w2(self, param, loaded, expert_id: int):
        lid = self._local_expert(expert_id)
        if lid is None:
            return
        I = self.intermediate_per_rank
        if self.use_ep:
            shard = loaded
        else:
            shard = loaded.narrow(1, get_tp_rank() * I, I)
        param.data[lid].copy_(shard)

    # ---- forward ----
    def forward(self, x: torch.Tensor,
                router_logits: torch.Tensor) -> torch.Tensor:
        weights, ids = ops.topk_softmax(router_logits, self.top_k,
                                        self.renormalize)  # [T,K], [T,K]
        return self.forward_routed(x, weights, ids)

    def forward_routed(self, x: torch.Tensor, weights: torch.Tensor,
                       ids: torch.Tensor) -> torch.Tensor:
        """Expert compute with externally computed routing (DeepSeek
        grouped-topk / routed scaling paths)."""
        from gllm_amd.parallel import get_dp_size
        if self.use_ep and get_dp_size() > 1:
            return self._forward_dp(x, weights, ids)
        out = self._expert_loop(x, weights, ids)
        if self.use_ep:
            from gllm_amd.parallel.state import ep_all_reduce
            out = ep_all_reduce(out)
        else:
            out = tensor_parallel_all_reduce(out)
        return out

    def routed_add_norm(self, x: torch.Tensor, weights: torch.Tensor,
                        ids: torch.Tensor, shared, residual: torch.Tensor,
                        norm):
        """(norm(residual + (forward_routed(...) + shared)), that sum): one
        kernel behind the experts where nothing has to be reduced over
        ranks first. ``shared``: a tensor, a gated feed-forward of x (beside
        the experts where that is the faster) or None."""
        one_rank = (get_ep_size() if self.use_ep else get_tp_size()) == 1
        if isinstance(shared, nn.Module):
            mlp = shared.weights_beside(x)
            if (mlp is not None and one_rank and get_tp_size() == 1
                    and self.activation == "silu_glu" and self._grouped(x)
                    and ops.moe_add_norm_ok(x, None, residual, norm.scale())
                    and ops.moe_shared_beside(x, self.w13_weight,
                                              self.w2_weight, ids.shape[1],
                                              *mlp)):
                out = ops.fused_moe(
                    x, self.w13_weight, self.w2_weight, weights, ids,
                    expert_start=self.expert_start,
                    num_global_experts=self.num_experts,
                    add_norm=(None, residual, norm.scale(), norm.eps),
                    shared_mlp=mlp)
                return out, residual
            shared = shared(x)
        if (one_rank and self._grouped(x)
                and ops.moe_add_norm_ok(x, shared, residual, norm.scale())):
            out = ops.fused_moe(
                x.contiguous(), self.w13_weight, self.w2_weight, weights,
                ids, expert_start=self.expert_start,
                num_global_experts=self.num_experts,
                activation=self.activation, act_args=self.act_args,
                add_norm=(shared, residual, norm.scale(), norm.eps))
            return out, residual
        out = self.forward_routed(x, weights, ids)
        if shared is not None:
            out = out + shared
        return norm(out, residual)

    def _grouped(self, x: torch.Tensor) -> bool:
        """Unquantized experts for the grouped bf16 product (it loads
        8-element vectors along K; odd widths take the segment loop)."""
        return (x.is_cuda and x.dtype == torch.bfloat16
                and ops.has_moe_kernels() and self.int4_packed is None
                and self.fp8_block is None and self.int4_cfg is None
                and x.shape[1] % 8 == 0
                and self.intermediate_per_rank % 8 == 0)

    def _expert_loop(self, x: torch.Tensor, weights: torch.Tensor,
                     ids: torch.Tensor) -> torch.Tensor:
        """Local expert shard over the (possibly DP-gathered) batch;
        returns the PARTIAL output (no collectives).

        GPU + bf16 experts -> the grouped MFMA GEMM pipeline
        (ops.fused_moe): device-side align, no host syncs, hipGraph-
        safe. CPU and quantized banks keep the sort+segment host loop.

        Host analogue of the reference's moe_align_block_size
        (_custom_ops.py): ONE stable sort groups the (token, expert)
        pairs by expert and ONE bincount transfer gives the segment
        table, so the loop only issues GEMMs for experts that actually
        received tokens — no per-expert device sync (the old
        ``sel.any()`` form synced once per expert: 256/layer on
        DeepSeek-V3). DP padding rows carry expert id -1 and land in
        segment 0 of the shifted bincount (skipped)."""
        if (x.is_cuda and x.dtype == torch.bfloat16
                and ops.has_moe_kernels()):
            if self.int4_packed is not None:
                # compressed-tensors int4 experts (Kimi-K2.5): run the
                # bf16 grouped MFMA GEMM over a one-time dequantized
                # shadow bank (288 GB HBM covers it; the group-32
                # native packed kernel is a ROADMAP item)
                if getattr(self, "_dq_stack", None) is None:
                    from gllm_amd.layers.quantization.int4 import                         dequant_ct_int4
                    g = self.int4_packed[1]
                    self._dq_stack = tuple(
                        torch.stack([
                            dequant_ct_int4(wp[e], ws[e], g, x.dtype)
                            for e in range(self.num_local_experts)
                        ]).contiguous()
                        for wp, ws in
                        ((self.w13_weight_packed, self.w13_weight_scale),
                         (self.w2_weight_packed, self.w2_weight_scale)))
                w13s, w2s = self._dq_stack
                return ops.fused_moe(
                    x.contiguous(), w13s, w2s, weights, ids,
                    expert_start=self.expert_start,
                    num_global_experts=self.num_experts)
            if self._grouped(x):
                return ops.fused_moe(
                    x.contiguous(), self.w13_weight, self.w2_weight,
                    weights, ids, expert_start=self.expert_start,
                    num_global_experts=self.num_experts,
                    activation=self.activation, act_args=self.act_args)
            if (self.fp8_block == (128, 128)
                    and x.shape[1] % 128 == 0
                    and self.intermediate_per_rank % 128 == 0):
                # e4m3-resident grouped GEMM (no dequant cache at all)
                return ops.fused_moe_fp8(
                    x.contiguous(), self.w13_weight,
                    self.w13_weight_scale_inv, self.w2_weight,
                    self.w2_weight_scale_inv, weights, ids,
                    expert_start=self.expert_start)
            if (self.int4_cfg is not None and self.int4_cfg[1] == 128
                    and x.shape[1] % 128 == 0
                    and self.intermediate_per_rank % 128 == 0):
                # packed-nibble grouped GEMM (w4a16, no dequant banks)
                if getattr(self, "_i4_banks", None) is None:
                    from gllm_amd.layers.quantization.int4 import \
                        repack_canonical_moe
                    w13c, w13sb, w2c, w2sb, _ = repack_canonical_moe(self)
                    self._i4_banks = (w13c.to(x.device), w13sb.to(x.device),
                                      w2c.to(x.device), w2sb.to(x.device))
                w13c, w13sb, w2c, w2sb = self._i4_banks
                return ops.fused_moe_int4(
                    x.contiguous(), w13c, w13sb, w2c, w2sb, weights, ids,
                    expert_start=self.expert_start)
        if not self.fp32_routing_weights:
            weights = weights.to(x.dtype)
        T = x.shape[0]
        out = torch.zeros_like(x)
        acc = torch.zeros(x.shape, dtype=torch.float32, device=x.device) \
            if weights.dtype != x.dtype else None
        flat_ids = ids.long().flatten()                    # [T*K]
        flat_rows = torch.arange(T, device=x.device).repeat_interleave(
            self.top_k)
        order = torch.argsort(flat_ids, stable=True)
        counts = torch.bincount(flat_ids + 1,
                                minlength=self.num_experts + 1)
        counts_host = counts.tolist()                      # single sync
        flat_w = weights.flatten()
        start = sum(counts_host[:self.expert_start + 1])
        for lid in range(self.num_local_experts):
            eid = self.expert_start + lid
            c = counts_host[eid + 1]
            if c == 0:
                continue
            sel = order.narrow(0, start, c)
            start += c
            rows = flat_rows[sel]
            xe = x.index_select(0, rows)
            if (self.fp8_block is not None or self.int4_cfg is not None
                    or self.int4_packed is not None):
                w13, w2 = self._dequant_expert(lid, x.dtype, x.device)
            else:
                w13, w2 = self.w13_weight[lid], self.w2_weight[lid]
            h = ops.linear(xe, w13)
            if self.activation == "swiglu_clamp":
                h = ops.clamp_swiglu(h, *self.act_args)
            else:
                h = ops.silu_and_mul(h) if self.gated else ops.relu2(h)
            ye = ops.linear(h, w2)
            w = flat_w[sel].unsqueeze(-1)
            if w.dtype != ye.dtype:       # fp32 routing weights
                acc.index_add_(0, rows, ye.float() * w)
            else:
                out.index_add_(0, rows, ye * w)
        if acc is not None:
            return acc.to(x.dtype)
        return out

    def _dequant_expert(self, lid: int, dtype, device):
        """Quantized expert weights dequantized into the compute dtype.

        The FULL local bank materializes on first touch (not lazily
        per-expert): the first forward is the model runner's profile
        run, so the dequant footprint is resident before KV-cache
        sizing and can never OOM mid-serving.
        The grouped fp8 MFMA GEMM consuming the packed layout directly
        replaces this."""
        if self._dq_cache is None:
            self._dq_cache = [None] * self.num_local_experts
            for other in range(self.num_local_experts):
                if other != lid:
                    self._dequant_expert(other, dtype, device)
        ent = self._dq_cache[lid]
        if ent is None:
            if self.int4_packed is not None:
                from gllm_amd.layers.quantization.int4 import \
                    dequant_ct_int4
                g = self.int4_packed[1]
                w13 = dequant_ct_int4(self.w13_weight_packed[lid],
                                      self.w13_weight_scale[lid], g,
                                      dtype).to(device)
                w2 = dequant_ct_int4(self.w2_weight_packed[lid],
                                     self.w2_weight_scale[lid], g,
                                     dtype).to(device)
            elif self.fp8_block is not None:
                from gllm_amd.layers.quantization.fp8 import \
                    dequant_block_fp8
                w13 = dequant_block_fp8(
                    self.w13_weight[lid], self.w13_weight_scale_inv[lid],
                    self.fp8_block, dtype).to(device)
                w2 = dequant_block_fp8(
                    self.w2_weight[lid], self.w2_weight_scale_inv[lid],
                    self.fp8_block, dtype).to(device)
            else:
                from gllm_amd.layers.quantization.int4 import (dequant_awq,
                                                               dequant_gptq)
                method, group = self.int4_cfg
                fn = dequant_gptq if method == "gptq" else dequant_awq
                w13 = fn(self.w13_qweight[lid], self.w13_qzeros[lid],
                         self.w13_scales[lid], group, dtype).to(device)
                w2 = fn(self.w2_qweight[lid], self.w2_qzeros[lid],
                        self.w2_scales[lid], group, dtype).to(device)
            ent = (w13, w2)
            self._dq_cache[lid] = ent
        return ent

    def _forward_dp(self, x: torch.Tensor, weights: torch.Tensor,
                    ids: torch.Tensor) -> torch.Tensor:
        """DP-attention MoE: experts span replicas (EP = DP x TP), so the
        routed batch is the union over replicas (reference
        models/utils.py:39-96 dp_ep_moe_routed). Every replica pads its
        rows to the round's max count (published by the engine's
        dp_meta_barrier), all-gathers tokens + routing over the DP
        group, computes its local expert shard on the GLOBAL batch, and
        one EP all-reduce over the stage yields the full output
        everywhere; each replica slices back its own rows. Padding rows
        carry expert id -1 (never matched) so they contribute zeros."""
        from gllm_amd.parallel import (dp_all_gather, get_dp_forward_counts,
                                       get_dp_rank)
        from gllm_amd.parallel.state import ep_all_reduce
        counts = get_dp_forward_counts()
        assert counts is not None, \
            "DP MoE forward entered without dp_meta_barrier counts"
        T = x.shape[0]
        maxc = max(counts + [T])

        def pad(t, fill):
            if T == maxc:
                return t.contiguous()
            tail = torch.full((maxc - T,) + tuple(t.shape[1:]), fill,
                              dtype=t.dtype, device=t.device)
            return torch.cat([t, tail], dim=0)

        gx = dp_all_gather(pad(x, 0))
        gw = dp_all_gather(pad(weights.to(x.dtype), 0))
        gids = dp_all_gather(pad(ids.long(), -1))
        out = self._expert_loop(gx, gw, gids)
        out = ep_all_reduce(out)
        start = get_dp_rank() * maxc
        return out[start:start + T]
