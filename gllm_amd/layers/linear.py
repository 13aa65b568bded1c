"""Megatron-style tensor-parallel linear layers.

Parity with the reference's layers/linear.py (Row/Column/Merged/QKV/
Replicated). GEMMs go through torch.nn.functional.linear → hipBLASLt on
ROCm (plain library GEMMs; the fused hot ops are the hand-written HIP
kernels in ops/). Weight sharding happens at load time via a
``weight_loader`` attribute attached to each parameter.
"""

from typing import List

import torch
import torch.nn as nn
import torch.nn.functional as F

from gllm_amd import ops
from gllm_amd.parallel import (get_tp_rank, get_tp_size,
                               tensor_parallel_all_reduce)


def _narrow_copy(param_data: torch.Tensor, loaded: torch.Tensor,
                 dim: int, rank: int, size: int):
    shard = loaded.shape[dim] // size
    param_data.copy_(loaded.narrow(dim, rank * shard, shard))


class LinearBase(nn.Module):
    def __init__(self, input_size: int, output_size: int, bias: bool,
                 params_dtype=None):
        super().__init__()
        self.input_size = input_size
        self.output_size = output_size
        dtype = params_dtype or torch.get_default_dtype()
        self.weight = nn.Parameter(
            torch.empty(output_size, input_size, dtype=dtype),
            requires_grad=False)
        if bias:
            self.bias = nn.Parameter(torch.empty(output_size, dtype=dtype),
                                     requires_grad=False)
        else:
            self.register_parameter("bias", None)
        # set by quantization/{fp8,int4}.py converters
        self.fp8_block = None
        self.int4_cfg = None
        self._w_dq = None

    def _gemm(self, x, bias=None):
        """GEMM entry for all subclasses.

        fp8-block weights on GPU run NATIVE: per-token-group activation
        quant + the block-scale fp8 MFMA weight-streaming kernel at
        decode sizes (weights stay e4m3-resident, halving the decode
        weight stream); large-M prefill calls dequantize per call (no
        resident cache — prefill is compute-bound and bursty). CPU and
        int4 keep the dequant path."""
        w = self.weight
        if not self.is_plain and self._native(ops.plain_rows(x)):
            op = self._few_rows(ops.plain_rows(x))
            if op is not None:
                return ops.quant_rows(x, op, self._bias32())
            return self._prefill_quant(ops.plain_rows(x), bias)
        x = ops.plain_rows(x)
        if self.fp8_block is not None:
            from gllm_amd.layers.quantization.fp8 import dequant_block_fp8
            if x.is_cuda:
                wd = dequant_block_fp8(w, self.weight_scale_inv,
                                       self.fp8_block, x.dtype)
                return ops.linear(x, wd, bias)
            if self._w_dq is None:
                self._w_dq = dequant_block_fp8(
                    w, self.weight_scale_inv, self.fp8_block,
                    x.dtype).to(x.device)
            w = self._w_dq
        elif self.int4_cfg is not None:
            if x.is_cuda:
                from gllm_amd.layers.quantization.int4 import dequant_layer
                return ops.linear(x, dequant_layer(self, x.dtype), bias)
            if self._w_dq is None:
                from gllm_amd.layers.quantization.int4 import dequant_layer
                self._w_dq = dequant_layer(self, x.dtype).to(x.device)
            w = self._w_dq
        return ops.linear(x, w, bias)

    @property
    def is_plain(self) -> bool:
        """Unquantized weights (the fused few-row forms take them)."""
        return self.fp8_block is None and self.int4_cfg is None

    def _native(self, x) -> bool:
        """Whether the quantized weight is used as it is stored."""
        if not (x.is_cuda and x.dim() == 2 and x.dtype == torch.bfloat16
                and ops.has_kernels()):
            return False
        if self.fp8_block is not None:
            return self.fp8_block == (128, 128) and x.shape[1] % 128 == 0
        return self.int4_cfg[1] == 128 and x.shape[1] % 256 == 0

    def _few_rows(self, x):
        """The quantized weight as ``ops.quant_rows`` takes it, None above
        64 rows: there the bf16 copy and the library's product are the
        faster ones (256 rows, gate_up: 103 us against 329)."""
        if self.int4_cfg is not None:
            # one-time canonical repack; sbt = transposed (scale, bias)
            if getattr(self, "_i4_canon", None) is None:
                from gllm_amd.layers.quantization.int4 import \
                    repack_canonical
                wq4, sb, grp = repack_canonical(self)
                sbt = sb.permute(1, 2, 0).contiguous()
                self._i4_canon = (wq4.to(x.device), sb.to(x.device),
                                  sbt.to(x.device), grp)
            wq4, _, sbt, _ = self._i4_canon
            return ("int4", wq4, sbt) if x.shape[0] <= 64 else None
        return ("fp8", self.weight, self.weight_scale_inv) \
            if x.shape[0] <= 64 else None

    def _fused_op(self, x):
        """``_few_rows`` where a fused form may take this layer, else
        None."""
        x = ops.plain_rows(x)
        if self.is_plain or x.shape[0] == 0 or not self._native(x):
            return None
        return self._few_rows(x)

    def takes_fp8(self, rows) -> bool:
        """Whether this layer quantizes as many rows to e4m3 as ``rows``
        has: what forms them may then hand them over as
        ``ops.Fp8Rows``."""
        rows = ops.plain_rows(rows)
        return (self.fp8_block == (128, 128) and rows.is_cuda
                and rows.dim() == 2 and rows.dtype == torch.bfloat16
                and 0 < rows.shape[0] <= 64
                and self.weight.shape[1] % 128 == 0 and ops.has_kernels())

    def _bias32(self):
        """fp32 bias cached once (the skinny epilogues add fp32)."""
        if self.bias is None:
            return None
        if getattr(self, "_bias_f32", None) is None:
            self._bias_f32 = self.bias.float()
        return self._bias_f32

    def _prefill_quant(self, x, bias):
        """Quantized rows above 64, three modes via
        GLLM_QUANT_PREFILL:

        - "cache" (default): dequantize ONCE into a resident bf16 copy
          and run the library GEMM. MI355X carries 288 GB HBM3E — for a
          32B model the bf16 shadow costs 64 GB and buys bf16-identical
          prefill speed, while decode keeps streaming the quantized
          weights (where the bandwidth win lives). Built during the
          profile run, so KV sizing accounts for it.
        - "stream": identity-routed grouped quant GEMM — no shadow
          copy; slower (dense M/64 weight re-reads) but memory-lean.
        - "dequant": dequantize per call, nothing cached.
        """
        import os
        from gllm_amd import ops
        mode = os.environ.get("GLLM_QUANT_PREFILL", "cache")
        if mode == "stream" and ops.has_kernels():
            if self.fp8_block is not None:
                return ops.fp8_prefill_linear(x, self.weight,
                                              self.weight_scale_inv,
                                              self.bias)
            wq4, sb, _, _ = self._i4_canon
            return ops.int4_prefill_linear(x, wq4, sb, self.bias)
        if mode == "cache":
            if self._w_dq is None:
                if torch.cuda.is_current_stream_capturing():
                    raise RuntimeError(
                        "quant prefill cache built during graph capture")
                self._w_dq = self._dequant_full(x.dtype).to(x.device)
            return ops.linear(x, self._w_dq, bias)
        return ops.linear(x, self._dequant_full(x.dtype), bias)

    def _dequant_full(self, dtype):
        if self.fp8_block is not None:
            from gllm_amd.layers.quantization.fp8 import dequant_block_fp8
            return dequant_block_fp8(self.weight, self.weight_scale_inv,
                                     self.fp8_block, dtype)
        from gllm_amd.layers.quantization.int4 import dequant_layer
        return dequant_layer(self, dtype)


class ReplicatedLinear(LinearBase):
    def __init__(self, input_size, output_size, bias=False, params_dtype=None):
        super().__init__(input_size, output_size, bias, params_dtype)
        self.weight.weight_loader = self._load
        if self.bias is not None:
            self.bias.weight_loader = self._load

    @staticmethod
    def _load(param, loaded):
        param.data.copy_(loaded)

    def forward(self, x):
        return self._gemm(x, self.bias)


class ColumnParallelLinear(LinearBase):
    """Y = XW^T with W sharded along its output dim; no collective."""

    def __init__(self, input_size, output_size, bias=False, params_dtype=None,
                 gather_output: bool = False):
        tp = get_tp_size()
        assert output_size % tp == 0, (output_size, tp)
        super().__init__(input_size, output_size // tp, bias, params_dtype)
        self.full_output_size = output_size
        self.gather_output = gather_output
        self.weight.weight_loader = self._load
        if self.bias is not None:
            self.bias.weight_loader = self._load

    @staticmethod
    def _load(param, loaded):
        _narrow_copy(param.data, loaded, 0, get_tp_rank(), get_tp_size())

    def forward(self, x):
        out = self._gemm(x, self.bias)
        if self.gather_output:
            from gllm_amd.parallel import tensor_parallel_all_gather
            out = tensor_parallel_all_gather(out, dim=-1)
        return out


class MergedColumnParallelLinear(LinearBase):
    """Several column-parallel projections fused into one GEMM
    (gate_proj + up_proj). Checkpoints hold them separately; the loader
    places each sub-weight's TP shard into its slice."""

    def __init__(self, input_size, output_sizes: List[int], bias=False,
                 params_dtype=None):
        tp = get_tp_size()
        for s in output_sizes:
            assert s % tp == 0
        self.output_sizes = output_sizes
        super().__init__(input_size, sum(output_sizes) // tp, bias,
                         params_dtype)
        self.weight.weight_loader = self._load
        if self.bias is not None:
            self.bias.weight_loader = self._load

    def _load(self, param, loaded, shard_id: int):
        tp_rank, tp = get_tp_rank(), get_tp_size()
        offset = sum(self.output_sizes[:shard_id]) // tp
        size = self.output_sizes[shard_id] // tp
        param.data.narrow(0, offset, size).copy_(
            loaded.narrow(0, tp_rank * size, size))

    def forward(self, x):
        return self._gemm(x, self.bias)

    def forward_silu(self, x, fp8=False):
        """silu(gate) * up of a gate | up projection; ``fp8``: as
        ``ops.Fp8Rows`` where the product can leave them."""
        if self.is_plain and self.bias is None and x.is_cuda \
                and x.dim() == 2:
            return ops.linear_silu(x, self.weight)
        if self.bias is None:
            op = self._fused_op(x)
            if op is not None:
                return ops.quant_silu(x, op, fp8)
        return ops.silu_and_mul(self(x))


class PackedLinear(LinearBase):
    """Several projections of one input as one GEMM, each block of output
    columns starting on a multiple of ``align`` (rows between blocks are
    zero), so that the blocks of a bf16 result can be read with 16 B
    accesses whatever the sizes are. Replicated (one rank)."""

    def __init__(self, input_size, output_sizes: List[int],
                 params_dtype=None, align: int = 8):
        self.output_sizes = list(output_sizes)
        self.offsets, off = [], 0
        for n in self.output_sizes:
            self.offsets.append(off)
            off += -(-n // align) * align
        super().__init__(input_size, off, False, params_dtype)
        self.weight.data.zero_()
        self.weight.weight_loader = self._load

    def _load(self, param, loaded, shard_id: int):
        dst = param.data.narrow(0, self.offsets[shard_id],
                                self.output_sizes[shard_id])
        assert dst.shape == loaded.shape, (dst.shape, loaded.shape)
        dst.copy_(loaded)

    def forward(self, x):
        out = self._gemm(x)
        return [out[:, o:o + n]
                for o, n in zip(self.offsets, self.output_sizes)]


class QKVParallelLinear(LinearBase):
    """Fused qkv projection, sharded by head. Handles GQA where kv heads
    replicate across TP ranks when tp > num_kv_heads."""

    def __init__(self, hidden_size, head_dim, num_heads, num_kv_heads,
                 bias=False, params_dtype=None):
        tp = get_tp_size()
        assert num_heads % tp == 0
        self.head_dim = head_dim
        self.total_num_heads = num_heads
        self.total_num_kv_heads = num_kv_heads
        self.num_heads = num_heads // tp
        if num_kv_heads >= tp:
            assert num_kv_heads % tp == 0
            self.num_kv_heads = num_kv_heads // tp
            self.kv_replication = 1
        else:
            assert tp % num_kv_heads == 0
            self.num_kv_heads = 1
            self.kv_replication = tp // num_kv_heads
        out_per_rank = (self.num_heads + 2 * self.num_kv_heads) * head_dim
        super().__init__(hidden_size, out_per_rank, bias, params_dtype)
        self.q_size = self.num_heads * head_dim
        self.kv_size = self.num_kv_heads * head_dim
        self.weight.weight_loader = self._load
        if self.bias is not None:
            self.bias.weight_loader = self._load

    def _load(self, param, loaded, shard_id: str):
        tp_rank = get_tp_rank()
        if shard_id == "q":
            offset, size, src_rank = 0, self.q_size, tp_rank
        elif shard_id == "k":
            offset, size = self.q_size, self.kv_size
            src_rank = tp_rank // self.kv_replication
        else:
            offset, size = self.q_size + self.kv_size, self.kv_size
            src_rank = tp_rank // self.kv_replication
        param.data.narrow(0, offset, size).copy_(
            loaded.narrow(0, src_rank * size, size))

    def project(self, x):
        """The merged q | k | v rows."""
        return self._gemm(x, self.bias)

    def parts(self, x):
        """The fp32 parts of the merged rows without the bias, for
        ``ops.qkv_rope_cache``, which adds it; None where ``project`` is
        the better one."""
        if self.is_plain:
            return ops.qkv_parts(x, self.weight, self.bias)
        op = self._fused_op(x)
        if op is None or not ops.plain_bias(
                self.bias, self.q_size + 2 * self.kv_size):
            return None
        return ops.quant_parts(x, op)

    def forward(self, x):
        return self.project(x).split(
            [self.q_size, self.kv_size, self.kv_size], dim=-1)


class RowParallelLinear(LinearBase):
    """Y = XW^T with W sharded along its input dim; output all-reduce
    across TP (2x per decoder layer: o_proj + down_proj)."""

    def __init__(self, input_size, output_size, bias=False, params_dtype=None,
                 reduce_results: bool = True):
        tp = get_tp_size()
        assert input_size % tp == 0
        super().__init__(input_size // tp, output_size, bias, params_dtype)
        self.reduce_results = reduce_results
        self.weight.weight_loader = self._load_w
        if self.bias is not None:
            self.bias.weight_loader = self._load_b

    @staticmethod
    def _load_w(param, loaded):
        _narrow_copy(param.data, loaded, 1, get_tp_rank(), get_tp_size())

    @staticmethod
    def _load_b(param, loaded):
        param.data.copy_(loaded)

    def forward_add_norm(self, x, residual, norm, fp8=False):
        """(norm(residual + self(x)), that sum): one kernel behind the
        product where nothing has to be reduced over ranks first. ``fp8``:
        the norm as ``ops.Fp8Rows`` where that kernel can leave them."""
        rows = ops.plain_rows(x)
        if (self.bias is None and rows.is_cuda and rows.dim() == 2
                and (get_tp_size() == 1 or not self.reduce_results)):
            if self.is_plain:
                return ops.linear_add_rmsnorm(x, self.weight, residual,
                                              norm.scale(), norm.eps)
            op = self._fused_op(x)
            if op is not None:
                return ops.quant_add_rmsnorm(x, op, residual, norm.scale(),
                                             norm.eps, fp8)
        return norm(self(x), residual)

    def forward(self, x):
        out = self._gemm(x)
        if self.reduce_results:
            out = tensor_parallel_all_reduce(out)
        # bias applied once, after the reduction
        if self.bias is not None:
            out = out + self.bias
        return out
