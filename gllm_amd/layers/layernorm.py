"""RMSNorm layers over the fused HIP kernels (reference: layers/layernorm.py)."""

from typing import Optional

import torch
import torch.nn as nn

from gllm_amd import ops


class RMSNorm(nn.Module):
    def __init__(self, hidden_size: int, eps: float = 1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.eps = eps

    def scale(self) -> torch.Tensor:
        """What the normed row is multiplied by."""
        return self.weight

    def forward(self, x: torch.Tensor,
                residual: Optional[torch.Tensor] = None):
        if residual is not None:
            return ops.fused_add_rmsnorm(x, residual, self.weight, self.eps)
        return ops.rmsnorm(x, self.weight, self.eps)


class GemmaRMSNorm(nn.Module):
    """(1 + w) convention (Qwen3.5/Gemma checkpoints store w - 1).

    The effective scale (1 + w) is cached after load so the hot path
    runs the same fused add+rmsnorm kernel as RMSNorm."""

    def __init__(self, hidden_size: int, eps: float = 1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.zeros(hidden_size))
        self.eps = eps
        self._w1 = None

    def scale(self) -> torch.Tensor:
        if self._w1 is None or self._w1.device != self.weight.device:
            self._w1 = (self.weight + 1.0).contiguous()
        return self._w1

    def forward(self, x: torch.Tensor,
                residual: Optional[torch.Tensor] = None):
        if residual is not None:
            return ops.fused_add_rmsnorm(x, residual, self.scale(),
                                         self.eps)
        return ops.rmsnorm(x, self.scale(), self.eps)


class LayerNorm(nn.Module):
    """LayerNorm with weight and (optional) bias over an fp32 residual
    stream.

    Sandwich-norm decoders (a norm before and after every sublayer) keep
    the stream in fp32 while sublayers run in the model dtype:

    * ``norm(x)``                       h = LN(x), x fp32 -> model dtype
    * ``norm.add_into(x, y, nxt)``      x += LN(y) in place and, when
      ``nxt`` (the next sublayer's pre-norm) is given, returns nxt(x) —
      one fused launch per boundary (ops.residual_layernorm)
    * ``norm.add_into(x, y, nxt, gate=g)``  the same with the sublayer
      result gated first: x += LN(y * sigmoid(g))

    The bias parameter is named ``bias`` (None with ``bias=False``);
    checkpoints that store it under another name map it in the model's
    load_weights.
    """

    def __init__(self, hidden_size: int, eps: float = 1e-5,
                 params_dtype=None, bias: bool = True):
        super().__init__()
        dtype = params_dtype or torch.get_default_dtype()
        self.weight = nn.Parameter(torch.ones(hidden_size, dtype=dtype),
                                   requires_grad=False)
        if bias:
            self.bias = nn.Parameter(torch.zeros(hidden_size, dtype=dtype),
                                     requires_grad=False)
        else:
            self.register_parameter("bias", None)
        self.eps = eps
        self._w32 = None

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return ops.layernorm_f32(x, self.weight, self.bias, self.eps,
                                 self.weight.dtype)

    def forward_f32(self, x: torch.Tensor) -> torch.Tensor:
        """LN(x) kept in fp32 (a norm whose result IS the residual
        stream, e.g. right after the embedding)."""
        if self.weight.dtype == torch.float32:
            return self.forward(x)
        if self._w32 is None or self._w32[0].device != x.device:
            self._w32 = (self.weight.float(), None if self.bias is None
                         else self.bias.float())
        return ops.layernorm_f32(x, self._w32[0], self._w32[1], self.eps,
                                 torch.float32)

    def add_into(self, x: torch.Tensor, y: torch.Tensor,
                 nxt: Optional["LayerNorm"] = None,
                 gate: Optional[torch.Tensor] = None):
        pre = (nxt.weight, nxt.bias) if nxt is not None else None
        return ops.residual_layernorm(x, y, self.weight, self.bias,
                                      self.eps, pre, gate)


class DynamicTanh(nn.Module):
    """tanh(alpha * x) * weight + bias in the place of a norm, over an
    fp32 residual stream (no statistics, so it fuses with whatever writes
    the stream). ``alpha`` is one learned number.

    * ``norm(x)``                      h = norm(x), x fp32 -> model dtype
    * ``DynamicTanh.boundary(x, y, pair, nxt)``  x += y, and x += s *
      (RMSnorm(l) * w_l + RMSnorm(r) * w_r) for ``pair`` = (l, w_l, r,
      w_r, s, eps), in place; returns nxt(x) with ``nxt``: one launch per
      layer boundary (ops.stream_tanh)
    * ``norm.open(ids, table, scale)``  (x, norm(x)) of a stream that
      opens with x = table[ids] * scale
    """

    def __init__(self, hidden_size: int, params_dtype=None):
        super().__init__()
        dtype = params_dtype or torch.get_default_dtype()
        self.weight = nn.Parameter(torch.ones(hidden_size, dtype=dtype),
                                   requires_grad=False)
        self.bias = nn.Parameter(torch.zeros(hidden_size, dtype=dtype),
                                 requires_grad=False)
        self.alpha = nn.Parameter(torch.ones((), dtype=torch.float32),
                                  requires_grad=False)
        self._alpha = None

    def args(self):
        # a launch argument (a captured graph keeps it): read once
        if self._alpha is None:
            self._alpha = float(self.alpha)
        return self._alpha, self.weight, self.bias

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return ops.stream_tanh(x, nxt=self.args())

    def open(self, ids: torch.Tensor, table: torch.Tensor, scale: float):
        x = torch.empty(ids.shape[0], table.shape[1], dtype=torch.float32,
                        device=table.device)
        h = ops.stream_tanh(x, nxt=self.args(), embed=(ids, table, scale))
        return x, h

    @staticmethod
    def boundary(x: torch.Tensor, y: Optional[torch.Tensor] = None,
                 pair=None, nxt: Optional["DynamicTanh"] = None):
        return ops.stream_tanh(x, y, pair,
                               nxt.args() if nxt is not None else None)


class StreamRMSNorm(nn.Module):
    """RMS norm (eps inside the root) over an fp32 residual stream, for
    decoders that norm a sublayer's result (and possibly its input) and
    add the normed result times a fixed multiplier:

    * ``norm(x)``                          h = RMSnorm(x) * w, model dtype
    * ``norm.add_into(x, y, nxt, mult)``   x += mult * RMSnorm(y) * w in
      place and, with ``nxt`` (the next sublayer's pre-norm), returns
      nxt(x): one launch per boundary (ops.stream_rmsnorm)
    * ``read=True`` instead of ``nxt``: the next sublayer reads the
      stream itself, returned in the model dtype by the same launch
    * ``y2``: the norm sees y + y2 (a routed and a shared result);
      ``y_scale``: it sees y_scale * (y + y2), the product formed in
      fp32; ``add`` (fp32 [width]): added to every row of x after the
      sublayer result and before ``nxt`` reads it
    * ``weight_offset``: the weight is stored as its distance from this
      number (1.0: a checkpoint that keeps w around zero); the sum is
      formed in fp32
    """

    def __init__(self, hidden_size: int, eps: float = 1e-5,
                 params_dtype=None, weight_offset: float = 0.0):
        super().__init__()
        dtype = params_dtype or torch.get_default_dtype()
        self.weight_offset = float(weight_offset)
        self.weight = nn.Parameter(
            torch.full((hidden_size,), 1.0 - self.weight_offset,
                       dtype=dtype), requires_grad=False)
        self.eps = eps

    def forward(self, x: torch.Tensor,
                add: Optional[torch.Tensor] = None) -> torch.Tensor:
        return ops.stream_rmsnorm(x, None, None, self.eps, add=add,
                                  pre_w=self.weight,
                                  pre_off=self.weight_offset)

    def add_into(self, x: torch.Tensor, y: torch.Tensor,
                 nxt: Optional["StreamRMSNorm"] = None, mult: float = 1.0,
                 y_scale: float = 1.0, y2: Optional[torch.Tensor] = None,
                 add: Optional[torch.Tensor] = None, read: bool = False):
        return ops.stream_rmsnorm(
            x, y, self.weight, self.eps, mult, y_scale, y2, add,
            nxt.weight if nxt is not None else None, self.weight_offset,
            nxt.weight_offset if nxt is not None else 0.0,
            self.weight.dtype if read and nxt is None else None)
