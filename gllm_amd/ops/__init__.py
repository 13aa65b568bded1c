"""Custom-op facade — the single switch point between backends.

Mirrors the role of the reference's ``_custom_ops.py`` ("single point
where we can swap backends", _custom_ops.py:1-10): every layer calls
through here. Dispatch rule:

* CUDA (= HIP/ROCm) tensors -> the in-tree gfx950 extension
  ``gllm_amd._kernels``. If the extension is missing on a GPU box this
  RAISES — no silent eager fallback (a GPU run must exercise the native
  kernels).
* CPU tensors -> the PyTorch reference implementations (ops.torch_ref),
  which double as the numerics oracle for the HIP kernels.
"""

import functools
import math
from typing import NamedTuple, Optional

import torch

from gllm_amd.ops import torch_ref

_K = None
_K_ERR: Optional[str] = None


def _load_kernels():
    global _K, _K_ERR
    if _K is not None or _K_ERR is not None:
        return _K
    try:
        from gllm_amd import _kernels  # built in-tree by setup.py
        _K = _kernels
    except ImportError as e:  # pragma: no cover
        _K_ERR = str(e)
    return _K


_KS = None
_KS_ERR: Optional[str] = None


def _load_seq_kernels():
    """The dtype-generic sequence-mixer module (setup.py SEQ_SOURCES):
    built on its own so a model that needs only these kernels serves
    from a checkout where the full extension was never compiled."""
    global _KS, _KS_ERR
    if _KS is not None or _KS_ERR is not None:
        return _KS
    try:
        from gllm_amd import _kernels_seq
        _KS = _kernels_seq
    except ImportError as e:  # pragma: no cover
        _KS_ERR = str(e)
    return _KS


class _SeqBacked:
    """Stand-in for the full extension when only the sequence-mixer
    module is built: serves the entry points both modules define (MoE
    grouped GEMM, gated activations) and fails loudly on the rest."""

    def __init__(self, mod):
        self._mod = mod

    def __getattr__(self, name):
        try:
            return getattr(self._mod, name)
        except AttributeError:
            raise RuntimeError(
                f"kernel {name!r} lives in gllm_amd._kernels, which is "
                f"not built (import error: {_K_ERR}); run `python "
                "setup.py build_ext --inplace`") from None


def _gpu_kernels():
    k = _load_kernels()
    if k is None:
        ks = _load_seq_kernels()
        if ks is not None:
            return _SeqBacked(ks)
        raise RuntimeError(
            "gllm_amd._kernels HIP extension not built but a CUDA tensor "
            "was passed — build with `python setup.py build_ext --inplace` "
            f"(PYTORCH_ROCM_ARCH=gfx950). Import error: {_K_ERR}")
    return k


def _seq_kernels():
    k = _load_seq_kernels()
    if k is None:
        raise RuntimeError(
            "gllm_amd._kernels_seq HIP extension not built but a CUDA "
            "tensor was passed — build with `GLLM_EXT=seq python setup.py "
            f"build_ext --inplace`. Import error: {_KS_ERR}")
    return k


def has_kernels() -> bool:
    return _load_kernels() is not None


def has_moe_kernels() -> bool:
    """The bf16 grouped MoE GEMM ships in both extension modules."""
    return _load_kernels() is not None or _load_seq_kernels() is not None


# --------------------------------------------------------------- norm
def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _gpu_kernels().rmsnorm(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor,
                      weight: torch.Tensor, eps: float):
    if x.is_cuda:
        _gpu_kernels().fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    return torch_ref.fused_add_rmsnorm(x, residual, weight, eps)


# --------------------------------------------------------------- activation
def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        d = x.shape[-1] // 2
        out = torch.empty(x.shape[:-1] + (d,), dtype=x.dtype, device=x.device)
        _gpu_kernels().silu_and_mul(out, x)
        return out
    return torch_ref.silu_and_mul(x)


def gelu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        d = x.shape[-1] // 2
        out = torch.empty(x.shape[:-1] + (d,), dtype=x.dtype, device=x.device)
        _gpu_kernels().gelu_and_mul(out, x)
        return out
    return torch_ref.gelu_and_mul(x)


# --------------------------------------------------------------- rope
def rotary_embedding(positions: torch.Tensor, q: torch.Tensor,
                     k: torch.Tensor, head_dim: int,
                     cos_sin_cache: torch.Tensor, is_neox: bool = True):
    if q.is_cuda:
        _gpu_kernels().rotary_embedding(positions, q, k, head_dim,
                                        cos_sin_cache, is_neox)
        return q, k
    return torch_ref.rotary_embedding(positions, q, k, head_dim,
                                      cos_sin_cache, is_neox)


# --------------------------------------------------------------- kv cache
def reshape_and_cache(k: torch.Tensor, v: torch.Tensor,
                      k_cache: torch.Tensor, v_cache: torch.Tensor,
                      slot_mapping: torch.Tensor):
    if k.is_cuda:
        _gpu_kernels().reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
        return
    torch_ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


# --------------------------------------------------------------- attention
def paged_attention(q: torch.Tensor, k_cache: torch.Tensor,
                    v_cache: torch.Tensor, block_table: torch.Tensor,
                    seq_lens: torch.Tensor, query_start_loc: torch.Tensor,
                    scale: float, max_query_len: int = 1,
                    out: Optional[torch.Tensor] = None,
                    sliding_window: int = 0,
                    single_rows: int = 0) -> torch.Tensor:
    """``single_rows``: how many of the sequences bring one query row
    beside longer portions, if the caller knows (those then go through
    the decode kernel)."""
    if q.is_cuda:
        kern = _gpu_kernels()
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        if max_query_len == 1:
            kern.paged_attention_decode(
                out, q, k_cache, v_cache, block_table, seq_lens, scale,
                sliding_window, None)
        else:
            qsl = query_start_loc.int()
            split = single_rows > 0 and kern.decode_rows_ok(
                k_cache, v_cache, q.shape[1])
            if split:
                kern.paged_attention_decode(
                    out, q, k_cache, v_cache, block_table, seq_lens, scale,
                    sliding_window, qsl)
            kern.paged_attention_prefill(
                out, q, k_cache, v_cache, block_table, seq_lens, qsl,
                max_query_len, scale, sliding_window, split)
        return out
    return torch_ref.paged_attention(q, k_cache, v_cache, block_table,
                                     seq_lens, query_start_loc, scale,
                                     out=out, sliding_window=sliding_window)


# --------------------------------------------------------------- moe
def topk_softmax(gating: torch.Tensor, topk: int, renormalize: bool = True):
    """MoE routing: softmax over all experts, then the top k (weights
    fp32 [T, k] in descending order, ids int32 [T, k]). Logits of up to
    512 experts on the GPU take one wave-per-row kernel (ties go to the
    lower index)."""
    if (gating.is_cuda and gating.dim() == 2 and gating.shape[1] <= 512
            and 0 < topk <= min(64, gating.shape[1])
            and gating.dtype in (torch.float32, torch.bfloat16,
                                 torch.float16) and has_moe_kernels()):
        gating = gating.contiguous()
        weights = torch.empty(gating.shape[0], topk, dtype=torch.float32,
                              device=gating.device)
        ids = torch.empty(gating.shape[0], topk, dtype=torch.int32,
                          device=gating.device)
        _gpu_kernels().softmax_topk_rows(weights, ids, gating, renormalize)
        return weights, ids
    return torch_ref.topk_softmax(gating, topk, renormalize)


def topk_then_softmax(logits: torch.Tensor, topk: int):
    """Top-k over raw router logits, softmax over the chosen only:
    (weights fp32 [T, k] in descending order of logit, ids int32
    [T, k]). fp32 logits of up to 512 experts on the GPU take one
    wave-per-row kernel (ties go to the lower index)."""
    if (logits.is_cuda and logits.dtype == torch.float32
            and logits.dim() == 2 and logits.shape[1] <= 512
            and topk <= min(64, logits.shape[1])):
        logits = logits.contiguous()
        weights = torch.empty(logits.shape[0], topk, dtype=torch.float32,
                              device=logits.device)
        ids = torch.empty(logits.shape[0], topk, dtype=torch.int32,
                          device=logits.device)
        _seq_kernels().topk_softmax_rows(weights, ids, logits)
        return weights, ids
    return torch_ref.topk_then_softmax(logits, topk)


def grouped_topk(scores, topk, n_group, topk_group, renormalize=True,
                 scoring="softmax", e_bias=None):
    # device-resident (a CPU round-trip here would sync every MoE
    # layer of every DeepSeek step)
    return torch_ref.grouped_topk(scores, topk, n_group, topk_group,
                                  renormalize, scoring, e_bias)


def fused_moe(x: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor,
              topk_weights: torch.Tensor, topk_ids: torch.Tensor,
              expert_start: int = 0,
              num_global_experts: Optional[int] = None,
              activation: str = "silu_glu",
              act_args: tuple = (),
              add_norm: Optional[tuple] = None,
              shared_mlp: Optional[tuple] = None) -> torch.Tensor:
    """Grouped-GEMM fused MoE on the gfx950 kernels (GPU, bf16).
    ``activation``: "silu_glu" (w13 = gate | up rows), "relu2"
    (ungated experts, w13 = up rows only, act = max(z, 0)^2) or
    "swiglu_clamp" (w13 = gate | up rows, ``act_args`` = (limit,
    alpha): min(g, limit) * sigmoid(alpha g) * (clamp(u) + 1)).

    Reference fused_experts_impl (fused_moe_triton/fused_moe.py:779):
    align -> GEMM1 + activation -> GEMM2 (weighted scatter) -> sum.
    Fully device-resident and hipGraph-safe (no host syncs; grids are
    sized by upper bound and gated on the device-side block count).
    Returns the PARTIAL output for this rank's expert shard (callers
    run their TP/EP all-reduce on top). ``add_norm`` = (shared or None,
    residual, norm weight, eps): the output (+ shared) is added to the
    residual, in place, and the norm of that is returned (one kernel; see
    ``moe_add_norm_ok``). ``shared_mlp`` = (gate over up rows, down weight)
    of a gated feed-forward that all rows pass: its output is the ``shared``
    of ``add_norm``, its products run beside the experts' (see
    ``moe_shared_beside``) where these are on wide tiles.
    """
    if shared_mlp is not None and (activation != "silu_glu" or add_norm is None
                                   or add_norm[0] is not None):
        raise ValueError("shared_mlp: beside gated experts, as the shared "
                         "part of add_norm")
    T, K = x.shape
    E_local, rows13, _ = w13.shape
    inter = w2.shape[2]
    topk = topk_ids.shape[1]
    n_pairs = T * topk
    dev = x.device
    k = _gpu_kernels()
    tw = topk_weights.float().contiguous()
    pair_out = torch.empty(n_pairs, K, dtype=x.dtype, device=dev)
    rpe = n_pairs / max(1, E_local)
    # (the wide tiles come to LDS in units of 16 B)
    x = x.clone() if x.data_ptr() % 16 else x
    if (K % 64 == 0 and inter % 64 == 0
            and w13.data_ptr() % 16 == 0 and w2.data_ptr() % 16 == 0):
        # row block by the rows per expert: while an expert's weights are
        # the cost, one block holds the rows of all but the most popular
        # experts (csrc/moe_tiled.hip has times on both sides of each line)
        block_m = _moe_block(rpe)
        ids32, tables, rows = _moe_tables(topk_ids, E_local, expert_start,
                                          block_m)
        act = torch.empty(rows, inter, dtype=x.dtype, device=dev)
        code = {"swiglu_clamp": 2, "relu2": 3}.get(activation, 1)
        limit, alpha = act_args if activation == "swiglu_clamp" \
            else (0.0, 0.0)
        if shared_mlp is not None:
            h = k.moe_gemm_tiled_shared(act, x, w13, *tables, None, n_pairs,
                                        topk, block_m, 1, x, shared_mlp[0])
            add_norm = (k.moe_gemm_tiled_shared(
                pair_out, act, w2, *tables, tw, n_pairs, topk, block_m, 0, h,
                shared_mlp[1]),) + add_norm[1:]
        else:
            k.moe_gemm_tiled(act, x, w13, *tables, None, n_pairs, topk,
                             block_m, code, limit, alpha)
            k.moe_gemm_tiled(pair_out, act, w2, *tables, tw, n_pairs, topk,
                             block_m, 0, 0.0, 0.0)
    else:
        if shared_mlp is not None:
            add_norm = (linear(linear_silu(x, shared_mlp[0]),
                               shared_mlp[1]),) + add_norm[1:]
        block_m = 16 if rpe < 12 else 32 if rpe < 40 else 64
        ids32, tables, rows = _moe_tables(topk_ids, E_local, expert_start,
                                          block_m)
        inter1 = torch.empty(rows, rows13, dtype=x.dtype, device=dev)
        k.moe_gemm(inter1, x, w13, *tables, None, n_pairs, topk, block_m,
                   False)
        if activation == "relu2":
            act = relu2(inter1)
        elif activation == "swiglu_clamp":
            act = clamp_swiglu(inter1, *act_args)
        else:
            act = silu_and_mul(inter1)
        k.moe_gemm(pair_out, act, w2, *tables, tw, n_pairs, topk, block_m,
                   True)
    if add_norm is not None:
        return k.moe_sum_norm(pair_out, ids32, expert_start, E_local, topk,
                              *add_norm)
    out = torch.empty(T, K, dtype=x.dtype, device=dev)
    k.moe_sum(out, pair_out, ids32, expert_start, E_local, topk)
    return out


def _moe_block(rows_per_expert: float) -> int:
    return (32 if rows_per_expert <= 12 else 64 if rows_per_expert <= 40
            else 128 if rows_per_expert <= 128 else 256)


def moe_shared_beside(x: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor,
                      topk: int, gate_up: torch.Tensor,
                      down: torch.Tensor) -> bool:
    """Whether ``fused_moe`` of gated experts runs a shared expert's products
    beside theirs: where they are aligned bf16 and ``_shared_beside`` takes
    their sizes."""
    T, K = x.shape
    inter, width = w2.shape[2], down.shape[1]
    if not (all(t.dtype == torch.bfloat16 and t.is_cuda and t.is_contiguous()
                and t.data_ptr() % 16 == 0
                for t in (x, w13, w2, gate_up, down))
            and T > 0 and K % 64 == 0 and inter % 64 == 0 and width % 64 == 0
            and down.shape[0] == K and gate_up.shape == (2 * width, K)):
        return False
    return _shared_beside(T, topk, max(1, w13.shape[0]), K, inter, width)


def _shared_beside(T: int, topk: int, experts: int, K: int, inter: int,
                   width: int) -> bool:
    """The sizes of ``moe_shared_beside``: rows, routed experts of K x inter,
    a shared one of K x width (us of experts, sum and norm, apart / beside).
    Up to 256 rows the products apart are a few launches that wait for
    weights: 64 experts of 2048 x 1408, shared 2816, 1 row 53 / 45, 32 rows
    203 / 194, 128 rows 214 / 207, 256 rows 241 / 231; 256 of 2048 x 512,
    shared 512, 8 rows 88 / 76, 128 rows 283 / 276; 64 of 7168 x 2048, shared
    2048, 64 rows 897 / 887. A shared expert wider than a routed one is a
    longer chain of K in a tile of the second product than any of those beside
    it, which they hide only while it is short (16 of 2048 x 3456, shared 5184,
    27 rows 145 / 154; 8 of 4096 x 2368, shared 4736, 14 rows 104 / 113); in
    blocks of 128 rows, of few experts, any chain has to be (8 of 4096 x 1856,
    shared 1856, 79 rows 134 / 168; 4 of 2048 x 704, shared 704, 100 rows 61 /
    47).
    Beyond, they fill rounds of tiles that either would leave: rows of 2048 at
    most, where rounds are short, and weights that are worth it (2048 x 1408 as
    above, 320 rows 260 / 240, 1000 rows 364 / 344, 3000 rows 600 / 578, 4096
    rows 661 / 624; 16 experts, shared 5632, 3000 rows 457 / 420; but 256 of
    2048 x 512, 512 rows 322 / 329, 64 of 7168 x 2048, 4096 rows 3363 / 3530).
    In blocks of less than 256 rows their tiles are slower than the library's
    or tile_gemm.hip's by themselves, so they are to be few, of narrow experts
    (32 of 2048 x 1088, shared 2176, 546 rows 176 / 146; 128 of 2048 x 1024,
    shared 2048, 1407 rows 470 / 489; 64 of 2048 x 2304, shared 4608, 1303 rows
    480 / 537). In blocks of 256 rows the rounds are counted: by themselves the
    shared tiles take the part of a round that they fill, at least half of one,
    and the routed ones whole rounds (8 of 2048 x 1856, shared 3712, 2498 rows
    457 / 412; 8 of 2048 x 1216, shared 2432, 1653 rows 144 / 157). That holds
    where most blocks have more than 128 rows, half of their products (32 of
    2048 x 2368, shared 2368, 2195 rows, 137 an expert, 336 / 354), where the
    shared products are a sixth of the routed ones or more (of 128 of 2048 x
    2304, shared 2304, 8 a row, 3376 rows 1024 / 1070) and whole multiples of
    theirs (4 of 2048 x 1728, shared 2560, 1566 rows 222 / 251), and from 1536
    to 5120 rows (level beyond). Over 175 sizes of these blocks this takes 121,
    in 0.92 of the time, three of them slower by 2 to 3 %."""
    # (what moe_gemm_tiled_shared takes of its two products)
    if max(T, 2 * width, K) >= 1 << 20 or 2 * width * K >= 1 << 30:
        return False
    per_expert = T * topk / experts
    block_m = _moe_block(per_expert)
    if T <= 256:
        short = (width <= inter and (block_m < 128 or inter <= 1024)
                 or block_m < 128 and K <= 2048
                 and width <= min(2 * inter, 3072))
        # (apart they are the streaming kernel's, and the second one's sums
        # over shares of K are the same beside)
        return (short and block_m < 256 and 2 * width >= 512
                and _use_skinny(T, 512, K) and _use_skinny(T, K, width)
                and _gpu_kernels().stream_slice(T, K, width) > 0)
    if K > 2048 or width * K < 4 << 20:
        return False
    if block_m < 256:
        return (T <= 1024 and inter <= 1600 and width <= 2 * inter
                and -(-T // block_m) * -(-width // 64) <= 384)
    # (offsets of tile_gemm.hip are 32 bits)
    if not (1536 <= T <= 5120 and per_expert >= 176
            and width % inter == 0 and 6 * width >= topk * inter
            and 2 * inter * K < 1 << 30
            and (T * topk + 256 * (experts + 1)) * max(inter, K) < 1 << 30):
        return False
    cus = _compute_units()
    rows, cols = -(-T // 256), -(-K // 256)
    blocks = experts * (per_expert / 256 + 0.5)
    up, down = rows * -(-width // 128), rows * cols
    routed_up, routed_down = blocks * -(-inter // 128), blocks * cols
    rounds = lambda tiles: math.ceil(tiles / cus)  # noqa: E731
    apart = (K * (max(0.5, up / cus) + rounds(routed_up))
             + width * max(0.5, down / cus) + inter * rounds(routed_down))
    beside = K * rounds(up + routed_up) + max(
        width, inter * rounds(down * width / inter + routed_down))
    return beside < apart


def moe_add_norm_ok(x: torch.Tensor, shared: Optional[torch.Tensor],
                    residual: torch.Tensor, norm_w: torch.Tensor) -> bool:
    """Whether ``fused_moe`` takes ``add_norm`` of these."""
    rows = [residual] + ([] if shared is None else [shared])
    return (x.is_cuda and x.dim() == 2 and x.shape[1] % 8 == 0
            and x.shape[1] <= 8192
            and all(t.dtype == torch.bfloat16 and t.shape == x.shape
                    and t.is_contiguous() and t.data_ptr() % 16 == 0
                    for t in rows)
            and norm_w.dtype in (torch.bfloat16, torch.float32)
            and norm_w.is_contiguous() and norm_w.data_ptr() % 16 == 0)


def _moe_tables(topk_ids: torch.Tensor, E_local: int, expert_start: int,
                block_m: int):
    """Sort the (token, expert) pairs by expert in blocks of ``block_m``
    rows: (int32 ids, (sorted_ids, expert_blocks, n_post), rows of a
    sorted buffer). Pairs of other ranks' experts, or of id -1, are in
    no block."""
    n_pairs = topk_ids.numel()
    dev = topk_ids.device
    cap = n_pairs + E_local * (block_m - 1) + 1
    max_blocks = (n_pairs + block_m - 1) // block_m + E_local
    ids32 = topk_ids.int().contiguous()
    tables = (torch.empty(cap, dtype=torch.int32, device=dev),
              torch.empty(max_blocks, dtype=torch.int32, device=dev),
              torch.empty(1, dtype=torch.int32, device=dev))
    _gpu_kernels().moe_align(ids32, E_local, expert_start, block_m, *tables)
    return ids32, tables, cap - 1 + block_m


# --------------------------------------------------------------- fp8
def per_token_group_quant_fp8(x: torch.Tensor, group: int = 128,
                              ue8m0: bool = False,
                              transposed: bool = False):
    """[T, K] bf16 -> (e4m3 [T, K], fp32 scales [T, K/group]).
    GPU kernel; CPU callers use the torch math in quantization/fp8.py.
    ``transposed=True`` additionally returns scales_t [K/group, T]
    (column-major) — the skinny GEMM stages a k-group's scales as ONE
    contiguous run instead of a strided 64-line gather."""
    assert x.is_cuda and group == 128
    T, K = x.shape
    q = torch.empty(T, K, dtype=torch.float8_e4m3fn, device=x.device)
    scales = torch.empty(T, K // group, dtype=torch.float32,
                         device=x.device)
    st = torch.empty(K // group, T, dtype=torch.float32,
                     device=x.device) if transposed else None
    _gpu_kernels().per_token_group_quant_fp8(
        x.contiguous(), q.view(torch.uint8), scales, st, ue8m0)
    if transposed:
        return q, scales, st
    return q, scales


def _quant_splitk(N: int, K: int, bk: int) -> int:
    """Parts along K of an fp8 product: the deepest power of two that
    leaves at least 8 stages of ``bk`` per part and at most 1024
    workgroups of 64 columns (us, 64 rows: 7168 x 5120 4 parts 16.7, 3
    17.6; 4096 x 14336 8 parts 18.3; 5120 x 27648 8 parts 38, 10 38)."""
    n_wg = -(-N // 64)
    s = 1
    while (s < 16 and n_wg * (s * 2) <= 1024
           and (K // bk) // (s * 2) >= 8):
        s *= 2
    k_slice = ((-(-K // s)) + bk - 1) // bk * bk
    return -(-K // k_slice)


def _quant_gemm(x: torch.Tensor, kind: str, w: torch.Tensor,
                ws: torch.Tensor, bias, form: int) -> torch.Tensor:
    splits = _quant_splitk(w.shape[0], plain_rows(x).shape[1], 128) \
        if kind == "fp8" else 0
    return _gpu_kernels().quant_gemm(*_quant_operands(x, kind, w, ws), bias,
                                     form, splits)


class Fp8Rows(NamedTuple):
    """bf16 rows with the e4m3 bytes and scales [columns / 128, rows] that
    an fp8 product takes of them, from the kernel that formed the rows
    (``per_token_group_quant_fp8`` would give the same)."""
    x: torch.Tensor
    q: torch.Tensor
    scales: torch.Tensor


def plain_rows(x):
    """The tensor of rows that may be ``Fp8Rows``."""
    return x.x if isinstance(x, Fp8Rows) else x


def _quant_operands(x, kind: str, w: torch.Tensor, ws: torch.Tensor):
    """(rows, their scales, weight bytes, weight scales) as
    csrc/quant_gemm.hip takes them; ``kind`` "fp8" (w [N, K] e4m3, ws fp32
    per 128 x 128 block; the rows are quantized per 128 columns) or "int4"
    (w [N, K / 2] packed, ws [K / 128, 2, N])."""
    if kind == "fp8" and isinstance(x, Fp8Rows):
        return x.q, x.scales, w.view(torch.uint8), ws.contiguous()
    x = plain_rows(x)
    if kind == "fp8":
        xq, _, xs = per_token_group_quant_fp8(x, transposed=True)
        return xq.view(torch.uint8), xs, w.view(torch.uint8), ws.contiguous()
    x = x.contiguous()
    return (x.clone() if x.data_ptr() % 16 else x), None, w, ws


def quant_rows(x: torch.Tensor, op, bias: Optional[torch.Tensor] = None):
    """x @ dequant(w).T (+ bias) for at most 256 rows; ``op`` = (kind, w,
    scales)."""
    return _quant_gemm(
        x, *op, bias.float().contiguous() if bias is not None else None, 1)


def quant_silu(x, op, fp8: bool = False):
    """silu(x @ w_gate.T) * (x @ w_up.T), w = gate rows over up rows. The
    one-kernel form cannot split K, so it is for weights with tiles enough
    without (28672 x 4096, 1 row, int4: 25 us against 20 + the second
    kernel's 5). ``fp8``: as ``Fp8Rows`` where the product can leave
    them."""
    N = op[1].shape[0]
    if N % 32 == 0 and N >= 16384:
        if fp8 and op[0] == "fp8":
            out = _gpu_kernels().quant_gemm_gated_fp8(
                *_quant_operands(x, *op))
            return Fp8Rows(*out) if len(out) == 3 else out[0]
        return _quant_gemm(x, *op, None, 0)
    return silu_and_mul(quant_rows(x, op))


def quant_parts(x: torch.Tensor, op) -> Optional[torch.Tensor]:
    """The fp32 parts [S, M, N] of x @ dequant(w).T, or None for an N that
    their readers do not take."""
    if op[1].shape[0] % 8:
        return None
    return _quant_gemm(x, *op, None, 2)


def quant_add_rmsnorm(x, op, residual: torch.Tensor, norm_w: torch.Tensor,
                      eps: float, fp8: bool = False):
    """residual += x @ dequant(w).T; (rmsnorm(residual), residual).
    ``fp8``: the norm as ``Fp8Rows`` where its kernel can leave them."""
    if _norm_parts_ok(op[1].shape[0], residual, norm_w):
        if fp8 and op[1].shape[0] % 128 == 0:
            return Fp8Rows(*_gpu_kernels().parts_add_norm_fp8(
                quant_parts(x, op), residual, norm_w, eps,
                op[0] == "fp8")), residual
        return _gpu_kernels().parts_add_norm(quant_parts(x, op), residual,
                                             norm_w, eps,
                                             op[0] == "fp8"), residual
    return fused_add_rmsnorm(quant_rows(x, op), residual, norm_w, eps)


def fp8_linear(x: torch.Tensor, w_q: torch.Tensor, w_scale: torch.Tensor,
               bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = x @ dequant(w_q).T via the fp8 weight-streaming kernel
    (M <= 256): per-token-group activation quant + block-scale fp8
    MFMA."""
    return quant_rows(x, ("fp8", w_q, w_scale), bias)


_IDENT: dict = {}


def _identity_tables(device, m_pad: int, block: int):
    """Routing tables that make the grouped MoE GEMM a plain dense
    GEMM: sorted_ids = arange (row i of the batch is 'pair' i, topk=1),
    every block belongs to expert 0. Cached per (device, m_pad) — the
    graph warmup pass populates the cache so capture never allocates."""
    key = (device.index or 0, m_pad, block)
    ent = _IDENT.get(key)
    if ent is None:
        if torch.cuda.is_current_stream_capturing():
            raise RuntimeError("identity tables built during graph capture")
        ids = torch.arange(m_pad, dtype=torch.int32, device=device)
        blocks = torch.zeros(m_pad // block, dtype=torch.int32,
                             device=device)
        n_post = torch.full((1,), m_pad, dtype=torch.int32, device=device)
        ent = (ids, blocks, n_post)
        _IDENT[key] = ent
    return ent


def fp8_prefill_linear(x: torch.Tensor, w_q: torch.Tensor,
                       w_scale: torch.Tensor,
                       bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Dense fp8 GEMM for M > 256: the grouped MoE fp8 kernel (wide
    BM64xBN256 prefill tile) with identity routing — weights stay e4m3,
    no per-call dequant materialization."""
    M, K = x.shape
    N = w_q.shape[0]
    aq, as_ = per_token_group_quant_fp8(x.contiguous())
    m_pad = (M + 63) // 64 * 64
    ids, blocks, n_post = _identity_tables(x.device, m_pad, 64)
    out_pad = torch.empty(m_pad, N, dtype=x.dtype, device=x.device)
    _gpu_kernels().moe_gemm_fp8(
        out_pad, aq.view(torch.uint8), as_,
        w_q.view(torch.uint8).view(1, N, K),
        w_scale.contiguous().view(1, w_scale.shape[0], w_scale.shape[1]),
        ids, blocks, n_post, None, M, 1, 164, False)
    out = out_pad.narrow(0, 0, M)
    if bias is not None:
        out = out.add_(bias)
    return out


def int4_prefill_linear(x: torch.Tensor, wq4: torch.Tensor,
                        sb: torch.Tensor,
                        bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Dense int4 (w4a16) GEMM for M > 256 via the grouped MoE int4
    kernel with identity routing — packed nibbles stream directly."""
    M, K2 = x.shape[0], wq4.shape[1]
    N = wq4.shape[0]
    m_pad = (M + 63) // 64 * 64
    ids, blocks, n_post = _identity_tables(x.device, m_pad, 64)
    out_pad = torch.empty(m_pad, N, dtype=x.dtype, device=x.device)
    _gpu_kernels().moe_gemm_int4(
        out_pad, x.contiguous(), wq4.view(1, N, K2),
        sb.view(1, N, -1, 2).contiguous() if sb.dim() == 3 else sb,
        ids, blocks, n_post, None, M, 1, 64, False)
    out = out_pad.narrow(0, 0, M)
    if bias is not None:
        out = out.add_(bias)
    return out


def fused_moe_fp8(x: torch.Tensor, w13: torch.Tensor, w13_scale,
                  w2: torch.Tensor, w2_scale,
                  topk_weights: torch.Tensor, topk_ids: torch.Tensor,
                  expert_start: int = 0) -> torch.Tensor:
    """fp8 grouped-GEMM MoE: same align/sum pipeline as fused_moe with
    block-scale fp8 GEMMs; expert weights stay e4m3-resident."""
    T, K = x.shape
    E_local, two_i, _ = w13.shape
    topk = topk_ids.shape[1]
    n_pairs = T * topk
    # same tile heuristic as the bf16 path (164 = BM64 x BN256 prefill)
    rpe = n_pairs / max(1, E_local)
    if n_pairs >= 4096:
        align_m, gemm_m = 64, 164
    elif rpe < 12:
        align_m = gemm_m = 16
    elif rpe < 40:
        align_m = gemm_m = 32
    else:
        align_m = gemm_m = 64
    dev = x.device
    k = _gpu_kernels()
    ids32, tables, rows_pad = _moe_tables(topk_ids, E_local, expert_start,
                                          align_m)
    aq, as_ = per_token_group_quant_fp8(x.contiguous())
    inter1 = torch.empty(rows_pad, two_i, dtype=x.dtype, device=dev)
    k.moe_gemm_fp8(inter1, aq.view(torch.uint8), as_,
                   w13.view(torch.uint8), w13_scale.contiguous(),
                   *tables, None, n_pairs, topk, gemm_m, False)
    act = silu_and_mul(inter1)
    actq, act_s = per_token_group_quant_fp8(act)
    pair_out = torch.empty(n_pairs, K, dtype=x.dtype, device=dev)
    k.moe_gemm_fp8(pair_out, actq.view(torch.uint8), act_s,
                   w2.view(torch.uint8), w2_scale.contiguous(), *tables,
                   topk_weights.float().contiguous(), n_pairs, topk,
                   gemm_m, True)
    out = torch.empty(T, K, dtype=x.dtype, device=dev)
    k.moe_sum(out, pair_out, ids32, expert_start, E_local, topk)
    return out


# --------------------------------------------------------------- gdn
def gdn_conv_update(x: torch.Tensor, weight: torch.Tensor,
                    conv_state: torch.Tensor,
                    slots: torch.Tensor) -> torch.Tensor:
    """Batched causal-conv1d decode step: x [B, C] one token per seq,
    conv_state pool rows indexed by ``slots`` roll in place."""
    out = torch.empty_like(x)
    _gpu_kernels().gdn_conv_update(out, x, weight, conv_state, slots)
    return out


def gdn_decode(qn: torch.Tensor, kn: torch.Tensor, v: torch.Tensor,
               g: torch.Tensor, beta: torch.Tensor, state: torch.Tensor,
               slots: torch.Tensor) -> torch.Tensor:
    """Batched fused recurrent gated-delta-rule step (one token per
    seq). qn/kn [B, Hv, 128] fp32 (normalized, q pre-scaled), v [B, Hv,
    Dv] fp32; state pool [slots, Hv, Dv, 128] fp32 updated in place."""
    B, Hv, Dv = v.shape
    o = torch.empty(B, Hv, Dv, dtype=torch.bfloat16, device=v.device)
    _gpu_kernels().gdn_decode(o, qn.contiguous(), kn.contiguous(),
                              v.contiguous(), g.contiguous(),
                              beta.contiguous(), state, slots)
    return o


def gdn_chunk_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                      g: torch.Tensor, beta: torch.Tensor,
                      states: torch.Tensor, scale: float) -> torch.Tensor:
    """WY chunk-parallel gated delta rule over a padded batch. q/k [B, T,
    Hk, 128], v [B, T, Hv, 128], g/beta [B, T, Hv] fp32, states [B, Hv,
    128, 128] fp32 updated IN PLACE. Falls back to the torch oracle
    off-GPU or for non-128 head dims."""
    B, T, Hk, Dk = q.shape
    Hv, Dv = v.shape[2], v.shape[3]
    if not (q.is_cuda and has_kernels() and Dk == 128 and Dv == 128
            and Hv % Hk == 0):
        from gllm_amd.ops import gdn_ref
        return gdn_ref.gated_delta_rule_chunked_batched(
            q, k, v, g, beta, scale, states)
    o = torch.empty(B, T, Hv, Dv, dtype=torch.bfloat16, device=q.device)
    _gpu_kernels().gdn_chunk_prefill(
        o, q.to(torch.bfloat16).contiguous(),
        k.to(torch.bfloat16).contiguous(),
        v.to(torch.bfloat16).contiguous(),
        g.float().contiguous(), beta.float().contiguous(),
        states, float(scale))
    return o


def gdn_rows_ok(qkvz: torch.Tensor, ba: torch.Tensor, conv_w: torch.Tensor,
                conv_state: torch.Tensor, state: torch.Tensor,
                norm_w: torch.Tensor, Dk: int, Dv: int) -> bool:
    """Whether ``gdn_rows`` takes this layer: bf16 on the GPU, heads of
    128, up to 8 taps."""
    return (qkvz.is_cuda and has_kernels() and _load_seq_kernels() is not None
            and all(t.dtype == torch.bfloat16 for t in
                    (qkvz, ba, conv_w, conv_state, norm_w))
            and state.dtype == torch.float32 and state.is_contiguous()
            and conv_state.is_contiguous() and conv_w.is_contiguous()
            and Dk == 128 and Dv == 128 and conv_w.shape[1] <= 8
            and qkvz.stride(1) == 1 and qkvz.stride(0) % 8 == 0
            and qkvz.data_ptr() % 16 == 0 and norm_w.data_ptr() % 16 == 0)


def gdn_reserve(like: torch.Tensor, rows: int, sequences: int, Hv: int):
    """Takes from ``like``'s device what the recurrence of ``gdn_rows`` works
    on for that many rows and sequences and gives it back (a profile run of a
    layer whose state is not there yet)."""
    if like.is_cuda and has_kernels():
        _gpu_kernels().gdn_reserve(like, rows, sequences, Hv)


def gdn_rows(qkvz: torch.Tensor, ba: torch.Tensor, conv_w: torch.Tensor,
             A_log: torch.Tensor, dt_bias: torch.Tensor,
             norm_w: torch.Tensor, eps: float, conv_state: torch.Tensor,
             state: torch.Tensor, slots: torch.Tensor,
             has_init: torch.Tensor, query_start_loc: torch.Tensor,
             max_query_len: int, carried: bool, Hk: int,
             scale: float) -> torch.Tensor:
    """A gated-delta layer between its projections over a ragged batch:
    short convolution, unit q and k, gates, recurrence (state in place),
    gated norm. qkvz rows are q | k | v | z, ba rows b | a; ``carried``:
    every sequence is one token on carried state. Returns [T, Hv * 128]."""
    k = _gpu_kernels()
    conv_dim = conv_w.shape[0]
    conv = causal_conv_silu(qkvz[:, :conv_dim], conv_w, conv_state, slots,
                            has_init, query_start_loc,
                            max_query_len=max_query_len)
    A = A_log.float()
    dt = dt_bias if dt_bias.dtype == torch.bfloat16 else dt_bias.float()
    if carried:
        o = k.gdn_step(conv, ba, A, dt, state, slots, Hk, scale)
    else:
        o = k.gdn_varlen(conv, ba, A, dt, state, slots, has_init,
                         query_start_loc, Hk, max_query_len, scale)
    return k.gdn_gate(o, qkvz[:, conv_dim:], norm_w, eps)


def rmsnorm_gated(x: torch.Tensor, z: torch.Tensor, weight: torch.Tensor,
                  eps: float) -> torch.Tensor:
    """out = rmsnorm(x) * w * silu(z) (fused, GPU)."""
    if not x.is_cuda:
        from gllm_amd.ops import gdn_ref
        return gdn_ref.rmsnorm_gated(x, z, weight, eps)
    out = torch.empty_like(x)
    _gpu_kernels().rmsnorm_gated(out, x.contiguous(), z.contiguous(),
                                 weight, eps)
    return out


def int4_linear(x: torch.Tensor, wq4: torch.Tensor, sbt: torch.Tensor,
                group: int,
                bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = x @ dequant(wq4).T via the int4 weight-streaming kernel
    (M <= 256): packed nibbles stream at 0.5 B/elem. ``sbt`` is the
    TRANSPOSED (scale, bias) bank [K/group, 2, N] (lane-contiguous
    staging; repack_canonical builds it), ``group`` 128."""
    if group != 128:
        raise RuntimeError("int4 gemm: group size 128")
    return quant_rows(x, ("int4", wq4, sbt), bias)


def fused_moe_int4(x: torch.Tensor, w13_c, w13_sb, w2_c, w2_sb,
                   topk_weights: torch.Tensor, topk_ids: torch.Tensor,
                   expert_start: int = 0) -> torch.Tensor:
    """int4 (w4a16) grouped-GEMM MoE: packed-nibble expert banks with
    in-fragment dequant — no bf16 materialization at all."""
    T, K = x.shape
    E_local, two_i, _ = w13_c.shape
    topk = topk_ids.shape[1]
    n_pairs = T * topk
    rpe = n_pairs / max(1, E_local)
    block_m = 16 if rpe < 12 else (32 if rpe < 40 else 64)
    dev = x.device
    k = _gpu_kernels()
    ids32, tables, rows_pad = _moe_tables(topk_ids, E_local, expert_start,
                                          block_m)
    inter1 = torch.empty(rows_pad, two_i, dtype=x.dtype, device=dev)
    k.moe_gemm_int4(inter1, x.contiguous(), w13_c, w13_sb, *tables, None,
                    n_pairs, topk, block_m, False)
    act = silu_and_mul(inter1)
    pair_out = torch.empty(n_pairs, K, dtype=x.dtype, device=dev)
    k.moe_gemm_int4(pair_out, act, w2_c, w2_sb, *tables,
                    topk_weights.float().contiguous(), n_pairs, topk,
                    block_m, True)
    out = torch.empty(T, K, dtype=x.dtype, device=dev)
    k.moe_sum(out, pair_out, ids32, expert_start, E_local, topk)
    return out


# --------------------------------------------------------------- sampling
def resolve_tokens(tokens: torch.Tensor, ring: torch.Tensor) -> torch.Tensor:
    """Negative token ids are places in ``ring`` (id -1 - i: its i-th
    entry) of tokens sampled by an earlier step."""
    if (tokens.is_cuda and tokens.dtype == torch.long
            and tokens.is_contiguous() and has_moe_kernels()):
        return _gpu_kernels().resolve_tokens(tokens, ring)
    flat = ring.view(-1)
    idx = (-tokens - 1).clamp_min(0)
    return torch.where(tokens < 0, flat[idx], tokens)


def greedy_argmax(logits: torch.Tensor) -> torch.Tensor:
    """logits.argmax(-1) of [B, V]: the first of equals, a NaN as the
    largest. (The kernel is in the core module only.)"""
    if (logits.is_cuda and logits.dim() == 2 and logits.is_contiguous()
            and logits.dtype in (torch.bfloat16, torch.float32)
            and 0 < logits.shape[1] < 2 ** 30
            and _load_kernels() is not None):
        return _gpu_kernels().greedy_argmax(logits)
    return logits.argmax(dim=-1)


def topk_topp_filter(probs: torch.Tensor, top_ks: torch.Tensor,
                     top_ps: torch.Tensor,
                     min_ps: Optional[torch.Tensor] = None):
    """In-place fused top-k/top-p/min-p filter + renormalize on [B, V]
    fp32 probs (GPU kernel; sorting-free 3-level radix select). CPU
    callers use the torch sort composite in layers/sampler.py."""
    assert probs.is_cuda
    _gpu_kernels().topk_topp_filter(
        probs, top_ks.int(), top_ps.float(),
        min_ps.float() if min_ps is not None else None)
    return probs


# --------------------------------------------------------------- mla
def apply_penalty_pool(logits, mask_pool, slots, penalties):
    """In-place repetition penalty against the persistent uint8 mask
    pool (GPU kernel; CPU callers use the inline torch math in
    layers/sampler.py)."""
    assert logits.is_cuda
    _gpu_kernels().apply_repetition_penalty(logits, mask_pool, slots,
                                            penalties)
    return logits


def cache_latent(k, k_cache, slot_mapping):
    """Scatter the absorbed-MLA latent row [T, 1, lora+rope] into the
    paged latent cache (the v 'cache' is a view of its first lora dims,
    so one write covers both). Reference concat_and_cache_mla
    (cache_kernels.py:161)."""
    if k.is_cuda:
        if k_cache.shape[-1] == 576:
            _gpu_kernels().cache_latent(
                k.reshape(k.shape[0], -1), k_cache, slot_mapping)
        else:  # non-standard latent width: plain K/V scatter, twice
            _gpu_kernels().reshape_and_cache(k, k, k_cache, k_cache,
                                             slot_mapping)
        return
    page_size = k_cache.shape[1]
    pages = torch.div(slot_mapping, page_size, rounding_mode="floor")
    offs = slot_mapping % page_size
    k_cache[pages, offs] = k.to(k_cache.dtype)


def mla_absorbed_ok(q: torch.Tensor, kv: torch.Tensor, w_kvb: torch.Tensor,
                    norm_w: torch.Tensor, k_cache: torch.Tensor,
                    cos_sin: torch.Tensor, nope: int, vdim: int) -> bool:
    """Whether ``mla_queries`` / ``mla_values`` take this layer: bf16 on
    the GPU with the latent 512 + 64, 128 unrotated query and 128 value
    dims a head (the sizes of every released checkpoint)."""
    return (q.is_cuda and q.dtype == torch.bfloat16
            and kv.dtype == torch.bfloat16 and w_kvb.dtype == torch.bfloat16
            and k_cache.dtype == torch.bfloat16 and k_cache.is_contiguous()
            and kv.shape[1] == 576 and k_cache.shape[-1] == 576
            and w_kvb.dim() == 2 and w_kvb.shape[1] == 512
            and w_kvb.is_contiguous() and nope == 128 and vdim == 128
            and norm_w.dtype in (torch.bfloat16, torch.float32)
            and cos_sin.dtype == torch.float32 and cos_sin.shape[-1] == 64
            and q.stride(1) == 1 and q.stride(0) % 8 == 0
            and kv.stride(1) == 1 and kv.stride(0) % 8 == 0
            and all(t.data_ptr() % 16 == 0
                    for t in (q, kv, w_kvb, norm_w, k_cache)))


def mla_queries(q, kv, norm_w, eps, positions, cos_sin, w_kvb, k_cache,
                slot_mapping):
    """Norm and rotate the latent rows ``kv`` [T, 576] into their cache
    slots; return the absorbed query rows [T, H, 576] of ``q`` [T, H *
    192] (rotate-half on the last 64 dims of a head)."""
    return _gpu_kernels().mla_queries(q, kv, norm_w, eps, positions, cos_sin,
                                      w_kvb, k_cache, slot_mapping)


def mla_prompts(q, kv, norm_w, eps, positions, cos_sin, w_kvb, k_cache,
                slot_mapping, query_start_loc, max_query_len, scale, out):
    """Latent attention of whole prompts (nothing of them is cached yet) in
    the per-head form: norm and rotate the latent rows ``kv`` [T, 576] into
    their cache slots, form the keys and values of every head, attend the
    prompts' own rows, into ``out`` [T, H * 128]. ``q`` [T, H * 192] is
    rotated in place. The two forms are one sum in another order; this one
    takes 320 products a pair of tokens and head where the absorbed one
    takes 1088 (4096 tokens, 16 heads, us: 102 for 380)."""
    kern = _gpu_kernels()
    lat, pe = kern.mla_prompt_rows(q, kv, norm_w, eps, positions, cos_sin,
                                   k_cache, slot_mapping)
    kern.mla_prompts(out, q, linear(lat, w_kvb), pe, query_start_loc,
                     max_query_len, scale)
    return out


def mla_values(o_lat, w_kvb):
    """Per-head values [T, H * 128] of the weighted latents [T, H, 512]."""
    return _gpu_kernels().mla_values(o_lat, w_kvb)


_MLA_GPU_WARNED = False


def mla_paged_attention(q, k_cache, v_cache, block_table, seq_lens,
                        query_start_loc, scale, topk_positions=None,
                        seq_lens_cpu=None, query_start_loc_cpu=None):
    """Varlen causal attention with asymmetric head dims (MLA).

    GPU + absorbed layout (Hkv=1, 576-dim latent) -> the gfx950 MQA
    MFMA kernel (one kernel serves decode w/ split-KV, chunked prefill
    and mixed batches — reference attention.py:366-446,653-925 roles).
    DSA sparse selection (topk_positions) and the non-absorbed debug
    layout stay on the torch path."""
    global _MLA_GPU_WARNED
    if (q.is_cuda and topk_positions is None and k_cache.shape[2] == 1
            and q.shape[-1] == 576 and v_cache.shape[-1] == 512
            and q.dtype == torch.bfloat16):
        qsl_h = query_start_loc_cpu or query_start_loc.tolist()
        max_q = max((qsl_h[i + 1] - qsl_h[i]
                     for i in range(seq_lens.shape[0])), default=1)
        T, H = q.shape[0], q.shape[1]
        out = torch.empty(T, H, 512, dtype=q.dtype, device=q.device)
        qsl_i = query_start_loc.int() \
            if query_start_loc.dtype != torch.int32 else query_start_loc
        _gpu_kernels().mla_paged_attention(
            out, q.contiguous(), k_cache, block_table, seq_lens, qsl_i,
            max_q, scale)
        return out
    if q.is_cuda and not _MLA_GPU_WARNED:
        from gllm_amd.logger import logger
        logger.warning("MLA attention falls back to the torch path on "
                       "GPU (sparse/non-absorbed layout)")
        _MLA_GPU_WARNED = True
    return torch_ref.mla_paged_attention(
        q, k_cache, v_cache, block_table, seq_lens, query_start_loc,
        scale, topk_positions=topk_positions, seq_lens_cpu=seq_lens_cpu,
        query_start_loc_cpu=query_start_loc_cpu)


# --------------------------------------------------------------- gemm
SKINNY_MAX_M = 256


def _rows_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """bf16 operands as csrc/stream_gemm.hip reads them: 16 B aligned
    rows, K a multiple of 64, N of 8."""
    return (x.is_cuda and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and x.dim() == 2 and w.dim() == 2
            and x.is_contiguous() and w.is_contiguous()
            and w.shape[1] % 64 == 0 and w.shape[0] % 8 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)


def plain_bias(bias, N: int) -> bool:
    return bias is None or (bias.dtype == torch.bfloat16
                            and bias.is_contiguous() and bias.numel() == N)


def skinny_gemm(x: torch.Tensor, w: torch.Tensor,
                bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = x @ w.T (+ bias) via the gfx950 weight-streaming kernel (at
    most 256 rows; an N or an address off its units goes to the library). A
    bias of another type is added to the bf16 product."""
    if not (x.is_cuda and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and x.is_contiguous()
            and w.is_contiguous() and w.shape[1] % 64 == 0
            and x.shape[0] <= 256):
        raise RuntimeError("skinny_gemm: contiguous bf16 on the GPU, K a "
                           "multiple of 64, at most 256 rows")
    if _rows_ok(x, w):
        run = _gpu_kernels().stream_gemm
    else:
        run = torch.nn.functional.linear
    if plain_bias(bias, w.shape[0]):
        return run(x, w, bias)
    out = run(x, w, None)
    out += bias
    return out


def _use_skinny(M: int, N: int, K: int) -> bool:
    """Measured against hipBLASLt (us, stream / library): up to 64 rows
    the stream wins wherever the product is more than a few workgroups (64
    x 5120 x 5120 18.9 / 21.5, 64 x 38016 x 5120 84 / 90, 64 x 5120 x 27648
    60 / 158); above that the library is level on wide weights (96 x 28672
    x 4096 53.7 / 55.0, 128 x 19008 x 5120 53.4 / 51.8, 128 x 38016 x 5120
    98 / 100) and, with 256 rows, ahead on the widest (28672 x 4096 82 /
    70, 38016 x 5120 158 / 111; 19008 x 5120 69 / 80, 16384 x 4096 54.7 /
    52.8), and it is behind on the rest (256 x 7168 x 5120 39 / 51, 256 x
    5120 x 27648 84 / 265)."""
    if K % 64 != 0 or N < 512 or M > SKINNY_MAX_M or M == 0:
        return False
    import os
    if os.environ.get("GLLM_DISABLE_SKINNY"):
        return False
    if M > (int(os.environ.get("GLLM_SKINNY_MAX_M", "0")) or SKINNY_MAX_M):
        return False
    return M <= 64 or N < 16384


def _streams(x: torch.Tensor, w: torch.Tensor) -> bool:
    return _rows_ok(x, w) and _use_skinny(x.shape[0], w.shape[0],
                                          w.shape[1])


def _tile_fits(M: int, N: int, K: int, gated: bool) -> bool:
    """Sizes that csrc/tile_gemm.hip takes (more rows than the streaming
    kernel's)."""
    return (M > SKINNY_MAX_M and K % 64 == 0 and N <= 1 << 20
            and K <= 1 << 21 and M <= 1 << 24
            and ((M + 127) // 128) * (N // 256 + 2) < 1 << 24
            and (not gated or N * K < 1 << 30))


@functools.lru_cache(maxsize=None)
def _compute_units() -> int:
    return torch.cuda.get_device_properties(
        torch.cuda.current_device()).multi_processor_count


def one_round(M: int, N: int) -> bool:
    """Whether an M x N product is a round of 256 x 256 tiles at most."""
    return -(-M // 256) * -(-N // 256) <= _compute_units()


@functools.lru_cache(maxsize=4096)
def _use_tile(M: int, N: int, K: int) -> bool:
    """Plain products for csrc/tile_gemm.hip: long K, where hipBLASLt keeps
    whole tiles and leaves CUs idle or falls to small ones, from 0.5 to 1.65
    PFLOP/s (us, library / tile): 4133 x 5120 x 27648 1448 / 810, 5000 x 5120
    x 27648 1667 / 1013, 4100 x 4096 x 14336 725 / 347, 512 x 4096 x 29568
    267 / 121. The library goes on where a tile's step of 1.33 us says less
    than 1.2 PFLOP/s (2800 x 4096 x 14336 236 / 291), with shorter K, where
    it is mostly 5 % ahead (4133 x 7168 x 5120 202 / 216), and where its own
    tiles fit: a last round of 256 x 256 tiles that is nearly full (8192 x
    4096 x 14336 605 / 642, 8192 x 2048 x 6144 131 / 142), a single one that
    is half to four fifths full (8192 x 1536 x 11904 222 / 278, 2304 x 5120 x
    15360 277 / 319), and, with K below 14336, any that is more than half
    full, below 9600 two fifths (10594 x 2560 x 7680 301 / 332; 4096 x 2048 x
    10944 154 / 142). Over 3977 sizes of 256 to 16384 rows this takes 915, in
    0.72 of the library's time, five of them slower by 3 to 7 %."""
    if K < 3 * N or not _tile_fits(M, N, K, False):
        return False
    tiles, cus = -(-M // 256) * -(-N // 256), _compute_units()
    last = ((tiles - 1) % cus + 1) / cus  # full part of the last round
    if last > 0.9 or (tiles <= cus and 0.5 < last <= 0.8) \
            or K < (0 if last <= 0.4 else 9600 if last <= 0.5 else 14336):
        return False
    us = 1.33 * _gpu_kernels().tile_gemm_cost(M, N, K, False)
    return us * 1.2e9 < 2.0 * M * N * K


@functools.lru_cache(maxsize=4096)
def _use_tile_gated(M: int, N: int, K: int) -> bool:
    """Gated products for csrc/tile_gemm.hip (us, library and the second
    kernel or, up to 256 rows, stream / tile).
    More than 256 rows: the tile kernel (512 x 5632 x 2048 31 / 26, 700 x
    55296 x 5120 415 / 342, 4133 x 55296 x 5120 1971 / 1750, 4133 x 9728 x
    2560 265 / 193), where hipBLASLt's tiles do not fit better:
      half a row block is left, of few of them (384 x 55296 x 5120 218 / 260,
      1152 x 43008 x 3840 332 / 367);
      a single round of tiles, less than 25 / 32 full (512 x 9728 x 2560 41 /
      46, 768 x 16384 x 11136 223 / 269);
      a second one, half full (714 x 32768 x 2560 126 / 142) or, with short
      K, less than a third (1242 x 16384 x 1536 75 / 81).
    With short K the second kernel weighs more, so a single round or an
    estimate (as in ``_use_tile``) of 1.1 PFLOP/s is enough, and so are few
    tiles of any K, where the library does not split it. Below 384 rows wide
    weights stay with the library (333 x 55296 x 5120 217 / 270). Over 3827
    sizes of 257 to 9000 rows this takes 1995, in 0.84 of the time, three of
    them slower by 4 %.
    One block of rows: weights of a round of tiles that is at least 25 / 32
    full, for K of 1024 to 14336 (256 x 51200 x 1024 34 / 32, 256 x 51200 x
    4096 119 / 104, 129 x 61440 x 14336 426 / 341; 256 x 49152 x 8192 223 /
    233, 256 x 28672 x 4096 67 / 80)."""
    if not (K % 64 == 0 and N <= 1 << 20 and M <= 1 << 24
            and N * K < 1 << 30):
        return False
    cus, cols = _compute_units(), -(-N // 256)
    if M <= SKINNY_MAX_M:
        return 128 < M and 25 * cus <= 32 * cols <= 32 * cus and K >= 1024
    if not _tile_fits(M, N, K, True) or (M < 384 and N >= 16384):
        return False
    tiles = -(-M // 256) * cols
    if tiles <= 20:
        return True
    if K <= 2048:
        us = 1.33 * _gpu_kernels().tile_gemm_cost(M, N, K, True)
        if tiles <= cus or us * 1.1e9 < 2.0 * M * N * K:
            return True
    if 0 < M % 256 <= 128 and M < 1600:
        return False
    if tiles <= cus:
        return 32 * tiles > 25 * cus
    if tiles <= 2 * cus:
        last = tiles / cus - 1
        return not 0.47 < last < 0.53 and (K > 2048 or last > 1 / 3)
    return True


def linear(x: torch.Tensor, w: torch.Tensor,
           bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """GEMM dispatch: the weight-streaming kernel for few rows, the tile
    kernel for many rows and long K, where measured faster; hipBLASLt
    otherwise."""
    import torch.nn.functional as F
    if _rows_ok(x, w):
        M, (N, K) = x.shape[0], w.shape
        if _use_skinny(M, N, K):
            return skinny_gemm(x, w, bias)
        if (_use_tile(M, N, K) and plain_bias(bias, N)
                and (bias is None or bias.data_ptr() % 16 == 0)
                and not (torch.is_grad_enabled()  # (the library's has one)
                         and any(t is not None and t.requires_grad
                                 for t in (x, w, bias)))):
            return _gpu_kernels().tile_gemm(x, w, bias, False)
    return F.linear(x, w, bias)


def linear_silu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x @ w_gate.T) * (x @ w_up.T), w = gate rows over up rows. Few
    rows: one kernel, the [rows, 2 ff] product is never written (above 64
    rows it is level with the library's product and saves the second
    kernel: 256 x 55296 x 5120 149 us against 154 + 9). Many rows, and one
    block of them on very wide weights: the tile kernel, again one, where it
    is the faster (see ``_use_tile_gated``)."""
    if (_rows_ok(x, w) and w.shape[0] % 16 == 0 and w.shape[0] >= 512):
        M, (N, K) = x.shape[0], w.shape
        few = _use_skinny(M, 512, K)
        if (few or M > SKINNY_MAX_M) and _use_tile_gated(M, N, K):
            return _gpu_kernels().tile_gemm(x, w, None, True)
        if few:
            return _gpu_kernels().stream_gemm_gated(x, w)
    return silu_and_mul(linear(x, w))


def _norm_parts_ok(N: int, residual: torch.Tensor,
                   norm_w: torch.Tensor) -> bool:
    return (N % 8 == 0 and N <= 8192 and residual.dtype == torch.bfloat16
            and residual.is_contiguous() and residual.data_ptr() % 16 == 0
            and norm_w.dtype in (torch.bfloat16, torch.float32))


def linear_add_rmsnorm(x: torch.Tensor, w: torch.Tensor,
                       residual: torch.Tensor, norm_w: torch.Tensor,
                       eps: float):
    """residual += x @ w.T; (rmsnorm(residual), residual). Few rows: the
    split product's parts are summed, added and normed by one kernel."""
    if _streams(x, w) and _norm_parts_ok(w.shape[0], residual, norm_w):
        return _gpu_kernels().stream_add_norm(x, w, residual, norm_w,
                                              eps), residual
    return fused_add_rmsnorm(linear(x, w), residual, norm_w, eps)


def qkv_parts(x: torch.Tensor, w: torch.Tensor,
              bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """The fp32 parts [S, M, N] of x @ w.T for ``qkv_rope_cache``, or None
    where the library's product is the better one."""
    if _streams(x, w) and plain_bias(bias, w.shape[0]):
        return _gpu_kernels().stream_parts(x, w)
    return None


def qkv_rope_cache_ok(k_cache: torch.Tensor, v_cache: torch.Tensor,
                      cos_sin: torch.Tensor, is_neox: bool) -> bool:
    return (is_neox and k_cache.is_cuda and k_cache.dim() == 4
            and k_cache.dtype == torch.bfloat16
            and v_cache.dtype == torch.bfloat16
            and v_cache.shape == k_cache.shape and k_cache.is_contiguous()
            and v_cache.is_contiguous() and k_cache.shape[3] % 8 == 0
            and cos_sin.device == k_cache.device
            and cos_sin.dtype == torch.float32 and cos_sin.is_contiguous()
            and cos_sin.shape[-1] % 8 == 0
            and cos_sin.shape[-1] <= k_cache.shape[3])


def qkv_rope_cache(src: torch.Tensor, bias, positions: torch.Tensor,
                   cos_sin: torch.Tensor, k_cache: torch.Tensor,
                   v_cache: torch.Tensor, slot_mapping: torch.Tensor,
                   num_heads: int, rounded: bool = False) -> torch.Tensor:
    """From a merged q|k|v projection (bf16 rows, or the fp32 parts of
    ``qkv_parts``): add the bias, rotate queries and keys, write keys and
    values to their cache slots, return the queries [M, heads * D]. One
    kernel for a bias, a rotation, a scatter and their copies.
    ``rounded``: the biased rows are rounded to bf16 first (fp8 weights)."""
    return _gpu_kernels().qkv_finish(src, bias, positions, cos_sin, k_cache,
                                     v_cache, slot_mapping, num_heads,
                                     rounded)


def qkv_norm_rope_cache_ok(src: torch.Tensor, q_w: torch.Tensor,
                           k_w: torch.Tensor, k_cache: torch.Tensor,
                           cos_sin: torch.Tensor) -> bool:
    """Whether ``qkv_norm_rope_cache`` takes these, with caches that
    ``qkv_rope_cache_ok`` takes."""
    return (has_kernels() and src.dtype == torch.bfloat16 and src.dim() == 2
            and src.stride(1) == 1 and src.stride(0) % 8 == 0
            and k_cache.shape[3] <= 128 and cos_sin.shape[-1] % 16 == 0
            and q_w.dtype == k_w.dtype
            and q_w.dtype in (torch.bfloat16, torch.float32)
            and all(t.is_contiguous() and t.numel() == k_cache.shape[3]
                    for t in (q_w, k_w))
            and all(t.data_ptr() % 16 == 0 for t in (src, q_w, k_w)))


def qkv_norm_rope_cache(src: torch.Tensor, q_w: torch.Tensor,
                        k_w: torch.Tensor, eps: float,
                        positions: torch.Tensor, cos_sin: torch.Tensor,
                        k_cache: torch.Tensor, v_cache: torch.Tensor,
                        slot_mapping: torch.Tensor,
                        num_heads: int) -> torch.Tensor:
    """``qkv_rope_cache`` of bf16 rows with an RMS norm of each query and key
    head in front of the rotation."""
    return _gpu_kernels().qkv_norm_finish(src, q_w, k_w, eps, positions,
                                          cos_sin, k_cache, v_cache,
                                          slot_mapping, num_heads)


def qkv_decode_ok(parts: torch.Tensor, k_cache: torch.Tensor,
                  num_heads: int, rounded: bool = False) -> bool:
    """Whether ``qkv_decode`` takes these rows and heads (with caches that
    ``qkv_rope_cache_ok`` takes) and is the faster form."""
    return parts.dim() == 3 and _gpu_kernels().qkv_decode_ok(
        k_cache, num_heads, parts.shape[1], rounded)


def qkv_decode(parts: torch.Tensor, bias, positions: torch.Tensor,
               cos_sin: torch.Tensor, k_cache: torch.Tensor,
               v_cache: torch.Tensor, slot_mapping: torch.Tensor,
               block_table: torch.Tensor, seq_lens: torch.Tensor,
               arrived: torch.Tensor, num_heads: int, scale: float,
               sliding_window: int = 0, rounded: bool = False,
               fp8: bool = False):
    """``qkv_rope_cache`` and the decode attention behind it, one token per
    sequence, as one kernel; the heads' outputs [B, heads * D]. Each slot is
    the last of its sequence. ``arrived``: int32 zeros, one per sequence and
    kv head, that are zeros again behind the launch (launches that may run
    at the same time need their own). ``fp8``: as ``Fp8Rows`` where a head
    is a group of 128."""
    args = (parts, bias, positions, cos_sin, k_cache, v_cache, slot_mapping,
            block_table, seq_lens, arrived, num_heads, scale, sliding_window,
            rounded)
    if fp8 and k_cache.shape[3] == 128:
        return Fp8Rows(*_gpu_kernels().qkv_decode_fp8(*args))
    return _gpu_kernels().qkv_decode(*args)


# --------------------------------------------------------------- layer norm
def layernorm_f32(x: torch.Tensor, w: torch.Tensor, b, eps: float,
                  dtype) -> torch.Tensor:
    """h = LayerNorm(x) with weight and optional bias (``b`` None =
    weight only); x is the fp32 residual stream, h comes out in
    ``dtype`` (the dtype of w and b)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=dtype, device=x.device)
        _seq_kernels().layernorm_f32(out, x, w, b, eps)
        return out
    return torch_ref.layernorm_f32(x, w, b, eps, dtype)


def residual_layernorm(x: torch.Tensor, y: torch.Tensor, w_post, b_post,
                       eps: float, pre=None, gate=None):
    """x (fp32, in place) += LN_post(y); with ``pre`` = (weight, bias)
    also returns LN_pre(x) in y's dtype — one launch per layer boundary
    of a sandwich-norm decoder. Biases may be None. ``gate`` ([rows,
    width] logits, row views allowed): LN_post sees y * sigmoid(gate),
    the product formed in fp32 inside the same launch."""
    if x.is_cuda:
        h = None
        if pre is not None:
            h = torch.empty(x.shape, dtype=y.dtype, device=x.device)
            _seq_kernels().residual_layernorm(x, y, w_post, b_post, h,
                                              pre[0], pre[1], eps, gate)
        else:
            _seq_kernels().residual_layernorm(x, y, w_post, b_post, None,
                                              None, None, eps, gate)
        return h
    return torch_ref.residual_layernorm(x, y, w_post, b_post, eps, pre,
                                        gate)


def stream_rmsnorm(x: torch.Tensor, y, w_post, eps: float,
                   mult: float = 1.0, y_scale: float = 1.0, y2=None,
                   add=None, pre_w=None, post_off: float = 0.0,
                   pre_off: float = 0.0, cast=None):
    """One launch per sublayer boundary of an RMS post- or sandwich-norm
    decoder over an fp32 stream x (in place):
        x += mult * RMSnorm(y_scale * (y + y2)) * (post_off + w_post)
                                                           (y given)
        x += add                                           (add: fp32 [width])
        returns RMSnorm(x) * (pre_off + pre_w) in pre_w's dtype
                                                           (pre_w given)
        or x itself in dtype ``cast``                      (cast given)
    y / y2 may be row views; statistics and sums are fp32."""
    if x.is_cuda:
        h = None
        if pre_w is not None:
            cast = pre_w.dtype
        if cast is not None:
            h = torch.empty(x.shape, dtype=cast, device=x.device)
        _seq_kernels().stream_rmsnorm(x, y, y2, w_post, add, h, pre_w,
                                      float(eps), float(mult),
                                      float(y_scale), float(post_off),
                                      float(pre_off))
        return h
    return torch_ref.stream_rmsnorm(x, y, w_post, eps, mult, y_scale, y2,
                                    add, pre_w, post_off, pre_off, cast)


def stream_tanh(x, y=None, pair=None, nxt=None, embed=None):
    """One launch per layer boundary of a decoder whose norms are dynamic
    tanhs over an fp32 stream x (in place):
        x = table[ids] * scale             (embed = (ids, table, scale))
        x += s * (RMSnorm(l) * w_l + RMSnorm(r) * w_r)
                                    (pair = (l, w_l, r, w_r, s, eps))
        x += y                                             (y given)
        returns tanh(alpha * x) * w + b in w's dtype
                                              (nxt = (alpha, w, b))
    alpha, scale and s are numbers; y, l and r may be row views."""
    if x.is_cuda:
        ids, table, scale = embed if embed is not None else (None, None, 1.0)
        l, w_l, r, w_r, s, eps = pair if pair is not None \
            else (None, None, None, None, 0.0, 0.0)
        alpha, w, b = nxt if nxt is not None else (0.0, None, None)
        h = None
        if w is not None:
            h = torch.empty(x.shape, dtype=w.dtype, device=x.device)
        _seq_kernels().stream_tanh(x, ids, table, float(scale), y, l, w_l, r,
                                   w_r, float(s), float(eps), h, w, b,
                                   float(alpha))
        return h
    return torch_ref.stream_tanh(x, y, pair, nxt, embed)


def embed_rmsnorm(ids, positions, table, pos, w, scale: float,
                  w_off: float, eps: float):
    """Token embedding of a decoder that norms it: returns (x, h) with
    x = RMSnorm(table[ids] * scale + pos[positions]) * (w_off + w) in fp32
    (the residual stream) and h its copy in the table's dtype. ``pos``
    (a learned position table) may be None."""
    if table.is_cuda:
        T, width = ids.shape[0], table.shape[1]
        x = torch.empty(T, width, dtype=torch.float32, device=table.device)
        h = torch.empty(T, width, dtype=table.dtype, device=table.device)
        _seq_kernels().embed_rmsnorm(x, h, ids, positions, table, pos, w,
                                     float(scale), float(w_off), float(eps))
        return x, h
    return torch_ref.embed_rmsnorm(ids, positions, table, pos, w, scale,
                                   w_off, eps)


def gated_act_mul(x: torch.Tensor, act: str = "silu") -> torch.Tensor:
    """x [rows, 2d] = gate | up -> act(gate) * up with act "silu" or
    "gelu_tanh"; any d, rows may be strided (bf16 or fp32)."""
    assert act in ("silu", "gelu_tanh")
    if x.is_cuda:
        out = torch.empty(x.shape[0], x.shape[1] // 2, dtype=x.dtype,
                          device=x.device)
        _seq_kernels().gated_act_mul(out, x, 0 if act == "silu" else 1)
        return out
    if act == "silu":
        return torch_ref.silu_and_mul(x)
    return torch_ref.gelu_tanh_and_mul(x)


def tanh_rows(x: torch.Tensor) -> torch.Tensor:
    """tanh of x [rows, n] (a column block of a wider buffer is fine),
    contiguous result in x's dtype."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq_kernels().tanh_rows(out, x)
        return out
    return torch.tanh(x.float()).to(x.dtype)


def sigmoid_group_topk(logits: torch.Tensor, correction, topk: int,
                       n_group: int = 1, keep: int = 1,
                       scale: float = 1.0):
    """Sigmoid router with a selection-only correction and group
    limits, one kernel on the GPU. logits fp32 [T, E]; returns (weights
    fp32 [T, topk], ids int32 [T, topk]). See torch_ref for the rule."""
    if logits.is_cuda:
        T = logits.shape[0]
        weights = torch.empty(T, topk, dtype=torch.float32,
                              device=logits.device)
        ids = torch.empty(T, topk, dtype=torch.int32, device=logits.device)
        _seq_kernels().sigmoid_group_topk(weights, ids, logits, correction,
                                          int(n_group), int(keep),
                                          float(scale))
        return weights, ids
    return torch_ref.sigmoid_group_topk(logits, correction, topk, n_group,
                                        keep, scale)


# --------------------------------------------------------------- windowed attn
def qk_norm_rope_store(q, k, v, q_w, k_w, positions, slot_mapping, freqs,
                       mag, rot_dims, k_cache, v_cache, H, G, D, Dv, eps,
                       half_layout=False, norm_last=False, do_norm=True,
                       v_freqs=None, norm_span=False, v_unit=False,
                       q_out=None):
    """Fused per-head q/k RMS norm, rotary (per-pair frequency table
    ``freqs`` fp64, cos/sin scaled by ``mag``) and paged K/V store.
    q [T, H*D] is updated in place (may be a column slice of a merged
    projection); k/v None = the layer reads another's cache.

    ``q_w``/``k_w`` None: unit-RMS heads without a weight.
    ``half_layout``: dimension i rotates with i + rot_dims/2 (the
    default pairs 2i with 2i+1). ``norm_last``: rotate, then norm.
    ``v`` may be ``k`` itself (values = keys as projected).
    ``do_norm`` False: rotary and store only. ``v_freqs`` (fp64
    [Dv/2]): each value row is turned by its own position over all of
    Dv (same pair layout) on its way into the cache.
    ``norm_span``: one RMS over all heads of a token's q (and of its k)
    with weights that cover the row ([H*D], [G*D]). ``v_unit``: each
    value head is divided by its RMS (eps inside the root, no weight)
    before it is stored. ``q_out`` ([T, H*D]): the prepared queries go
    there and q stays as it came (required with ``norm_span``)."""
    if q.is_cuda:
        _seq_kernels().qk_norm_rope_store(
            q, k, v, q_w, k_w, positions, slot_mapping, freqs, mag,
            rot_dims, k_cache, v_cache, H, G, D, Dv, eps,
            bool(half_layout), bool(norm_last), bool(do_norm), v_freqs,
            bool(norm_span), bool(v_unit), q_out)
        return
    torch_ref.qk_norm_rope_store(q, k, v, q_w, k_w, positions,
                                 slot_mapping, freqs, mag, rot_dims,
                                 k_cache, v_cache, H, G, D, Dv, eps,
                                 half_layout, norm_last, do_norm, v_freqs,
                                 norm_span, v_unit, q_out)


def rotate_scale_rows(x, positions, freqs, heads, D, sign=1.0, scale=1.0,
                      half_layout=False, out=None) -> torch.Tensor:
    """Turn the pairs of every head row of x [T, heads*D] by
    sign * position * freqs[m] and scale the result (sign -1 undoes the
    turn that rotated values carry). ``out`` may be a column block of a
    wider buffer."""
    if x.is_cuda:
        if out is None:
            out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq_kernels().rotate_scale_rows(out, x, positions, freqs, heads, D,
                                         float(sign), float(scale),
                                         bool(half_layout))
        return out
    return torch_ref.rotate_scale_rows(x, positions, freqs, heads, D, sign,
                                       scale, half_layout, out)


def rms_weight_store(x, w, eps, cache=None, slot_mapping=None):
    """x / rms(x) * w per row (fp32 inside, x's dtype out); with
    ``cache`` [pages, page, 1, n] the normed rows are also scattered
    into their paged slots (a cached low-rank latent)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq_kernels().rms_weight_store(out, x, w, eps, cache, slot_mapping)
        return out
    return torch_ref.rms_weight_store(x, w, eps, cache, slot_mapping)


def latent_rope_store(q, ckv, w, eps, positions, slot_mapping, freqs, mag,
                      cache, H, D, R, Dr) -> None:
    """What a latent-attention layer prepares per token, in one launch:
    cache row <- [RMSnorm(ckv[:R]) * w | ckv[R:] turned by the position],
    and the last Dr columns of every head of q [T, H*(D+Dr)] turned in
    place (pairs (2i, 2i+1), fp64 frequencies, cos / sin times mag)."""
    if q.is_cuda:
        _seq_kernels().latent_rope_store(q, ckv, w, float(eps), positions,
                                         slot_mapping, freqs, float(mag),
                                         cache, H, D, R, Dr)
        return
    torch_ref.latent_rope_store(q, ckv, w, eps, positions, slot_mapping,
                                freqs, mag, cache, H, D, R, Dr)


def latent_attention(q_lat, q_rot, cache, block_table, seq_lens,
                     query_start_loc, scale, window=0, sinks=None,
                     max_query_len=0) -> torch.Tensor:
    """Ragged attention of H query heads over ONE cached row per token,
    [latent (R) | rotated key part (Dr)] in ``cache`` [pages, page, 1,
    R + Dr]: score = (q_lat . latent + q_rot . rotated) * scale, position
    i sees 0 <= i - j < window (window <= 0: every j <= i), ``sinks``
    (fp32 [H]) join the softmax denominator, and the result per head is
    the weighted latent. q_lat [H, T, R], q_rot [T, H, Dr] (views are
    fine); returns [H, T, R].

    bf16 with R <= 512, R + Dr <= 576 and 8-aligned sizes runs the MFMA
    kernel (prompt portions, mixed batches and, with the keys split,
    decoding); fp32 and other sizes the generic windowed kernel."""
    H, T, R = q_lat.shape
    if q_lat.is_cuda and q_lat.dtype == torch.bfloat16:
        out = torch.empty(H, T, R, dtype=q_lat.dtype, device=q_lat.device)
        if _seq_kernels().latent_attention_mfma(
                out, q_lat, q_rot, cache, block_table, seq_lens,
                query_start_loc, float(scale), int(window), sinks,
                int(max_query_len)):
            return out
    q = torch.cat([q_lat.transpose(0, 1), q_rot], -1).reshape(T, -1)
    # (the generic kernel holds up to 512 value columns)
    parts = [window_attention(q, None, cache, cache[..., c:min(c + 512, R)],
                              block_table, seq_lens, query_start_loc, scale,
                              window, 0, False, max_query_len,
                              sinks=sinks).view(T, H, -1)
             for c in range(0, R, 512)]
    o = parts[0] if len(parts) == 1 else torch.cat(parts, -1)
    return o.transpose(0, 1)


def head_gate(x, gate=None) -> torch.Tensor:
    """x [H, T, D] (head major) -> [T, H*D], each element times
    sigmoid(gate [T, H*D]) when a gate is given (row views are fine)."""
    H, T, D = x.shape
    if x.is_cuda:
        out = torch.empty(T, H * D, dtype=x.dtype, device=x.device)
        _seq_kernels().head_gate(out, x, gate)
        return out
    return torch_ref.head_gate(x, gate)


# --------------------------------------------------------------- streams
def hyper_streams(xs, y=None, y2=None, gate=None, mix=None, out_w=None,
                  read=None, dtype=None):
    """Hyper-connection residual xs [S, T, W] fp32.

    Write (``y`` given, in place): x_t <- sum_s mix[s, t] x_s +
    out_w[t] * (y + sigmoid(gate) * y2), all streams from the old ones;
    y2 / gate ([T, 1] logits) optional. Read (``read`` = (in_w [S],
    gain [1], eps)): returns gain * u / rms(u) in ``dtype`` with
    u = sum_s in_w[s] x_s — of the updated streams when both are asked
    for (one launch per sublayer boundary)."""
    if xs.is_cuda:
        h = None
        in_w = gain = None
        eps = 0.0
        if read is not None:
            in_w, gain, eps = read
            h = torch.empty(xs.shape[1:], dtype=dtype, device=xs.device)
        _seq_kernels().hyper_streams(xs, y, y2, gate, mix, out_w, h, in_w,
                                     gain, eps)
        return h
    return torch_ref.hyper_streams(xs, y, y2, gate, mix, out_w, read, dtype)


# --------------------------------------------------------------- minGRU
def mingru_varlen(zx, gp, state, slots, has_init, query_start_loc,
                  scale=1.0, max_query_len=0, out=None) -> torch.Tensor:
    """Ragged minGRU (prompt portions and decode tokens in one
    launch): zx [T, 2C] update-gate | candidate pre-activations, gp
    [T, C] read-out gate logits, fp32 state [slots, C] in place.
    Returns scale * S_t * silu(gp_t) in zx's dtype ([T, C]; ``out`` may
    be a column block of a wider buffer)."""
    if zx.is_cuda:
        if out is None:
            out = torch.empty(gp.shape, dtype=zx.dtype, device=zx.device)
        _seq_kernels().mingru_varlen(out, zx, gp, state, slots, has_init,
                                     query_start_loc, float(scale),
                                     int(max_query_len))
        return out
    return torch_ref.mingru_varlen(zx, gp, state, slots, has_init,
                                   query_start_loc, scale, out)


def clamp_swiglu(x: torch.Tensor, limit: float, alpha: float = 1.702,
                 out=None) -> torch.Tensor:
    """x [rows, 2d] = gate | up -> min(g, limit) * sigmoid(alpha g) *
    (clamp(u, -limit, limit) + 1); ``out`` may be a column block of a
    wider buffer."""
    if x.is_cuda:
        if out is None:
            out = torch.empty(x.shape[0], x.shape[1] // 2, dtype=x.dtype,
                              device=x.device)
        _seq_kernels().clamp_swiglu(out, x, float(limit), float(alpha))
        return out
    res = torch_ref.clamp_swiglu(x, limit, alpha)
    if out is not None:
        out.copy_(res)
        return out
    return res


def window_attention(q, gate, k_cache, v_cache, block_table, seq_lens,
                     query_start_loc, scale, window=0, keep_first=0,
                     sink=False, max_query_len=0, sinks=None,
                     softcap=0.0, out=None, bias=None,
                     temp=(0.0, 0)) -> torch.Tensor:
    """Ragged paged attention over K [pages, page, G, D] / V [.., Dv]:
    sliding window with kept first tokens, optional softmax sink (+1 in
    the denominator; ``sinks`` fp32 [H]: exp(sinks[h]) instead), tanh
    score cap (``softcap`` > 0: cap * tanh(s / cap)) and fused sigmoid
    output gate. K and V may be the same tensor (attention over a
    cached latent). ``bias`` (fp32 [H, L]): bias[h, min(i - j, L - 1)]
    is added to the scaled (and capped) score. ``temp`` = (coef, every)
    with every > 0: the query at position p is multiplied by 1 + coef *
    ln(floor((p + 1) / every) + 1). Returns [T, H*Dv]; ``out`` may be a
    column block of a wider buffer.

    Batches that hold prompt portions (``max_query_len`` > 1) in bf16
    with D and Dv multiples of 8 up to 128 run the MFMA tile kernel
    shared with paged_attention (128 query rows per workgroup, K/V
    streamed through LDS); decode-only bf16 batches of these sizes with
    up to 16 query heads per kv head run the split-KV decode kernels;
    fp32 and every other head geometry run the generic
    one-workgroup-per-(token, head) kernel."""
    if q.is_cuda:
        T = q.shape[0]
        D, Dv = k_cache.shape[3], v_cache.shape[3]
        H = q.shape[1] // D
        if out is None:
            out = torch.empty(T, H * Dv, dtype=q.dtype, device=q.device)
        coef, every = float(temp[0]), int(temp[1])
        rows = (q.dtype == torch.bfloat16 and k_cache.is_contiguous()
                and v_cache.is_contiguous())
        if (max_query_len > 1 and rows and D % 8 == 0 and Dv % 8 == 0
                and D <= 128 and Dv <= 128):
            _seq_kernels().window_attention_mfma(
                out, q, gate, k_cache, v_cache, block_table, seq_lens,
                query_start_loc, max_query_len, scale, window, keep_first,
                sink, sinks, softcap, bias, coef, every)
            return out
        if (max_query_len == 1 and rows
                and _seq_kernels().window_attention_decode(
                    out, q, gate, k_cache, v_cache, block_table, seq_lens,
                    scale, window, keep_first, sink, sinks, softcap, bias,
                    coef, every)):
            # decode-only batch on the split-KV kernels shared with
            # paged_attention (one workgroup per GQA group and KV split)
            return out
        _seq_kernels().window_attention(
            out, q, gate, k_cache, v_cache, block_table, seq_lens,
            query_start_loc, scale, window, keep_first, sink, sinks,
            softcap, bias, coef, every)
        return out
    res = torch_ref.window_attention(q, gate, k_cache, v_cache,
                                     block_table, seq_lens,
                                     query_start_loc, scale, window,
                                     keep_first, sink, sinks, softcap,
                                     bias, temp)
    if out is not None:
        out.copy_(res)
        return out
    return res


# --------------------------------------------------------------- talking heads
def talking_attention(q, k_cache, v_cache, block_table, seq_lens,
                      query_start_loc, scale, talk, sink=None,
                      max_query_len=0) -> torch.Tensor:
    """Ragged paged causal attention with cross-head score mixing:
    s_g = scale * q_g . k_kv(g) for all H heads, s'_h = sum_g
    talk[h, g] s_g, softmax over the keys per head with exp(sink[h])
    added to the denominator (``sink`` None: plain softmax), output
    head h = weights . v_kv(h). K [pages, page, G, D], V [.., Dv];
    talk [H, H] and sink [H] fp32. Returns [T, H*Dv].

    All heads of a query are handled together (the mix couples them).
    bf16 batches with prompt portions and D == Dv a multiple of 32
    run the MFMA tile kernel; bf16 decode-only batches the split-KV
    kernel; fp32 and other shapes the generic kernel."""
    if q.is_cuda:
        T = q.shape[0]
        D, Dv = k_cache.shape[3], v_cache.shape[3]
        H = q.shape[1] // D
        out = torch.empty(T, H * Dv, dtype=q.dtype, device=q.device)
        _seq_kernels().talking_attention(
            out, q, k_cache, v_cache, block_table, seq_lens,
            query_start_loc, scale, talk, sink, max_query_len)
        return out
    return torch_ref.talking_attention(q, k_cache, v_cache, block_table,
                                       seq_lens, query_start_loc, scale,
                                       talk, sink)


# --------------------------------------------------------------- activations
def xielu(x: torch.Tensor, a_pos: float, a_neg: float) -> torch.Tensor:
    """xIELU: z > 0 -> a_pos z^2 + z/2, else a_neg (e^z - 1 - z) + z/2."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _seq_kernels().xielu(out, x, a_pos, a_neg)
        return out
    return torch_ref.xielu(x, a_pos, a_neg)


def relu2(x: torch.Tensor) -> torch.Tensor:
    """max(x, 0)^2."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _seq_kernels().relu2(out, x)
        return out
    return torch_ref.relu2(x)


def gelu_erf(x: torch.Tensor) -> torch.Tensor:
    """Exact gelu: z * Phi(z)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq_kernels().gelu_erf(out, x)
        return out
    return torch_ref.gelu_erf(x)


def token_gate(z, table, ids, col0: int) -> torch.Tensor:
    """gelu_tanh(z [T, n]) * table[ids, col0:col0 + n]."""
    if z.is_cuda:
        out = torch.empty(z.shape, dtype=z.dtype, device=z.device)
        _seq_kernels().token_gate(out, z, table, ids, int(col0))
        return out
    return torch_ref.token_gate(z, table, ids, col0)


# --------------------------------------------------------------- delta rule
def causal_conv_silu(x, w, conv_state, slots, has_init, query_start_loc,
                     activation=True, max_query_len=0, bias=None):
    """Ragged short causal conv (+ ``bias`` [C]) + silu (``activation``
    False: the plain convolution); rolls ``conv_state`` rows ``slots`` in place. x may be
    a column slice of a merged projection. ``max_query_len`` == 1
    (decode-only batch): the state is rolled by the same launch."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq_kernels().causal_conv_silu(out, x, w, conv_state, slots,
                                        has_init, query_start_loc,
                                        bool(activation),
                                        int(max_query_len), bias)
        return out
    from gllm_amd.ops import gdn_ref
    return gdn_ref.causal_conv_silu(x, w, conv_state, slots, has_init,
                                    query_start_loc, activation, bias)


def delta_rule_varlen(q, k, v, a, b, A_log, dt_bias, state, slots,
                      has_init, query_start_loc, q_scale,
                      max_query_len=0) -> torch.Tensor:
    """Ragged gated delta rule (prompt portions and decode tokens in one
    launch); fp32 state [slots, H, Dk, Dv] in place; returns fp32
    [T, H, Dv]. ``max_query_len`` == 1 (decode-only batch) keeps the
    operands in registers; anything else stages token tiles through
    LDS — same arithmetic per token either way."""
    if q.is_cuda:
        H, _, Dv = state.shape[1:]
        o = torch.empty(q.shape[0], H, Dv, dtype=torch.float32,
                        device=q.device)
        _seq_kernels().delta_rule_varlen(o, q, k, v, a, b, A_log, dt_bias,
                                         state, slots, has_init,
                                         query_start_loc, q_scale,
                                         max_query_len)
        return o
    from gllm_amd.ops import gdn_ref
    return gdn_ref.delta_rule_varlen(q, k, v, a, b, A_log, dt_bias, state,
                                     slots, has_init, query_start_loc,
                                     q_scale)


def rms_gate(o, z, w, H, eps, dtype, gate="silu", scale=1.0,
             out=None) -> torch.Tensor:
    """Per head scale * o / rms(o) * w * act(z): fp32 [T, H, Dv] ->
    [T, H*Dv]. ``w`` [Dv] serves every head, [H*Dv] gives each head its
    own; ``gate`` "silu" or "sigmoid"; ``out`` may be a column block of
    a wider buffer."""
    assert gate in ("silu", "sigmoid")
    if o.is_cuda:
        if out is None:
            out = torch.empty(o.shape[0], o.shape[1] * o.shape[2],
                              dtype=dtype, device=o.device)
        _seq_kernels().rms_gate(out, o, z, w, H, eps, gate == "sigmoid",
                                float(scale))
        return out
    from gllm_amd.ops import gdn_ref
    return gdn_ref.rms_gate(o, z, w, H, eps, dtype, gate, scale, out)


def general_delta_rule(r, k, v, w_logit, a_logit, w0, decay_scale, state,
                       slots, has_init, query_start_loc,
                       max_query_len=0) -> torch.Tensor:
    """Ragged generalized delta rule with per-channel decay and removal
    (prompt portions and decode tokens in one launch). Per head, with
    w = exp(-decay_scale * sigmoid(w_logit + w0)), a = sigmoid(a_logit),
    u = k / sqrt(|k|^2 + 1e-6):
        S <- diag(w) S - (a u)(u^T S) + k v^T,   o = S^T r
    fp32 state [slots, H, D, Dv] in place; decay, removal rate and the
    unit key are formed in fp32 from the projections. Returns fp32
    [T, H, Dv]."""
    if r.is_cuda:
        H, _, Dv = state.shape[1:]
        o = torch.empty(r.shape[0], H, Dv, dtype=torch.float32,
                        device=r.device)
        _seq_kernels().general_delta_rule(
            o, r, k, v, w_logit, a_logit, w0, float(decay_scale), state,
            slots, has_init, query_start_loc, int(max_query_len))
        return o
    from gllm_amd.ops import gdn_ref
    return gdn_ref.general_delta_rule(r, k, v, w_logit, a_logit, w0,
                                      decay_scale, state, slots, has_init,
                                      query_start_loc)


def channel_delta_rule(q, k, v, a, b, A_log, dt_bias, state, slots,
                       has_init, query_start_loc, q_scale,
                       max_query_len=0) -> torch.Tensor:
    """Ragged gated delta rule with a decay per (value head, key
    channel), prompt portions and decode tokens in one launch. q, k
    [T, G*Dk] raw (unit norms, q_scale, decays and write strengths are
    formed in fp32 here), v [T, H*Dv], a [T, H*Dk] decay logits, b [T, H]
    write-strength logits. Per head, g = exp(-exp(A_log) softplus(a +
    dt_bias)), beta = sigmoid(b):
        S <- diag(g) S;  S <- S + k (beta (v - S^T k))^T;  o = S^T q
    fp32 state [slots, H, Dk, Dv] in place; returns fp32 [T, H, Dv].
    ``max_query_len`` == 1 (decode-only batch) with Dv a multiple of 64
    runs the one-token kernel; anything else stages token tiles in LDS."""
    if q.is_cuda:
        H, _, Dv = state.shape[1:]
        o = torch.empty(q.shape[0], H, Dv, dtype=torch.float32,
                        device=q.device)
        _seq_kernels().channel_delta_rule(
            o, q, k, v, a, b, A_log, dt_bias, state, slots, has_init,
            query_start_loc, float(q_scale), int(max_query_len))
        return o
    from gllm_amd.ops import gdn_ref
    return gdn_ref.channel_delta_rule(q, k, v, a, b, A_log, dt_bias, state,
                                      slots, has_init, query_start_loc,
                                      q_scale)


def token_shift(h, mu, state, slots, has_init, query_start_loc,
                max_query_len=0):
    """Ragged token shift h_t + (h_(t-1) - h_t) * mu: the row before a
    portion's first comes from ``state`` [slots, width] (zeros when the
    sequence starts here), which is left at the portion's last incoming
    row. ``mu`` [width] -> [T, width]; [mixes, width] -> [mixes, T,
    width], every mix from the same two rows."""
    if h.is_cuda:
        out = torch.empty(tuple(mu.shape[:-1]) + tuple(h.shape),
                          dtype=h.dtype, device=h.device)
        _seq_kernels().token_shift(out, h, mu, state, slots, has_init,
                                   query_start_loc, int(max_query_len))
        return out
    return torch_ref.token_shift(h, mu, state, slots, has_init,
                                 query_start_loc)


# --------------------------------------------------------------- scans
def wkv_scan(r, k, v, w_logit, w0, u, state, slots, has_init,
             query_start_loc, max_query_len=0) -> torch.Tensor:
    """Ragged outer-product recurrence with a decay per (head, key
    channel) and a bonus for the current token (prompt portions and
    decode tokens in one launch). Per head, w = exp(-exp(w_logit + w0)):
        o = (S + diag(u) k v^T)^T r;   S <- diag(w) S + k v^T
    r, k, w_logit [T, H*Dk], v [T, H*Dv], w0 and u fp32 [H*Dk]; fp32 state
    [slots, H, Dk, Dv] in place; returns fp32 [T, H, Dv]."""
    if r.is_cuda:
        H, _, Dv = state.shape[1:]
        o = torch.empty(r.shape[0], H, Dv, dtype=torch.float32,
                        device=r.device)
        _seq_kernels().wkv_scan(o, r, k, v, w_logit, w0, u, state, slots,
                                has_init, query_start_loc,
                                int(max_query_len))
        return o
    from gllm_amd.ops import gdn_ref
    return gdn_ref.wkv_scan(r, k, v, w_logit, w0, u, state, slots, has_init,
                            query_start_loc)


def state_space_scan(x, B, C, dt_logit, A_log, dt_bias, D, state, slots,
                     has_init, query_start_loc,
                     max_query_len=0) -> torch.Tensor:
    """Ragged state-space recurrence with a scalar decay per head. With
    dt = softplus(dt_logit + dt_bias):
        S <- exp(-exp(A_log) dt) S + dt B x^T;   y = S^T C + D x
    x [T, H*P], B and C [T, G*N] (head h reads group h // (H / G)),
    dt_logit [T, H], the per-head numbers fp32 [H]; fp32 state [slots, H,
    N, P] in place; returns fp32 [T, H, P]."""
    if x.is_cuda:
        H, _, P = state.shape[1:]
        y = torch.empty(x.shape[0], H, P, dtype=torch.float32,
                        device=x.device)
        _seq_kernels().state_space_scan(y, x, B, C, dt_logit, A_log,
                                        dt_bias, D, state, slots, has_init,
                                        query_start_loc, int(max_query_len))
        return y
    from gllm_amd.ops import gdn_ref
    return gdn_ref.state_space_scan(x, B, C, dt_logit, A_log, dt_bias, D,
                                    state, slots, has_init, query_start_loc)


def gate_rms(y, z, w, parts, eps, dtype, out=None) -> torch.Tensor:
    """(y * silu(z)) divided by its root mean square in ``parts`` equal
    parts of the row, times w: y fp32 [T, H, P], z [T, H*P], w [H*P] ->
    [T, H*P]; ``out`` may be a column block of a wider buffer."""
    if y.is_cuda:
        if out is None:
            out = torch.empty(z.shape, dtype=dtype, device=y.device)
        _seq_kernels().gate_rms(out, y, z, w, int(parts), float(eps))
        return out
    from gllm_amd.ops import gdn_ref
    return gdn_ref.gate_rms(y, z, w, parts, eps, dtype, out)
