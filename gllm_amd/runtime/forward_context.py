"""Per-forward batch metadata handed through the model to every layer.

Equivalent in role to the reference's InputData (gllm/input_data.py) GPU
tensors, but passed explicitly down ``model.forward`` instead of being
read from a global.
"""

import dataclasses
from typing import Dict, List, Optional

import torch


@dataclasses.dataclass
class ForwardContext:
    # --- ragged batch geometry ---
    num_tokens: int
    positions: torch.Tensor          # [T] int64
    slot_mapping: torch.Tensor       # [T] int64 (flat KV slot per new token)
    block_table: torch.Tensor        # [B, max_pages] int32
    seq_lens: torch.Tensor           # [B] int32 (total context incl. chunk)
    query_start_loc: torch.Tensor    # [B+1] int32
    max_query_len: int               # 1 => pure decode
    max_seq_len: int
    # sequences of this batch that bring one query row beside portions of
    # more (0: unknown or none)
    single_rows: int = dataclasses.field(default=0, kw_only=True)
    # --- KV cache (this stage's layers) ---
    k_caches: List[torch.Tensor]     # per local layer [pages, page, Hkv, D]
    v_caches: List[torch.Tensor]
    # --- sampling metadata (set on the last PP stage) ---
    # rows of the hidden states whose logits we need: query_start_loc[1:]-1
    logits_indices: Optional[torch.Tensor] = None
    # profile/warmup run: attention may be skipped (no KV yet)
    is_profile_run: bool = False
    # (rows, sequences) of the largest batch, in the profile run
    largest_batch: Optional[tuple] = dataclasses.field(default=None,
                                                       kw_only=True)
    # overlap mode: token ids contain negative ring placeholders
    has_placeholders: bool = False
    # hybrid GDN models: per-seq SSM state slots (core/ssm.py)
    ssm_pool: Optional[object] = None
    ssm_slots: Optional[List[int]] = None
    ssm_has_init: Optional[List[bool]] = None
    # graph-replay path: persistent device slot buffer (all rows are
    # initialized decode steps; padding rows point at the dummy slot)
    ssm_slots_dev: Optional[object] = None
    # device copies of ssm_slots (int64) / ssm_has_init (int32) for the
    # ragged state kernels (causal_conv_silu, delta_rule_varlen)
    ssm_slots_t: Optional[torch.Tensor] = None
    ssm_has_init_t: Optional[torch.Tensor] = None
    # multimodal: rows of this batch whose embeddings come from the
    # vision tower (replaced after embed_tokens on the first stage)
    mm_rows: Optional[torch.Tensor] = None     # [N] long
    mm_embeds: Optional[torch.Tensor] = None   # [N, hidden]
    # Qwen3-VL deepstack: [N, D*hidden] multiscale features added at the
    # image rows after decoder layers 0..D-1
    mm_deepstack: Optional[torch.Tensor] = None
    # DSA (DeepSeek-V3.2): per-layer paged index-K caches
    # [pages, page_size, index_head_dim] (models/deepseek_v32.py)
    idx_caches: Optional[List[torch.Tensor]] = None
    # host copies of the ragged geometry (filled by the batch builder
    # from its numpy staging for free) so per-seq torch paths — DSA
    # selection, GDN chunking, prompt logprobs — iterate without a
    # device sync per int() read
    seq_lens_cpu: Optional[List[int]] = None
    query_start_loc_cpu: Optional[List[int]] = None

    _prompts_from: Optional[int] = dataclasses.field(default=None,
                                                     kw_only=True)
    _per_head_from: Optional[tuple] = dataclasses.field(default=None,
                                                        kw_only=True)

    # zeros of the owner of a captured forward, who keeps them as long as the
    # graph (see arrivals)
    arrived: Optional[torch.Tensor] = dataclasses.field(default=None,
                                                        kw_only=True)
    _arrivals: Dict[int, torch.Tensor] = dataclasses.field(
        default_factory=dict, kw_only=True)

    def arrivals(self, kv_heads: int) -> torch.Tensor:
        """Zeros that split decode attention counts its workgroups in and
        leaves as zeros. The layers of a forward follow one another and share
        them; forwards on two streams do not, and a graph may outlive this
        context, so what a capture counts in is ``arrived`` or the graph's
        own."""
        n = self.seq_lens.shape[0] * kv_heads
        zeros = self.arrived
        if zeros is not None and zeros.numel() >= n:
            return zeros
        if torch.cuda.is_current_stream_capturing():
            return torch.zeros(n, dtype=torch.int32,
                               device=self.seq_lens.device)
        stream = torch.cuda.current_stream().cuda_stream
        zeros = self._arrivals.get(stream)
        if zeros is None or zeros.numel() < n:
            zeros = self._arrivals[stream] = torch.zeros(
                n, dtype=torch.int32, device=self.seq_lens.device)
        return zeros

    def prompts_from(self) -> int:
        """The first sequence from which on all are whole prompts: two rows
        or more and nothing in the cache (their number if there are none)."""
        if self._prompts_from is None:
            s = self.seq_lens.shape[0]
            if self.max_query_len > 1:
                qsl, lens = self.host_qsl(), self.host_seq_lens()
                while s > 0 and lens[s - 1] > 1 and \
                        lens[s - 1] == qsl[s] - qsl[s - 1]:
                    s -= 1
            self._prompts_from = s
        return self._prompts_from

    def per_head_from(self, heads: int) -> int:
        """The first sequence from which on latent attention of ``heads``
        heads takes the per-head form, which only whole prompts can (their
        number where the absorbed form of everything is the faster one; us
        of an attention layer of 16 heads, absorbed / the two forms):
        prompts of 8 rows and more on average (64 of 8 55 / 41, 300 of 2 72
        / 86); behind decode rows if one of those has 512 keys, for which the
        absorbed form of a mixed batch is one long chain (16 of 1000 keys and
        32 rows 114 / 80, of 200 keys 52 / 72), or if the mixed batch's tiles
        fill the chip (64 of 200 keys and 192 rows 152 / 86); behind portions
        of prompts, which stay absorbed, if there is much to save (256 rows
        after 2000 and 64 rows 250 / 281, 2048 rows 413 / 367)."""
        if self._per_head_from is None or self._per_head_from[0] != heads:
            self._per_head_from = (heads, self._choose_per_head(heads))
        return self._per_head_from[1]

    def _choose_per_head(self, heads: int) -> int:
        n, s = self.seq_lens.shape[0], self.prompts_from()
        if s == n:
            return n
        qsl, lens = self.host_qsl(), self.host_seq_lens()
        rows = qsl[n] - qsl[s]
        if rows < 8 * (n - s):
            return n
        if qsl[s] > s:
            return s if rows * heads >= 32768 else n
        if s > 0 and max(lens[:s]) < 512 \
                and n * max(lens[s:n]) * heads < 65536:
            return n
        return s

    @property
    def is_pure_decode(self) -> bool:
        return self.max_query_len == 1

    def host_qsl(self) -> List[int]:
        if self.query_start_loc_cpu is None:
            self.query_start_loc_cpu = self.query_start_loc.tolist()
        return self.query_start_loc_cpu

    def host_seq_lens(self) -> List[int]:
        if self.seq_lens_cpu is None:
            self.seq_lens_cpu = self.seq_lens.tolist()
        return self.seq_lens_cpu
