"""hipGraph-captured decode buckets.

Parity: reference CUDA-graph capture (model_runner.py:1525-1615) with
the dummy-page padding trick (input_data.py:611-671), re-done on HIP:
torch.cuda.CUDAGraph IS hipGraph on ROCm. Pure-decode batches replay a
captured graph for the smallest bucket >= B; everything else runs eager.

Capture covers embed -> layers -> final norm (hidden out). Logits GEMM
and sampling stay eager (cheap, metadata-dependent). All graphs share
one memory pool; inputs live in persistent device buffers fed from
persistent pinned staging.

Nothing on the way from a scheduled batch to its sampled tokens waits for
the device, so the next step is staged while this one runs: the staging is
a ring of STAGES sets, each re-used only once its copies are done. All
per-row numbers and the used columns of the block table, packed, travel in
one copy; the columns are spread over the table's rows on the device. (A copy
of a strided block from the host goes through pageable memory, and from a few
hundred KB on it waits for the device.) The packing itself grows with the
page tables: 0.13 ms for 64 requests of 64 pages, 0.5 ms for 256.
"""

import contextlib
import gc
from typing import Dict, List, Optional

import numpy as np
import torch

from gllm_amd.logger import logger
from gllm_amd.runtime.forward_context import ForwardContext

STAGES = 4  # steps that may be staged ahead of the device
DECODE_BUCKETS = [1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512]


@contextlib.contextmanager
def _collector_held():
    """A graph that is destroyed while another one is captured ends the
    process, and the graphs of an engine that is no longer used go when the
    cyclic collector runs (its parts refer to each other): it waits."""
    enabled = gc.isenabled()
    gc.disable()
    try:
        yield
    finally:
        if enabled:
            gc.enable()


class GraphRunner:
    # what the captured forwards' decode attention counts in; the graphs are
    # replayed one behind the other
    arrived: Optional[torch.Tensor] = None

    def __init__(self, runner):
        self.runner = runner
        cfg = runner.config
        self.device = cfg.device
        self.buckets = [b for b in DECODE_BUCKETS if b <= cfg.max_graph_bs]
        self.graphs: Dict[int, torch.cuda.CUDAGraph] = {}
        self.hidden_out: Dict[int, torch.Tensor] = {}
        self.captured = False
        self.max_bs = self.buckets[-1]
        max_len = cfg.model_max_length or 32768
        self.pages_cap = -(-max_len // cfg.page_size)
        # the reserved scratch page (never allocated to a real seq)
        self.dummy_page = runner.num_kv_pages_total - 1

        B = self.max_bs
        dev = self.device
        self.uses_mrope = bool(getattr(runner, "uses_mrope", False))
        pshape = (3, B) if self.uses_mrope else (B,)
        # one device buffer behind every per-row input of the graphs
        n_pos = 3 * B if self.uses_mrope else B
        at = [0]

        def take(words):
            at[0] += words
            return at[0] - words
        o_ids, o_pos, o_slots = take(B), take(n_pos), take(B)
        o_ssm, o_lens = take(B), take(-(-B // 2))
        words = take(-(-B * self.pages_cap // 2))  # the packed table's place

        def views(flat):
            return (flat[o_ids:o_ids + B],
                    flat[o_pos:o_pos + n_pos].view(pshape),
                    flat[o_slots:o_slots + B], flat[o_ssm:o_ssm + B],
                    flat[o_lens:words].view(torch.int32)[:B],
                    flat[words:].view(torch.int32))
        self.table_at = words
        self.flat = torch.zeros(at[0], dtype=torch.long, device=dev)
        (self.in_ids, self.positions, self.slots, ssm, self.seq_lens,
         self.packed_table) = views(self.flat)
        self.seq_lens.fill_(1)
        self.block_table = torch.zeros((B, self.pages_cap),
                                       dtype=torch.int32, device=dev)
        self.qsl = torch.arange(B + 1, dtype=torch.int32, device=dev)
        # hybrid (GDN/SSM) models: device slots of the recurrent state;
        # all captured rows are initialized decode steps, padding rows
        # point at the pool's dummy scratch slot
        self.ssm_slots_dev = None
        if runner.ssm_pool is not None:
            self.ssm_slots_dev = ssm
            ssm.fill_(runner.ssm_pool.dummy_slot)
        # pinned staging sets: the tensor, its numpy views, and the event
        # behind the last copy out of it
        self.staging = []
        for _ in range(STAGES):
            flat = torch.zeros(at[0], dtype=torch.long).pin_memory()
            self.staging.append((flat, [v.numpy() for v in views(flat)],
                                 torch.cuda.Event()))
        self.next_stage = 0

    def _fctx_for(self, bs: int) -> ForwardContext:
        pos = self.positions[:, :bs] if self.uses_mrope \
            else self.positions[:bs]
        fctx = ForwardContext(
            num_tokens=bs,
            positions=pos,
            slot_mapping=self.slots[:bs],
            block_table=self.block_table[:bs],
            seq_lens=self.seq_lens[:bs],
            query_start_loc=self.qsl[:bs + 1],
            max_query_len=1, max_seq_len=1,
            k_caches=self.runner.k_caches,
            v_caches=self.runner.v_caches,
            arrived=self.arrived)
        if self.ssm_slots_dev is not None:
            fctx.ssm_pool = self.runner.ssm_pool
            fctx.ssm_slots_dev = self.ssm_slots_dev[:bs]
        return fctx

    @torch.no_grad()
    def capture_all(self):
        runner = self.runner
        # dummy metadata: every row points at the scratch page
        self.block_table.fill_(0)
        self.block_table[:, 0] = self.dummy_page
        self.seq_lens.fill_(1)
        base = self.dummy_page * runner.config.page_size
        ps = runner.config.page_size
        self.slots.copy_(base + torch.arange(self.max_bs) % ps)
        heads = max((c.shape[2] for c in runner.k_caches
                     if c is not None and c.dim() == 4), default=0)
        self.arrived = self.seq_lens.new_zeros(self.max_bs * heads)
        pool = torch.cuda.graphs.graph_pool_handle()
        stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        with _collector_held():
            self._capture_buckets(pool, stream)
        torch.cuda.synchronize()
        self.captured = True
        logger.info("hipGraph capture done: %d decode buckets (max bs %d)",
                    len(self.graphs), self.max_bs)

    def _capture_buckets(self, pool, stream):
        runner = self.runner
        # capture largest first so the shared pool is sized once
        for bs in reversed(self.buckets):
            fctx = self._fctx_for(bs)
            with torch.cuda.stream(stream):
                pos = self.positions[:, :bs] if self.uses_mrope \
                    else self.positions[:bs]
                for _ in range(2):  # warmup outside capture
                    ids = runner.resolve_tokens(self.in_ids[:bs])
                    runner.model(ids, pos, fctx)
            torch.cuda.current_stream().wait_stream(stream)
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, pool=pool, stream=stream):
                ids = runner.resolve_tokens(self.in_ids[:bs])
                hidden, _ = runner.model(ids, pos, fctx)
            self.graphs[bs] = g
            self.hidden_out[bs] = hidden

    # ------------------------------------------------------------------
    def can_replay(self, batch) -> bool:
        if not self.captured:
            return False
        items = batch.items
        if len(items) > self.max_bs:
            return False
        if not all(it.num_tokens == 1 and it.start >= it.seq.prompt_len
                   for it in items):
            return False
        if self.ssm_slots_dev is not None:
            # a pending recurrent-state restore (prefix hit on a fresh
            # slot) needs the eager path's host-side copy
            if not all(it.seq.ssm_slot >= 0 and it.seq.ssm_state_ready
                       for it in items):
                return False
        return True

    def _bucket(self, n: int) -> int:
        for b in self.buckets:
            if b >= n:
                return b
        raise AssertionError

    def _stage(self, items) -> int:
        """Send a step's inputs on their way to the captured buffers; the
        bucket that takes them."""
        B = len(items)
        bs = self._bucket(B)
        ps = self.runner.config.page_size
        flat, (ids, pos, slots, ssm, seq_lens, bt), done = \
            self.staging[self.next_stage]
        self.next_stage = (self.next_stage + 1) % STAGES
        done.synchronize()   # the copy of STAGES steps ago
        npg = max(1, max(len(it.seq.page_table) for it in items))
        bt = bt[:bs * npg].reshape(bs, npg)
        for i, it in enumerate(items):
            seq = it.seq
            ids[i] = seq.token_ids[it.start]
            if self.uses_mrope:
                # decode rows: all three sections advance together from
                # the prompt's mrope delta (batch_builder.py math)
                pos[:, i] = (seq.mrope_delta + (it.start - seq.prompt_len)
                             if seq.mrope_positions is not None
                             else it.start)
            else:
                pos[i] = it.start
            page_tab = seq.page_table
            bt[i, :len(page_tab)] = page_tab
            slots[i] = page_tab[it.start // ps] * ps + it.start % ps
            seq_lens[i] = it.start + 1
        dummy_base = self.dummy_page * ps
        for i in range(B, bs):
            ids[i] = 0
            if self.uses_mrope:
                pos[:, i] = 0
            else:
                pos[i] = 0
            bt[i, 0] = self.dummy_page
            slots[i] = dummy_base + i % ps
            seq_lens[i] = 1
        if self.ssm_slots_dev is not None:
            dummy = self.runner.ssm_pool.dummy_slot
            for i, it in enumerate(items):
                ssm[i] = it.seq.ssm_slot
            ssm[B:bs] = dummy
        # H2D into the captured buffers
        used = self.table_at + -(-bs * npg // 2)
        self.flat[:used].copy_(flat[:used], non_blocking=True)
        self.block_table[:bs, :npg].copy_(
            self.packed_table[:bs * npg].view(bs, npg))
        done.record()
        return bs

    @torch.no_grad()
    def replay(self, batch):
        items = batch.items
        bs = self._stage(items)
        self.graphs[bs].replay()
        hidden = self.hidden_out[bs][:len(items)]
        fctx = self._fctx_for(bs)
        fctx.logits_indices = None  # hidden already one row per seq
        return self.runner._sample(batch, hidden, fctx)
