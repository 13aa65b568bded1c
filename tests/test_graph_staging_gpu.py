"""Captured decode steps staged ahead of the device."""

import json

import pytest
import torch

pytestmark = pytest.mark.gpu

CFG = {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2",
       "hidden_size": 512, "intermediate_size": 1024,
       "num_hidden_layers": 3, "num_attention_heads": 8,
       "num_key_value_heads": 2, "vocab_size": 4096,
       "max_position_embeddings": 2048, "rms_norm_eps": 1e-6,
       "rope_theta": 10000.0, "tie_word_embeddings": False,
       "eos_token_id": 0}


def _run(tmp_path, graph, steps):
    """Logits of ``steps`` decode steps of three requests, launched one
    after the other without waiting for the device in between."""
    from gllm_amd.config import EngineConfig
    from gllm_amd.engine.llm import LLM
    from gllm_amd.sequence import SamplingParams
    (tmp_path / "config.json").write_text(json.dumps(CFG))
    llm = LLM(config=EngineConfig(
        model=str(tmp_path), load_format="dummy", device="cuda:0",
        dtype="bfloat16", page_size=16, use_graph=graph, max_graph_bs=4,
        enable_prefix_caching=False, enable_overlap=False),
        num_pages_override=64)
    seen = []
    llm.runner.sampler.register_forward_pre_hook(
        lambda m, a: seen.append(a[0].clone()))
    sp = SamplingParams(temperature=0.0, ignore_eos=True, max_tokens=500)
    seqs = [llm.allocate_seq(list(range(2 + i, 30 + 17 * i)), sp)
            for i in range(3)]
    sched = llm.scheduler
    batch = sched.schedule_scripted([(s, s.prompt_len) for s in seqs])
    llm.runner.step_first_stage(batch)
    sched.commit_scripted(batch)
    torch.cuda.synchronize()
    del seen[:]
    for step in range(steps):
        live = seqs[:1 + step % 3]      # buckets change from step to step
        for i, s in enumerate(live):
            s.append_token(5 + 7 * step + i)
        batch = sched.schedule_scripted([(s, 1) for s in live])
        assert graph == (llm.runner.graph_runner is not None and
                         llm.runner.graph_runner.can_replay(batch))
        llm.runner.step_first_stage(batch)
        sched.commit_scripted(batch)
    torch.cuda.synchronize()
    return seen


def test_steps_staged_ahead_match_eager(tmp_path):
    steps = 24                           # more than the staging sets hold
    staged = _run(tmp_path, True, steps)
    eager = _run(tmp_path, False, steps)
    assert len(staged) == len(eager) == steps
    for a, b in zip(staged, eager):
        # a padded bucket has another split of its products: bf16 rounding
        # of the activations through three layers
        err = (a.float() - b.float()).norm() / b.float().norm()
        assert err < 0.02, err


@pytest.mark.parametrize("rows,pages", [(1, 2048), (3, 5), (500, 2047),
                                        (512, 2048)])
def test_staging_waits_for_its_own_copies_only(rows, pages):
    """With the device far behind, STAGES steps are staged at once and the
    next one only when the first one's copies are done; every step sees its
    own numbers."""
    from types import SimpleNamespace

    from gllm_amd.runtime.graph_runner import STAGES, GraphRunner
    runner = GraphRunner(SimpleNamespace(
        config=SimpleNamespace(device="cuda:0", max_graph_bs=512,
                               model_max_length=32768, page_size=16),
        num_kv_pages_total=5000, ssm_pool=None))
    steps = STAGES + 2
    torch.manual_seed(rows)

    def items(step):
        out = []
        for i in range(rows):
            n = pages if i == rows // 2 else 1 + (i + step) % 3
            table = torch.randint(0, 4999, (n,)).tolist()
            start = n * 16 - 1 - (i + step) % 16
            out.append(SimpleNamespace(start=start, seq=SimpleNamespace(
                token_ids={start: 7 * i + step}, page_table=table,
                mrope_positions=None)))
        return out
    work = [items(s) for s in range(steps)]
    seen = torch.zeros(steps, *runner.block_table.shape, dtype=torch.int32,
                       device="cuda")
    nums = torch.zeros(steps, runner.flat.numel(), dtype=torch.long,
                       device="cuda")

    def stage(s):
        bs = runner._stage(work[s])
        seen[s].copy_(runner.block_table)
        nums[s].copy_(runner.flat)
        return bs
    for s in range(steps):              # (what is set up once)
        bs = stage(s)
    torch.cuda.synchronize()
    seen.zero_()
    a = torch.ones(8192, 8192, device="cuda").bfloat16()
    behind = torch.cuda.Event()
    for _ in range(300):                # about 0.2 s
        torch.mm(a, a)
    behind.record()
    for s in range(steps):
        stage(s)
        assert behind.query() == (s >= STAGES), s
    torch.cuda.synchronize()
    B = runner.max_bs
    for s in range(steps):
        ids, pos, slots = nums[s, :3 * B].view(3, B).cpu()
        lens = nums[s, 4 * B:].view(torch.int32)[:B].cpu()
        for i, it in enumerate(work[s]):
            t = it.seq.page_table
            assert int(ids[i]) == 7 * i + s and int(pos[i]) == it.start
            assert int(lens[i]) == it.start + 1
            assert int(slots[i]) == t[it.start // 16] * 16 + it.start % 16
        got = seen[s].cpu()
        for i, it in enumerate(work[s]):
            t = it.seq.page_table
            assert got[i, :len(t)].tolist() == t
        for i in range(rows, bs):       # padding: the scratch page
            assert int(got[i, 0]) == 4999 and int(lens[i]) == 1


@pytest.mark.parametrize("n", [1, 255, 257])
def test_resolve_tokens(n):
    from gllm_amd import ops
    ring = torch.randint(0, 1000, (4, 100), device="cuda")
    tokens = torch.randint(-400, 1000, (n,), device="cuda")
    want = torch.where(tokens < 0, ring.view(-1)[(-tokens - 1).clamp_min(0)],
                       tokens)
    assert torch.equal(ops.resolve_tokens(tokens, ring), want)
