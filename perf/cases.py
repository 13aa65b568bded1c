"""Serving steps whose time and results are measured.

A case is one engine step of a decoder that this package serves: a batch
of running requests that decode one token each, a batch of prompts, or
both in one batch. It goes through the engine's own path: the scheduler's
batch record -> ``ModelRunner.step_first_stage`` (captured decode
buckets, or the eager forward when the batch holds prompt portions) ->
logits -> sampler. The decoders are the ones of the benchmark, cut to a
stack of 2 to 8 of their 24 to 64 equal layers (about what one stage of a
pipeline holds), with the vocabulary cut in the same proportion so that
the head keeps its share of a step.

Requests are greedy. Weights, prompts and the keys / values (or
recurrent state) that earlier steps would have left are random and
depend on the seed alone.
"""

import gc
import json
import math
import os
import tempfile
import zlib

import torch

PAGE = 16

# Sizes of the benchmark's models. "of" is the full depth: the vocabulary
# is scaled by layers / of.
GEOMETRY = {
    # Qwen2.5-32B
    "dense-32b": dict(
        arch="Qwen2ForCausalLM", kind="qwen2", width=5120, ff=27648,
        heads=40, kv=8, dim=128, bias=True, theta=1e4, eps=1e-6,
        vocab=152064, layers=8, of=64),
    # Llama-3-8B
    "dense-8b": dict(
        arch="LlamaForCausalLM", kind="llama", width=4096, ff=14336,
        heads=32, kv=8, dim=128, bias=False, theta=1e4, eps=1e-5,
        vocab=128256, layers=8, of=32),
    # Mixtral-8x7B
    "moe-8x7b": dict(
        arch="MixtralForCausalLM", kind="mixtral", width=4096, ff=14336,
        heads=32, kv=8, dim=128, bias=False, theta=1e4, eps=1e-5,
        vocab=32000, layers=4, of=32, experts=8, top=2, renorm=True),
    # DeepSeek-V2-Lite: latent attention, 64 experts and two shared ones
    "mla-lite": dict(
        arch="DeepseekV2ForCausalLM", kind="deepseek_v2", width=2048,
        ff=10944, heads=16, lora=512, nope=128, rope=64, vdim=128,
        theta=1e4, eps=1e-6, vocab=102400, layers=6, of=27, experts=64,
        top=6, expert_ff=1408, shared=2, first_dense=1, renorm=False),
    # Qwen3-Next-9B hybrid: three gated-delta layers to one of attention
    "hybrid-9b": dict(
        arch="Qwen3NextForCausalLM", kind="qwen3_next", width=2048,
        ff=5504, heads=16, kv=2, dim=128, rot=32, theta=1e4, eps=1e-6,
        vocab=151936, layers=8, of=24, lin_v=16, lin_k=8, lin_dim=128,
        taps=4, every=4),
}


def listed():
    return [
        # One user in an interactive session: latency of a single token.
        dict(name="8b decode 1", model="dense-8b", quant="none",
             decode=1, context=600, prompts=0, tokens=0),
        # The flagship serving batch of the benchmark's README table.
        dict(name="32b decode 64", model="dense-32b", quant="none",
             decode=64, context=1024, prompts=0, tokens=0),
        # The default benchmark's batch: saturated offline throughput.
        dict(name="32b decode 256", model="dense-32b", quant="none",
             decode=256, context=1024, prompts=0, tokens=0),
        # A throttled scheduler tick while requests arrive: portions of
        # prompts beside the requests that already decode.
        dict(name="32b mixed", model="dense-32b", quant="none",
             decode=37, context=1024, prompts=5, tokens=4096),
        # A long document for a few users: attention over long caches.
        dict(name="8b decode 24 long", model="dense-8b", quant="none",
             decode=24, context=5400, prompts=0, tokens=0),
        # Block-quantized fp8 checkpoint, decode.
        dict(name="32b fp8 decode 64", model="dense-32b", quant="fp8",
             decode=64, context=1024, prompts=0, tokens=0),
        # int4 (GPTQ) checkpoint, decode, a batch between two buckets.
        dict(name="32b int4 decode 29", model="dense-32b", quant="int4",
             decode=29, context=1024, prompts=0, tokens=0),
        # Few large experts, decode.
        dict(name="moe decode 64", model="moe-8x7b", quant="none",
             decode=64, context=1024, prompts=0, tokens=0),
        # Few large experts, prompts of unequal lengths.
        dict(name="moe prefill", model="moe-8x7b", quant="none",
             decode=0, context=0, prompts=7, tokens=5000),
        # Latent attention and many small experts, decode.
        dict(name="mla decode 128", model="mla-lite", quant="none",
             decode=128, context=1024, prompts=0, tokens=0),
        # Latent attention and many small experts, prompts.
        dict(name="mla prefill", model="mla-lite", quant="none",
             decode=0, context=0, prompts=4, tokens=4096),
        # Recurrent layers: new prompts beside nothing else.
        dict(name="hybrid prefill", model="hybrid-9b", quant="none",
             decode=0, context=0, prompts=4, tokens=4096),
    ]


def draw(rng):
    model, quant = rng.choice([
        ("dense-8b", "none"), ("dense-32b", "none"), ("dense-32b", "fp8"),
        ("dense-32b", "int4"), ("moe-8x7b", "none"), ("mla-lite", "none"),
        ("hybrid-9b", "none")])

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    # quantized checkpoints and the hybrid stack are drawn for the
    # directions that the listed cases hold for them, plus hybrid decode
    phase = "decode" if quant != "none" else rng.choice(
        ["decode", "decode", "prefill"] +
        (["mixed"] if model.startswith("dense") else []))
    case = dict(model=model, quant=quant, decode=0, context=0, prompts=0,
                tokens=0)
    if phase != "prefill":
        case["decode"] = spread(1, 32 if phase == "mixed" else
                                64 if quant != "none" else 256)
        case["context"] = spread(64, min(5400, 262144 // case["decode"]))
    if phase != "decode":
        case["tokens"] = spread(48, 4096)
        case["prompts"] = rng.randint(1, min(8, case["tokens"] // 8))
    return case


# ------------------------------------------------------------ the inputs
def _geometry(case):
    g = dict(GEOMETRY[case["model"]])
    if case["quant"] == "fp8":
        # activations are rounded to fp8 in front of every product: two
        # layers keep what two correct implementations may differ by
        # (that rounding, met anew in every layer) within a few percent
        g["layers"] = 2
    g["vocab"] = -(-g["vocab"] * g["layers"] // g["of"] // 64) * 64
    return g


def _lengths(n, mean):
    """``n`` unequal lengths between half and one and a half times
    ``mean``, the same for every seed."""
    return [max(1, int(mean * (0.5 + (0.5 + 0.618034 * i) % 1.0)))
            for i in range(n)]


def _portions(case):
    """Prompt lengths that add up to ``tokens``."""
    n, total = case["prompts"], case["tokens"]
    if not n:
        return []
    cut = _lengths(n, total / n)
    cut = [max(1, c * total // sum(cut)) for c in cut]
    cut[-1] += total - sum(cut)
    return cut


def _rand(seed, name, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    gen = torch.Generator(device="cuda")
    gen.manual_seed((seed * 1000003 + zlib.crc32(name.encode()))
                    % (1 << 62))
    t = torch.empty(shape, dtype=dtype, device="cuda")
    return t.normal_(mean, std, generator=gen)


def _prefers(seed, g, layer):
    """Router input of each token id in one layer, [vocab, experts]: a
    trained router follows the token, so every id has ``top`` experts of
    its own (some experts more popular than others) well above the rest."""
    E, k = g["experts"], g["top"]
    pop = _rand(seed, "popular.%d" % layer, (E,), 0.5, dtype=torch.float32)
    taste = _rand(seed, "taste.%d" % layer, (g["vocab"], E),
                  dtype=torch.float32)
    ids = (taste + pop).topk(k, dim=1).indices
    base = taste.mul(0.3).clamp(-1.0, 1.0)
    first = torch.linspace(4.0, 3.5, k, device="cuda").expand(ids.shape)
    return base.scatter(1, ids, first).to(torch.bfloat16)


class _Weights:
    """Checkpoint tensors by their checkpoint names, each made on demand
    from the seed. ``dense`` gives a projection's values as the stored
    format holds them, in 64 bits."""

    def __init__(self, case, seed):
        self.g, self.seed, self.quant = _geometry(case), seed, case["quant"]
        g = self.g
        self.routed = [i for i in range(g["layers"])
                       if "experts" in g and i >= g.get("first_dense", 0)]
        # coordinates of the stream that carry the token's preferences;
        # the sublayers do not write there
        self.quiet = len(self.routed) * g.get("experts", 0)

    def rand(self, name, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return _rand(self.seed, name, shape, std, mean, dtype)

    # -- unquantized tensors
    def norm(self, name, n):
        return self.rand(name, (n,), 0.1, 1.0)

    def matrix(self, name, out, inp, gain=1.0, writes=False):
        w = self.rand(name, (out, inp), gain * inp ** -0.5)
        if writes and self.quiet:
            w[:self.quiet] = 0
        return w

    def embedding(self):
        g = self.g
        e = self.rand("embed", (g["vocab"], g["width"]))
        for n, layer in enumerate(self.routed):
            e[:, n * g["experts"]:(n + 1) * g["experts"]] = _prefers(
                self.seed, g, layer)
        return e

    def router(self, layer):
        g = self.g
        n = self.routed.index(layer)
        w = self.rand("router.%d" % layer, (g["experts"], g["width"]),
                      0.1 * g["width"] ** -0.5)
        at = torch.arange(g["experts"], device="cuda")
        w[at, n * g["experts"] + at] = 1.0
        return w

    # -- quantized projections
    def fp8(self, name, out, inp, gain):
        w = self.rand(name, (out, inp), 100.0).clamp(-440, 440)
        s = self.rand(name + ".s", (-(-out // 128), -(-inp // 128)), 0.1,
                      1.0, torch.float32).clamp(0.5, 1.5)
        return (w.to(torch.float8_e4m3fn),
                s * (gain * inp ** -0.5 / 100.0))

    def int4(self, name, out, inp, gain):
        """GPTQ tensors: q [in/8, out], stored zeros [in/128, out/8] and
        scales [in/128, out]."""
        def pack(v, dim):
            n = v.shape[dim] // 8
            v = v.view((n, 8, -1) if dim == 0 else (-1, n, 8)).to(torch.int64)
            p = sum(v.select(1 if dim == 0 else 2, i) << (4 * i)
                    for i in range(8))
            return torch.where(p >= 1 << 31, p - (1 << 32), p).to(torch.int32)
        q = self.rand(name, (inp, out), 2.7, 8.0).round().clamp(0, 15)
        z = self.rand(name + ".z", (inp // 128, out), 0.8, 8.0).round() \
            .clamp(1, 15)
        s = self.rand(name + ".s", (inp // 128, out), 0.1, 1.0,
                      torch.float32).clamp(0.5, 1.5)
        s = (s * (gain * inp ** -0.5 / 2.7)).to(torch.float16)
        return q, z, s, pack(q, 0), pack(z - 1, 1)

    def projection(self, name, out, inp, gain=1.0, writes=False):
        """(checkpoint name, tensor) pairs of one linear layer."""
        if self.quant == "fp8":
            w, s = self.fp8(name, out, inp, gain)
            return [(name + ".weight", w), (name + ".weight_scale_inv", s)]
        if self.quant == "int4":
            _, _, s, qw, qz = self.int4(name, out, inp, gain)
            return [(name + ".qweight", qw), (name + ".qzeros", qz),
                    (name + ".scales", s)]
        return [(name + ".weight", self.matrix(name, out, inp, gain,
                                               writes))]

    def dense(self, name, out, inp, gain=1.0, writes=False):
        if self.quant == "fp8":
            w, s = self.fp8(name, out, inp, gain)
            s = s.double().repeat_interleave(128, 0)[:out] \
                .repeat_interleave(128, 1)[:, :inp]
            return w.double() * s
        if self.quant == "int4":
            q, z, s, _, _ = self.int4(name, out, inp, gain)
            at = torch.arange(inp, device="cuda") // 128
            return ((q.double() - z.double()[at]) * s.double()[at]).t()
        return self.matrix(name, out, inp, gain, writes).double()

    # -- shapes of a layer's projections: (name, out, in, gain, writes)
    def attention(self, i):
        g, p = self.g, "layers.%d.self_attn." % i
        D, q = g["dim"], 1.0 if "rot" in g else 2.0
        return [(p + "q_proj", g["heads"] * D, g["width"], q, False),
                (p + "k_proj", g["kv"] * D, g["width"], 1.0, False),
                (p + "v_proj", g["kv"] * D, g["width"], 1.0, False),
                (p + "o_proj", g["width"], g["heads"] * D, 1.0, True)]

    def latent(self, i):
        g, p = self.g, "layers.%d.self_attn." % i
        H, W = g["heads"], g["width"]
        return [(p + "q_proj", H * (g["nope"] + g["rope"]), W, 2.0, False),
                (p + "kv_a_proj_with_mqa", g["lora"] + g["rope"], W, 1.0,
                 False),
                (p + "kv_b_proj", H * (g["nope"] + g["vdim"]), g["lora"],
                 1.0, False),
                (p + "o_proj", W, H * g["vdim"], 1.0, True)]

    def linear_attention(self, i):
        g, p = self.g, "layers.%d.linear_attn." % i
        qk, v = g["lin_k"] * g["lin_dim"], g["lin_v"] * g["lin_dim"]
        return [(p + "in_proj_qkvz", 2 * qk + 2 * v, g["width"], 1.0, False),
                (p + "in_proj_ba", 2 * g["lin_v"], g["width"], 0.5, False),
                (p + "out_proj", g["width"], v, 1.0, False)]

    def mlp(self, prefix, ff):
        W = self.g["width"]
        return [(prefix + "gate_proj", ff, W, 1.0, False),
                (prefix + "up_proj", ff, W, 1.0, False),
                (prefix + "down_proj", W, ff, 1.0, True)]

    def experts(self, i):
        """Stacked expert matrices gate, up [E, ff, W] and down [E, W, ff]."""
        g = self.g
        E, W, F = g["experts"], g["width"], g.get("expert_ff", g["ff"])
        gate = self.rand("experts.%d.g" % i, (E, F, W), W ** -0.5)
        up = self.rand("experts.%d.u" % i, (E, F, W), W ** -0.5)
        down = self.rand("experts.%d.d" % i, (E, W, F), F ** -0.5)
        down[:, :self.quiet] = 0
        return gate, up, down

    def vectors(self, i):
        """The small tensors of a gated-delta layer."""
        g, p = self.g, "layers.%d.linear_attn." % i
        H = g["lin_v"]
        ch = 2 * g["lin_k"] * g["lin_dim"] + H * g["lin_dim"]
        rate = self.rand(p + "A", (H,), dtype=torch.float32)
        return {p + "conv1d.weight": self.rand(p + "conv", (ch, 1,
                                                            g["taps"]), 0.5),
                p + "A_log": rate.clamp(-2, 2) - 2.0,
                p + "dt_bias": self.rand(p + "dt", (H,), 0.5, -1.0,
                                         torch.float32),
                p + "norm.weight": self.norm(p + "norm", g["lin_dim"])}

    def is_linear(self, i):
        return "every" in self.g and (i + 1) % self.g["every"] != 0

    def layer_norms(self, i):
        p = "layers.%d." % i
        return {p + n: self.norm(p + n, self.g["width"]) for n in (
            "input_layernorm.weight", "post_attention_layernorm.weight")}

    def head_norms(self, i):
        p = "layers.%d.self_attn." % i
        return {p + n: self.norm(p + n, self.g["dim"])
                for n in ("q_norm.weight", "k_norm.weight")}

    # -- the checkpoint
    def checkpoint(self):
        g = self.g
        gemma = "every" in g       # this family stores norm weights - 1
        off = 1.0 if gemma else 0.0
        yield "model.embed_tokens.weight", self.embedding()
        for i in range(g["layers"]):
            m, p = "model.", "layers.%d." % i
            for n, w in self.layer_norms(i).items():
                yield m + n, w - off
            if self.is_linear(i):
                for s in self.linear_attention(i):
                    yield from ((m + n, w) for n, w in self.projection(*s))
                for n, w in self.vectors(i).items():
                    yield m + n, w
            elif "lora" in g:
                for s in self.latent(i):
                    yield from ((m + n, w) for n, w in self.projection(*s))
                n = p + "self_attn.kv_a_layernorm.weight"
                yield m + n, self.norm(n, g["lora"])
            else:
                for s in self.attention(i):
                    yield from ((m + n, w) for n, w in self.projection(*s))
                if g.get("bias"):
                    for s in self.attention(i)[:3]:
                        yield (m + s[0] + ".bias",
                               self.rand(s[0] + ".bias", (s[1],), 0.1))
                if gemma:
                    for n, w in self.head_norms(i).items():
                        yield m + n, w - off
            if i in self.routed:
                mixtral = "shared" not in g
                q = m + p + ("block_sparse_moe." if mixtral else "mlp.")
                yield q + "gate.weight", self.router(i)
                names = ("w1", "w3", "w2") if mixtral else (
                    "gate_proj", "up_proj", "down_proj")
                for n, t in zip(names, self.experts(i)):
                    for e in range(g["experts"]):
                        yield "%sexperts.%d.%s.weight" % (q, e, n), t[e]
                if not mixtral:
                    for s in self.mlp(p + "mlp.shared_experts.",
                                      g["shared"] * g["expert_ff"]):
                        yield from ((m + n, w)
                                    for n, w in self.projection(*s))
            else:
                for s in self.mlp(p + "mlp.", g["ff"]):
                    yield from ((m + n, w) for n, w in self.projection(*s))
        yield "model.norm.weight", self.norm("norm", g["width"]) - off
        yield "lm_head.weight", self.matrix("lm_head", g["vocab"],
                                            g["width"])


def _requests(case, seed, vocab):
    """Token ids of the decoding requests' contexts (the last id is the
    one they feed now) and of the prompts."""
    gen = torch.Generator().manual_seed(seed)

    def ids(n):
        return torch.randint(1, vocab - 1, (n,), generator=gen).tolist()
    return ([ids(n + 1) for n in _lengths(case["decode"], case["context"])],
            [ids(n) for n in _portions(case)])


def _cached(seed, layer, request, n, heads, dim, what):
    """Keys or values that earlier steps of one request left, [n, heads,
    dim] (rotated keys and projected values are close to normal)."""
    return _rand(seed, "cache.%s.%d.%d" % (what, layer, request),
                 (n, heads, dim))


def _carried(seed, g, layer, rows):
    """Recurrent state and convolution inputs of the decoding requests."""
    H, D = g["lin_v"], g["lin_dim"]
    ch = (2 * g["lin_k"] + H) * D
    return (_rand(seed, "state.%d" % layer, (rows, H, D, D), 0.1,
                  dtype=torch.float32),
            _rand(seed, "conv.%d" % layer, (rows, ch, g["taps"] - 1)))


def _config(g, quant):
    c = {"architectures": [g["arch"]], "model_type": g["kind"],
         "hidden_size": g["width"], "intermediate_size": g["ff"],
         "num_hidden_layers": g["layers"],
         "num_attention_heads": g["heads"],
         "num_key_value_heads": g.get("kv", g["heads"]),
         "vocab_size": g["vocab"], "max_position_embeddings": 32768,
         "rms_norm_eps": g["eps"], "rope_theta": g["theta"],
         "tie_word_embeddings": False, "eos_token_id": 0}
    if "lora" in g:
        c.update(moe_intermediate_size=g["expert_ff"],
                 first_k_dense_replace=g["first_dense"],
                 n_routed_experts=g["experts"], n_shared_experts=g["shared"],
                 num_experts_per_tok=g["top"], n_group=1, topk_group=1,
                 routed_scaling_factor=1.0, scoring_func="softmax",
                 norm_topk_prob=g["renorm"], q_lora_rank=None,
                 kv_lora_rank=g["lora"], qk_nope_head_dim=g["nope"],
                 qk_rope_head_dim=g["rope"], v_head_dim=g["vdim"])
    elif "experts" in g:
        c.update(num_local_experts=g["experts"],
                 num_experts_per_tok=g["top"])
    if "every" in g:
        c.update(head_dim=g["dim"], linear_num_value_heads=g["lin_v"],
                 linear_num_key_heads=g["lin_k"],
                 linear_key_head_dim=g["lin_dim"],
                 linear_value_head_dim=g["lin_dim"],
                 linear_conv_kernel_dim=g["taps"],
                 full_attention_interval=g["every"], num_experts=0,
                 partial_rotary_factor=g["rot"] / g["dim"])
    if quant == "fp8":
        c["quantization_config"] = {"quant_method": "fp8",
                                    "weight_block_size": [128, 128]}
    elif quant == "int4":
        c["quantization_config"] = {"quant_method": "gptq", "bits": 4,
                                    "group_size": 128}
    return c


class _KeepLogits:
    """Pre-hook of the engine's sampler: the logits it was given."""
    logits = None

    def __call__(self, module, args):
        self.logits = args[0]


def prepare(case, seed):
    """A serving engine with its weights loaded and its decode buckets
    captured, and a scheduled batch of requests."""
    from gllm_amd.config import EngineConfig
    from gllm_amd.engine.llm import LLM
    from gllm_amd.runtime.graph_runner import DECODE_BUCKETS, GraphRunner
    from gllm_amd.sequence import SamplingParams
    weights = _Weights(case, seed)
    g = weights.g
    running, prompts = _requests(case, seed, g["vocab"])
    rows = len(running) + len(prompts)
    pages = sum(-(-len(t) // PAGE) for t in running + prompts) + 2
    bucket = min([b for b in DECODE_BUCKETS if b >= case["decode"]])
    with tempfile.TemporaryDirectory(prefix="perf_model_") as d:
        with open(os.path.join(d, "config.json"), "w") as f:
            json.dump(_config(g, case["quant"]), f)
        config = EngineConfig(
            model=d, load_format="dummy", dtype="bfloat16",
            device="cuda:0", page_size=PAGE, maxp=8192, maxd=512,
            use_graph=False, enable_overlap=False,
            enable_prefix_caching=False, max_state_slots=rows,
            max_graph_bs=bucket)
        # every parameter of the model in the serving type, norms included
        torch.set_default_dtype(torch.bfloat16)
        try:
            llm = LLM(config=config, num_pages_override=pages)
        finally:
            torch.set_default_dtype(torch.float32)
    llm.scheduler.log = False
    runner, sched = llm.runner, llm.scheduler
    runner.model.load_weights(weights.checkpoint())
    if not case["prompts"]:
        # a graph must not be destroyed while another one is captured:
        # engines that are no longer used go first
        gc.collect()
        runner.graph_runner = GraphRunner(runner)
        runner.graph_runner.capture_all()
    greedy = SamplingParams(temperature=0.0, ignore_eos=True,
                            max_tokens=4096)

    # the requests that decode: their contexts are in the caches
    chunks = []
    seqs = [llm.allocate_seq(t[:-1], greedy) for t in running]
    if seqs:
        sched.commit_scripted(sched.schedule_scripted(
            [(s, s.prompt_len) for s in seqs]))
        for i, (s, t) in enumerate(zip(seqs, running)):
            s.append_token(t[-1])
            table = torch.tensor(s.page_table, device="cuda")
            at = torch.arange(s.prompt_len, device="cuda")
            at = table[at // PAGE] * PAGE + at % PAGE
            for layer, (k, v) in enumerate(zip(runner.k_caches,
                                               runner.v_caches)):
                for what, c in (("k", k), ("v", v)):
                    if what == "v" and "lora" in g:
                        continue        # the values are part of the keys
                    c.view(-1, *c.shape[2:])[at] = _cached(
                        seed, layer, i, s.prompt_len, c.shape[2],
                        c.shape[3], what)
        chunks += [(s, 1) for s in seqs]
    if runner.ssm_pool is not None and seqs:
        pool = runner.ssm_pool
        slots = [pool.ensure(s) for s in seqs]
        for s in seqs:
            s.ssm_state_ready = True
        for layer in range(pool.spec.num_ssm_layers):
            state, conv = _carried(seed, g, layer, len(seqs))
            pool.ssm_state[layer][slots] = state
            pool.conv_state[layer][slots] = conv
    chunks += [(s, s.prompt_len)
               for s in (llm.allocate_seq(t, greedy) for t in prompts)]
    keep = _KeepLogits()
    runner.sampler.register_forward_pre_hook(keep)
    return {"llm": llm, "batch": sched.schedule_scripted(chunks),
            "keep": keep, "rows": rows}


def run(state):
    """One engine step. Logits of each request's next token, the last
    layer's keys and values (one page is the engine's scratch page) and
    the recurrent state."""
    runner = state["llm"].runner
    runner.step_first_stage(state["batch"])
    out = {"logits": state["keep"].logits,
           "keys": runner.k_caches[-1][:-1],
           "values": runner.v_caches[-1][:-1]}
    if runner.ssm_pool is not None:
        out["state"] = runner.ssm_pool.ssm_state[:, :state["rows"]]
    return out


# ----------------------------------------------------------- what it costs
def work(case):
    g = _geometry(case)
    W, V, L = g["width"], g["vocab"], g["layers"]
    wb = {"none": 2.0, "fp8": 1.0 + 4 / 16384, "int4": 0.5 + 2.5 / 128}[
        case["quant"]]
    weights = _Weights.__new__(_Weights)
    weights.g, weights.quant = g, case["quant"]
    weights.routed = [i for i in range(L)
                      if "experts" in g and i >= g.get("first_dense", 0)]
    contexts = _lengths(case["decode"], case["context"])
    portions = _portions(case)
    T, rows = len(contexts) + sum(portions), len(contexts) + len(portions)
    pairs = sum(n + 1 for n in contexts) + sum(n * (n + 1) // 2
                                               for n in portions)
    held = sum(contexts)
    bytes_ = T * W * 2 + V * W * 2 + rows * V * 2
    flops = 2.0 * rows * V * W
    for i in range(L):
        if weights.is_linear(i):
            shapes = weights.linear_attention(i)
            D = g["lin_dim"]
            state = g["lin_v"] * D * D * 4
            bytes_ += state * (2 * len(contexts) + len(portions))
            flops += 6.0 * T * g["lin_v"] * D * D
        elif "lora" in g:
            shapes = weights.latent(i)
            row = g["lora"] + g["rope"]
            bytes_ += 2 * row * (held + T)
            # prompts: per-head keys and values; decoding: the latent
            own = sum(n * (n + 1) // 2 for n in portions)
            flops += 2.0 * own * g["heads"] * (g["nope"] + g["rope"] +
                                               g["vdim"])
            flops += 2.0 * (pairs - own) * g["heads"] * (row + g["lora"])
        else:
            shapes = weights.attention(i)
            bytes_ += 4 * g["kv"] * g["dim"] * (held + T)
            flops += 4.0 * pairs * g["heads"] * g["dim"]
        if i in weights.routed:
            E, k = g["experts"], g["top"]
            one = 3 * W * g.get("expert_ff", g["ff"])
            bytes_ += 2 * one * E * (1 - (1 - k / E) ** T) + 2 * E * W
            flops += 2.0 * T * (k * one + E * W)
            if "shared" in g:
                shapes = shapes + weights.mlp("", g["shared"] *
                                              g["expert_ff"])
        else:
            shapes = shapes + weights.mlp("", g["ff"])
        bytes_ += wb * sum(s[1] * s[2] for s in shapes)
        flops += 2.0 * T * sum(s[1] * s[2] for s in shapes)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # bf16 activations through the stack: against exact() the logits are
    # off by 0.008 (4 expert layers), 0.013 (8 dense layers) and 0.035
    # (fp8 activations); the 8-layer stack with its products summed in
    # another order differs from itself by 0.016 to 0.02, at most 0.12 of
    # the result's size at any one value
    return {"rel": 0.03, "max": 0.5}


# --------------------------------------------------- the step in 64 bits
def _rms(x, w, eps):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * w.double()


def _rope(x, pos, dims, theta):
    """Rotate-half on the first ``dims`` of [T, heads, D]."""
    f = theta ** (-torch.arange(0, dims, 2, device="cuda",
                                dtype=torch.float64) / dims)
    a = (pos.double()[:, None] * f)[:, None]
    h = dims // 2
    x1, x2 = x[..., :h], x[..., h:dims]
    return torch.cat([x1 * a.cos() - x2 * a.sin(),
                      x2 * a.cos() + x1 * a.sin(), x[..., dims:]], -1)


def _attend(q, k, v, scale):
    """Causal attention of the last len(q) positions: q [n, H, D], k
    [m, G, D], v [m, G, E]."""
    n, H, m, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    mask = torch.arange(m, device="cuda")[None] > \
        torch.arange(m - n, m, device="cuda")[:, None]
    out = torch.empty(n, H, v.shape[2], dtype=torch.float64, device="cuda")
    r = H // G
    for j in range(G):
        s = torch.matmul(q[:, j * r:(j + 1) * r].transpose(0, 1),
                         k[:, j].t().contiguous()) * scale
        s = s.masked_fill(mask, -math.inf).softmax(-1)
        out[:, j * r:(j + 1) * r] = torch.matmul(s, v[:, j].contiguous()) \
            .transpose(0, 1)
    return out


def _swiglu(w, specs, x):
    g, u, d = (w.dense(*s) for s in specs)
    return (torch.nn.functional.silu(x @ g.t()) * (x @ u.t())) @ d.t()


def _delta(w, i, n_lin, x, spans, seed, new_state):
    """One gated-delta layer over every request's span of rows."""
    g, p = w.g, "layers.%d.linear_attn." % i
    D, Hk, H = g["lin_dim"], g["lin_k"], g["lin_v"]
    qk, taps = Hk * D, g["taps"]
    qkvz, ba, out = (w.dense(*s) for s in w.linear_attention(i))
    v = {n[len(p):]: t.double() for n, t in w.vectors(i).items()}
    y, ba = x @ qkvz.t(), x @ ba.t()
    z = y[:, 2 * qk + H * D:].view(-1, H, D)
    beta = ba[:, :H].sigmoid()
    decay = (-v["A_log"].exp() * torch.nn.functional.softplus(
        ba[:, H:] + v["dt_bias"])).exp()
    mixed, B = y[:, :2 * qk + H * D], len(spans)
    live = [s for s in spans if s[2]]
    S = torch.zeros(B, H, D, D, dtype=torch.float64, device="cuda")
    past = torch.zeros(B, mixed.shape[1], taps - 1, dtype=torch.float64,
                       device="cuda")
    if live:
        s0, c0 = _carried(seed, g, n_lin, len(live))
        S[:len(live)], past[:len(live)] = s0.double(), c0.double()
    longest = max(b - a for a, b, _ in spans)
    pad = torch.zeros(B, longest, 2 * qk + H * D, dtype=torch.float64,
                      device="cuda")
    gate = torch.zeros(2, B, longest, H, dtype=torch.float64, device="cuda")
    gate[0] = 1.0                      # rows past a span change nothing
    kernel = v["conv1d.weight"].squeeze(1)
    for j, (a, b, _) in enumerate(spans):
        line = torch.cat([past[j].t(), mixed[a:b]])
        pad[j, :b - a] = torch.nn.functional.silu(sum(
            line[t:t + b - a] * kernel[:, t] for t in range(taps)))
        gate[0, j, :b - a], gate[1, j, :b - a] = decay[a:b], beta[a:b]
    q, k, u = pad.split([qk, qk, H * D], -1)

    def unit(t):
        t = t.view(B, longest, Hk, D)
        t = t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt()
        return t.repeat_interleave(H // Hk, 2)
    q, k, u = unit(q) * D ** -0.5, unit(k), u.view(B, longest, H, D)
    o = torch.empty_like(u)
    for t in range(longest):
        S = S * gate[0, :, t, :, None, None]
        kt = k[:, t].unsqueeze(-1)
        d = (u[:, t].unsqueeze(-1) - S @ kt) * gate[1, :, t, :, None, None]
        S = S + d * kt.transpose(-1, -2)
        o[:, t] = (S @ q[:, t].unsqueeze(-1)).squeeze(-1)
    new_state.append(S)
    o = torch.cat([o[j, :b - a] for j, (a, b, _) in enumerate(spans)])
    o = _rms(o, v["norm.weight"], g["eps"]) * torch.nn.functional.silu(z)
    return o.reshape(-1, H * D) @ out.t()


def _experts(w, i, x):
    g, k = w.g, w.g["top"]
    prob = (x @ w.router(i).double().t()).softmax(-1)
    share, ids = prob.topk(k, -1)
    if g["renorm"]:
        share = share / share.sum(-1, keepdim=True)
    gate, up, down = w.experts(i)
    y = torch.zeros_like(x)
    for e in range(g["experts"]):
        row, col = (ids == e).nonzero(as_tuple=True)
        if len(row):
            h = x[row]
            h = torch.nn.functional.silu(h @ gate[e].double().t()) * (
                h @ up[e].double().t())
            y[row] += (h @ down[e].double().t()) * share[row, col, None]
    if "shared" in g:
        y = y + _swiglu(w, w.mlp("layers.%d.mlp.shared_experts." % i,
                                 g["shared"] * g["expert_ff"]), x)
    return y


def exact(case, seed):
    w = _Weights(case, seed)
    g = w.g
    running, prompts = _requests(case, seed, g["vocab"])
    ids, pos, spans = [], [], []
    for t in running:
        spans.append((len(ids), len(ids) + 1, len(t) - 1))
        ids.append(t[-1])
        pos.append(len(t) - 1)
    for t in prompts:
        spans.append((len(ids), len(ids) + len(t), 0))
        ids += t
        pos += range(len(t))
    ids = torch.tensor(ids, device="cuda")
    pos = torch.tensor(pos, device="cuda")
    x = w.embedding()[ids].double()
    T, state, n_lin, n_kv = len(ids), [], 0, 0
    for i in range(g["layers"]):
        p = "layers.%d." % i
        norms = w.layer_norms(i)
        h = _rms(x, norms[p + "input_layernorm.weight"], g["eps"])
        if w.is_linear(i):
            x = x + _delta(w, i, n_lin, h, spans, seed, state)
            n_lin += 1
        elif "lora" in g:
            wq, wa, wb, wo = (w.dense(*s) for s in w.latent(i))
            H, dn, dr, C = g["heads"], g["nope"], g["rope"], g["lora"]
            q = (h @ wq.t()).view(T, H, dn + dr)
            a = h @ wa.t()
            n = p + "self_attn.kv_a_layernorm.weight"
            c = _rms(a[:, :C], w.norm(n, C), g["eps"])
            kr = _rope(a[:, None, C:], pos, dr, g["theta"])[:, 0]
            q = torch.cat([q[..., :dn],
                           _rope(q[..., dn:], pos, dr, g["theta"])], -1)
            wb = wb.view(H, dn + g["vdim"], C)
            o = torch.empty(T, H, g["vdim"], dtype=torch.float64,
                            device="cuda")
            for j, (s, e, past) in enumerate(spans):
                lat, rk = c[s:e], kr[s:e]
                if past:
                    old = _cached(seed, n_kv, j, past, 1, C + dr,
                                  "k")[:, 0].double()
                    lat = torch.cat([old[:, :C], lat])
                    rk = torch.cat([old[:, C:], rk])
                kv = torch.matmul(lat, wb.transpose(1, 2).contiguous())
                kv = kv.transpose(0, 1)
                k = torch.cat([kv[..., :dn],
                               rk[:, None].expand(-1, H, -1)], -1)
                o[s:e] = _attend(q[s:e], k, kv[..., dn:],
                                 (dn + dr) ** -0.5)
            x = x + o.reshape(T, -1) @ wo.t()
            n_kv += 1
        else:
            D, G = g["dim"], g["kv"]
            specs = w.attention(i)
            q, k, v = (h @ w.dense(*s).t() for s in specs[:3])
            if g.get("bias"):
                q, k, v = (t + w.rand(s[0] + ".bias", (s[1],), 0.1).double()
                           for t, s in zip((q, k, v), specs))
            q, k, v = q.view(T, -1, D), k.view(T, G, D), v.view(T, G, D)
            if "every" in g:
                hn = w.head_norms(i)
                q = _rms(q, hn[p + "self_attn.q_norm.weight"], g["eps"])
                k = _rms(k, hn[p + "self_attn.k_norm.weight"], g["eps"])
            rot = g.get("rot", D)
            q, k = _rope(q, pos, rot, g["theta"]), _rope(k, pos, rot,
                                                         g["theta"])
            o = torch.empty_like(q)
            for j, (s, e, past) in enumerate(spans):
                ks, vs = k[s:e], v[s:e]
                if past:
                    ks = torch.cat([_cached(seed, n_kv, j, past, G, D,
                                            "k").double(), ks])
                    vs = torch.cat([_cached(seed, n_kv, j, past, G, D,
                                            "v").double(), vs])
                o[s:e] = _attend(q[s:e], ks, vs, D ** -0.5)
            x = x + o.reshape(T, -1) @ w.dense(*specs[3]).t()
            n_kv += 1
        h = _rms(x, norms[p + "post_attention_layernorm.weight"], g["eps"])
        x = x + (_experts(w, i, h) if i in w.routed else
                 _swiglu(w, w.mlp(p + "mlp.", g["ff"]), h))
    last = torch.tensor([e - 1 for _, e, _ in spans], device="cuda")
    h = _rms(x[last], w.norm("norm", g["width"]), g["eps"])
    out = {"logits": h @ w.matrix("lm_head", g["vocab"],
                                  g["width"]).double().t(),
           "keys": None, "values": None}
    if state:
        out["state"] = torch.stack(state)
    return out
