"""Latent attention against fp64 at the edges of its row and key tiles."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(q_lens, ctx, H, page=16, seed=0):
    torch.manual_seed(seed)
    lens = [c + n for c, n in zip(ctx, q_lens)]
    need = [-(-n // page) for n in lens]
    pages = torch.randperm(sum(need) + 3)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n].int()
        at += n
    cache = torch.randn(sum(need) + 3, page, 1, 576).bfloat16()
    q = torch.randn(sum(q_lens), H, 576).bfloat16()
    qsl = torch.tensor([0] + q_lens).cumsum(0).int()
    return q, cache, table, torch.tensor(lens).int(), qsl


def _ref(q, cache, table, lens, qsl, scale):
    out = torch.empty(q.shape[0], q.shape[1], 512, dtype=torch.float64)
    for i, n in enumerate(lens.tolist()):
        a, b = int(qsl[i]), int(qsl[i + 1])
        k = cache[table[i].long()].reshape(-1, 576)[:n].double()
        s = q[a:b].double() @ k.t() * scale           # [n, H, keys]
        pos = torch.arange(n - (b - a), n)
        hide = torch.arange(n)[None] > pos[:, None]
        s = s.masked_fill(hide[:, None], -float("inf"))
        out[a:b] = s.softmax(-1) @ k[:, :512]
    return out


@pytest.mark.parametrize("q_lens,ctx,H,page", [
    ([1], [0], 16, 16),                    # one key
    ([1, 1, 1], [63, 64, 65], 16, 16),     # edges of a key tile
    ([1] * 5, [127, 1000, 1, 300, 64], 5, 16),
    ([1, 1], [200, 2000], 17, 16),         # more rows than one tile
    ([1, 1], [70, 500], 128, 16),
    ([1] * 600, [40] * 600, 16, 16),       # no split
    ([70, 1, 3], [0, 130, 64], 16, 16),    # portions beside a decode
    ([1] * 7, [30, 31, 32, 94, 95, 96, 1500], 16, 16),  # 32 keys
    ([2, 1, 2], [31, 33, 700], 8, 16),     # two rows a head
    ([3] * 300, [64] * 300, 5, 16),        # the same, no split
    ([33], [100], 5, 48),                  # page size not a power of two
    ([64, 65], [0, 0], 16, 1),
])
def test_mla_attention_tiles(q_lens, ctx, H, page):
    from gllm_amd import ops
    args = _case(q_lens, ctx, H, page)
    scale = 192 ** -0.5
    ref = _ref(*args, scale)
    q, cache, table, lens, qsl = (t.cuda() for t in args)
    out = ops.mla_paged_attention(q, cache, cache[..., :512], table, lens,
                                  qsl, scale)
    # weights and the result are rounded to bf16 (2^-9 each)
    err = (out.cpu().double() - ref).norm() / ref.norm()
    assert err < 3 * 2 ** -9, err


def test_mla_attention_reads_as_many_offsets_as_lengths():
    """Offsets past the sequences' own (buffers of a larger batch) are not
    looked at."""
    from gllm_amd import ops
    q, cache, table, lens, qsl = (
        t.cuda() for t in _case([1, 1, 1, 9], [5, 900, 64, 0], 16))
    want = ops.mla_paged_attention(q[:3], cache, cache[..., :512], table[:3],
                                   lens[:3], qsl[:4], 0.1)
    out = ops.mla_paged_attention(q[:3], cache, cache[..., :512], table[:3],
                                  lens[:3], qsl, 0.1)
    assert torch.equal(out, want)


def test_mla_decode_captured_serves_longer_batches():
    """The split count does not depend on the lengths seen at capture."""
    from gllm_amd import ops
    scale = 192 ** -0.5
    q, cache, table, lens, qsl = (
        t.cuda() for t in _case([1] * 4, [5, 900, 64, 300], 16))
    short = torch.ones_like(lens)
    run = lambda: ops.mla_paged_attention(  # noqa: E731
        q, cache, cache[..., :512], table, buf, qsl, scale,
        seq_lens_cpu=[1] * 4, query_start_loc_cpu=[0, 1, 2, 3, 4])
    buf = short.clone()
    run()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = run()
    for want in (lens, short, lens):
        buf.copy_(want)
        eager = ops.mla_paged_attention(q, cache, cache[..., :512], table,
                                        want, qsl, scale)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("T,H,strided,wdtype", [
    (1, 16, False, torch.bfloat16), (64, 3, True, torch.float32),
    (65, 16, False, torch.float32), (130, 128, True, torch.bfloat16)])
def test_mla_queries_and_values(T, H, strided, wdtype):
    """Latent rows, absorbed queries and per-head values against fp64."""
    from gllm_amd import ops
    torch.manual_seed(T)
    wide = 8 if strided else 0        # rows of a wider projection
    q = torch.randn(T, H * 192 + wide, device="cuda").bfloat16()[
        :, :H * 192]
    kv = torch.randn(T, 576 + wide, device="cuda").bfloat16()[:, :576]
    norm = (1 + 0.1 * torch.randn(512, device="cuda")).to(wdtype)
    w = (torch.randn(H * 256, 512, device="cuda") * 512 ** -0.5).bfloat16()
    pos = torch.randint(0, 4096, (T,), device="cuda")
    ang = torch.arange(4096).double()[:, None] * 10000.0 ** (
        -torch.arange(0, 64, 2).double() / 64)
    cs = torch.cat([ang.cos(), ang.sin()], -1).float().cuda()
    cache = torch.zeros(T // 16 + 2, 16, 1, 576, device="cuda").bfloat16()
    slots = torch.randperm(cache.shape[0] * 16, device="cuda")[:T]
    assert ops.mla_absorbed_ok(q, kv, w, norm, cache, cs, 128, 128)
    qf = ops.mla_queries(q, kv, norm, 1e-6, pos, cs, w, cache, slots)

    def turn(x):
        c, s = cs[pos].double().chunk(2, -1)
        if x.dim() == 3:
            c, s = c[:, None], s[:, None]
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    q64, kv64 = q.double().view(T, H, 192), kv.double()
    wv = w.double().view(H, 256, 512)
    lat = torch.matmul(q64[..., :128].transpose(0, 1).contiguous(),
                       wv[:, :128].contiguous()).transpose(0, 1)
    want = torch.cat([lat, turn(q64[..., 128:])], -1)
    c = kv64[:, :512]
    c = c * (c.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * norm.double()
    row = torch.cat([c, turn(kv64[:, 512:])], -1)
    got = cache.view(-1, 576)[slots].double()
    values = ops.mla_values(qf[..., :512].contiguous(), w)
    vref = torch.matmul(
        qf[..., :512].double().transpose(0, 1).contiguous(),
        wv[:, 128:].transpose(1, 2).contiguous()).transpose(0, 1)
    # one bf16 rounding of the result each
    for a, b in ((qf.double(), want), (got, row),
                 (values.double().view(T, H, 128), vref)):
        assert (a - b).norm() / b.norm() < 2 ** -8
    untouched = torch.ones(cache.shape[0] * 16, dtype=torch.bool)
    untouched[slots.cpu()] = False
    assert not cache.view(-1, 576)[untouched.cuda()].any()
