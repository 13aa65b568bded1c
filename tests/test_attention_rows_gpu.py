"""One-row sequences of a mixed batch on the decode kernel, and the decode
kernel's unsplit form."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(q_lens, ctx, Hq, Hkv, D, page=16):
    torch.manual_seed(sum(q_lens) + Hq)
    lens = [c + n for c, n in zip(ctx, q_lens)]
    need = [-(-n // page) for n in lens]
    pages = torch.randperm(sum(need) + 2)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n].int()
        at += n
    kc, vc = (torch.randn(sum(need) + 2, page, Hkv, D).bfloat16().cuda()
              for _ in range(2))
    q = torch.randn(sum(q_lens), Hq, D).bfloat16().cuda()
    qsl = torch.tensor([0] + q_lens).cumsum(0).int().cuda()
    return q, kc, vc, table.cuda(), torch.tensor(lens).int().cuda(), qsl


def _ref(q, kc, vc, table, lens, qsl, scale, window):
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    r = q.shape[1] // kc.shape[2]
    for i, n in enumerate(lens.tolist()):
        a, b = int(qsl[i]), int(qsl[i + 1])
        k, v = (c[table[i].long()].flatten(0, 1)[:n].double()
                .repeat_interleave(r, 1).transpose(0, 1).contiguous()
                for c in (kc, vc))
        s = torch.matmul(q[a:b].double().transpose(0, 1).contiguous(),
                         k.transpose(1, 2).contiguous()) * scale
        pos = torch.arange(n - (b - a), n, device="cuda")[:, None]
        key = torch.arange(n, device="cuda")[None]
        hide = (key > pos) | ((key <= pos - window) if window else False)
        s = s.masked_fill(hide, -float("inf")).softmax(-1)
        out[a:b] = torch.matmul(s, v).transpose(0, 1)
    return out


@pytest.mark.parametrize("window", [0, 48])
@pytest.mark.parametrize("q_lens,ctx,Hq,Hkv,D", [
    ([1, 70, 1, 3, 1], [40, 0, 300, 64, 0], 8, 2, 128),
    ([130, 1], [5, 31], 40, 8, 128),
    ([1] * 9 + [2], [33 * i for i in range(10)], 16, 1, 64),
    ([1, 64], [100, 0], 17, 1, 128),     # more heads than it takes
])
def test_mixed_batch(q_lens, ctx, Hq, Hkv, D, window):
    from gllm_amd import ops
    case = _case(q_lens, ctx, Hq, Hkv, D)
    scale = D ** -0.5
    ref = _ref(*case, scale, window)
    for single in (0, sum(n == 1 for n in q_lens)):
        out = ops.paged_attention(
            *case, scale, max_query_len=max(q_lens), sliding_window=window,
            single_rows=single)
        # weights and the result rounded to bf16
        err = (out.double() - ref).norm() / ref.norm()
        assert err < 3 * 2 ** -9, (single, err)


@pytest.mark.parametrize("B,Hkv", [(1030, 1), (515, 2)])
def test_unsplit_decode(B, Hkv):
    """A batch that fills the chip in one split (the result is written by
    the attention kernel itself), with gate, sink and learned sinks."""
    from gllm_amd import ops
    G, D = 4, 64
    q, kc, vc, table, lens, qsl = _case(
        [1] * B, [i % 90 for i in range(B)], Hkv * G, Hkv, D)
    ref = _ref(q, kc, vc, table, lens, qsl, D ** -0.5, 0)
    out = ops.paged_attention(q, kc, vc, table, lens, qsl, D ** -0.5)
    assert (out.double() - ref).norm() / ref.norm() < 3 * 2 ** -9
    k = ops._seq_kernels()
    rows = q.reshape(B, -1)
    gate = torch.randn_like(rows)
    sinks = torch.randn(Hkv * G, device="cuda")
    for sink, learned in ((False, None), (True, None), (False, sinks)):
        def run(a, b):
            o = torch.empty_like(rows[a:b])
            assert k.window_attention_decode(
                o, rows[a:b], gate[a:b].contiguous(), kc, vc,
                table[a:b].contiguous(), lens[a:b].contiguous(), D ** -0.5,
                0, 0, sink, learned, 0.0, None, 0.0, 0)
            return o
        whole = run(0, B)
        parts = torch.cat([run(a, min(a + 7, B)) for a in range(0, B, 7)])
        # the split form rounds its weights against another maximum
        err = (whole.double() - parts.double()).norm() / parts.double().norm()
        assert err < 3 * 2 ** -9, err


def test_decode_reads_as_many_lengths_as_rows():
    """A step's tables may be longer than the step (buffers of a larger
    batch): the first rows count."""
    from gllm_amd import ops
    q, kc, vc, table, lens, qsl = _case([1] * 5, [3, 200, 64, 17, 90], 8, 2,
                                        128)
    ref = ops.paged_attention(q, kc, vc, table, lens, qsl, 0.1)
    for n in (1, 3):
        for t in (table, table[:n]):
            out = ops.paged_attention(q[:n], kc, vc, t, lens, qsl, 0.1)
            # (the splits follow the rows)
            err = (out - ref[:n]).float().norm() / ref[:n].float().norm()
            assert err < 3 * 2 ** -9, err
    with pytest.raises(RuntimeError):           # lengths for fewer rows
        ops.paged_attention(q, kc, vc, table, lens[:4], qsl, 0.1)
