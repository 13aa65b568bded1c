"""Wide-tile grouped MoE GEMM, token alignment and the softmax router
against plain fp32 / fp64 formulas, at the edges of their tiles."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(x, w13, w2, weights, ids, start, activation, args):
    x, w13, w2 = x.double(), w13.double(), w2.double()
    out = torch.zeros_like(x)
    for e in range(w13.shape[0]):
        row, col = (ids.long() == e + start).nonzero(as_tuple=True)
        if not len(row):
            continue
        h = x[row] @ w13[e].t()
        if activation == "relu2":
            a = h.clamp_min(0).square()
        else:
            g, u = h.chunk(2, dim=-1)
            if activation == "swiglu_clamp":
                g, u = g.clamp_max(args[0]), u.clamp(-args[0], args[0])
                a = g * torch.sigmoid(args[1] * g) * (u + 1)
            else:
                a = torch.nn.functional.silu(g) * u
        out.index_add_(0, row, (a @ w2[e].t()) *
                       weights[row, col].double()[:, None])
    return out


@pytest.mark.parametrize("case", [
    # T, E, topk, hidden, inter, activation, first local expert, experts
    (1, 8, 2, 64, 64, "silu_glu", 0, 8),        # one stage, one row
    (48, 8, 2, 128, 192, "silu_glu", 0, 8),     # 12 rows per expert: 32
    (53, 8, 2, 192, 320, "silu_glu", 0, 8),     # just over: 64
    (33, 16, 4, 256, 512, "silu_glu", 4, 8),    # a shard of the experts
    (160, 8, 2, 64, 128, "swiglu_clamp", 0, 8),  # 40 rows: 64
    (165, 8, 2, 128, 1408, "relu2", 0, 8),      # just over: 128
    (512, 8, 2, 192, 64, "silu_glu", 0, 8),     # 128 rows: 128
    (517, 8, 2, 128, 320, "silu_glu", 0, 8),    # just over: 256
    (600, 8, 2, 320, 192, "swiglu_clamp", 2, 3),
    (300, 2, 2, 64, 448, "relu2", 0, 2),
    (40, 8, 2, 72, 64, "silu_glu", 0, 8),       # 64 does not divide K
])
def test_fused_moe_tiles(case):
    from gllm_amd import ops
    T, E, topk, H, I, activation, start, local = case
    torch.manual_seed(T + I)
    args = (7.0, 1.702) if activation == "swiglu_clamp" else ()
    rows = I if activation == "relu2" else 2 * I
    x = torch.randn(T, H, device="cuda").bfloat16()
    w13 = (torch.randn(local, rows, H, device="cuda") * H ** -0.5).bfloat16()
    w2 = (torch.randn(local, H, I, device="cuda") * I ** -0.5).bfloat16()
    weights, ids = ops.topk_softmax(torch.randn(T, E, device="cuda"), topk)
    ids[T // 2, 0] = -1  # a padding pair contributes nothing
    out = ops.fused_moe(x, w13, w2, weights, ids, expert_start=start,
                        num_global_experts=E, activation=activation,
                        act_args=args)
    ref = _ref(x, w13, w2, weights, ids, start, activation, args)
    # bf16 roundings: the activation (2^-9 per term, averaged over the
    # contraction), each pair's result and their sum (2^-9 each)
    err = (out.double() - ref).norm() / ref.norm().clamp_min(1e-9)
    assert err < 4 * 2 ** -9, err


@pytest.mark.parametrize("N,E,start,block", [
    (1, 1, 0, 32), (65, 64, 0, 32), (1000, 64, 16, 128), (5000, 1024, 0, 64),
    (4096, 7, 0, 256)])
def test_moe_align_tables(N, E, start, block):
    from gllm_amd import ops
    torch.manual_seed(N)
    ids = torch.randint(-1, E + 2 * start, (N, 1), device="cuda").int()
    _, (sid, blocks, n_post), rows = ops._moe_tables(ids, E, start, block)
    ids, n = ids.view(-1).cpu(), int(n_post)
    assert n % block == 0 and n <= rows
    sid, blocks = sid[:n].cpu().view(-1, block), blocks[:n // block].cpu()
    seen = []
    for row, e in zip(sid, blocks):
        live = row[row < N]
        assert (ids[live.long()] == int(e) + start).all()
        assert len(live) and (row[:len(live)] < N).all()  # padding last
        seen += live.tolist()
    local = ((ids >= start) & (ids < start + E)).nonzero().view(-1)
    assert sorted(seen) == local.tolist()
    assert (blocks[1:] >= blocks[:-1]).all()


@pytest.mark.parametrize("rows,E,k,dtype", [
    (1, 8, 2, torch.bfloat16), (130, 64, 6, torch.bfloat16),
    (5, 512, 64, torch.float32), (7, 1, 1, torch.float32),
    (9, 65, 8, torch.float16)])
@pytest.mark.parametrize("renorm", [False, True])
def test_softmax_topk(rows, E, k, dtype, renorm):
    from gllm_amd import ops
    from gllm_amd.ops import torch_ref
    torch.manual_seed(E)
    # distinct logits in every row: the choice is unambiguous
    logits = torch.stack([torch.randperm(E) for _ in range(rows)]) \
        .sub(E / 2).mul(0.25).to(dtype).cuda()
    w, ids = ops.topk_softmax(logits, k, renorm)
    rw, rids = torch_ref.topk_softmax(logits.double(), k, renorm)
    assert torch.equal(ids, rids) and w.dtype == torch.float32
    # fp32 exponentials and sums of at most 512 terms
    assert torch.allclose(w, rw.float(), rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("E,k", [(8, 2), (64, 6), (100, 64)])
def test_softmax_topk_rows_that_are_not_finite(E, k):
    """Whatever the logits, the ids are k different experts; rows beside
    them are as ever."""
    from gllm_amd import ops
    from gllm_amd.ops import torch_ref
    torch.manual_seed(E)
    x = torch.stack([torch.randperm(E) for _ in range(9)]).float()
    ref, rids = torch_ref.topk_softmax(x.double(), k)
    x[0] = float("nan")
    x[2, 1], x[2, E - 1] = float("nan"), float("nan")
    x[4, 0], x[4, E // 2] = float("inf"), float("inf")
    x[6] = float("-inf")
    w, ids = ops.topk_softmax(x.cuda(), k)
    for out in (ids, ops.topk_then_softmax(x.cuda(), k)[1],
                ops.sigmoid_group_topk(x.cuda(), None, k)[1]):
        for row in out.tolist():
            assert len(set(row)) == k and 0 <= min(row) and max(row) < E
    good = [1, 3, 5, 7, 8]
    assert torch.equal(ids.cpu()[good], rids[good])
    assert torch.allclose(w.cpu()[good], ref[good].float(), rtol=1e-5,
                          atol=1e-9)
    assert w[[0, 2, 4, 6]].isnan().all()


@pytest.mark.parametrize("which", ["x", "w13", "w2", "activation"])
def test_fused_moe_takes_what_the_general_form_takes(which):
    """Operands that do not start on 16 bytes, and a gated activation by
    another name."""
    from gllm_amd import ops
    torch.manual_seed(3)
    T, E, H, I = 40, 8, 128, 192
    arg = {"x": torch.randn(T, H, device="cuda").bfloat16(),
           "w13": (torch.randn(E, 2 * I, H, device="cuda") * 0.1).bfloat16(),
           "w2": (torch.randn(E, H, I, device="cuda") * 0.1).bfloat16()}
    weights, ids = ops.topk_softmax(torch.randn(T, E, device="cuda"), 2)
    ref = _ref(arg["x"], arg["w13"], arg["w2"], weights, ids, 0, "", ())
    kind = "silu_glu"
    if which == "activation":
        kind = "silu"
    else:
        t = arg[which]
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")
        arg[which] = buf[4:4 + t.numel()].view(t.shape).copy_(t)
    out = ops.fused_moe(arg["x"], arg["w13"], arg["w2"], weights, ids,
                        activation=kind)
    assert (out.double() - ref).norm() / ref.norm() < 4 * 2 ** -9
