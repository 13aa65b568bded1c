"""Few-row products with quantized weights (csrc/quant_gemm.hip) against the
exact weights in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def make(kind, M, N, K):
    """(x, op, exact product [M, N] in fp64, a bound on |x| |w|)."""
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K).to(torch.bfloat16)
    if kind == "int4":
        q = torch.randint(0, 16, (N, K))
        s = torch.rand(K // 128, N) * 0.01 + 0.001
        z = torch.randint(0, 16, (K // 128, N))
        sbt = torch.stack([s, -z * s], 1).contiguous()
        rep = [t.t().repeat_interleave(128, 1).double()
               for t in (s, sbt[:, 1])]
        w = q.double() * rep[0] + rep[1]
        packed = (q[:, ::2] | (q[:, 1::2] << 4)).to(torch.uint8)
        op = ("int4", packed.cuda(), sbt.cuda())
        xe = x.double()
    else:
        wq = (torch.randn(N, K) * 20).to(torch.float8_e4m3fn)
        ws = torch.rand(-(-N // 128), K // 128) * 0.01 + 0.001
        w = wq.double() * ws.double().repeat_interleave(
            128, 0)[:N].repeat_interleave(128, 1)
        from gllm_amd import ops
        xq, xs = [t.cpu() for t in ops.per_token_group_quant_fp8(x.cuda())]
        xe = (xq.double().view(M, -1, 128) * xs.double()[..., None]).view(
            M, K)
        op = ("fp8", wq.cuda(), ws.cuda())
    return x.cuda(), op, xe @ w.t(), xe.abs() @ w.abs().t()


def close(out, ref, size, bf16=True, kind="int4"):
    # sums in 32 bits: 1e-5 of the terms' sizes (their rounding and, int4,
    # the offset of 16 in front of each; the e4m3 matrix instruction lines
    # its 32 products up with the largest before it adds them and drops
    # what falls below its adder: 2^-15); a bf16 result: half a step, 2^-8
    bound = (1e-5 if kind == "int4" else 2 ** -15) * size \
        + (2 ** -8 * ref.abs() if bf16 else 0)
    assert ((out.cpu().double() - ref).abs() <= bound).all()


# tiles of 16, 32 and 64 rows, of 64, 128 and 256 columns, with remainders in
# both, split and unsplit; more than one block of 64 rows; N of no multiple
# of 8
@pytest.mark.parametrize("kind", ["int4", "fp8"])
@pytest.mark.parametrize("M,N,K", [
    (1, 264, 512), (16, 72, 2560), (17, 200, 1024), (29, 520, 2048),
    (32, 16648, 256), (33, 1032, 768), (64, 136, 5120), (64, 36104, 256),
    (5, 16392, 512), (100, 264, 1024), (256, 136, 512), (3, 100, 512),
    (20, 27, 256)])
def test_rows_parts_and_norm(kind, M, N, K):
    from gllm_amd import ops
    x, op, ref, size = make(kind, M, N, K)
    bias = torch.randn(N)
    close(ops.quant_rows(x, op), ref, size, kind=kind)
    out = ops.quant_rows(x, op, bias.cuda())
    close(out, ref + bias.double(), size, kind=kind)
    part = ops.quant_parts(x, op)
    if N % 8:
        assert part is None
        return
    close(part.double().sum(0), ref, size, bf16=False, kind=kind)
    if N <= 8192:
        res = torch.randn(M, N).to(torch.bfloat16)
        w = torch.rand(N) + 0.5
        got = res.cuda()
        h, r = ops.quant_add_rmsnorm(x, op, got, w.cuda(), 1e-6)
        s = ref + res.double()
        # (fp8: the product is rounded to bf16 before it is added)
        near = 2 ** -8 * ref.abs() if kind == "fp8" else 0
        assert ((r.cpu().double() - s).abs() <= 2 ** -15 * size + near
                + 2 ** -8 * (s.abs() + near)).all()
        rr = r.cpu().double()
        n = rr * torch.rsqrt(rr.pow(2).mean(-1, keepdim=True) + 1e-6) * w
        assert ((h.cpu().double() - n).abs() <= 2 ** -7 * n.abs() + 1e-5).all()


@pytest.mark.parametrize("kind", ["int4", "fp8"])
@pytest.mark.parametrize("M", [1, 16, 31, 64])
@pytest.mark.parametrize("N", [16416, 36096, 512])
def test_gated(kind, M, N):
    from gllm_amd import ops
    x, op, ref, size = make(kind, M, N, 256)
    ref, size = ref * 0.05, size * 0.05   # (silu in its curved range)
    op = (op[0], op[1], op[2] * 0.05)
    g, u = ref.split(N // 2, 1)
    want = torch.nn.functional.silu(g) * u
    sg, su = size.split(N // 2, 1)
    out = ops.quant_silu(x, op).cpu().double()
    # |d silu| <= 1.1; a small N rounds gate, up and the result to bf16
    err = (1e-5 if kind == "int4" else 2 ** -15) * (1.1 * sg * u.abs() + g.abs() * su) \
        + 4 * 2 ** -8 * (want.abs() + g.abs() * u.abs() * 0.3) + 1e-6
    assert ((out - want).abs() <= err).all()


def test_int4_rows_that_are_not_finite():
    """An infinity or a NaN in a row gives what the weights one by one give,
    and the other rows are not touched."""
    from gllm_amd import ops
    x, op, ref, size = make("int4", 20, 264, 512)
    x[3, 130], x[5, 7], x[6, 9] = float("inf"), float("nan"), 3e38
    out = ops.quant_rows(x, op).cpu().double()
    rest = [i for i in range(20) if i not in (3, 5, 6)]
    close(out[rest], ref[rest], size[rest])
    q = op[1].cpu()
    s, b = op[2].cpu()[1, 0], op[2].cpu()[1, 1]       # group of column 130
    w = (q[:, 65] & 15).float() * s + b
    want = torch.where(w > 0, float("inf"), float("-inf")).double()
    some = w.abs() > 1e-6                             # (0 * inf is NaN)
    assert torch.equal(out[3][some], want[some])
    assert out[5].isnan().all()
    w6 = (q[:, 4] >> 4).float() * op[2].cpu()[0, 0] + op[2].cpu()[0, 1]
    assert torch.equal(out[6][w6.abs() > 1e-6] > 0, w6[w6.abs() > 1e-6] > 0)


@pytest.mark.parametrize("M,N,K", [(4, 272, 512), (20, 272, 512),
                                   (29, 16640, 256), (40, 1040, 768)])
def test_int4_large_values_that_cancel(M, N, K):
    """The sum of a group's activations may be small where the terms of the
    offset form are past 32 bits."""
    from gllm_amd import ops
    x, op, _, _ = make("int4", M, N, K)
    x[2] = 0
    x[2, 10], x[2, 11] = 2e37, -2e37
    x[3, 128:256:2], x[3, 129:256:2] = 3e36, -3e36
    q = torch.stack([op[1].cpu() & 15, op[1].cpu() >> 4], -1).view(N, K)
    s, b = (op[2][:, i].cpu().t().repeat_interleave(128, 1).double()
            for i in (0, 1))
    w = q.double() * s + b
    ref, size = (a @ v.t() for a, v in (
        (x.cpu().double(), w), (x.cpu().double().abs(), w.abs())))
    rest = [i for i in range(M) if i not in (2, 3)]
    for out in (ops.quant_rows(x, op), ops.quant_parts(x, op).sum(0)):
        out = out.cpu().double()
        close(out[rest], ref[rest], size[rest])
        # (these rows may take weights rounded to bf16)
        assert ((out - ref).abs() <= 2 ** -7 * size)[2:4].all()
    # gate and up of a size that silu and their product leave finite
    small = (op[0], op[1], op[2] * 1e-30)
    g, u = (ref * 1e-30).split(N // 2, 1)
    want = torch.nn.functional.silu(g) * u
    sg, su = (size * 1e-30).split(N // 2, 1)
    out = ops.quant_silu(x, small).cpu().double()
    err = 2 ** -6 * (sg * u.abs() + g.abs() * su + want.abs()) + 1e-30
    assert ((out - want).abs() <= err)[2:4].all()


def test_refusals():
    from gllm_amd import ops
    x, op, _, _ = make("int4", 4, 64, 256)
    with pytest.raises(RuntimeError):
        ops.int4_linear(x, op[1], op[2], 64)
    with pytest.raises(RuntimeError):       # K of 128
        ops.quant_rows(x[:, :128], ("int4", op[1][:, :64].contiguous(),
                                    op[2][:1]))
    with pytest.raises(RuntimeError):       # more than 256 rows
        ops.quant_rows(torch.zeros(257, 256, dtype=torch.bfloat16,
                                   device="cuda"), op)
    assert ops.quant_rows(x[:0], op).shape == (0, 64)
