"""Few-row products and what is fused behind them, against fp64, at the
edges of their tiles and splits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    return x, w, x.double() @ w.double().t()


def _close(got, want, tol=2 ** -8):
    # one bf16 rounding of the result
    err = (got.double() - want).norm() / want.norm()
    assert err < tol, err


SHAPES = [
    (1, 512, 64), (16, 520, 128), (17, 2048, 2048), (32, 4096, 576),
    (33, 1000, 5120), (64, 512, 8192), (65, 1024, 1024), (128, 7168, 320),
    (128, 8192, 640), (100, 512, 2048), (129, 1536, 1024), (256, 512, 4096),
    (256, 5120, 192), (24, 36000, 256), (64, 40008, 128), (128, 36008, 192),
]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_stream_gemm(M, N, K):
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    b = torch.randn(N, device="cuda").bfloat16()
    _close(ops.skinny_gemm(x, w), ref)
    _close(ops.skinny_gemm(x, w, b), ref + b.double())
    if N % 16 == 0:
        g, u = ref.chunk(2, dim=-1)
        _close(ops.linear_silu(x, w), torch.nn.functional.silu(g) * u)


@pytest.mark.parametrize("M,N,K", [(256, 36000, 128), (200, 16384, 192),
                                   (129, 40000, 64)])
def test_stream_gemm_gated_wide(M, N, K):
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    g, u = ref.chunk(2, dim=-1)
    _close(ops.linear_silu(x, w), torch.nn.functional.silu(g) * u)


@pytest.mark.parametrize("M,N,K,wdtype", [
    (1, 512, 4096, torch.float32), (3, 2048, 2048, torch.bfloat16),
    (64, 2056, 1024, torch.float32), (33, 5120, 27648, torch.float32),
    (256, 6152, 512, torch.bfloat16), (16, 8192, 64, torch.float32),
    (300, 1024, 512, torch.bfloat16)])     # the library's product
def test_linear_add_rmsnorm(M, N, K, wdtype):
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    res = torch.randn(M, N, device="cuda").bfloat16()
    norm = (1 + 0.1 * torch.randn(N, device="cuda")).to(wdtype)
    want = res.double() + ref
    out, new = ops.linear_add_rmsnorm(x, w, res.clone(), norm, 1e-6)
    _close(new, want)
    want = new.double()
    want = want * (want.square().mean(-1, keepdim=True) + 1e-6).rsqrt()
    _close(out, want * norm.double())


@pytest.mark.parametrize("parts", [False, True])
@pytest.mark.parametrize("M,Hq,Hkv,D,rot,K", [
    (1, 8, 8, 64, 64, 512), (37, 40, 8, 128, 128, 1024),
    (64, 16, 2, 128, 32, 512), (130, 4, 1, 96, 96, 256),
    (5, 6, 3, 80, 40, 4096)])
def test_qkv_rope_cache(M, Hq, Hkv, D, rot, K, parts):
    from gllm_amd import ops
    N = (Hq + 2 * Hkv) * D
    x, w, ref = _operands(M, N, K)
    bias = torch.randn(N, device="cuda").bfloat16()
    src = ops.qkv_parts(x, w, bias) if parts else (x @ w.t())
    if not parts:
        ref = src.double()
    ref = (ref + bias.double()).view(M, -1, D)
    pos = torch.randint(0, 2000, (M,), device="cuda")
    ang = torch.arange(2000).double()[:, None] * 10000.0 ** (
        -torch.arange(0, rot, 2).double() / rot)
    cs = torch.cat([ang.cos(), ang.sin()], -1).float().cuda()
    kc = torch.zeros(M // 16 + 2, 16, Hkv, D, device="cuda").bfloat16()
    vc = torch.zeros_like(kc)
    slots = torch.randperm(kc.shape[0] * 16, device="cuda")[:M]
    assert ops.qkv_rope_cache_ok(kc, vc, cs, True)
    q = ops.qkv_rope_cache(src, bias, pos, cs, kc, vc, slots, Hq)
    c, s = cs[pos].double()[:, None].chunk(2, -1)
    h = ref[:, :Hq + Hkv]
    a, b = h[..., :rot // 2], h[..., rot // 2:rot]
    h = torch.cat([a * c - b * s, b * c + a * s, h[..., rot:]], -1)
    _close(q.view(M, Hq, D), h[:, :Hq])
    _close(kc.view(-1, Hkv, D)[slots], h[:, Hq:])
    _close(vc.view(-1, Hkv, D)[slots], ref[:, Hq + Hkv:])
    free = torch.ones(kc.shape[0] * 16, dtype=torch.bool, device="cuda")
    free[slots] = False
    assert not kc.view(-1, Hkv, D)[free].any()
    assert not vc.view(-1, Hkv, D)[free].any()


@pytest.mark.parametrize("M,N,K", [(8, 1024, 4096), (100, 2056, 128)])
def test_bias_of_another_type(M, N, K):
    """An fp32 bias is added to the bf16 product; the result stays bf16."""
    from gllm_amd import ops
    x, w, ref = _operands(M, N, K)
    bias = torch.randn(N, device="cuda")
    for f in (ops.skinny_gemm, ops.linear):
        out = f(x, w, bias)
        assert out.dtype == torch.bfloat16
        # two roundings
        _close(out, ref + bias.double(), 2 ** -7)
    # an N that the kernel does not take
    _close(ops.skinny_gemm(x, w[:N - 3], bias[:N - 3]),
           ref[:, :N - 3] + bias[:N - 3].double(), 2 ** -7)
    for bad in ((x.float(), w.float()), (x.t(), w[:, :M].contiguous()),
                (x.repeat(300, 1), w)):
        with pytest.raises(RuntimeError):
            ops.skinny_gemm(*bad)
