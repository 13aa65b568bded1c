"""Many-row products on 256-row tiles against fp64, at the edges of their
tiles, row blocks, splits along K and of the dispatch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,bias,gated", [
    (1, 8, 64, False, False),            # one stage, one row, one unit
    (257, 264, 128, True, False),        # a row and 8 columns into a tile
    (128, 512, 320, False, False),       # a whole half block
    (129, 248, 192, True, False),
    (385, 1040, 64, False, True),        # half block last, ragged columns
    (300, 16, 128, False, True),
    (2049, 1024, 640, True, False),      # many tiles of one row more
    (640, 4096, 4160, True, False),      # split along K
    (700, 4112, 4160, False, True),
    (4133, 2048, 1088, False, False),    # whole tiles, then split ones
])
def test_tile_gemm(M, N, K, bias, gated):
    from gllm_amd import ops
    k = ops._gpu_kernels()
    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda").bfloat16() if bias else None
    out = k.tile_gemm(x, w, b, gated)
    y = x.double() @ w.double().t()
    if bias:
        y = y + b.double()
    if gated:
        g, u = y.chunk(2, dim=-1)
        y = torch.nn.functional.silu(g) * u
    assert out.shape == y.shape and torch.isfinite(out).all()
    # one rounding to bf16 of fp32 sums; exponentials to a few 2^-23
    err = ((out.double() - y).abs() / y.abs().clamp_min(
        y.square().mean().sqrt())).max()
    assert err < 1.1 * 2 ** -8, err
    assert torch.equal(out, k.tile_gemm(x, w, b, gated))


def test_rows_past_the_last_are_left_alone():
    """Infinities and NaN in one row stay in it."""
    from gllm_amd import ops
    x = torch.randn(390, 192, device="cuda").bfloat16()
    w = torch.randn(520, 192, device="cuda").bfloat16()
    clean = ops._gpu_kernels().tile_gemm(x, w, None, False)
    x[17], x[388] = float("inf"), float("nan")
    out = ops._gpu_kernels().tile_gemm(x, w, None, False)
    keep = torch.ones(390, dtype=torch.bool)
    keep[17] = keep[388] = False
    assert torch.equal(out[keep], clean[keep])
    assert out[388].isnan().all() and not out[17].isfinite().any()


@pytest.mark.parametrize("M", [256, 257, 384, 500])
def test_dispatch(M):
    """The same numbers whichever kernel a row count is sent to: the stream
    and the library, gated the stream and the tile kernel."""
    from gllm_amd import ops
    torch.manual_seed(M)
    x = torch.randn(M, 3072, device="cuda").bfloat16()
    w = (torch.randn(1024, 3072, device="cuda") * 3072 ** -0.5).bfloat16()
    b = torch.randn(1024, device="cuda").bfloat16()
    ref = x.double() @ w.double().t()
    for out, y in ((ops.linear(x, w, b), ref + b.double()),
                   (ops.linear(x, w), ref)):
        assert ((out.double() - y).norm() / y.norm()) < 2 ** -8
    # a bias of another type, off 16 bytes or a strided view: refused or
    # taken as before
    off = torch.cat([b[:1], b])[1:]
    assert torch.allclose(ops.linear(x, w, off).float(),
                          ops.linear(x, w, b).float(), atol=0.05)
    half = ops.linear(x[:, ::2], w[:, ::2])
    y = x[:, ::2].double() @ w[:, ::2].double().t()
    assert ((half.double() - y).norm() / y.norm()) < 2 ** -8
    g, u = ref.chunk(2, dim=-1)
    y = torch.nn.functional.silu(g) * u
    out = ops.linear_silu(x, w)
    assert ((out.double() - y).norm() / y.norm()) < 2 ** -7


@pytest.mark.parametrize("M,N,K", [
    (32, 9216, 8192),        # the stream's last row count
    (33, 9216, 8192), (64, 9216, 8192),    # long streams
    (65, 5128, 5120), (128, 5120, 5120),   # half a block, ragged columns
    (129, 5128, 5120), (256, 5120, 5120),  # two blocks of 128 rows
    (129, 9208, 8192), (200, 5120, 27648),  # one block
])
@pytest.mark.parametrize("gated", [False, True])
def test_few_rows(M, N, K, gated):
    """Parts of wide weights, and the gated form on very wide ones."""
    from gllm_amd import ops
    if gated:
        N, K = {5120: 65536, 5128: 49152}.get(N, 49168), 4096
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    y = x.double() @ w.double().t()
    if gated:
        g, u = y.chunk(2, dim=-1)
        y = torch.nn.functional.silu(g) * u
        out = ops.linear_silu(x, w).double()
        bound = 1.1 * 2 ** -8   # one rounding to bf16
    else:
        part = ops._gpu_kernels().stream_parts(x, w)
        assert part.shape[1:] == (M, N)
        out = part.double().sum(0)
        bound = 2 ** -23 * K ** 0.5  # fp32 sums: a rounding per 32 columns
    err = (out - y).abs() / y.abs().clamp_min(y.square().mean().sqrt())
    assert err.max() < bound, err.max()


@pytest.mark.parametrize("M,N,K,stream", [
    (256, 1024, 28736, True), (160, 2048, 16448, True),  # CUs would idle
    (256, 2560, 12864, False),
    (96, 3072, 12352, True), (96, 3584, 8256, False),
    (128, 6144, 4096, True), (128, 8192, 3584, True),    # short parts
    (128, 5120, 5120, False), (136, 6144, 4096, False),
])
def test_lines_of_parts(M, N, K, stream):
    """Sizes whose parts come from the stream kernel: as many as for rows
    that are apart in memory, which only that kernel takes."""
    from gllm_amd import ops
    k = ops._gpu_kernels()
    torch.manual_seed(M + N)
    x = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    apart, part = k.stream_parts(x, w), k.stream_parts(x.contiguous(), w)
    if stream:
        assert torch.equal(apart, part)
    else:
        assert apart.shape != part.shape or not torch.equal(apart, part)
    y = x.double() @ w.double().t()
    err = (part.double().sum(0) - y).abs() / y.abs().clamp_min(
        y.square().mean().sqrt())
    assert err.max() < 2 ** -23 * K ** 0.5  # fp32 sums


@pytest.mark.parametrize("M,N,K,tile", [
    (4096, 1024, 17408, True), (500, 4096, 28672, True),
    (8200, 1024, 17408, False),    # a round that is half full
    (4096, 2048, 10944, True), (4096, 2048, 9472, False),
    (8192, 2048, 6144, False),     # nearly full
    (10600, 2560, 7680, False),    # the second one, K short
    (4096, 1024, 3008, False),     # K below 3 N
    (2000, 512, 2048, False),      # slow for either
])
def test_long_contractions(M, N, K, tile):
    """Which sizes ops.linear sends to the tile kernel, and its bias there:
    one off 16 bytes, of another type or strided goes to the library."""
    from gllm_amd import ops
    assert ops._use_tile(M, N, K) == tile
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    b = torch.randn(N + 1, device="cuda").bfloat16()
    y = x.double() @ w.double().t()
    lib = torch.nn.functional.linear
    for bias in (None, b[:N], b[1:], b[:N].repeat(2).view(2, N).t()[:, 0],
                 b[:1].expand(N)):
        ours = tile and (bias is None or (bias.is_contiguous()
                                          and bias.data_ptr() % 16 == 0))
        out = ops.linear(x, w, bias)
        if ours:
            assert torch.equal(
                out, ops._gpu_kernels().tile_gemm(x, w, bias, False))
        else:
            assert torch.equal(out, lib(x, w, bias))
        ref = y if bias is None else y + bias.double()
        assert ((out.double() - ref).norm() / ref.norm()) < 2 ** -8


def test_long_contractions_have_gradients():
    from gllm_amd import ops
    torch.manual_seed(0)
    M, N, K = 4096, 1024, 17408
    assert ops._use_tile(M, N, K)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    g = torch.randn(M, N, device="cuda").bfloat16()
    for operand in (x, w):
        operand.requires_grad_()
        out = ops.linear(x, w)
        ref = torch.nn.functional.linear(x, w)
        got, want = (torch.autograd.grad(o, operand, g)[0]
                     for o in (out, ref))
        assert torch.equal(got, want)
        with torch.no_grad():
            assert not ops.linear(x, w).requires_grad
        operand.requires_grad_(False)


@pytest.mark.parametrize("M,N,K,tile", [
    (128, 55296, 4096, False), (129, 55296, 4096, True),
    (256, 51200, 1024, True), (256, 51184, 1088, True),
    (256, 50944, 1024, False), (200, 65536, 1024, True),
    (200, 65552, 1024, False),               # more than a round
    (200, 51200, 960, False),
    (300, 5632, 2048, True), (300, 16384, 2048, False),
    (257, 2048, 4096, True),                 # few tiles
    (512, 9728, 2560, False), (768, 16384, 11136, False),  # part of a round
    (1000, 13312, 2560, True),
    (384, 55296, 5120, False), (512, 55296, 5120, True),   # half row blocks
    (1152, 43008, 3840, False), (1664, 43008, 3840, True),
    (714, 32768, 2560, False), (700, 37888, 3584, True),   # second rounds
    (1242, 16384, 1536, False), (1242, 21888, 2048, True),
])
def test_lines_of_gated(M, N, K, tile):
    """Which sizes ops.linear_silu sends to the tile kernel; up to 256 rows
    the others are the stream's, above the library's."""
    from gllm_amd import ops
    assert ops._use_tile_gated(M, N, K) == tile
    k = ops._gpu_kernels()
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    if tile:
        ref = k.tile_gemm(x, w, None, True)
    elif M <= 256:
        ref = k.stream_gemm_gated(x, w)
    else:
        ref = ops.silu_and_mul(torch.nn.functional.linear(x, w))
    assert torch.equal(ops.linear_silu(x, w), ref)
    g, u = (x[:3].double() @ w.double().t()).chunk(2, dim=-1)
    y = torch.nn.functional.silu(g) * u
    assert ((ref[:3].double() - y).norm() / y.norm()) < 2 ** -7
