"""e4m3 rows from the kernels that form the rows: what quantizing their bf16
result gives, bit for bit."""

import pytest
import torch

from test_qkv_decode_gpu import _step

pytestmark = pytest.mark.gpu


def _same(rows, x):
    from gllm_amd import ops
    q, _, st = ops.per_token_group_quant_fp8(x, transposed=True)
    assert torch.equal(rows.x, x)
    assert torch.equal(rows.scales, st)
    assert torch.equal(rows.q, q.view(torch.uint8))


def _fp8(N, K):
    w = (torch.randn(N, K, device="cuda") * 20).to(torch.float8_e4m3fn)
    ws = torch.rand(-(-N // 128), K // 128, device="cuda") * 0.01 + 0.001
    return "fp8", w, ws


@pytest.mark.parametrize("M,N", [(1, 128), (3, 2048), (64, 2176), (5, 4224),
                                 (33, 5120), (2, 8192)])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
def test_norm(M, N, wdtype):
    from gllm_amd import ops
    torch.manual_seed(M + N)
    x = torch.randn(M, 256, device="cuda").bfloat16()
    op, res = _fp8(N, 256), torch.randn(M, N, device="cuda").bfloat16()
    res[0, :128] = float("-inf") if M == 2 else 0
    w = (1 + 0.1 * torch.randn(N, device="cuda")).to(wdtype)
    want, r0 = ops.quant_add_rmsnorm(x, op, res.clone(), w, 1e-6)
    got, r1 = ops.quant_add_rmsnorm(x, op, res.clone(), w, 1e-6, fp8=True)
    assert torch.equal(r0, r1)
    if M == 2:
        want, got = want[1:], ops.Fp8Rows(
            got.x[1:], got.q[1:], got.scales[:, 1:].contiguous())
    _same(got, want)


@pytest.mark.parametrize("M", [1, 17, 32, 33, 64])
@pytest.mark.parametrize("N", [36096, 36864, 16384, 36000])
def test_gated(M, N):
    from gllm_amd import ops
    torch.manual_seed(M + N)
    x = torch.randn(M, 256, device="cuda").bfloat16()
    x[M // 2] = 0                       # a row of smallest scales
    op = _fp8(N, 256)
    want = ops.quant_silu(x, op)
    got = ops.quant_silu(x, op, fp8=True)
    if M > 16 and N in (36096, 36864):  # whole groups in a tile
        _same(got, want)
    else:
        assert torch.equal(got, want)


@pytest.mark.parametrize("B,Hq,Hkv,lens", [
    (1, 32, 8, [600]), (3, 40, 8, [1, 33, 2000]),
    (64, 40, 8, [512 + 16 * i for i in range(64)]), (2, 16, 1, [70, 1500])])
def test_attention(B, Hq, Hkv, lens):
    from gllm_amd import ops
    s = _step(B, Hq, Hkv, 128, 128, 4, lens)
    arrived = torch.zeros(B * Hkv, dtype=torch.int32, device="cuda")
    args = [s[n] for n in ("parts", "bias", "positions", "cos_sin", "k", "v",
                           "slots", "table", "lens")]
    want = ops.qkv_decode(*args, arrived, Hq, 128 ** -0.5, rounded=True)
    got = ops.qkv_decode(*args, arrived, Hq, 128 ** -0.5, rounded=True,
                         fp8=True)
    _same(got, want)


def test_products_take_them():
    from gllm_amd import ops
    torch.manual_seed(0)
    x = torch.randn(20, 512, device="cuda").bfloat16()
    q, _, st = ops.per_token_group_quant_fp8(x, transposed=True)
    rows = ops.Fp8Rows(x, q.view(torch.uint8), st)
    op = _fp8(264, 512)
    assert torch.equal(ops.quant_rows(rows, op), ops.quant_rows(x, op))
    assert torch.equal(ops.quant_parts(rows, op), ops.quant_parts(x, op))
