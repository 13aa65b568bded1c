"""int4 products of small weights by waves, of larger ones by pairs."""

import pytest

from test_quant_gemm_gpu import close, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    # 20 M values, and a column or a group less
    (1, 4096, 5120), (16, 4095, 5120), (16, 4088, 5120), (7, 4096, 4864),
    (9, 10240, 2048), (16, 10232, 2048)])
def test_int4(M, N, K):
    from gllm_amd import ops
    x, op, ref, size = make("int4", M, N, K)
    close(ops.quant_rows(x, op), ref, size)
    if N % 8 == 0:
        close(ops.quant_parts(x, op).sum(0), ref, size, bf16=False)
