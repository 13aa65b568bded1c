"""Grouped products on 256-row blocks with operands of 2 GiB and more."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["gather", "scatter"])
def test_two_gib(form):
    from gllm_amd import ops
    torch.manual_seed(0)
    k, dev, E, T = ops._gpu_kernels(), "cuda", 3, (1 << 16) + 70
    wide, narrow = 1 << 14, 64
    ids = torch.randint(0, E, (T, 1), device=dev)
    ids32, tables, rows = ops._moe_tables(ids, E, 0, 256)
    place = torch.empty(T, dtype=torch.long, device=dev)  # of a pair's row
    pair = tables[0][:tables[2].item()].long()
    used = (pair < T).nonzero().flatten()
    place[pair[used]] = used
    at = torch.tensor([0, 1, 255, 256, T // 2, T - 256, T - 2, T - 1])
    if form == "gather":    # x [T, wide] past 2 GiB
        x = torch.randn(T, wide, dtype=torch.bfloat16, device=dev)
        w = torch.randn(E, narrow, wide, dtype=torch.bfloat16,
                        device=dev) * wide ** -0.5
        out = torch.empty(rows, narrow, dtype=torch.bfloat16, device=dev)
        k.moe_gemm_tiled(out, x, w, *tables, None, T, 1, 256, 3, 0.0, 0.0)
        out, x = out[place[at]], x[at.to(dev)]
    else:                   # the result [T, wide]
        act = torch.randn(rows, narrow, dtype=torch.bfloat16, device=dev)
        w = torch.randn(E, wide, narrow, dtype=torch.bfloat16,
                        device=dev) * narrow ** -0.5
        out = torch.empty(T, wide, dtype=torch.bfloat16, device=dev)
        k.moe_gemm_tiled(out, act, w, *tables, None, T, 1, 256, 0, 0.0, 0.0)
        out, x = out[at.to(dev)], act[place[at]]
    e = ids[at.to(dev), 0]
    ref = torch.stack([w[i].double() @ r.double() for i, r in zip(e, x)])
    if form == "gather":
        ref = ref.clamp_min(0) ** 2
    err = (out.double() - ref).abs()
    # one rounding to bf16 of fp32 sums (squared: twice their error)
    assert (err <= ref.abs() * 2 ** -8 * 1.02 + 1e-4).all(), err.max()
