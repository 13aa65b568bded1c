"""Whole latent-attention prompts in their per-head form against fp64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _attend(q, k, v, scale):
    """q [n, H, D] (the last n positions), k [m, G, D], v [m, G, E], fp64."""
    n, H, m, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    k, v = (t.repeat_interleave(H // G, 1) for t in (k, v))
    s = (q.transpose(0, 1) @ k.permute(1, 2, 0).contiguous()) * scale
    hide = torch.arange(m)[None] > torch.arange(m - n, m)[:, None]
    s = s.masked_fill(hide, -float("inf")).softmax(-1)
    return (s @ v.transpose(0, 1).contiguous()).transpose(0, 1)


@pytest.mark.parametrize("rows,H", [
    ([2], 1), ([63, 64, 65], 16), ([127, 129, 1000], 5), ([7] * 300, 2)])
def test_latent_prompts(rows, H):
    """The per-head form: the cache rows are the absorbed form's own, the
    result that of its definition."""
    from gllm_amd import ops
    torch.manual_seed(len(rows))
    T, dev = sum(rows), "cuda"
    q = torch.randn(T, H * 192).bfloat16().to(dev)
    kv = torch.randn(T, 576).bfloat16().to(dev)
    w = (torch.randn(H * 256, 512) * 512 ** -0.5).bfloat16().to(dev)
    norm = torch.rand(512).bfloat16().to(dev) + 0.5
    pos = torch.cat([torch.arange(n) for n in rows]).to(dev)
    ang = torch.arange(max(rows))[:, None] * 1e4 ** (-torch.arange(32) / 32)
    cos_sin = torch.cat([ang.cos(), ang.sin()], 1).float().to(dev)
    slots = torch.randperm(T // 16 * 16 + 32)[:T].to(dev)
    qsl = torch.tensor([0] + rows).cumsum(0).int().to(dev)
    caches = [torch.zeros(T // 16 + 2, 16, 1, 576, dtype=torch.bfloat16,
                          device=dev) for _ in range(2)]
    qf = ops.mla_queries(q, kv, norm, 1e-6, pos, cos_sin, w, caches[0],
                         slots)
    out = torch.full((T + 1, H * 128), 7.0, dtype=torch.bfloat16, device=dev)
    ops.mla_prompts(q, kv, norm, 1e-6, pos, cos_sin, w, caches[1], slots,
                    qsl, max(rows), 192 ** -0.5, out[:T])
    assert torch.equal(caches[0], caches[1]) and (out[T] == 7).all()
    assert torch.equal(q.view(T, H, 192)[..., 128:], qf[..., 512:])
    lat = caches[1].view(-1, 576)[slots].double().cpu()
    qd, wd = q.double().cpu().view(T, H, 192), w.double().cpu()
    heads = (lat[:, :512] @ wd.t()).view(T, H, 256)
    k = torch.cat([heads[..., :128],
                   lat[:, None, 512:].expand(T, H, 64)], -1)
    ref = torch.cat([_attend(qd[a:b], k[a:b], heads[a:b, :, 128:],
                             192 ** -0.5)
                     for a, b in zip(qsl.tolist(), qsl.tolist()[1:])])
    # keys and values are rounded to bf16 besides
    err = (out[:T].cpu().double().view(T, H, 128) - ref).norm() / ref.norm()
    assert err < 4 * 2 ** -9, err
