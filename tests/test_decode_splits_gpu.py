"""Decode attention from a projection's parts against fp64, in the ranges where
the number of splits depends on a sequence's length: sequences of very unlike
lengths, without keys, and on both sides of where a sequence is split."""

import pytest
import torch

from test_qkv_decode_gpu import _step

pytestmark = pytest.mark.gpu


def _reference(s, Hq, rounded):
    """fp64 attention over the rotated bf16 rows (that the caches and queries
    are those of the separate kernel is compared bit for bit elsewhere)."""
    from gllm_amd import ops
    k, v = s["k"].clone(), s["v"].clone()
    Hkv, D = k.shape[2:]
    q = ops.qkv_rope_cache(s["parts"], s["bias"], s["positions"],
                           s["cos_sin"], k, v, s["slots"], Hq,
                           rounded=rounded)
    q = q.view(-1, Hkv, Hq // Hkv, D).double()
    out = torch.zeros_like(q)
    for b, n in enumerate(s["lens"].tolist()):
        if n == 0:
            continue
        pages = s["table"][b, :-(-n // 16)].long()
        ks, vs = (c[pages].flatten(0, 1)[:n].double() for c in (k, v))
        for h in range(Hkv):
            p = (q[b, h] @ ks[:, h].t() * D ** -0.5).softmax(-1)
            out[b, h] = p @ vs[:, h]
    return out.flatten(1), k, v


CASES = [
    # a workgroup a CU: whole up to 8 tiles of 32, a split of 4 at least
    (1, 32, 8, 128, [3000]), (2, 16, 8, 64, [256, 257]),
    (2, 16, 8, 64, [4000, 1]), (2, 16, 8, 64, [0, 700]),
    # two a CU: up to 16, 8 at least
    (4, 40, 8, 128, [512, 513, 3900, 1]), (16, 32, 8, 128,
     [4000] + [100] * 14 + [0]), (32, 16, 8, 64, [544 + i for i in range(32)]),
    # more: up to 32, 24 at least
    (6, 16, 8, 128, [1024, 1025, 2049, 4090, 33, 0]),
    (24, 40, 8, 128, [4000, 3000, 0] + [60 * i + 1 for i in range(21)]),
    (31, 14, 2, 64, [4096] + [50] * 30),
    # sequences that nearly fill a round: up to 40
    (45, 8, 8, 128, [1280, 1281, 2561] + [30 * i for i in range(42)]),
    (60, 40, 8, 128, [4096, 0] + [100 + 20 * i for i in range(58)]),
    # one split
    (64, 16, 8, 128, [4000, 0] + [40] * 62)]


@pytest.mark.parametrize("rounded", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,D,lens", CASES)
def test_against_fp64(B, Hq, Hkv, D, lens, rounded):
    from gllm_amd import ops
    s = _step(B, Hq, Hkv, D, D, 3, lens)
    want, k, v = _reference(s, Hq, rounded)
    arrived = torch.zeros(B * Hkv, dtype=torch.int32, device="cuda")
    args = (s["positions"], s["cos_sin"], s["k"], s["v"], s["slots"],
            s["table"], s["lens"], arrived, Hq, D ** -0.5)
    got = ops.qkv_decode(s["parts"], s["bias"], *args, rounded=rounded)
    assert torch.equal(s["k"], k) and torch.equal(s["v"], v)
    assert not arrived.any()
    for b, n in enumerate(lens):
        if n == 0:
            assert not got[b].any()
        else:
            # weights and results are rounded to bf16 once each, 2^-9 relative
            err = (got[b].double() - want[b]).norm() / want[b].norm()
            assert err < 2 ** -7, (b, n, err)
    err = (got.double() - want).norm() / want.norm()
    assert err < 2 ** -8, err
    # another launch on the same counters: the same bits
    assert torch.equal(got, ops.qkv_decode(s["parts"], s["bias"], *args,
                                           rounded=rounded))


def test_fp8_rows_of_no_keys():
    from gllm_amd import ops
    lens = [0, 33, 700, 0]
    s = _step(4, 16, 2, 128, 128, 3, lens)
    arrived = torch.zeros(8, dtype=torch.int32, device="cuda")
    got = ops.qkv_decode(s["parts"], s["bias"], s["positions"], s["cos_sin"],
                         s["k"], s["v"], s["slots"], s["table"], s["lens"],
                         arrived, 16, 128 ** -0.5, rounded=True, fp8=True)
    q, _, st = ops.per_token_group_quant_fp8(got.x, transposed=True)
    assert torch.equal(got.scales, st)
    assert torch.equal(got.q, q.view(torch.uint8))
    assert not got.x[0].any() and not got.q[3].any()


@pytest.mark.parametrize("B,Hkv,rounded,ok", [
    # two rounds of workgroups of 256 CUs; rounded and split, one
    (128, 8, False, True), (129, 8, False, False), (128, 8, True, True),
    (129, 8, True, False), (33, 8, False, True), (33, 8, True, False),
    (32, 8, True, True)])
def test_limits(B, Hkv, rounded, ok):
    from gllm_amd import ops
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are counted in CUs")
    cache = torch.empty(1024, 16, Hkv, 64, dtype=torch.bfloat16,
                        device="cuda")
    parts = torch.empty(1, B, 3 * Hkv * 64, device="cuda")
    assert ops.qkv_decode_ok(parts, cache, Hkv, rounded) == ok
