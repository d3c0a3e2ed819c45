"""Ops.splits over batches, heads, lengths and record formats: every split keeps two pages per wave, the grid
stays within two workgroups per CU (the work-buffer bound), one split where the pairs fill the CUs, and every
workgroup resident at once where a page ring takes over half a CU's LDS."""
import pytest

from kushkash_amd import Ops, record_bytes
from kushkash_amd._ops import DECODE_WAVES


@pytest.mark.parametrize("D,bits,G", [(128, 4, 4), (128, 8, 4), (64, 8, 2), (256, 4, 16), (256, 8, 4), (128, 4, 20)])
def test_split_policy(D, bits, G):
    ops = Ops.__new__(Ops)
    ops.D, ops.bits, ops.G, ops.gpu, ops.sms = D, bits, G, True, 256
    single = 16 * record_bytes(D, bits) + 4096 > 80 * 1024
    chunks = -(-G // 16)
    for pairs in [*range(1, 40), 63, 64, 100, 128, 144, 160, 200, 255, 256, 700]:
        for pages in (0, 1, 7, 8, 40, 125, 1000, 4096):
            ns = ops.splits(pairs, 1, pages)
            assert 1 <= ns <= 256 and (ns == 1 or pages // ns >= 2 * DECODE_WAVES)
            assert pairs * ns <= max(pairs, 2 * ops.sms)
            if pairs * chunks >= ops.sms:
                assert ns == 1
            if G > 16:
                assert ns & (ns - 1) == 0
            if single:
                assert ns == 1 or pairs * chunks * ns <= ops.sms
    assert ops.splits(0, 8, 100) == 1
    assert ops.splits(8, 8, 4096) == (4 if chunks == 1 else 2)


# sequences, kv heads, D, bits, tokens and the counts within a few percent of the fastest one, as measured
@pytest.mark.parametrize("S,H,D,bits,tokens,good", [
    (12, 4, 128, 4, 1000, (2, 3)), (4, 8, 128, 4, 4096, (8,)), (2, 8, 128, 4, 131072, (16,)),
    (1, 8, 128, 4, 131072, (26, 32)), (8, 8, 128, 4, 131072, (3, 4)), (3, 8, 64, 4, 32768, (10, 21)),
    (2, 8, 64, 4, 65536, (16,)), (1, 4, 256, 8, 4096, (8, 16)), (34, 2, 128, 8, 721, (1,))])
def test_small_batches_fill_the_chip(S, H, D, bits, tokens, good):
    ops = Ops.__new__(Ops)
    ops.D, ops.bits, ops.G, ops.gpu, ops.sms = D, bits, 4, True, 256
    assert ops.splits(S, H, tokens // 32) in good


@pytest.mark.gpu
@pytest.mark.parametrize("D,bits,G,waves", [(128, 4, 7, 4), (128, 8, 4, 2), (256, 4, 16, 4), (64, 8, 2, 4)])
@pytest.mark.parametrize("ns", [3, 5, 6, 7, 13])
def test_any_split_count(D, bits, G, waves, ns):
    """A step's append and decode in any number of splits, splits without pages and the token's page in any of them:
    records and tails equal, outputs as in one split within their roundings."""
    import torch
    from test_gpu_append_decode import _state
    lens = [0, 31, 95, 96, 160, 700, 1311, 2559]                        # before the token
    S, H, dev = len(lens), 2, "cuda"
    ops = Ops(torch.device(dev), D, bits, G, torch.bfloat16)
    g = torch.Generator().manual_seed(ns)
    k, v, q = (torch.randn(S, h, D, generator=g).to(torch.bfloat16).to(dev) for h in (H, H, H * G))
    sl = torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=dev)
    got = []
    for n in (1, ns):
        cache, bt, tail_k, tail_idx = _state(ops, lens, H, D, torch.bfloat16, seed=D + bits)
        out, work = torch.empty_like(q), torch.empty(S * H * n * G * (D + 2), device=dev)
        ops.append_decode(k, v, q, out, cache, bt, sl, tail_idx, tail_k, D ** -0.5, n, work, waves=waves)
        got.append((cache, tail_k, out.float()))
    (c1, t1, a), (c2, t2, b) = got
    assert torch.equal(c1, c2) and torch.equal(t1, t2)
    # a weight is rounded to fp16 once per launch, relative to another split's largest score (unit roundoff 2^-11, two
    # launches, values' code part below 6), and each output once to bf16 (2^-8 of it, both)
    assert ((a - b).abs() <= 2 * 2.0 ** -11 * 6 + 2.0 ** -7 * torch.maximum(a.abs(), b.abs())).all()
