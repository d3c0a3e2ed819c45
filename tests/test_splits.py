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
