"""The decode launch's own handling of a step's new token (the copies it keeps in LDS of a token that does not
complete its page) and of a rotated q, at the slots and sizes where they change path: the first and last slots
of a page, no full page at all, the table's prefetch bound, wave splits. Records, K tails and outputs equal the
append's and the decode's by themselves; a rotated decode equals the plain one on q rotated by Ops.fwht, its
output rotated back, within that output's own rounding."""
import pytest
import torch

import kushkash_amd as kk
from test_gpu_append_decode import _state

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [0, 1, 29, 30, 31, 32, 33, 62, 63, 64, 1300, 32767, 32768, 32800]     # before the token; 1,024 pages = the prefetch


@pytest.mark.parametrize("rot", [False, True])
@pytest.mark.parametrize("D,bits,dtype", [(64, 8, torch.float16), (64, 4, torch.float32), (128, 4, torch.bfloat16),
                                          (128, 8, torch.float32), (256, 4, torch.bfloat16), (256, 8, torch.float16)])
@pytest.mark.parametrize("G,ns,waves", [(3, 1, 4), (9, 1, 2), (8, 8, 4)])
def test_token_in_the_launch(D, bits, dtype, G, ns, waves, rot, monkeypatch):
    if ns > 1:
        monkeypatch.setenv("KUSHKASH_AMD_WAVE_SPLITS", "1")
    H, S = 1, len(LENS)
    ops = kk.Ops(torch.device(DEV), D, bits, G, dtype)
    states = [_state(ops, LENS, H, D, dtype, seed=D + bits) for _ in range(2)]
    g = torch.Generator().manual_seed(5)
    k, v, q = (torch.randn(S, h, D, generator=g).to(dtype).to(DEV) for h in (H, H, H * G))
    sl = torch.tensor([n + 1 for n in LENS], dtype=torch.int32, device=DEV)
    work = torch.empty(S * H * ns * G * (D + 2), dtype=torch.float32, device=DEV)
    outs = [torch.empty_like(q) for _ in range(2)]
    for i, (cache, bt, tail_k, tail_idx) in enumerate(states):
        args = (cache, bt, sl, tail_idx, tail_k, D ** -0.5, ns, work)
        if i == 0:
            ops.append_decode(k, v, q, outs[i], *args, waves=waves, rot=rot)
        else:
            ops.append(k, v, sl, tail_idx, cache, bt, tail_k, -1, False, rot=rot)
            ops.decode(q, outs[i], *args, waves=waves, rot=rot)
    assert torch.equal(states[0][0], states[1][0]) and torch.equal(states[0][2], states[1][2])
    assert torch.equal(outs[0], outs[1])
    if rot:
        plain = torch.empty_like(q)
        ops.decode(ops.fwht(q), plain, *args, waves=waves)
        back = ops.fwht(plain).float()
        # plain and back are each rounded to dtype (unit roundoff u), and a q entry on the edge between two values
        # may round the other way: within 4 u of the largest output
        u = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 2.0 ** -17}[dtype]
        assert (outs[1].float() - back).abs().max() <= 4 * u * back.abs().max() + 2 * u
