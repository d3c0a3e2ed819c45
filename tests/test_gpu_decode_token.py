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


@pytest.mark.parametrize("rot", [False, True])
@pytest.mark.parametrize("D,bits,dtype", [(64, 8, torch.float16), (128, 4, torch.bfloat16), (128, 8, torch.float32),
                                          (256, 4, torch.float32)])
def test_tokens_of_special_values(D, bits, dtype, rot):
    """A new token of zeros of both signs, equal values, one outlier, subnormals, values whose range overflows fp16, and
    infinities and NaN in K or V: the bytes and outputs of the append and the decode by themselves."""
    kinds = ["zeros", "signed zeros", "equal", "outlier", "subnormal", "huge", "inf", "nan", "all nan", "-inf all"]
    H, S, G = 2, 2 * len(kinds), 4
    ops = kk.Ops(torch.device(DEV), D, bits, G, dtype)
    lens = [37 + s for s in range(S)]                                    # never a completed page: 38 .. 57 tokens
    g = torch.Generator().manual_seed(9)
    k, v, q = (torch.randn(S, h, D, generator=g).to(dtype) for h in (H, H, H * G))
    big = 3e4 if dtype == torch.float16 else 3e30
    for i, kind in enumerate(kinds):
        for x, s in ((k, 2 * i), (v, 2 * i + 1)):
            if kind == "zeros":
                x[s] = 0
            elif kind == "signed zeros":
                x[s] = torch.where(torch.arange(D) % 3 == 0, -0.0, 0.0).to(dtype)
            elif kind == "equal":
                x[s] = -1.25
            elif kind == "outlier":
                x[s, :, D - 1] = 300
            elif kind == "subnormal":
                x[s] = x[s] * torch.finfo(dtype).smallest_normal / 4
            elif kind == "huge":
                x[s] = torch.where(torch.arange(D) % 2 == 0, -big, big).to(dtype)
            elif kind == "inf":
                x[s, :, 3] = float("inf")
            elif kind == "nan":
                x[s, :, D // 2 + 1] = float("nan")
            else:
                x[s] = float("nan") if kind == "all nan" else float("-inf")
    k, v, q = (x.to(DEV) for x in (k, v, q))
    sl = torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=DEV)
    got = []
    for fused in (True, False):
        cache, bt, tail_k, tail_idx = _state(ops, lens, H, D, dtype, seed=D)
        out = torch.empty_like(q)
        args = (cache, bt, sl, tail_idx, tail_k, D ** -0.5)
        if fused:
            ops.append_decode(k, v, q, out, *args, rot=rot)
        else:
            ops.append(k, v, sl, tail_idx, cache, bt, tail_k, -1, False, rot=rot)
            ops.decode(q, out, *args, rot=rot)
        got.append((cache, tail_k, out))
    raw = {2: torch.int16, 4: torch.int32}[k.element_size()]
    (c0, t0, o0), (c1, t1, o1) = got
    # a NaN is a NaN, whatever its sign and payload: in the K tail, in a record's scales and biases, and in an output
    same = (t0.view(raw) == t1.view(raw)) | (t0.isnan() & t1.isnan())
    assert bool(same.all())
    codes = c0.shape[-1] - 4 * D - 128
    assert torch.equal(c0[..., :codes], c1[..., :codes])
    m0, m1 = (c[..., codes:].contiguous().view(torch.float16) for c in (c0, c1))
    assert bool(((m0.view(torch.int16) == m1.view(torch.int16)) | (m0.isnan() & m1.isnan())).all())
    assert bool(((o0 == o1) | (o0.isnan() & o1.isnan())).all())
