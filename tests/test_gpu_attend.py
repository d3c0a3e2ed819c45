"""The prefill attention kernel (_attend.attend) against 64-bit attention at the edges of its tiles -- rows
and keys of one, a tile, a tile and one, a ragged last tile -- for every head size, dtype, workgroup size and
key split, with rows that are strided views; and what it leaves to the other paths."""
import math

import pytest
import torch

from kushkash_amd import _attend

DEV = "cuda"
# Relative 2-norm error of a correct kernel: the output's rounding and P's, u / sqrt(3) each for uniform rounding
# errors at unit roundoff u = 2^-9 (bf16) / 2^-12 (fp16), P's at most that of a single key; twice their sum
# leaves room for small samples.
BOUND = {torch.bfloat16: 4 * 2.0 ** -9 / math.sqrt(3), torch.float16: 4 * 2.0 ** -12 / math.sqrt(3)}


def _exact(q, k, v, causal, scale):
    """Attention and log-sum-exp of one sequence, q [T, Hq, D], k, v [N, Hk, D], in 64 bits."""
    T, N, G = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    qd, kd, vd = (x.double().cpu() for x in (q, k, v))
    s = torch.stack([qd[:, h] @ kd[:, h // G].t() for h in range(q.shape[1])], 1) * scale            # [T, Hq, N]
    if causal:
        s.masked_fill_((torch.arange(N)[None] > torch.arange(T)[:, None] + N - T)[:, None], -math.inf)
    p = torch.softmax(s, -1)
    return torch.stack([p[:, h] @ vd[:, h // G] for h in range(q.shape[1])], 1), torch.logsumexp(s, -1)


def _rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm()).item()


def _rows(shape, dt):
    """Rows that are a slice of wider ones (16-byte aligned)."""
    return torch.randn(*shape[:-2], shape[-2] + 1, shape[-1], device=DEV).to(dt)[..., 1:, :]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("T,N,Hk,G,causal", [
    (1, 1, 1, 1, True), (1, 64, 2, 3, True), (32, 65, 1, 4, True), (33, 63, 2, 4, False), (65, 200, 1, 7, True),
    (129, 130, 1, 2, True), (9, 1000, 2, 16, False), (300, 300, 1, 1, True)])
def test_attention_at_tile_edges(D, dtype, T, N, Hk, G, causal, monkeypatch):
    torch.manual_seed(T * N + D)
    B, scale = 2, D ** -0.5
    q, k, v = _rows((B, T, Hk * G, D), dtype), _rows((B, N, Hk, D), dtype) * 2, _rows((B, N, Hk, D), dtype)
    assert _attend.takes(q, k, v, scale)
    want = [_exact(q[b], k[b], v[b], causal, scale) for b in range(B)]
    for waves, chunk in ((4, 0), (8, 0), (4, 1), (8, 3), (4, 5)):
        print(D, dtype, T, N, Hk, G, causal, waves, chunk, flush=True)
        monkeypatch.setattr(_attend, "plan", lambda *a: (waves, chunk))
        out = _attend.attend(q, k, v, causal, scale)
        out32, lse = _attend.attend(q, k, v, causal, scale, lse=True)
        assert out.dtype == dtype and out.shape == q.shape and out32.dtype == torch.float32
        for b in range(B):
            assert _rel(out[b], want[b][0]) < BOUND[dtype]
            assert _rel(out32[b], want[b][0]) < BOUND[dtype]
            # log of a sum of weights each rounded to dtype (relative u) and fp32 scores (a few 1e-6)
            assert (lse[b].double().cpu() - want[b][1]).abs().max() < BOUND[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("chunk", [0, 2])
def test_ragged_rows(chunk, monkeypatch):
    torch.manual_seed(3)
    T, N = [5, 64, 1, 200, 17], [5, 300, 129, 200, 1017]
    Hk, G, D, scale = 2, 4, 128, 0.11
    q, k, v = (torch.randn(sum(n), h, D, device=DEV).bfloat16() for n, h in ((T, Hk * G), (N, Hk), (N, Hk)))
    cu = [torch.tensor([0] + x, device=DEV).cumsum(0).to(torch.int32) for x in (T, N)]
    monkeypatch.setattr(_attend, "plan", lambda *a: (4, chunk))
    out = torch.empty_like(q)
    got = _attend.attend(q, k, v, True, scale, cu=(*cu, max(T), max(N)), spans=list(zip(T, N)), out=out)
    assert got is out
    for i in range(len(T)):
        a, b, c, d = *cu[0][i:i + 2].tolist(), *cu[1][i:i + 2].tolist()
        assert _rel(out[a:b], _exact(q[a:b], k[c:d], v[c:d], True, scale)[0]) < BOUND[torch.bfloat16], i


@pytest.mark.gpu
def test_inputs_left_to_the_other_paths():
    def rows(D=128, dt=torch.bfloat16):
        return [torch.randn(1, 8, 2, D, device=DEV).to(dt) for _ in range(3)]

    q, k, v = rows()
    assert _attend.takes(q, k, v, 0.1)
    assert not _attend.takes(*rows(96), 0.1) and not _attend.takes(*rows(dt=torch.float32), 0.1)
    assert not any(_attend.takes(q, k, v, s) for s in (0.0, -1.0, math.inf, math.nan))
    assert not _attend.takes(torch.randn(1, 8, 2, 129, device=DEV).bfloat16()[..., 1:], k, v, 0.1)    # misaligned
    assert not _attend.takes(q, k.half(), v, 0.1) and not _attend.takes(q, k[..., :64], v[..., :64], 0.1)
    assert not _attend.takes(q, k[:, :1].expand(1, 8, 2, 128), v, 0.1)                                # rows that repeat
    assert not _attend.takes(q.requires_grad_(), k, v, 0.1)
    with torch.no_grad():
        assert _attend.takes(q, k, v, 0.1)


def _same(got, want, bound):
    """NaN in the same places, the rest within the bound."""
    got = got.double().cpu()
    assert torch.equal(got.isnan(), want.isnan())
    at = ~want.isnan()
    assert not at.any() or ((got[at] - want[at]).norm() / want[at].norm()).item() < bound


@pytest.mark.gpu
@pytest.mark.parametrize("waves,chunk", [(4, 0), (8, 0), (4, 1), (8, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("what", ["nan key", "inf key", "-inf keys", "no finite score", "nan query", "nan value"])
def test_values_that_are_not_finite(what, dtype, waves, chunk, monkeypatch):
    """Causal, 150 queries over 200 keys: a NaN score makes the rows that see it NaN and no other, +inf too, -inf scores
    weigh nothing, a row of nothing else is NaN with log-sum-exp -inf, and a query's NaN stays in its row."""
    torch.manual_seed(11)
    T, N, Hk, G, D, scale = 150, 200, 2, 2, 128, 0.09
    q, k, v = (torch.randn(1, n, h, D, device=DEV).to(dtype) for n, h in ((T, Hk * G), (N, Hk), (N, Hk)))
    q[..., 5] = q[..., 5].abs() + 0.5                                   # an infinite k[..., 5] gives scores of its sign
    if what == "nan key":
        k[:, 130, 1, 7] = math.nan
    elif what == "inf key":
        k[:, 130, 1, 5] = math.inf
    elif what == "-inf keys":
        k[:, 20:128, 0, 5] = -math.inf                                  # a whole key tile among them
    elif what == "no finite score":
        k[:, :, 0, 5] = -math.inf
    elif what == "nan query":
        q[:, 77, 3, 64] = math.nan
    else:
        v[:, 190, 0, 3] = math.nan
    monkeypatch.setattr(_attend, "plan", lambda *a: (waves, chunk))
    out = _attend.attend(q, k, v, True, scale)
    out32, lse = _attend.attend(q, k, v, True, scale, lse=True)
    want, logs = _exact(q[0], k[0], v[0], True, scale)
    if what == "nan value":
        # the product of a zero weight and NaN is NaN: what rows that do not see the key hold is not defined (a tile's
        # rows have it, others not); those that see it are NaN in that dim, and all other dims are whole
        assert out[0, 140:, :G, 3].isnan().all()
        keep = [d for d in range(D) if d != 3]
        out, out32, want = out[..., keep], out32[..., keep], want[..., keep]
    _same(out[0], want, BOUND[dtype])
    _same(out32[0], want, BOUND[dtype])
    finite = logs.isfinite()
    # (of a row with a +inf score, whose output is NaN, the kernel's is inf - inf, 64 bits' is inf: neither is used)
    assert torch.equal(lse[0].cpu().isfinite(), finite) and torch.equal(lse[0].cpu() == -math.inf, logs == -math.inf)
    assert (lse[0].double().cpu()[finite] - logs[finite]).abs().max() < BOUND[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(2,), (0,), (0, 2)])
def test_rows_that_repeat_over_heads_or_batches(dims):
    """k and v expanded over heads or batches (strides of 0), and q over batches."""
    torch.manual_seed(12)
    B, T, N, Hk, G, D, scale = 3, 70, 130, 2, 3, 64, 0.1
    q = torch.randn(1 if 0 in dims else B, T, Hk * G, D, device=DEV).bfloat16().expand(B, -1, -1, -1)
    k, v = (torch.randn(*(1 if i in dims else n for i, n in enumerate((B, N, Hk))), D, device=DEV).bfloat16().expand(B, N, Hk, D)
            for _ in range(2))
    assert _attend.takes(q, k, v, scale)
    out = _attend.attend(q, k, v, True, scale)
    for b in range(B):
        assert _rel(out[b], _exact(q[b], k[b], v[b], True, scale)[0]) < BOUND[torch.bfloat16]


@pytest.mark.gpu
def test_split_keys_in_a_captured_graph():
    """A call whose keys are split (partials from the allocator, a second launch), replayed on new inputs with eager work
    between: the eager call's bits each time."""
    torch.manual_seed(13)
    T, N, Hk, G, D, scale = 40, 4000, 2, 4, 128, 0.09
    rows = [torch.randn(1, n, h, D, device=DEV).bfloat16() for n, h in ((T, Hk * G), (N, Hk), (N, Hk))]
    assert _attend.plan(((T, N, 1),), G, Hk, D, T)[1] > 0
    _attend.attend(*rows, True, scale)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        out = _attend.attend(*rows, True, scale)
    for _ in range(4):
        for x in rows:
            x.copy_(torch.randn_like(x))
        want = _attend.attend(*rows, True, scale)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_a_trace_is_not_plain():
    """torch.jit.trace records torch's operators only: under it nothing is the kernel's."""
    x, seen = torch.randn(2, 4), []
    torch.jit.trace(lambda t: seen.append(_attend._plain(t)) or t + 1, x, check_trace=False)
    assert seen == [False] and _attend._plain(x)


@pytest.mark.gpu
def test_a_traced_prompt_attends_its_own_inputs():
    """(One q head per kv head: torch cannot trace repeat_interleave, which the path left to torch needs for more.)"""
    from kushkash_amd.hf import prompt_attention
    torch.manual_seed(7)
    first, second = ([torch.randn(1, h, 70, 128, device=DEV).bfloat16() for h in (2, 2, 2)] for _ in range(2))
    traced = torch.jit.trace(lambda q, k, v: prompt_attention(q, k, v, 0.09), first, check_trace=False)
    for x in (first, second):
        want = _exact(*(t[0].transpose(0, 1) for t in x), True, 0.09)[0].transpose(0, 1)
        assert _rel(traced(*x)[0], want) < BOUND[torch.bfloat16]


@pytest.mark.gpu
@pytest.mark.parametrize("N", [40, 64, 100, 150])
def test_a_prompt_over_keys_of_another_length(N):
    """prompt_attention with more or fewer keys than queries: query t sees keys 0 .. t, as the paths around the kernel
    have it (the kernel aligns the queries with the last keys, and takes no causal call of fewer keys than queries)."""
    from kushkash_amd.hf import prompt_attention
    torch.manual_seed(N)
    T, scale = 100, 0.09
    q, k, v = (torch.randn(1, h, n, 128, device=DEV).bfloat16() for h, n in ((4, T), (2, N), (2, N)))
    got = prompt_attention(q, k, v, scale)
    s = torch.stack([q[0, h].double().cpu() @ k[0, h // 2].double().cpu().t() for h in range(4)]) * scale
    s.masked_fill_(torch.arange(N) > torch.arange(T)[:, None], -math.inf)
    p = torch.softmax(s, -1)
    want = torch.stack([p[h] @ v[0, h // 2].double().cpu() for h in range(4)])
    assert got.dtype == q.dtype and _rel(got[0], want) < BOUND[torch.bfloat16]


@pytest.mark.gpu
@pytest.mark.parametrize("history", [0, 75])
@pytest.mark.parametrize("N", [20, 50])
def test_a_chunk_of_more_or_fewer_keys_than_queries(history, N):
    """attend_chunk where k and v do not hold one row per query: every query sees the whole history, and the chunk's keys
    up to N - T + t, as before the history and the chunk were attended in one call."""
    import kushkash_amd as kk
    torch.manual_seed(history + N)
    T, H, G = 33, 2, 2
    c = kk.KushCache(1, H, H * G, 128, bits=8, device=DEV, dtype=torch.bfloat16, rotate=False)
    hk, hv = torch.zeros(2, H, 0, 128, dtype=torch.float64)
    if history:
        c.write(0, *(torch.randn(1, H, history, 128, device=DEV).bfloat16() for _ in range(2)))
        hk, hv = (x[0].double().cpu() for x in c.dequantize(0))
    q, k, v = (torch.randn(1, h, n, 128, device=DEV).bfloat16() for h, n in ((H * G, T), (H, N), (H, N)))
    got = c.attend_chunk(0, q, k, v)[0]
    keys, vals = (torch.cat([h, x[0].double().cpu()], 1).repeat_interleave(G, 0) for h, x in ((hk, k), (hv, v)))
    s = q[0].double().cpu() @ keys.transpose(1, 2) * c.scale
    s[:, :, history:].masked_fill_(torch.arange(N) > torch.arange(T)[:, None] + N - T, -math.inf)
    want = torch.nan_to_num(torch.softmax(s, -1)) @ vals                # (no key at all: 0)
    # the blocks' outputs are rounded to bf16 before their merge: one rounding more
    assert _rel(got, want) < 1.5 * BOUND[torch.bfloat16]


@pytest.mark.parametrize("G", [1, 4, 7, 16])
def test_the_plan_covers_the_keys_and_bounds_its_scratch(G):
    """Whatever the shape: 4 or 8 waves, a split (if any) of at least 12 key tiles that leaves more than one
    part, within the scratch bound, and no split where the row tiles fill the chip evenly."""
    for D in (64, 128, 256):
        for hkv in (1, 8):
            for T, N, c in ((1, 1, 1), (16, 8016, 1), (256, 8256, 4), (2048, 34816, 1), (3001, 3001, 2), (1, 200000, 64)):
                waves, chunk = _attend.plan(((T, N, c),), G, hkv, D, T * c)
                nt = -(-N // 64)
                assert waves in ((4, 8) if D < 256 else (4,)) and (chunk == 0 or 12 <= chunk < nt)
                if chunk:
                    assert -(-nt // chunk) * T * c * hkv * G * (D + 2) * 4 <= 2 * _attend.PARTIAL_BYTES
    assert _attend.plan(((3001, 3001, 2),), 7, 4, 128, 6002) == (4, 0)
    assert _attend.plan(((2048, 34816, 1),), 4, 8, 128, 2048) == (8, 0)


# spans, q heads per kv head, kv heads, D: splitting the keys measured slower than whole, or at least 1.2 times as fast
@pytest.mark.parametrize("spans,G,hkv,D,split", [
    ([(2048, 2048, 1)], 4, 8, 128, False), ([(2048, 2048, 1)], 4, 8, 64, False), ([(3072, 3072, 1)], 4, 8, 128, False),
    ([(1600, 1600, 1)], 4, 8, 256, False), ([(2826, 2826, 4)], 2, 4, 128, False), ([(4225, 4225, 1)], 12, 2, 128, False),
    ([(256, 8000, 1)], 4, 8, 128, True), ([(512, 34816, 1)], 4, 8, 128, True), ([(1280, 8192, 1)], 4, 8, 64, True),
    ([(64, 34816, 4)], 4, 8, 128, True), ([(41, 34187, 1)], 7, 1, 128, True), ([(239, 10522, 1)], 4, 8, 256, True), ([(512, 1600, 1)], 4, 8, 256, True)])
def test_the_plan_splits_keys_where_that_pays(spans, G, hkv, D, split):
    assert (_attend.plan(spans, G, hkv, D, sum(t * c for t, _, c in spans))[1] > 0) == split


def test_the_plan_keeps_its_partials_within_the_scratch():
    """Every part's rows together within PARTIAL_BYTES, and within what the caller gives where that is less."""
    split = 0
    for D in (64, 128, 256):
        for G, hkv in ((1, 1), (4, 8), (16, 2)):
            for T in (1, 16, 100, 256, 500, 700, 1100):
                for N in (1600, 8000, 34816, 200000):
                    for c in (1, 3):
                        for scratch in (1 << 30, 1 << 28, 1 << 24, 1 << 20, 0):
                            waves, chunk = _attend.plan(((T, N, c),), G, hkv, D, T * c, False, scratch)
                            parts = -(-(-(-N // 64)) // chunk) if chunk else 0
                            assert parts * T * c * hkv * G * (D + 2) * 4 <= min(scratch, _attend.PARTIAL_BYTES)
                            split += parts > 1
    assert split > 100
    # one long sequence among many rows: half its keys' partials are 1.2 times the bound
    assert _attend.plan([(1000, 15000, 1), (1000, 1000, 9)], 4, 8, 128, 10000) == (4, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["chunk", "first chunk", "prompt"])
def test_split_keys_within_block_bytes(what, monkeypatch):
    """The callers' memory bound reaches the plan: no partials past it, and the answer stays."""
    import kushkash_amd as kk
    from kushkash_amd.hf import prompt_attention
    torch.manual_seed(2)
    T = 512 if what == "chunk" else 1700
    q, k, v = (torch.randn(1, h, T, 128, device=DEV).bfloat16() for h in (8, 2, 2))
    c = kk.KushCache(1, 2, 8, 128, bits=8, device=DEV, dtype=torch.bfloat16)
    if what == "chunk":
        c.write(0, *(torch.randn(1, 2, 4096, 128, device=DEV).bfloat16() for _ in range(2)))
    plans = []
    real = _attend.plan
    monkeypatch.setattr(_attend, "plan", lambda *a: plans.append((a, real(*a))) or plans[-1][1])
    outs = []
    for bound in (1 << 28, 1 << 22):
        plans.clear()
        outs.append(prompt_attention(q, k, v, 0.09, bound) if what == "prompt" else c.attend_chunk(0, q, k, v, bound))
        for a, (waves, chunk) in plans:
            nt = -(-max(n for _, n, _ in a[0]) // 64)
            assert (-(-nt // chunk) if chunk else 0) * a[4] * 8 * 130 * 4 <= bound and plans
    assert _rel(outs[0], outs[1].double().cpu()) < 3 * BOUND[torch.bfloat16]


@pytest.mark.parametrize("T,waves", [(2048, 8), (3584, 8), (4096, 8), (6144, 8), (2049, 4), (2176, 4), (3072, 4), (4352, 4)])
def test_the_plan_takes_8_waves_for_full_rounds(T, waves):
    """Over many keys, 8-wave workgroups only where their last round of row tiles fills most of the chip."""
    assert _attend.plan(((T, 34816, 1),), 4, 8, 128, T)[0] == waves


@pytest.mark.parametrize("T,N", [(8192, 2016), (4096, 2048), (3000, 1600), (70000, 20000)])
def test_the_plan_of_an_unmasked_call_counts_every_key(T, N):
    """Without a mask all rows see all keys, also where there are more rows than keys: row tiles that fill the chip take
    them whole (8,192 rows over 2,016 keys, 4 x 8 heads: 311 us, 387 with its keys split)."""
    assert _attend.plan(((T, N, 1),), 4, 8, 128, T, False)[1] == 0


def test_kernels_keep_their_wait_states(tmp_path):
    """On the assembly: every read or overwrite of a 32x32x16 MFMA's result waits, on every control-flow path,
    the 12 states that the compiler keeps in straight-line code (a branch join once broke this in the
    decode), and m0 is only the LDS DMA's base, one wait state ahead of its load."""
    import re
    import shutil
    import subprocess
    from pathlib import Path

    import test_isa
    from kushkash_amd.build import FLAGS, ROOT
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    subprocess.run([hipcc, *(f for f in FLAGS if f not in ("-shared", "-fPIC")), f"-I{ROOT / 'include'}", "-S",
                    "--cuda-device-only", str(ROOT / "kushkash_amd/csrc/kush_attend.hip"), "-o",
                    str(tmp_path / "a.s")], check=True, capture_output=True)
    text = (tmp_path / "a.s").read_text().replace("13attend_kernel", "13decode_kernel")     # as kernels() finds them
    found = test_isa.kernels(text)
    assert len(found) == 10                                                # 3 head sizes x 2 dtypes, 8 waves for two
    need = dict(test_isa.MFMA_WAIT, v_mfma_f32_32x32x16_bf16=12, v_mfma_f32_32x32x16_f16=12)
    for name, lines in found.items():
        saved = dict(test_isa.MFMA_WAIT)
        test_isa.MFMA_WAIT.update(need)
        try:
            assert not test_isa.mfma_short_paths(lines), name
        finally:
            test_isa.MFMA_WAIT.clear()
            test_isa.MFMA_WAIT.update(saved)
        live = [l for l in lines if l]
        for i, ins in enumerate(live):
            if "m0" in ins:
                assert re.match(r"s_mov_b32 m0, s\d+$", ins) and live[i + 1] == "s_nop 0" and live[i + 2].endswith(" lds"), ins
