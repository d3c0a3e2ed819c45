"""The native host side of decode, append_decode and write (csrc/kush_fastcall.cpp) against the Python path it
stands in for: the same bytes and outputs, with and without splits, order and waves, and the same exception with the
same text for every kind of argument that the checks refuse (each handed on to the Python path)."""
import types

import pytest
import torch

import kushkash_amd as kk
from test_gpu_append_decode import _state

pytestmark = pytest.mark.gpu
DEV, D, H, G = "cuda", 128, 2, 4
LENS = [40, 95, 31, 0, 700]


def _ops(native):
    ops = kk.Ops(torch.device(DEV), D, 4, G, torch.bfloat16, validate=False)
    assert ops._fast is not None, "build() makes _fastcall.so"
    if not native:
        ops._fast = None
    return ops


def _step(ops, ns):
    S = len(LENS)
    cache, bt, tail_k, tail_idx = _state(ops, LENS, H, D, torch.bfloat16, seed=4)
    g = torch.Generator().manual_seed(6)
    k, v, q = (torch.randn(S, h, D, generator=g).bfloat16().to(DEV) for h in (H, H, H * G))
    return dict(k=k, v=v, q=q, out=torch.empty_like(q), cache=cache, block_table=bt,
                seq_lens=torch.tensor([n + 1 for n in LENS], dtype=torch.int32, device=DEV), tail_idx=tail_idx,
                tail_k=tail_k, scale=0.09, n_splits=ns, work=torch.empty(S * H * ns * G * (D + 2), device=DEV))


@pytest.mark.parametrize("ns,waves,order,rot", [(1, None, False, False), (1, 2, True, True), (4, None, True, False),
                                                (8, 4, False, True)])
def test_the_same_calls(ns, waves, order, rot, monkeypatch):
    got = []
    for native in (True, False):
        ops = _ops(native)
        a = _step(ops, ns)
        opt = dict(waves=waves, rot=rot,
                   order=torch.arange(len(LENS), dtype=torch.int32, device=DEV).flip(0).contiguous() if order else None)
        calls, taken = [], []
        if native:                                               # the extension's answers: 0 is a launch of its own
            fast = ops._fast
            monkeypatch.setattr(ops, "_fast", types.SimpleNamespace(NOT_TAKEN=fast.NOT_TAKEN, **{
                n: lambda *x, f=getattr(fast, n): taken.append(f(*x)) or taken[-1] for n in ("decode", "write")}))
        monkeypatch.setattr(ops, "_decode", lambda *x: calls.append(x) or kk.Ops._decode(ops, *x))
        ops.append_decode(**a, **opt)
        first = a["out"].clone()
        ops.decode(**{n: x for n, x in a.items() if n not in "kv"}, **opt)
        assert len(calls) == (0 if native else 2)
        n = sum(LENS)
        js, jp = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in zip(*((s, p) for s, m in enumerate(LENS) for p in range(-(-m // 32)))))
        rows = torch.randn(n, H, D, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
        qsl = torch.tensor([0] + LENS, device=DEV).cumsum(0).to(torch.int32)
        ops.write(rows, rows.flip(0).contiguous(), qsl, torch.tensor(LENS, dtype=torch.int32, device=DEV), a["tail_idx"], js, jp,
                  a["cache"], a["block_table"], a["tail_k"], fused=True, rot=rot)
        assert taken == ([0, 0, 0] if native else [])
        got.append((first, a["out"], a["cache"], a["tail_k"]))
    assert all(torch.equal(x, y) for x, y in zip(*got))


REFUSED = {
    "q dtype": lambda a: a.update(q=a["q"].half()), "out shape": lambda a: a.update(out=a["out"][:2]),
    "k head stride": lambda a: a.update(k=a["k"].transpose(0, 1).contiguous().transpose(0, 1)),
    "short v": lambda a: a.update(v=a["v"][:1]), "lens dtype": lambda a: a.update(seq_lens=a["seq_lens"].long()),
    "short lens": lambda a: a.update(seq_lens=a["seq_lens"][:2]), "host lens": lambda a: a.update(seq_lens=a["seq_lens"].cpu()),
    "table dtype": lambda a: a.update(block_table=a["block_table"].long()),
    "tail shape": lambda a: a.update(tail_k=a["tail_k"][:, :, :16].contiguous()),
    "cache alignment": lambda a: a.update(cache=torch.zeros(a["cache"].numel() + 1, dtype=torch.uint8, device=DEV)[1:].view_as(a["cache"])),
    "small work": lambda a: a.update(n_splits=4, work=a["work"][:8]), "no work": lambda a: a.update(n_splits=2, work=None),
    "no splits": lambda a: a.update(n_splits=0), "waves": lambda a: a.update(waves=3),
    "short order": lambda a: a.update(order=torch.zeros(2, dtype=torch.int32, device=DEV)),
}


@pytest.mark.parametrize("what", sorted(REFUSED))
def test_the_same_errors(what):
    said = []
    for native in (True, False):
        ops = _ops(native)
        a = _step(ops, 1)
        REFUSED[what](a)
        with pytest.raises((ValueError, RuntimeError)) as e:
            ops.append_decode(**a)
        said.append((type(e.value), str(e.value)))
    assert said[0] == said[1]


@pytest.mark.parametrize("name", ["q", "seq_lens"])
def test_a_tensor_without_storage(name):
    """What torch.vmap passes is a torch.Tensor by type: refused as on the Python path, before any launch."""
    said = []
    for native in (True, False):
        ops = _ops(native)
        a = _step(ops, 1)
        with pytest.raises(RuntimeError) as e:
            torch.vmap(lambda x: ops.append_decode(**{**a, name: x}))(a[name][None])
        said.append(str(e.value))
    assert said[0] == said[1]
