"""The prefill attention kernel (csrc/kush_attend.hip, include/kushkash_amd_attend.h): which inputs it takes,
how a call is spread over the chip, and the call. Half-precision rows on the GPU, any batch and row strides,
GQA, causal with the queries at the end of the keys or not, ragged rows packed end to end; forward only.
Reference: the varlen flash attention of kushkash/vllm/backend.py:837-880."""
from __future__ import annotations

import ctypes
import math

import torch

from . import _lib

CUS = 256                        # MI355X compute units
KEYS = 64                        # keys per tile
PARTIAL_BYTES = 1 << 28          # at most this much scratch for split keys
SLOTS = {64: 4 * CUS, 128: 2 * CUS, 256: CUS}       # 4-wave workgroups the chip holds at once, by head_dim
TILE_US = {64: 1.26, 128: 2.14, 256: 2.88}          # a key tile's time with all of them taken
_Strides = ctypes.c_int64 * 15
# torch.jit.trace, a vmap / grad / functionalize level, and dispatch modes (read on every call)
_tracing, _transform, _modes = (torch._C._get_tracing_state, torch._C._functorch.peek_interpreter_stack,
                                torch._C._len_torch_dispatch_stack)


def _plain(*ts: torch.Tensor) -> bool:
    """Whether the tensors are what a kernel can be handed: no subclass, no tracing or transform around
    them, and no derivative asked for (the kernel has none)."""
    if any(type(t) not in (torch.Tensor, torch.nn.Parameter) for t in ts):
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        return False
    return not (torch.compiler.is_compiling() or _tracing() is not None or _transform() is not None or _modes()
                or torch.autograd.forward_ad._current_level >= 0)


def _row_strides(t: torch.Tensor, D: int) -> tuple[int, int, int]:
    """(batch, row, head) strides of [.., rows, heads, D]; a dim of one entry counts as packed."""
    st = [0 if t.dim() == 3 or t.shape[0] == 1 else t.stride(0), t.stride(-3), t.stride(-2)]
    if t.shape[-3] == 1:
        st[1] = D
    if t.shape[-2] == 1:
        st[2] = D
    return tuple(st)


def takes(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> bool:
    """Whether the kernel takes q [B, T, Hq, D] (or packed [rows, Hq, D]) over k, v [B, N, Hk, D]: anything
    else is the caller's other paths' (torch's flash kernel, fp32 products)."""
    D = q.shape[-1]
    if (not q.is_cuda or q.dtype not in (torch.bfloat16, torch.float16) or D not in (64, 128, 256)
            or not (k.dtype == v.dtype == q.dtype and k.device == v.device == q.device)
            or not (0.0 < scale < math.inf) or k.shape != v.shape or k.shape[-1] != D or q.dim() != k.dim()
            or (q.dim() == 4 and q.shape[0] != k.shape[0]) or not _plain(q, k, v)):
        return False
    T, Hq, Hk = q.shape[-3], q.shape[-2], k.shape[-2]
    if not q.numel() or not k.numel() or Hq % Hk or T * (Hq // Hk) > 1 << 22 or k.shape[-3] > 1 << 30:
        return False
    for t in (q, k, v):
        st = _row_strides(t, D)
        if t.stride(-1) != 1 or t.data_ptr() % 16 or any(s % 8 or s < 0 for s in st):
            return False
        if t is not q and not D <= st[1] <= 1 << 23:
            return False
    return True


def plan(spans, group: int, hkv: int, D: int, total_q: int, causal: bool = True,
         scratch: int = PARTIAL_BYTES) -> tuple[int, int]:
    """(waves, chunk) of a call whose sequences have (T, N, count) query rows and keys. A row tile is 32 waves
    query rows (group heads of each token) of one kv head; 4 waves fill half a CU (a whole one at D 256, a
    quarter at D 64), 8 a whole one.
      8 waves  share each K / V tile among twice the rows, one workgroup to a CU: 1,048 us against 1,097 at 2,048
               tokens x 4 heads over 34,816 keys (8 kv heads, D 128), 3-7 % less from 16,384 keys on at D 64 and 128;
               at 8,192 keys between 2 % more and 4 % less, and 6-20 % more at 2,048. Only where the last round of row
               tiles fills the chip: 3,584 tokens (448 row tiles, 0.88 of two rounds) 1,843 us against 1,996, 3,072
               (384, 0.75) 1,811 against 1,647, 2,176 (272, 0.53) 1,836 against 1,573.
      chunk    split the keys of a row tile where the row tiles leave the chip idle, into as many parts as fill it
               (256 tokens over 8,000 keys: 162 -> 68 us), or, where the longest would run on alone, into
               halves (nine chunks of 61-395 tokens over 800-8,300 keys: 295 -> 268 us), if that gains more than the
               partials cost: half of what the longest row tile is over an even share (the workgroups left have
               more of a CU by then; 0.7 at D 256, one workgroup to a CU) against their bytes out and in at 2.5
               TB/s. The constants are from 700 drawn calls of both sides; without the condition 118 of them were
               2-32 % slower than whole (3,072 tokens over themselves: 101 -> 129 us, 2,048 at D 64: 43 -> 52), with
               it 7 (up to 13 %), and 9 of the splits that it leaves out would have gained 2-13 %.
               Not below 24 tiles (1,000 tokens over themselves: 31 us whole, 31-34 split), and into no more parts
               than min(scratch, PARTIAL_BYTES) holds the partials of."""
    longest = max([n for _, n, _ in spans])
    nt = -(-longest // KEYS)
    if nt < 24:
        return 4, 0
    if D <= 128 and longest >= 16384:
        wide = sum(c * (-(-t * group // 256)) for t, _, c in spans) * hkv              # row tiles of 8 waves
        if wide >= CUS and wide >= 0.8 * CUS * -(-wide // CUS):
            return 8, 0
    tasks = units = 0
    for t, n, c in spans:
        tiles = -(-t * group // 128) * c
        tasks += tiles
        units += tiles * -(-(n - t // 2 if causal else n) // KEYS)       # (causal: the mean over the rows, N >= T)
    tasks, units = tasks * hkv, units * hkv
    if not tasks:
        return 4, 0
    slots = SLOTS[D]
    if 2 * tasks <= slots:
        chunk = -(-nt // (slots // tasks))
    else:
        chunk = -(-max(2 * units // slots, nt) // 2)
    row = total_q * hkv * group * (D + 2) * 4
    parts = min(scratch, PARTIAL_BYTES) // row                          # at most, in the scratch
    if parts < 2:
        return 4, 0
    chunk = max(chunk, 12, -(-nt // parts))
    gain = (0.7 if D == 256 else 0.5) * (nt - units / slots) * TILE_US[D]
    if chunk >= nt or gain <= -(-nt // chunk) * row * 2 / 2.5e6:
        return 4, 0
    return 4, chunk


def attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: bool, scale: float, lse: bool = False,
           cu: tuple | None = None, spans=None, out: torch.Tensor | None = None, scratch: int = PARTIAL_BYTES):
    """Attention of inputs that takes() accepts: out in q's shape and type (the given one, its rows 16-byte
    aligned, or a new one), or with lse the pair (out fp32, lse fp32 [.., Hq]). cu = (cu_q, cu_k, max_q, max_k)
    and spans = [(T, N)] for packed rows: the offsets as int32 device tensors, the lengths on the host. scratch: the
    bytes that partials of split keys may take."""
    D, Hq, Hk = q.shape[-1], q.shape[-2], k.shape[-2]
    group = Hq // Hk
    if cu is None:
        seqs, n_q, n_k, total = q.shape[0], q.shape[1], k.shape[1], q.shape[0] * q.shape[1]
        cq = ck = None
        waves, chunk = plan(((n_q, n_k, seqs),), group, Hk, D, total, causal, scratch)
    else:
        cq, ck, n_q, n_k = cu[0].data_ptr(), cu[1].data_ptr(), cu[2], cu[3]
        seqs, total = len(spans), q.shape[0]
        waves, chunk = plan([(t, n, 1) for t, n in spans], group, Hk, D, total, causal, scratch)
    dev = q.device
    if out is None:
        out = torch.empty(q.shape, dtype=torch.float32 if lse else q.dtype, device=dev)
    logs = torch.empty(q.shape[:-1], dtype=torch.float32, device=dev) if lse else None
    ls = _row_strides(logs.unsqueeze(-1), 1) if lse else (0, 0, 0)
    strides = _Strides(*_row_strides(q, D), *_row_strides(k, D), *_row_strides(v, D), *_row_strides(out, D), *ls)
    rows = -(-(-(-n_k // KEYS)) // chunk) * total * Hq if chunk else 0          # partial rows: every split's
    part = torch.empty(rows * (D + 2), dtype=torch.float32, device=dev) if chunk else None
    with torch.cuda.device(dev):
        rc = _lib.lib().kush_attend(
            D, 1 if q.dtype == torch.float16 else 2, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
            logs.data_ptr() if lse else None, ctypes.addressof(strides), cq, ck, n_q, n_k, total, seqs, Hk, group, scale,
            int(causal), int(lse), waves, chunk, part.data_ptr() if chunk else None,
            part.data_ptr() + rows * D * 4 if chunk else None, torch.cuda.current_stream(dev).cuda_stream)
    if rc:
        raise RuntimeError(f"kush_attend failed ({rc}): {(_lib.lib().kush_last_error() or b'').decode(errors='replace')}")
    return (out, logs) if lse else out
