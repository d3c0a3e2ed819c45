"""The native host side of the per-step calls (csrc/kush_fastcall.cpp) on the CPU: the file built without its
device check, around entry points that only count their calls. A tensor without storage (what torch.vmap passes: its
type is torch.Tensor itself) is not taken in any place, whatever thread state the failure meets, and the caller's
Python path raises the error."""
import shutil
import subprocess
import sys

import pytest

SCRIPT = r"""
import ctypes, importlib.util, sys
import torch
spec = importlib.util.spec_from_file_location("_fastcall", sys.argv[1])
m = importlib.util.module_from_spec(spec)
spec.loader.exec_module(m)

P, I, L, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
DECODE = [I, I, I, I, P, P, P, L, L, P, P, P, P, L, I, F, I, P, P, I, P]
EXT = [I, P, I, P, I]
WRITE = [I, I, I, P, P, L, L, P, P, P, P, P, I, I, P, L, L, P, P, L, I, P, I]
calls = []
def entry(name, args):
    return ctypes.CFUNCTYPE(I, *args)(lambda *a: calls.append((name, a)) or 0)
fns = [entry("decode", DECODE + EXT), entry("append_decode", DECODE + [P, P, L, L] + EXT), entry("write", WRITE)]
S, H, G, D, B = 3, 2, 4, 64, 5
sync = torch.zeros(64, dtype=torch.int32)
# a dtype of 0 is fp32; the device index of a CPU tensor is -1
cfg = m.make_config(D, 4, G, 0, -1, sync.data_ptr(), *(ctypes.cast(f, P).value for f in fns))
i32 = dict(dtype=torch.int32)
t = dict(k=torch.randn(S, H, D), v=torch.randn(S, H, D), q=torch.randn(S, H * G, D), out=torch.zeros(S, H * G, D),
         cache=torch.zeros(B, H, 2560, dtype=torch.uint8), table=torch.zeros(S, 2, **i32), lens=torch.ones(S, **i32),
         tidx=torch.arange(S, **i32), tail=torch.zeros(S, H, 32, D), work=torch.zeros(S * H * 2 * G * (D + 2)),
         order=torch.arange(S, **i32), qsl=torch.arange(S + 1, **i32), js=torch.arange(S, **i32), jp=torch.zeros(S, **i32))

def decode(x, ns=2):
    return m.decode(cfg, x["k"], x["v"], x["q"], x["out"], x["cache"], x["table"], x["lens"], x["tidx"], x["tail"], 0.1,
                    ns, x["work"], 4, x["order"], False, 64, 0)
def alone(x):
    return decode(dict(x, k=None, v=None), 1)
def write(x):
    return m.write(cfg, x["k"], x["v"], x["qsl"], x["lens"], x["tidx"], x["js"], x["jp"], x["cache"], x["table"], x["tail"],
                   False, 0)

CALLS = [(decode, "k v q out cache table lens tidx tail work order"), (alone, "q out cache table lens tidx tail order"),
         (write, "k v qsl lens tidx js jp cache table tail")]
for fn, names in CALLS:
    assert fn(t) == 0 and calls, fn.__name__                       # the plain call is taken ...
    want = {t[n].data_ptr() for n in names.split()}
    assert want <= set(calls.pop()[1]), fn.__name__                # ... with every tensor's address
    for n in names.split():                                        # ... and none without one
        print(fn.__name__, n, flush=True)
        def body(x):
            assert type(x) is torch.Tensor
            assert fn(dict(t, **{n: x})) == m.NOT_TAKEN
            return torch.zeros(1)
        torch.vmap(body)(t[n][None])
    assert not calls
print("every call answered")
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    import importlib
    build = importlib.import_module("kushkash_amd.build")
    tmp = tmp_path_factory.mktemp("fastcall")
    src = (build.PKG / "csrc" / build.FAST_SOURCE).read_text()
    check = "t.is_cuda() && t.get_device() == c.device && "
    assert src.count(check) == 1
    (tmp / build.FAST_SOURCE).write_text(src.replace(check, ""))
    out = tmp / "_fastcall.so"
    cmd = build.fastcall_command(out)
    at = cmd.index(str(build.PKG / "csrc" / build.FAST_SOURCE))
    subprocess.run([*cmd[:at], str(tmp / build.FAST_SOURCE), *cmd[at + 1:]], check=True, capture_output=True)
    return out


def test_an_extension_of_another_abi_is_refused(monkeypatch):
    """Built for another revision of the library whose addresses it would call: an error that says so, before any call."""
    import types

    import kushkash_amd
    from kushkash_amd import _lib
    for old in (types.SimpleNamespace(), types.SimpleNamespace(ABI=_lib.ABI_VERSION - 1)):
        monkeypatch.setitem(sys.modules, "kushkash_amd._fastcall", old)
        monkeypatch.setattr(kushkash_amd, "_fastcall", old, raising=False)
        _lib.fastcall.cache_clear()
        with pytest.raises(RuntimeError, match=f"expected {_lib.ABI_VERSION}; rebuild it"):
            _lib.fastcall()
    monkeypatch.undo()
    _lib.fastcall.cache_clear()
    assert _lib.fastcall() is None or _lib.fastcall().ABI == _lib.ABI_VERSION


def test_the_extension_has_a_source_digest():
    """Its source, the header whose entry points it calls, and its flags decide it; the build records it."""
    import importlib
    build = importlib.import_module("kushkash_amd.build")
    assert build.source_digest(build.FAST_SOURCE) not in (None, build.source_digest(build.CPU_SOURCE))
    assert build.built_digest(build.FAST_SOURCE) in (None, build.source_digest(build.FAST_SOURCE))
    seen = set()
    build._includes(build.PKG / "csrc" / build.FAST_SOURCE, seen)
    assert {f.name for f in seen} == {build.FAST_SOURCE, "kushkash_amd.h"}


def test_tensors_without_storage(library, tmp_path):
    (tmp_path / "calls.py").write_text(SCRIPT)
    r = subprocess.run([sys.executable, str(tmp_path / "calls.py"), str(library)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "every call answered" in r.stdout, (r.returncode, r.stdout[-300:], r.stderr[-2000:])
