"""csrc/moa_host.cpp without a GPU: a copy that takes CPU tensors, in front of entry points that do nothing, in a process of its
own (a fault in compiled code would end this one)."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PREAMBLE = """
import ctypes, importlib.util, sys
import torch
from moa_amd import _lib
spec = importlib.util.spec_from_file_location("_host", sys.argv[1])
host = importlib.util.module_from_spec(spec)
spec.loader.exec_module(host)
NAMES = ("moa_decode_workspace_bytes", "moa_decode_fwd_counted", "moa_rope_cache_append", "moa_cache_append", "moa_prefill_fwd_tokens")
seen = []

def entry(name):
    result, args = _lib.SIGNATURES[name]
    def call(*a):
        seen.append((name, a))
        return 0
    return ctypes.CFUNCTYPE(result, *args)(call)

entries = [entry(n) for n in NAMES]

def refuse(code):
    raise AssertionError(code)

def connect(scratch):
    host.setup(*(ctypes.cast(e, ctypes.c_void_p).value for e in entries), lambda device: 7, refuse, scratch, 16)

def calls():
    "A call of every function, as (function, arguments); the tensors are new ones."
    f, i = (lambda *s: torch.zeros(*s, dtype=torch.float16)), (lambda *s: torch.zeros(*s, dtype=torch.int64))
    B, Hq, H, D, C, N = 2, 4, 2, 64, 30, 130
    def layer():
        return [f(B, C, D), f(B, C, D), i(B, C), i(B, H), i(B, H), i(H), i(H), i(H), i(H)]
    return {
        "decode": (host.attend, [f(B, Hq, 1, D), f(B, C, D), f(B, C, D), 0.1, i(B, H), i(B, H), None, None]),
        "prefill": (host.attend, [f(B, Hq, N, D), f(B, H, N, D), f(B, H, N, D), 0.1, None, None, i(H), i(H)]),
        "rope_append": (host.rope_append, [f(B, Hq, 1, D), f(B, H, 1, D), f(B, H, 1, D), f(1, 1, D), f(1, 1, D), f(B, 1, Hq, D), *layer(), 5]),
        "append": (host.append, [f(B, H, 1, D), f(B, H, 1, D), *layer(), 5]),
    }
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    from moa_amd import build
    tree = tmp_path_factory.mktemp("host")
    csrc = tree / "moa_amd" / "csrc"
    csrc.mkdir(parents=True)
    shutil.copytree(os.path.join(ROOT, "include"), tree / "include")
    text = open(build.HOST_SOURCE).read()
    assert text.count(".is_cuda()") == 1
    (csrc / "moa_host.cpp").write_text(text.replace(".is_cuda()", ".is_cpu()"))
    built = str(tree / "_host.so")
    with pytest.MonkeyPatch.context() as m:
        m.setattr(build, "HOST_SOURCE", str(csrc / "moa_host.cpp"))
        m.setattr(build, "HOST_PATH", built)
        build._build_host()

    def script(body):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + body, built], cwd=ROOT, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    return script


def test_a_tensor_without_an_address_is_an_exception(run):
    """A tensor that throws when it is asked for its address (any of a call's, one after the other): the exception comes out,
    nothing was launched, and the interpreter goes on."""
    run("""
connect(lambda device, stream, nbytes: (4096, 256, None))
for name, (call, args) in calls().items():
    assert call(*args) is not None, name
for name in calls():
    for place in range(len(calls()[name][1])):
        call, args = calls()[name]
        if not torch.is_tensor(args[place]):
            continue
        torch._C._set_throw_on_mutable_data_ptr(args[place])
        del seen[:]
        try:
            call(*args)
        except RuntimeError as e:
            assert "data pointer" in str(e), e
        else:
            raise AssertionError((name, place))
        assert all(n == "moa_decode_workspace_bytes" for n, _ in seen), (name, place)
""")


def test_a_recorded_decode_brings_its_own_workspace(run):
    """No counters in the scratch say that the call is being recorded: it does not take the stream's workspace."""
    run("""
for counters in (8192, None):
    connect(lambda device, stream, nbytes: (4096, 256, counters))
    call, args = calls()["decode"]
    assert call(*args) is not None
    name, a = seen.pop()
    assert name == "moa_decode_fwd_counted" and a[6] == counters, a
    assert (a[4] == 4096) == (counters is not None), a
""")


@pytest.mark.parametrize("found", ["for another torch", "no module", "nothing"])
def test_a_module_that_does_not_fit_is_not_loaded(tmp_path, monkeypatch, found):
    """Torch's C++ classes differ between versions: a module that was built for another one is stale, and is not loaded. The
    calls are left to the Python code then, as they are without any module, and it says so once."""
    import warnings

    import torch

    from moa_amd import _lib, build
    path = tmp_path / "_host.so"
    if found == "for another torch":
        built = open(_lib.HOST_PATH, "rb").read()
        assert built.count(torch.__version__.encode() + b",") == 1
        path.write_bytes(built.replace(torch.__version__.encode() + b",", b"1" * len(torch.__version__) + b","))
    elif found == "no module":
        path.write_bytes(b"")
    assert _lib.host_fits()
    for module in (_lib, build):
        monkeypatch.setattr(module, "HOST_PATH", str(path))
    monkeypatch.setattr(_lib, "_host", None)
    assert build.is_stale()
    with pytest.warns(RuntimeWarning, match="not built for torch " + torch.__version__.split("+")[0]):
        host = _lib.host()
    assert host.attend(*range(8)) is None and host.rope_append(*range(17)) is None and host.append(*range(12)) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.host() is host
