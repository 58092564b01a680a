"""The native host path (csrc/kvc_host.cpp) where it cannot serve, on the
CPU: arguments without storage that pass for GPU tensors (each case in a
process of its own, since what it guards against ends the process), and an
extension that is absent or does not load."""
import pathlib
import subprocess
import sys
import warnings

import pytest
import torch

from nanovllm_amd import _native

PROLOGUE = f"""
import sys
sys.path.insert(0, {str(_native.PKG_ROOT)!r})
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from nanovllm_amd import _native
from nanovllm_amd.kernels.paged_attention import paged_decode_append, paged_decode_attention
from nanovllm_amd.layers.rotary import qk_norm_rope_store
_native.stream_of = lambda t: 0
host, served = _native.host(), []

def spy(fn):
    def call(*a):
        served.append(fn(*a))
        return served[-1]
    return call

class Spy:
    decode = staticmethod(spy(host.decode))
    rope = staticmethod(spy(host.rope))

_native.host = lambda: Spy

def bf(*shape, dtype=torch.bfloat16):
    return torch.empty((2,) + shape, dtype=dtype, device="cuda")
"""

VMAPPED = """
def one(q, k, v, kc, vc, tables, lens, positions, cos_sin):
    assert type(q) is torch.Tensor and q.is_cuda
    if call == "append":
        return paged_decode_append(q, k, v, kc, vc, lens, tables, lens, 0.1)
    if call == "decode":
        return paged_decode_attention(q, kc, vc, tables, lens, 0.1, 256)
    return qk_norm_rope_store(q, k, v, positions, cos_sin)

with FakeTensorMode():
    args = (bf(3, 16, 128), bf(3, 8, 128), bf(3, 8, 128), bf(4, 64, 8, 128), bf(4, 64, 8, 128),
            bf(3, 4, dtype=torch.int32), bf(3, dtype=torch.int32), bf(3, dtype=torch.int64),
            bf(512, 128, dtype=torch.float32))
    try:
        torch.vmap(one)(*args)
    except RuntimeError as e:
        assert "storage" in str(e) or "data pointer" in str(e), e
        print("refused", served)
"""


@pytest.mark.parametrize("call", ["append", "decode", "rope"])
def test_tensors_without_storage_are_refused(call):
    # vmap's tensors are exact torch.Tensors without storage: data_ptr()
    # throws, and the Python function then raises as it would by itself.
    run = subprocess.run([sys.executable, "-c", PROLOGUE + f"call = {call!r}\n" + VMAPPED],
                         capture_output=True, text=True, timeout=300,
                         cwd=pathlib.Path(__file__).parent)
    assert run.returncode == 0, (run.returncode, run.stderr[-2000:])
    assert run.stdout.strip() == "refused [None]"


@pytest.mark.parametrize("broken", ["absent", "not a library", "another torch"])
def test_calls_take_the_python_path_without_the_extension(monkeypatch, tmp_path, broken):
    path = tmp_path / "_kvc_host.so"
    if broken == "not a library":
        path.write_bytes(b"not ELF")
    elif broken == "another torch":
        path = _native.HOST_PATH
        monkeypatch.setattr(torch, "__version__", "1.0.0")
    monkeypatch.setattr(_native, "HOST_PATH", path)
    monkeypatch.setattr(_native, "_host", None)
    with pytest.warns(RuntimeWarning, match="host path"):
        host = _native.host()
    assert host.decode(*range(11)) is None and host.rope(*range(13)) is None
    with warnings.catch_warnings():           # said once
        warnings.simplefilter("error")
        assert _native.host() is host
    with pytest.raises(RuntimeError):
        _native.load_host()
