"""The native host path (csrc/kvc_host.cpp) on calls that it cannot serve, on
the CPU: arguments without storage that pass for GPU tensors.  Each case runs
in a process of its own, since what it guards against ends the process."""
import pathlib
import subprocess
import sys

import pytest

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
