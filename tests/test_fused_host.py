"""Host side of the Q/K RMSNorm + RoPE calls: what a launch reads stays alive until it is enqueued (no GPU)."""

import contextlib
import gc
import weakref
from types import SimpleNamespace

import pytest
import torch

from qwen_image_kernel_amd import fused


class _DeviceTensor(torch.Tensor):
    """A CPU tensor that passes for a device one in the host code's checks."""

    is_cuda = True

    @staticmethod
    def make(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape).to(dtype).as_subclass(_DeviceTensor)


@pytest.mark.parametrize("cached", [0, 61, 62, 63, 64])
@pytest.mark.parametrize("pair", [True, False])
def test_prepared_tensors_outlive_the_launch(monkeypatch, cached, pair):
    """With any number of prepared calls cached (a 65th clears the others) and no cos/sin table
    cached, the tensors behind the pointers of Q's and K's argument structs (the fp32 copy of a
    16-bit norm weight, cos and sin) are alive when the library is called."""
    held = {}  # data pointer -> weak references of the tensors it belonged to

    real = fused._prepare

    def prepare(*a):
        fused._cos_sin_cache.clear()
        ent = real(*a)
        for t in ent.keep[1:2] + ent.keep[3:]:
            held.setdefault(t.data_ptr(), []).append(weakref.ref(t))
        return ent

    seen = []

    def launch(*a):
        gc.collect()
        for s in a[:-1]:
            args = s._obj
            seen.append([all(r() is not None for r in held[p]) for p in (args.weight, args.cos, args.sin)])
        return 0

    lib = SimpleNamespace(qik_rms_rope=launch, qik_rms_rope_pair=launch)
    monkeypatch.setattr(fused, "_prepare", prepare)
    monkeypatch.setattr(fused._lib, "load", lambda: lib)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "device", contextlib.nullcontext)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda idx: 0, raising=False)
    monkeypatch.setattr(fused, "_CALLS", {i: None for i in range(cached)})
    monkeypatch.setattr(fused, "_cos_sin_cache", {})

    q, k = _DeviceTensor.make(1, 5, 3, 32), _DeviceTensor.make(1, 5, 2, 32)
    norms = [SimpleNamespace(weight=torch.randn(32).bfloat16(), eps=1e-6) for _ in range(2)]
    freqs = torch.polar(torch.ones(5, 16), torch.randn(5, 16))
    if pair:
        fused._rms_rope_qk(q, k, norms[0], norms[1], freqs)
    else:
        for x, n in ((q, norms[0]), (k, norms[1])):
            fused.fused_rms_norm_rope(x, n.weight, freqs, n.eps)
    assert seen == [[True] * 3] * 2
