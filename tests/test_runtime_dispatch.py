"""Which calls of the runtime go to the library's kernels, and how they are
launched, on the CPU: the library is replaced by a recorder, so nothing here
needs a GPU.
"""
import contextlib

import pytest
import torch

from santa_amd import runtime
from santa_amd.runtime import LlamaShape, NHDCache, _FusedOps

BF = torch.bfloat16


class _Recorder:
    """A library whose functions only note the device that is current."""

    def __init__(self, current):
        self.current, self.calls = current, []

    def __getattr__(self, name):
        def fn(*args):
            self.calls.append((name, self.current[-1]))
            return 0

        return fn


@pytest.fixture
def recorder(monkeypatch):
    current = ["another device"]

    @contextlib.contextmanager
    def device(d):
        current.append(d)
        yield
        current.pop()

    class stream:
        cuda_stream = 0  # a device's default stream: the current device's null stream to the runtime

    rec = _Recorder(current)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: stream)
    monkeypatch.setattr(_FusedOps, "_lib", rec)
    return rec


def _ops():
    x, w = torch.ones(2, 64, dtype=BF), torch.ones(48, 64, dtype=BF)
    qkv, cs = torch.ones(1, 2, 64, dtype=BF), torch.ones(2, 16, dtype=BF)
    cache = NHDCache(LlamaShape(hidden=32, intermediate=8, heads=2, kv_heads=1, layers=1, vocab=8), 1, 4, BF, "cpu")
    kv = torch.ones(1, 4, 1, 128, dtype=BF)
    q = torch.ones(1, 4, 2, 128, dtype=BF)
    return {
        "add_rms_norm": lambda: _FusedOps.add_rms_norm(x, x.clone(), x[0], 1e-5),
        "rope_table": lambda: _FusedOps.rope_table(3, 16, 1e4, x),
        "rope_write": lambda: _FusedOps.rope_write(qkv[0, :1], cs[0], cs[0], cache, 0, 1, 2, 1, 16),
        "rope_write_rows": lambda: _FusedOps.rope_write_rows(qkv, cs, cs, cache.k[0], cache.v[0], 2, 1, 16),
        "linear": lambda: _FusedOps.linear(x, w),
        "linear_f32": lambda: _FusedOps.logits(x, w),
        "linear_rope": lambda: _FusedOps.linear_rope(x[:1], torch.ones(64, 64, dtype=BF), cs[0], cs[0], cache, 0, 1, 2,
                                                     1, 16),
        "argmax": lambda: _FusedOps.argmax(x.float()),
        "silu_mul": lambda: _FusedOps.silu_mul(x),
        "causal_attention": lambda: _FusedOps.causal_attention(q, kv, kv),
        "exact_decode": lambda: _FusedOps.exact_decode(q[:, 0], kv, kv, 3),
    }


@pytest.mark.parametrize("op", sorted(_ops()))
def test_launches_on_the_tensors_device(op, recorder):
    """Every kernel is launched with its tensors' device current: a default
    stream is 0, which the runtime takes as the current device's."""
    _ops()[op]()
    launches = [c for c in recorder.calls if not c[0].endswith("workspace_size")]
    assert [name for name, _ in launches] == ["santa_rt_" + op]
    assert launches[0][1] == torch.device("cpu")
