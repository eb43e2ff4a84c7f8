"""Failures of the native tensor calls (Zefr.residual_at / residual_vjp), with the library
replaced by a stand-in that refuses: one native call, and its message is the one raised."""

from __future__ import annotations

import pytest
import torch

from zefr_amd import zefr


class _Refuses:
    """Fails every launch with a message of its own; dims are those of two 2x4x9 elements."""

    def __init__(self):
        self.calls, self.n = [], 0

    def __getattr__(self, name):
        def call(*a):
            self.calls.append(name)
            if name == "zefr_get_dims":
                a[1][0], a[1][1], a[1][3] = 2, 9, 4
                return 0
            if name == "zefr_synchronize":
                return 0
            self.n += 1
            return 1
        return call


class _Cuda(torch.Tensor):
    is_cuda = True


@pytest.mark.parametrize("call", ["residual_at", "residual_vjp"])
@pytest.mark.parametrize("shape,error", [((2, 4, 9), RuntimeError), ((3, 4, 9), ValueError)])
def test_a_failed_native_call_is_not_tried_again(monkeypatch, call, shape, error):
    L = _Refuses()
    monkeypatch.setattr(zefr, "lib", lambda: L)
    monkeypatch.setattr(zefr, "last_error", lambda: f"failure {L.n}")
    monkeypatch.setattr(zefr, "check", lambda rc: rc and (_ for _ in ()).throw(RuntimeError(zefr.last_error())))
    monkeypatch.setattr(zefr, "current_stream", lambda: 0)
    z = zefr.Zefr.__new__(zefr.Zefr)
    z._h, z._owned = 1, False
    monkeypatch.setattr(z, "_ready", lambda *ts: True, raising=False)
    ts = [torch.zeros(shape, dtype=torch.float64).as_subclass(_Cuda) for _ in range(2 if call == "residual_at" else 3)]
    with pytest.raises(error) as e:
        getattr(z, call)(*ts)
    if error is RuntimeError:
        assert str(e.value) == "failure 1"
    assert [c for c in L.calls if "residual" in c] == [f"zefr_{'residual' if call == 'residual_at' else call}_tensor"]
