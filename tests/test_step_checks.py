"""What AttentionStep.run refuses before it calls the library (no GPU needed: a
step whose device side is replaced by its description)."""
from types import SimpleNamespace

import pytest
import torch

from kunserve_amd import AttentionStep, _lib


@pytest.fixture
def step(monkeypatch):
    def no_call(name, *args):
        raise AssertionError(f"{name} was called")

    monkeypatch.setattr(_lib, "call", no_call)
    s = object.__new__(AttentionStep)
    s.pool = SimpleNamespace(num_layers=1, num_kv_heads=2, head_dim=64, dtype=torch.float16,
                             device=torch.device("cuda", 0), desc=lambda: None)
    s.layer_offset, s.num_tokens, s.num_qo_heads = 0, 3, 4
    s._device, s._q_shape, s._kv_shape = s.pool.device, (3, 4, 64), (3, 2, 64)
    s._device_index, s._step_ref = 0, None
    return s


def _tensors(device):
    return [torch.empty((3, h, 64), dtype=torch.float16, device=device) for h in (4, 2, 2, 4)]


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_tensors_of_another_device_are_refused(step, device):
    q, k, v, out = _tensors(device)
    with pytest.raises(ValueError, match="q is on"):
        step.run(0, q, k, v, out=out)
    with pytest.raises(ValueError, match="q is on"):
        step.run(0, q, k, v)


@pytest.mark.parametrize("rope", [(None,), (None, False, 1), ()])
def test_rope_is_a_pair(step, rope):
    q, k, v, out = _tensors("meta")
    with pytest.raises(ValueError, match="unpack"):
        step.run(0, q, k, v, out=out, rope=rope)
