"""The native host module on tensors it must leave to the per-call path, and its
checks of grads.  No kernel is launched here."""
from __future__ import annotations

import pytest
import torch

from slideformer_amd import LayerAdam, _lib

CALL = (1 << 19, 1, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, 0, 0)    # an id that no test creates: a library call would fail


def _cpu(n=8, dtype=torch.float32):
    return torch.zeros(n, dtype=dtype)


def test_update_leaves_host_tensors_and_other_objects_to_the_caller():
    h = _lib.host_calls()
    p, g, m, v = _cpu(), _cpu(), _cpu(), _cpu()
    assert h.update(*CALL, p, g, m, v, None, None) is None
    assert h.update(*CALL, torch.nn.Parameter(p), g, m, v, _cpu(dtype=torch.bfloat16), _cpu(1)) is None
    assert h.update(*CALL, torch.empty(8, device="meta"), g, m, v, None, None) is None
    assert h.update(*CALL, "p", g, m, v, None, None) is None
    assert h.update(*CALL[:2], torch.tensor(1e-3), *CALL[3:], p, g, m, v, None, None) is None
    for lr in ("1e-3", None, 10 ** 400):                    # not a number: the per-call path raises
        assert h.update(*CALL[:2], lr, *CALL[3:], p, g, m, v, None, None) is None
    assert h.update_multi(*CALL, [(p, g, m, v)] * 2, None) is None
    assert h.update_multi(*CALL, [], None) is None
    assert h.update_multi(*CALL, [(p, g, m)], None) is None
    with pytest.raises(TypeError):
        h.update(*CALL, p)
    with pytest.raises(TypeError):
        h.update_multi(*CALL, ((p, g, m, v),), None)


@pytest.mark.parametrize("step", [-1, 2 ** 64 + 7])
def test_a_step_number_beyond_64_bits_wraps_as_in_the_per_call_path(step):
    h = _lib.host_calls()
    p, g, m, v = _cpu(), _cpu(), _cpu(), _cpu()
    assert h.update(CALL[0], step, *CALL[2:], p, g, m, v, None, None) is None
    assert h.update_multi(CALL[0], step, *CALL[2:], [(p, g, m, v)] * 2, None) is None


def test_check_grads_names_the_first_refused_grad():
    h = _lib.host_calls()
    assert h.check_grads([], 0) is None
    assert h.check_grads([_cpu()], 0) == (0, 0)
    with pytest.raises(TypeError):
        h.check_grads([None], 0)


def test_a_host_tensor_is_refused_without_a_device_and_the_scalars_stay(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_available", lambda: False)
    adam = LayerAdam(lr=1e-3)
    adam.add_layer_params(0, [torch.nn.Parameter(_cpu()), torch.nn.Parameter(_cpu())])
    for q in adam.param_groups[0]["params"]:
        q.grad = _cpu()
    with pytest.raises(RuntimeError, match="HIP device"):
        adam.step(0)
    sc = adam._scalars(1, 1e-3, 0.9, 0.999, 1e-8, 0.0, True)     # the first call that advances the powers of beta
    assert sc.step == 1 and sc.beta1_t == sc.beta1 and sc.beta2_t == sc.beta2


@pytest.mark.parametrize("overlap", [False, True])
@pytest.mark.parametrize("streamers", [1, 2])
def test_a_step_over_host_tensors_waits_for_every_streamer(streamers, overlap):
    """The last call waits for its own device's streamer; a second one (grads on another device) is waited for too."""
    calls = []

    class Queued(LayerAdam):
        def __init__(self):
            self.overlap_host_chunks = overlap
            self._streamers = dict.fromkeys(range(streamers))

        def _checked_update(self, *args):
            calls.append(args[-1])

        def _synchronize_streamers(self):
            calls.append("all")

    entries = [(_cpu(), _cpu(), _cpu(), _cpu()) for _ in range(3)] + [(_cpu(0),) * 4]
    group = {"step": 1, "lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8, "weight_decay": 0.0, "bias_correction": True}
    adam = Queued()     # kept: its end synchronizes once more
    adam._update_tensors(group, entries)
    waits = [False, False, not overlap, False]
    assert calls == waits + (["all"] if streamers > 1 and not overlap else [])
