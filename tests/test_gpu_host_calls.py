"""LayerAdam's calls through the native host module: the per-tensor step equals
one call per tensor bit for bit, whatever decides its route."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from slideformer_amd import LayerAdam
from tests import _hip as H

pytestmark = pytest.mark.gpu

SIZES = [(5,), (64, 3), (1,), (700, 11), (0,), (4099,)]


def _layer(dev, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    params, grads = [], []
    for shape in SIZES:
        params.append(torch.nn.Parameter((torch.randn(shape, generator=gen) * 0.02).to(dtype).to(dev)))
        grads.append((torch.randn(shape, generator=gen) * 1e-3).to(dtype).to(dev))
    return params, grads


def _bits(t):
    return H.to_np_bits(t, {torch.float32: "f32", torch.bfloat16: "bf16"}[t.dtype])


@pytest.mark.parametrize("form", ["plain", "subclass", "overlap", "mixed grads", "pageable", "pinned", "half on host"])
def test_step_equals_one_call_per_tensor(form, hip_device):
    """Plain tensors and a tensor subclass (batched), two tensors that share memory
    and grads of two types (one call each), host tensors (queued, the last one
    waits) and a layer whose second half is on the host."""
    dtype = torch.bfloat16 if form == "plain" else torch.float32
    coef = torch.tensor([0.5], device=hip_device)
    results = []
    for route in ("step", "calls"):
        params, grads = _layer(hip_device, dtype, 3)
        if form == "overlap":
            flat = torch.cat([p.detach().reshape(-1) for p in params])
            params[0] = torch.nn.Parameter(flat[:5].view(5))
            params[1] = torch.nn.Parameter(flat[3:3 + 192].view(64, 3))
        if form == "subclass":
            class Named(torch.Tensor):
                pass
            grads = [g.as_subclass(Named) for g in grads]
        if form == "mixed grads":
            grads[3] = grads[3].bfloat16()
        if form in ("pageable", "pinned"):
            params = [torch.nn.Parameter(p.detach().cpu()) for p in params]
            grads = [g.cpu() for g in grads]
        if form == "pinned":
            params = [torch.nn.Parameter(p.detach().pin_memory()) for p in params]
            grads = [g.pin_memory() for g in grads]
        if form == "half on host":
            params[3:] = [torch.nn.Parameter(p.detach().cpu()) for p in params[3:]]
            grads[3:] = [g.cpu() for g in grads[3:]]
        adam = LayerAdam(lr=1e-3, weight_decay=0.01, moments_device=hip_device if form == "half on host" else None)
        adam.add_layer_params(0, params)
        print(f"host calls {form} {route}", flush=True)
        for step in (1, 2, 3):
            if route == "step":
                adam.step_with_grad_views(0, dict(zip(params, grads)), clip_coef=coef)
                assert form not in ("pageable", "pinned") or adam.last_stream_stats is not None
            else:
                for p, g in zip(params, grads):
                    st = adam.state[p]
                    adam.adam_update(step, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, p, g, st["exp_avg"], st["exp_avg_sq"],
                                     clip_coef=coef)
        torch.cuda.synchronize()
        results.append([_bits(t) for t in (*params, adam.exp_avg_flat[0], adam.exp_avg_sq_flat[0])])
    for a, b in zip(*results):
        assert np.array_equal(a, b)


class _Recorded:
    """The native host module, with what its update_multi calls returned."""

    def __init__(self, host):
        self.host, self.returned = host, []

    def __getattr__(self, name):
        return getattr(self.host, name)

    def update_multi(self, *args):
        self.returned.append(self.host.update_multi(*args))
        return self.returned[-1]


def _step(dev, params, grads, coef=None, **group):
    """One step(layer) of params with grads: what its batched call returned and every bit of the result."""
    adam = LayerAdam(lr=1e-3, weight_decay=0.01)
    adam._host = _Recorded(adam._host)
    adam.add_layer_params(0, params)
    adam.param_groups[0].update(group)
    adam.step_with_grad_views(0, dict(zip(params, grads)), clip_coef=coef)
    return adam._host.returned, [_bits(t) for t in (*params, adam.exp_avg_flat[0], adam.exp_avg_sq_flat[0])]


@pytest.mark.parametrize("kind", ["np.float32", "tensor", "device tensor", "np array"])
def test_hyper_parameters_of_any_number_type_keep_the_batched_launch(kind, hip_device):
    lr = {"np.float32": np.float32(1e-3), "tensor": torch.tensor(1e-3), "np array": np.array(1e-3, np.float32),
          "device tensor": torch.tensor(1e-3, device=hip_device)}[kind]
    returned, got = _step(hip_device, *_layer(hip_device, torch.float32, 4), lr=lr, betas=(np.float32(0.9), 0.999))
    assert returned == [0]
    for a, b in zip(got, _step(hip_device, *_layer(hip_device, torch.float32, 4))[1]):
        assert np.array_equal(a, b)


class _Scale(torch.nn.Parameter):
    pass


class _View(torch.Tensor):
    pass


class _Elsewhere(torch.Tensor):
    """A subclass with an answer of its own."""

    def data_ptr(self):
        return super().data_ptr()


@pytest.mark.parametrize("kind,batched", [("parameter", True), ("grad and clip", True), ("own answer", False)])
def test_tensor_subclasses_keep_the_batched_launch(kind, batched, hip_device):
    """Subclasses that leave torch's methods as they are go in one launch, as plain tensors do; one that answers
    for itself is asked, call by call."""
    params, grads = _layer(hip_device, torch.float32, 6)
    coef = torch.tensor([0.5], device=hip_device)
    if kind == "parameter":
        params = [_Scale(p.detach()) for p in params]
    elif kind == "grad and clip":
        grads, coef = [g.as_subclass(_View) for g in grads], coef.as_subclass(_View)
    else:
        grads[1] = grads[1].as_subclass(_Elsewhere)
    returned, got = _step(hip_device, params, grads, coef)
    assert returned == [0 if batched else None]
    plain = _step(hip_device, *_layer(hip_device, torch.float32, 6), torch.tensor([0.5], device=hip_device))[1]
    for a, b in zip(got, plain):
        assert np.array_equal(a, b)


def test_refused_calls_still_raise_and_complete_what_was_queued(hip_device):
    adam = LayerAdam(lr=1e-3)
    p, m, v = (torch.zeros(16, device=hip_device) for _ in range(3))
    g = torch.ones(32, device=hip_device)
    hp = (1, 1e-3, 0.9, 0.999, 1e-8, 0.0, True)
    with pytest.raises(RuntimeError, match="grads must be contiguous"):
        adam.adam_update(*hp, p, g[::2], m, v)
    with pytest.raises(RuntimeError, match="size mismatch"):
        adam.adam_update(*hp, p, g, m, v)
    with pytest.raises(RuntimeError, match="not supported"):
        adam.adam_update(*hp, p, g[:16], m.half(), v.half())
    with pytest.raises(RuntimeError, match="bf16_out"):
        adam.adam_update(*hp, p, g[:16], m, v, bf16_out=torch.zeros(16, device=hip_device))
    with pytest.raises(RuntimeError, match="clip_coef"):
        adam.adam_update(*hp, p, g[:16], m, v, clip_coef=torch.zeros(1))
    with pytest.raises(RuntimeError, match="contiguous"):
        adam.clip_grad_norm([g, g[::2]], 1.0)
    with pytest.raises(RuntimeError, match="expected"):
        adam.clip_grad_norm([g, torch.ones(3)], 1.0)
    with pytest.raises(RuntimeError, match="dtype"):
        adam.clip_grad_norm([g.double()], 1.0)
    # a layer on the host whose second tensor is refused: the first is complete
    a, b = torch.zeros(100_000), torch.zeros(64)
    adam.add_layer_params(0, [torch.nn.Parameter(a), torch.nn.Parameter(b)])
    params = adam.param_groups[0]["params"]
    with pytest.raises(RuntimeError, match="contiguous"):
        adam.step_with_grad_views(0, {params[0]: torch.ones(100_000), params[1]: torch.ones(128)[::2]})
    assert (a < 0).all() and (b == 0).all()
