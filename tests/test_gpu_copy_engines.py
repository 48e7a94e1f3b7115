"""The copy-engine path of the streaming pipeline: where the caller asks for it (the
choice of LayerAdam and of a pipeline), where page-locked memory out of the kernels'
reach lies beside staged arrays, and the tests of the pipeline once more on it."""
from __future__ import annotations

import ctypes
import itertools

import numpy as np
import pytest
import torch

from oracle import oracle as O
import slideformer_amd.layer_adam as layer_adam
from slideformer_amd import LayerAdam, _lib
from slideformer_amd.layer_adam import HostStreamer
from tests import _hip as H
from tests import test_gpu_layer_adam as pipeline_tests
from tests import test_gpu_pipeline_property as property_tests

pytestmark = pytest.mark.gpu

HP = (1e-3, 0.9, 0.999, 1e-8, 0.01, True)


def direct(stats):
    """The direct path reports one span for the three stages; the copy-engine path one per stream."""
    return stats.h2d_ms == stats.compute_ms == stats.d2h_ms


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("engines", [True, False])
def test_the_caller_chooses_the_path(engines, pinned, hip_device):
    """LayerAdam(copy_engines=True) leaves page-locked state and staged pageable state to the copy engines; without
    it kernels take both.  Three steps, several chunks, bit-exact with the oracle."""
    n = 70_003
    rng = np.random.default_rng(int(pinned))
    ph = rng.normal(0, 0.02, n).astype(np.float32)
    mh, vh = np.zeros(n, np.float32), np.zeros(n, np.float32)
    adam = LayerAdam(lr=1e-3, weight_decay=0.01, pin_host_state=pinned, stream_chunk_elems=16384, copy_engines=engines)
    p = torch.from_numpy(ph.copy())
    if pinned:
        p = p.pin_memory()
    adam.add_layer_params(0, [torch.nn.Parameter(p)])
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    for step in (1, 2, 3):
        g = torch.from_numpy(rng.normal(0, 1e-3, n).astype(np.float32)).bfloat16()
        print(f"engines={engines} pinned={pinned} step={step}", flush=True)
        group = adam.begin_chunk_step(0)
        adam.step_chunk(p, g.pin_memory() if pinned else g, adam.exp_avg_flat[0], adam.exp_avg_sq_flat[0], group)
        assert direct(adam.last_stream_stats) == (not engines)
        adam.end_chunk_step(0)
        orc.update(step, *HP, ph, H.to_np_bits(g, "bf16"), mh, vh, g16="bf16")
    for t, x in ((p, ph), (adam.exp_avg_flat[0], mh), (adam.exp_avg_sq_flat[0], vh)):
        assert np.array_equal(H.to_np_bits(t, "f32"), x.view(np.uint32))


PORTABLE = 0x1    # a hipHostMalloc flag that makes the memory coarse-grained


@pytest.mark.parametrize("overlap", [False, True])
@pytest.mark.parametrize("pageable", ["moments and grads", "grads"])
def test_coarse_master_beside_staged_arrays(pageable, overlap, hip_device):
    """A page-locked master that kernels cannot reach beside pageable arrays that go through the staging: the copy
    engines move both.  Many chunks over two slots, so that every twin is filled again and again: what its last
    copy-in reads and what its last copy-out owes must be done first.  With pageable grads alone nothing is owed."""
    n, chunk = 150 * 1024 + 19, 1024
    rng = np.random.default_rng(17)
    ph = rng.normal(0, 0.02, n).astype(np.float32)
    mh, vh = rng.normal(0, 1e-3, n).astype(np.float32), np.abs(rng.normal(0, 1e-6, n)).astype(np.float32)
    rt, ptr = _lib._hip(), ctypes.c_void_p()
    assert rt.hipHostMalloc(ctypes.byref(ptr), 4 * n, PORTABLE) == 0
    raw = np.frombuffer((ctypes.c_uint8 * (4 * n)).from_address(ptr.value), dtype=np.uint8).view(np.float32)
    raw[:] = ph
    p = torch.from_numpy(raw)
    m, v = torch.from_numpy(mh.copy()), torch.from_numpy(vh.copy())
    if pageable == "grads":
        m, v = m.to(hip_device), v.to(hip_device)
    out = torch.empty(n, dtype=torch.bfloat16)
    if pageable == "grads":
        out = out.pin_memory()
    adam = LayerAdam(lr=1e-3, weight_decay=0.01, overlap_host_chunks=overlap)
    adam._streamers[hip_device] = HostStreamer(hip_device, chunk_elems=chunk, slots=2, host_threads=2)
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    call = 40 * 1024
    for step in (1, 2, 3):
        print(f"coarse master, pageable {pageable}, overlap={overlap}, step {step}", flush=True)
        g = torch.from_numpy(rng.normal(0, 1e-3, n).astype(np.float32)).bfloat16()
        for lo in range(0, n, call):
            hi = min(n, lo + call)
            adam.step_chunk(p[lo:hi], g[lo:hi], m[lo:hi], v[lo:hi], dict(adam.defaults, step=step), bf16_out=out[lo:hi])
            st = adam.last_stream_stats
            assert overlap == (st is None)
            assert overlap or (not direct(st) and st.staged_bytes == (hi - lo) * (2 if pageable == "grads" else 20))
            orc.update(step, *HP, ph[lo:hi], H.to_np_bits(g[lo:hi], "bf16"), mh[lo:hi], vh[lo:hi], g16="bf16")
        adam.synchronize()
        for t, x in ((p, ph), (m, mh), (v, vh)):
            assert np.array_equal(H.to_np_bits(t, "f32"), x.view(np.uint32)), step
        assert np.array_equal(H.to_np_bits(out, "bf16"), O.f32_to_bf16(ph)), step
    del p, t, raw
    rt.hipHostFree(ptr)


def _calls(test):
    """Every call of a test that pytest's parametrize marks make of it."""
    sets = []
    for mark in (m for m in getattr(test, "pytestmark", []) if m.name == "parametrize"):
        names = [x.strip() for x in mark.args[0].split(",")]
        sets.append([dict(zip(names, x if len(names) > 1 else (x,))) for x in mark.args[1]])
    return [{k: v for part in combination for k, v in part.items()} for combination in itertools.product(*sets)]


@pytest.mark.parametrize("name", [
    "test_host_tensors_are_staged_through_hbm",
    "test_pipeline_matches_oracle",
    "test_pipeline_with_clip_and_odd_tail",
    "test_runtime_protocol_on_host_state_with_shared_grad_buffer",
    "test_pinned_host_state_layer_step",
    "test_pageable_state_staged_through_page_locked_twins",
    "test_overlapped_host_chunks_in_the_runtime_protocol",
    "test_overlapped_calls_keep_device_temporaries_alive",
    "test_pipeline_mixed_placements_match_oracle",
    "test_staged_grads_only_wait_for_the_twins_copy_in",
    "test_moments_in_hbm_in_the_runtime_protocol",
    "test_moments_hbm_budget_splits_layers",
    "test_pipeline_other_triples_staged_and_overlapped",
    "test_async_pipeline_calls_with_changing_layouts",
    "test_c5_streamed_full_size_matches_resident",
    "test_pipeline_equals_resident_on_random_layouts",
])
def test_pipeline_tests_on_the_copy_engines(name, hip_device, monkeypatch):
    """The pipeline's tests of results and hazards, whose arrays kernels could reach, with every pipeline asked for
    the copy engines."""
    routes = []

    class Engines(HostStreamer):
        def __init__(self, device, *args, **kwargs):
            super().__init__(device, *args, **dict(kwargs, copy_engines=True))

        def step(self, *args, **kwargs):
            stats = super().step(*args, **kwargs)
            if stats is not None:
                routes.append(direct(stats))
            return stats

    monkeypatch.setattr(layer_adam, "HostStreamer", Engines)
    monkeypatch.setattr(property_tests, "HostStreamer", Engines)
    test = getattr(pipeline_tests, name, None) or getattr(property_tests, name)
    for arguments in _calls(test):
        print(f"{name} {arguments}", flush=True)
        test(**arguments, hip_device=hip_device)
    assert not any(routes)
