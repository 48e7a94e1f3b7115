"""The streaming pipeline's direct path (kernels on page-locked host memory)
and the rule that chooses it, against the CPU checker, bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from slideformer_amd import LayerAdam, _lib
from slideformer_amd.layer_adam import HostStreamer
from tests import _hip as H

pytestmark = pytest.mark.gpu

HP = (1e-3, 0.9, 0.999, 1e-8, 0.01, True)
# hipHostMalloc flags
PORTABLE, MAPPED, WRITE_COMBINED, COHERENT, NONCOHERENT = 0x1, 0x2, 0x4, 0x40000000, 0x80000000


class Case:
    """One layer on the host: the same numbers for the library and the checker."""

    def __init__(self, n, seed):
        rng = np.random.default_rng(seed)
        self.n = n
        self.p = rng.normal(0, 0.02, n).astype(np.float32)
        self.m = rng.normal(0, 1e-3, n).astype(np.float32)
        self.v = np.abs(rng.normal(0, 1e-6, n)).astype(np.float32)
        self.rng = rng
        self.orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
        self.ref = [self.p.copy(), self.m.copy(), self.v.copy()]

    def grads(self):
        return torch.from_numpy(self.rng.normal(0, 1e-3, self.n).astype(np.float32)).bfloat16()

    def expect(self, step, g, lo=0, hi=None):
        hi = self.n if hi is None else hi
        p, m, v = (x[lo:hi] for x in self.ref)
        self.orc.update(step, *HP, p, H.to_np_bits(g[lo:hi], "bf16"), m, v, g16="bf16")

    def check(self, p, m, v, out=None):
        for t, x in zip((p, m, v), self.ref):
            assert np.array_equal(H.to_np_bits(t, "f32"), x.view(np.uint32))
        if out is not None:
            assert np.array_equal(H.to_np_bits(out, "bf16"), O.f32_to_bf16(self.ref[0]))


def direct(stats):
    """The direct path reports one span for the three stages; the copy-engine path one per stream."""
    return stats.h2d_ms == stats.compute_ms == stats.d2h_ms


def streamed(dev, **shape):
    overlap = shape.pop("overlap", False)
    adam = LayerAdam(lr=1e-3, weight_decay=0.01, overlap_host_chunks=overlap)
    adam._streamers[dev] = HostStreamer(dev, **shape)
    return adam


def flagged(x, flags, shift=0):
    """x in a hipHostMalloc allocation of the given flags, `shift` bytes off its start; the tensor and its owner."""
    rt = _lib._hip()
    ptr = ctypes.c_void_p()
    assert rt.hipHostMalloc(ctypes.byref(ptr), x.nbytes + 64, flags) == 0
    raw = np.frombuffer((ctypes.c_uint8 * (x.nbytes + 64)).from_address(ptr.value), dtype=np.uint8)
    raw[shift:shift + x.nbytes] = x.view(np.uint8)
    return raw, ptr


@pytest.mark.parametrize("flags,shift,is_direct", [(0, 0, True), (MAPPED, 4, True), (COHERENT, 12, True),
                                                   (PORTABLE, 0, False), (WRITE_COMBINED, 0, False),
                                                   (NONCOHERENT, 0, False), (0, 2, False)])
def test_route_of_page_locked_memory(flags, shift, is_direct, hip_device):
    """Coherent page-locked state takes the direct path, at any element
    alignment; coarse-grained memory and arrays that start inside an element
    keep the copy engines, which take both.  Repeated steps with the host
    rewriting the master in between: nothing stale is read."""
    c = Case(70_001, flags % 97 + shift)
    raw, ptr = flagged(c.p, flags, shift)
    L = _lib.load()
    handle = ctypes.c_void_p()
    _lib.check(L.la_pipeline_create(16384, 3, ctypes.byref(handle)), "la_pipeline_create")
    mask = _lib.LA_ON_HOST_P | _lib.LA_ON_HOST_G
    ws = torch.empty(L.la_pipeline_workspace_bytes(16384, 3, 0, 1, 0, mask), dtype=torch.uint8, device=hip_device)
    m, v = torch.from_numpy(c.m).to(hip_device), torch.from_numpy(c.v).to(hip_device)
    opt = H.HipAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    for step in range(1, 6):
        g = c.grads().pin_memory()
        sc, st = _lib.LaScalars(), _lib.LaPipelineStats()
        _lib.check(L.la_scalars(opt.id, step, *HP[:5], 1, ctypes.byref(sc)), "la_scalars")
        print(f"route flags={flags:#x} shift={shift} step={step}", flush=True)
        _lib.check(L.la_pipeline_step(handle, ctypes.byref(sc), 0, ptr.value + shift, 1, g.data_ptr(), 0, m.data_ptr(),
                                      v.data_ptr(), c.n, None, mask, None, ws.data_ptr(), ws.numel(),
                                      torch.cuda.current_stream().cuda_stream, 1, ctypes.byref(st)),
                   "la_pipeline_step")
        assert direct(st) == is_direct
        c.expect(step, g)
        now = raw[shift:shift + 4 * c.n].copy().view(np.uint32)
        assert np.array_equal(now, c.ref[0].view(np.uint32)), step
        c.ref[0] *= np.float32(-0.5)                       # the host's own write between steps
        raw[shift:shift + 4 * c.n] = c.ref[0].view(np.uint8)
    c.check(torch.from_numpy(c.ref[0]), m, v)
    L.la_pipeline_destroy(handle)
    del raw
    _lib._hip().hipHostFree(ptr)


# one sub-chunk, the smallest split, its remainder, and more sub-chunks than twins
@pytest.mark.parametrize("n", [17, 65_536, 65_537, 8 * 65_536 + 5, 3_000_001, 9 * 1_048_576 + 3])
@pytest.mark.parametrize("pageable", ["state", "grads"])
def test_staged_sub_chunks(n, pageable, hip_device):
    c = Case(n, n)
    adam = streamed(hip_device, chunk_elems=4 * 1024 * 1024, slots=2, host_threads=5)
    host = [torch.from_numpy(x.copy()) for x in (c.p, c.m, c.v)]
    if pageable == "grads":
        host = [t.pin_memory() for t in host]
    out = torch.empty(n, dtype=torch.bfloat16, device=hip_device)
    for step in (1, 2, 3):
        g = c.grads()
        adam.step_chunk(host[0], g if pageable == "grads" else g.pin_memory(), host[1], host[2],
                        dict(adam.defaults, step=step), bf16_out=out)
        assert direct(adam.last_stream_stats)
        assert adam.last_stream_stats.staged_bytes == n * (2 if pageable == "grads" else 24)
        c.expect(step, g)
        c.check(*host, out)


def test_queued_calls_of_every_route_on_one_pipeline(hip_device):
    """Calls that return once queued, in turn page-locked (direct), pageable
    through the twins (direct), pageable without staging and coarse-grained
    (copy engines), on disjoint parts of one layer and then on the same parts
    again: each switch completes what it must."""
    n, part = 120_000, 20_000
    c = Case(n, 5)
    adam = streamed(hip_device, chunk_elems=4096, slots=3, overlap=True, host_threads=3)
    streamer = adam._streamers[hip_device]
    coarse, owner = flagged(c.p, PORTABLE)
    kinds = ["locked", "staged", "locked", "unstaged", "staged", "coarse"]
    parts = []
    for i, kind in enumerate(kinds):
        lo, hi = i * part, (i + 1) * part
        p, m, v = (torch.from_numpy(x[lo:hi].copy()) for x in (c.p, c.m, c.v))
        if kind in ("locked", "coarse"):
            p, m, v = p.pin_memory(), m.pin_memory(), v.pin_memory()
        if kind == "coarse":
            p = torch.from_numpy(coarse[:4 * n].view(np.float32))[lo:hi]
        parts.append((kind, lo, hi, p, m, v))
    for step in (1, 2, 3):
        g = c.grads()
        gd = g.to(hip_device)
        for repeat in range(2):                     # the second round meets unsettled bytes of the first
            for kind, lo, hi, p, m, v in parts:
                streamer.stage_pageable = kind not in ("unstaged", "coarse")
                adam.step_chunk(p, gd[lo:hi], m, v, dict(adam.defaults, step=2 * step - 1 + repeat))
                c.expect(2 * step - 1 + repeat, g, lo, hi)
        adam.synchronize()
        for kind, lo, hi, p, m, v in parts:
            for t, x in zip((p, m, v), c.ref):
                assert np.array_equal(H.to_np_bits(t, "f32"), x[lo:hi].view(np.uint32)), (step, kind)
    del parts, p, m, v, t, adam, streamer, coarse
    _lib._hip().hipHostFree(owner)


@pytest.mark.parametrize("triple,offsets", [
    (("bf16", "bf16", "f32"), (1, 3, 2, 1, 5)),      # odd elements, no head aligns all: the misphased form
    (("bf16", "bf16", "bf16"), (1, 2, 5, 7, 3)),
    (("f16", "f16", "f16"), (3, 3, 3, 3, 3)),        # one odd phase for all: a head of 5
    (("f16", "f32", "f32"), (1, 0, 1, 3, 0)),
    (("f32", "bf16", "f32"), (1, 3, 0, 2, 7)),
])
@pytest.mark.parametrize("n", [1, 31, 4097, 100_003])
def test_page_locked_arrays_at_odd_elements(triple, offsets, n, hip_device):
    """Host arrays of every element size that start at odd elements, which the kernel reads and writes over the link
    in place, the host's bf16 copy included; what lies beside them stays as it is.  Bit-exact with the checker."""
    rng = np.random.default_rng(n + offsets[0])
    kinds = (triple[0], triple[1], triple[2], triple[2], "bf16")
    k16 = [None if k == "f32" else k for k in triple]
    values = [rng.normal(0, 0.02, n), None, rng.normal(0, 1e-3, n), np.abs(rng.normal(0, 1e-5, n)), np.zeros(n)]
    pads, arrays = [], []
    for x, kind, off in zip(values, kinds, offsets):
        pad = torch.full((off + n + 9,), 7.0, dtype=H.TD[kind]).pin_memory()
        pads.append((pad, off))
        arrays.append(pad[off:off + n])
        if x is not None:
            arrays[-1].copy_(torch.from_numpy(x.astype(np.float32)).to(H.TD[kind]))
    p, g, m, v, out = arrays
    ref = [H.to_np_bits(t, k) for t, k in zip(arrays, kinds)]
    view = lambda b, k: b.view(np.float32) if k == "f32" else b
    adam = streamed(hip_device, chunk_elems=16384, slots=2)
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    for step in (1, 2, 3):
        print(f"odd elements {triple} {offsets} n={n} step={step}", flush=True)
        g.copy_(torch.from_numpy(rng.normal(0, 1e-3, n).astype(np.float32)).to(g.dtype))
        adam.step_chunk(p, g, m, v, dict(adam.defaults, step=step), bf16_out=out)
        assert direct(adam.last_stream_stats)
        orc.update(step, *HP, view(ref[0], kinds[0]), view(H.to_np_bits(g, kinds[1]), kinds[1]), view(ref[2], kinds[2]),
                   view(ref[3], kinds[3]), p16=k16[0], g16=k16[1], s16=k16[2], p_bf16_out=ref[4])
        for j in (0, 2, 3, 4):
            assert np.array_equal(H.to_np_bits(arrays[j], kinds[j]), ref[j]), (step, j)
    for pad, off in pads:
        assert (pad[:off] == 7.0).all() and (pad[off + n:] == 7.0).all()


# around one trip of 32 and of 64 workgroups, and several
@pytest.mark.parametrize("n", [5, 32_768, 32_785, 65_536, 65_551, 200_003])
@pytest.mark.parametrize("triple,host", [(("f32", "bf16", "f32"), "g"), (("bf16", "bf16", "f32"), "p"),
                                         (("f16", "f16", "f32"), "go"), (("bf16", "bf16", "bf16"), "g")])
def test_calls_that_read_few_bytes_over_the_link(triple, host, n, hip_device):
    """Only the grads or 16-bit parameters (and the bf16 copy) in page-locked memory, the rest in HBM: the launch
    shape for waves that read at most 512 bytes of host memory per trip, and the all-16-bit triple, which reads more.
    Bit-exact with the checker."""
    rng = np.random.default_rng(n)
    kinds = dict(p=triple[0], g=triple[1], m=triple[2], v=triple[2], o="bf16")
    scale = dict(p=0.02, m=1e-3, v=1e-5, o=0.0)
    place = lambda t, name: t.pin_memory() if name in host else t.to(hip_device)
    make = lambda s, k: torch.from_numpy(rng.normal(0, 1, n).astype(np.float32) * np.float32(s)).to(H.TD[k])
    t = {k: place(make(scale[k], kinds[k]).abs() if k == "v" else make(scale[k], kinds[k]), k) for k in "pmvo"}
    ref = {k: H.to_np_bits(t[k], kinds[k]) for k in "pmvo"}
    k16 = {k: None if x == "f32" else x for k, x in kinds.items()}
    view = lambda b, k: b.view(np.float32) if k == "f32" else b
    adam = streamed(hip_device, chunk_elems=16384, slots=2)
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    for step in (1, 2):
        print(f"few bytes over the link {triple} {host} n={n} step={step}", flush=True)
        g = make(1e-3, kinds["g"])
        adam.step_chunk(t["p"], place(g, "g"), t["m"], t["v"], dict(adam.defaults, step=step), bf16_out=t["o"])
        assert direct(adam.last_stream_stats)
        orc.update(step, *HP, view(ref["p"], kinds["p"]), view(H.to_np_bits(g, kinds["g"]), kinds["g"]),
                   view(ref["m"], kinds["m"]), view(ref["v"], kinds["v"]), p16=k16["p"], g16=k16["g"], s16=k16["m"],
                   p_bf16_out=ref["o"])
        for k in "pmvo":
            assert np.array_equal(H.to_np_bits(t[k], kinds[k]), ref[k]), (step, k)
