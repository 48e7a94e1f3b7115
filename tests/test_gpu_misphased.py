"""Streams that disagree in alignment phase, against the CPU checker, bit for bit.

The update kernels' misphased form masks the lanes of a partial last run
itself, so the sizes sit around one run (256 elements, 512 for the all-16-bit
triples) and around the reference's 16-element tail, and the elements before
and after each array must stay as they were.
"""
from __future__ import annotations

import zlib

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import _golden as G
from tests import _hip as H

pytestmark = pytest.mark.gpu

TRIPLES = [("f32", "bf16", "f32"), ("f32", "f32", "f32"), ("f32", "f16", "f32"), ("bf16", "bf16", "f32"),
           ("bf16", "f32", "f32"), ("bf16", "bf16", "bf16"), ("f16", "f16", "f32"), ("f16", "f32", "f32"),
           ("f16", "f16", "f16")]
# element offsets of p, g, m, v, out from a 256-byte boundary; no head aligns all five
PHASES = [(0, 3, 0, 0, 3), (1, 0, 3, 3, 2), (0, 0, 1, 2, 0), (5, 1, 3, 7, 0), (0, 0, 0, 0, 1)]
SIZES = (1, 15, 17, 18, 19, 255, 256, 259, 272, 512, 515, 531, 8_191, 70_001)
HP = (1e-3, 0.9, 0.999, 1e-8, 0.01, True)
K16 = {"bf16": "bf16", "f16": "f16", "f32": None}
GUARD = 8


def _host(bits, kind):
    return bits.view(np.float32) if kind == "f32" else bits


def _draw(rng, kind, std, n, positive=False):
    x = rng.normal(0, std, n).astype(np.float32)
    return torch.from_numpy(np.abs(x) if positive else x).to(H.TD[kind])


@pytest.mark.parametrize("route", ["single", "grid_stride", "multi"])
@pytest.mark.parametrize("triple", TRIPLES, ids="-".join)
def test_misphased_streams(triple, route, hip_device):
    pk, gk, sk = triple
    lib = H.load_small_grid() if route == "grid_stride" else None
    opt = H.HipAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True, lib=lib)
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    rng = np.random.default_rng(zlib.crc32(repr(triple).encode()))
    coef = torch.tensor([0.625], device=hip_device)
    calls = []
    for n in SIZES:
        for off in PHASES + ([(0, 0, 0, 0, 0)] if route == "multi" else []):   # aligned tensors in the same batch
            src = [_draw(rng, pk, 0.02, n + 2 * GUARD), _draw(rng, gk, 1e-3, n + 2 * GUARD),
                   _draw(rng, sk, 1e-3, n + 2 * GUARD), _draw(rng, sk, 1e-3, n + 2 * GUARD, True),
                   torch.zeros(n + 2 * GUARD, dtype=torch.bfloat16)]
            dev = [t.to(hip_device) for t in src]
            bits = [H.to_np_bits(t, k) for t, k in zip(src, (pk, gk, sk, sk, "bf16"))]
            calls.append((n, off, dev, bits))
    views = [[t[o:o + n] for t, o in zip(dev, off)] for n, off, dev, _ in calls]
    print(f"misphased {triple} {route}: {len(calls)} calls", flush=True)
    if route == "multi":
        opt.update_multi(1, *HP, [tuple(v) for v in views], coef=coef)
    else:
        for p, g, m, v, out in views:
            opt.update(1, *HP, p, g, m, v, out=out, coef=coef)
    torch.cuda.synchronize()
    for n, off, dev, bits in calls:
        p, g, m, v, out = (_host(b, k)[o:o + n] for b, k, o in zip(bits, (pk, gk, sk, sk, "bf16"), off))
        orc.update(1, *HP, p, g, m, v, p16=K16[pk], g16=K16[gk], s16=K16[sk], p_bf16_out=out, clip_coef=0.625)
        for t, b, k in zip(dev, bits, (pk, gk, sk, sk, "bf16")):
            assert G.same_bits(H.to_np_bits(t, k), b, k).all(), (n, off, k)
