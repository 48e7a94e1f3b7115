"""The update around the size up to which a launch runs without a residency cap
(8192 waves: 2,097,152 elements, 4,194,304 of the all-16-bit triples), single
and batched, against the CPU checker, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import _golden as G
from tests import _hip as H

pytestmark = pytest.mark.gpu

HP = (1e-3, 0.9, 0.999, 1e-8, 0.01, True)
K16 = {"bf16": "bf16", "f16": "f16", "f32": None}


def _host(bits, kind):
    return bits.view(np.float32) if kind == "f32" else bits


@pytest.mark.parametrize("extra", [-1, 0, 1, 257])
@pytest.mark.parametrize("triple", [("f32", "bf16", "f32"), ("bf16", "bf16", "bf16")], ids="-".join)
def test_update_around_one_round_of_waves(triple, extra, hip_device):
    pk, gk, sk = triple
    n = 8192 * (512 if pk == "bf16" else 256) + extra
    rng = np.random.default_rng(n)
    src = [torch.from_numpy(x.astype(np.float32)).to(H.TD[k]) for x, k in (
        (rng.normal(0, 0.02, n), pk), (rng.normal(0, 1e-3, n), gk), (rng.normal(0, 1e-3, n), sk),
        (np.abs(rng.normal(0, 1e-6, n)), sk))]
    bits = [H.to_np_bits(t, k) for t, k in zip(src, (pk, gk, sk, sk))]
    orc = O.OracleAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
    orc.update(1, *HP, *(_host(b, k) for b, k in zip(bits, (pk, gk, sk, sk))), p16=K16[pk], g16=K16[gk], s16=K16[sk])
    for route in ("single", "batched"):
        print(f"one round {triple} {extra} {route}", flush=True)
        dev = [t.to(hip_device) for t in src]
        opt = H.HipAdam(1e-3, (0.9, 0.999), 1e-8, 0.01, True)
        if route == "single":
            opt.update(1, *HP, *dev)
        else:
            opt.update_multi(1, *HP, [(*dev, None)])
        torch.cuda.synchronize()
        for t, b, k in zip(dev, bits, (pk, gk, sk, sk)):
            assert G.same_bits(H.to_np_bits(t, k), b, k).all(), (route, k)
