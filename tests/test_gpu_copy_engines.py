"""Host arrays over the copy engines where the caller asks for them: the choice of LayerAdam and of a pipeline."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from slideformer_amd import LayerAdam
from tests import _hip as H

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
