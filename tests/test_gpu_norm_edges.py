"""The grad norm at the edges of its launch rules, against the CPU checker's
compensated float64 sum (1e-12 relative; the coefficient bit for bit)."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from slideformer_amd import _lib
from tests import _hip as H

pytestmark = pytest.mark.gpu

ONE = 131_072        # most elements that one workgroup takes, fold included


def _bits(g, kind):
    b = H.to_np_bits(g, kind)
    return b.view(np.float32) if kind == "f32" else b


@pytest.mark.parametrize("kind", ["bf16", "f32", "f16"])
@pytest.mark.parametrize("n", [1, ONE - 1, ONE, ONE + 1, ONE + 7])
def test_norm_around_the_one_workgroup_limit(n, kind, hip_device):
    """Both sides of the limit, from an odd element on, overwriting and adding
    to a running sum; the partials' workspace is poisoned (a result that read a
    partial no launch wrote would be NaN)."""
    g = (torch.randn(n + 3, device=hip_device) * 1e-2).to(H.TD[kind])[3:]
    L = _lib.load()
    need = L.la_grad_sqnorm_workspace(n)
    assert (need == 8) == (n <= ONE)
    ws = torch.full((need // 8,), float("nan"), dtype=torch.float64, device=hip_device)
    sq = torch.full((1,), 2.5, dtype=torch.float64, device=hip_device)
    cn = torch.zeros(2, device=hip_device)
    exact = O.grad_sqnorm(_bits(g, kind), None if kind == "f32" else kind)
    print(f"norm n={n} {kind}", flush=True)
    for accumulate, want in ((1, 2.5 + exact), (0, exact)):
        _lib.check(L.la_grad_norm_clip(H.CODE[kind], g.data_ptr(), n, ws.data_ptr(), need, sq.data_ptr(), accumulate,
                                       1.0, cn.data_ptr(), cn.data_ptr() + 4,
                                       torch.cuda.current_stream().cuda_stream), "la_grad_norm_clip")
        got = sq.item()
        assert abs(got - want) <= 1e-12 * want
        coef, norm = O.clip_coef(got, 1.0)
        assert cn[0].item() == np.float32(coef) and cn[1].item() == np.float32(norm)
