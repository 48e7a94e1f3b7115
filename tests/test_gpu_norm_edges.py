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


@pytest.mark.parametrize("kind", ["bf16", "f32", "f16"])
@pytest.mark.parametrize("sizes", [(5, 0, 3), (256, 1, 255, 257), (0, 0, 0), (4099,) * 32, (700_001, 3, 1_048_576, 9),
                                   (1_500_000, 64, 131_073, 2_000_003)])
def test_norm_over_buffers_whose_runs_share_trips(sizes, kind, hip_device):
    """la_grad_norm_multi numbers the 256-element runs of all buffers in one
    sequence: empty buffers, buffers of scalars only, partial runs and odd
    starts, on one workgroup and on many; also a sum within 1e-12 when the
    buffers are given in the other order, and single buffers with the bits of
    la_grad_norm_clip."""
    L = _lib.load()
    bufs = [(torch.randn(n + 8, device=hip_device) * 1e-2).to(H.TD[kind])[k % 4:k % 4 + n]
            for k, n in enumerate(sizes)]
    exact = sum(O.grad_sqnorm(_bits(g, kind), None if kind == "f32" else kind) for g in bufs if g.numel())
    need = L.la_grad_sqnorm_workspace(max(1, sum(sizes)))
    stream = torch.cuda.current_stream().cuda_stream

    def run(order):
        ws = torch.full((need // 8,), float("nan"), dtype=torch.float64, device=hip_device)
        sq = torch.full((1,), float("nan"), dtype=torch.float64, device=hip_device)
        cn = torch.zeros(2, device=hip_device)
        flat = [x for g in order for x in (g.data_ptr(), g.numel())]
        arr = ctypes.cast((ctypes.c_uint64 * len(flat))(*flat), ctypes.POINTER(_lib.LaGradBuffer))
        _lib.check(L.la_grad_norm_multi(H.CODE[kind], arr, len(order), ws.data_ptr(), need, sq.data_ptr(), 0, 0.5,
                                        cn.data_ptr(), cn.data_ptr() + 4, stream), "la_grad_norm_multi")
        return sq.item(), cn

    print(f"multi norm {sizes[:6]} {kind}", flush=True)
    for order in (bufs, bufs[::-1]):
        got, cn = run(order)
        assert abs(got - exact) <= 1e-12 * exact
        coef, norm = O.clip_coef(got, 0.5)
        assert cn[0].item() == np.float32(coef) and cn[1].item() == np.float32(norm)
    for g in bufs:
        if g.numel():
            assert run([g])[0] == H.norm_clip(g, 0.5)[0].item()


def test_norms_of_more_runs_than_one_launch_numbers(hip_device):
    """The small-grid build numbers at most 4096 runs per launch (the product
    build 2^31): a larger buffer is summed in parts and a larger list buffer by
    buffer, to the same 1e-12, with the coefficient written once."""
    L = H.load_small_grid()
    stream = torch.cuda.current_stream().cuda_stream
    ws = torch.full((2,), float("nan"), dtype=torch.float64, device=hip_device)
    big = (torch.randn(5_000_009, device=hip_device) * 1e-2).bfloat16()[1:]
    bufs = [big, big[:700_001], big[3:2_000_000], big[:0], big[5:10]]
    for which in ("single", "multi"):
        sq = torch.full((1,), float("nan"), dtype=torch.float64, device=hip_device)
        cn = torch.zeros(2, device=hip_device)
        if which == "single":
            exact = O.grad_sqnorm(_bits(big, "bf16"), "bf16")
            rc = L.la_grad_norm_clip(1, big.data_ptr(), big.numel(), ws.data_ptr(), 16, sq.data_ptr(), 0, 0.5,
                                     cn.data_ptr(), cn.data_ptr() + 4, stream)
        else:
            exact = sum(O.grad_sqnorm(_bits(g, "bf16"), "bf16") for g in bufs if g.numel())
            flat = [x for g in bufs for x in (g.data_ptr(), g.numel())]
            arr = ctypes.cast((ctypes.c_uint64 * len(flat))(*flat), ctypes.POINTER(_lib.LaGradBuffer))
            rc = L.la_grad_norm_multi(1, arr, len(bufs), ws.data_ptr(), 16, sq.data_ptr(), 0, 0.5, cn.data_ptr(),
                                      cn.data_ptr() + 4, stream)
        assert rc == 0
        got = sq.item()
        print(f"norm in parts, {which}", flush=True)
        assert abs(got - exact) <= 1e-12 * exact
        coef, norm = O.clip_coef(got, 0.5)
        assert cn[0].item() == np.float32(coef) and cn[1].item() == np.float32(norm)


def test_gathered_norm_reads_changes_and_second_finish(hip_device):
    """The accumulator's partials over calls of one and of many workgroups and of
    several dtypes: a sum read between two adds, one changed in place (as an
    all-reduce over ranks does) before finish, more adds after a finish."""
    from slideformer_amd import LayerAdam

    def make(n, kind):
        return (torch.randn(n + 1, device=hip_device) * 1e-2).to(H.TD[kind])[1:]

    def exact(grads):
        return sum(O.grad_sqnorm(_bits(g, k), None if k == "f32" else k) for g, k in grads if g.numel())

    acc = LayerAdam().grad_norm_begin(hip_device)
    assert acc.sqnorm.item() == 0.0
    grads = [(make(n, k), k) for n, k in [(ONE, "bf16"), (ONE + 1, "f32"), (0, "bf16"), (2_000_003, "f16"), (5, "f32")]]
    acc.add(grads[0][0])
    acc.add([g for g, _ in grads[1:]])
    want = exact(grads)
    for _ in range(2):
        assert abs(acc.sqnorm.item() - want) <= 1e-12 * want
    acc.sqnorm.mul_(4.0)
    for more in ([], [(make(700_001, "bf16"), "bf16"), (make(9, "bf16"), "bf16")]):
        before = exact(grads) * 4.0
        for g, _ in more:
            acc.add(g)
        coef, norm = acc.finish(0.5)
        want = before + exact(more)
        got = acc.sqnorm.item()
        print(f"gathered norm, {len(more)} more", flush=True)
        assert abs(got - want) <= 1e-12 * want
        c_ref, n_ref = O.clip_coef(got, 0.5)
        assert coef.item() == np.float32(c_ref) and norm.item() == np.float32(n_ref)


def test_gathered_norm_in_a_replayed_graph(hip_device):
    """add, add, finish captured on an accumulator made before: every replay is the norm of the grads of its time."""
    from slideformer_amd import LayerAdam

    a, b = (torch.zeros(n, device=hip_device, dtype=torch.bfloat16) for n in (1_000_003, 77))
    adam = LayerAdam()
    warm, acc = adam.grad_norm_begin(hip_device), adam.grad_norm_begin(hip_device)
    warm.add(a)
    warm.add([b, a])
    warm.finish(1.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        acc.add(a)
        acc.add([b, a])
        coef, norm = acc.finish(1.0)
    for replay, scale in enumerate((1e-2, 1.0, 1e-3)):
        for t in (a, b):
            t.copy_(torch.randn(t.numel(), device=hip_device) * scale)
        graph.replay()
        torch.cuda.synchronize()
        if replay:              # the sum that the replay left, finished outside the graph
            eager = acc.finish(1.0)
            assert torch.equal(eager[0], coef) and torch.equal(eager[1], norm)
        sq = 2 * O.grad_sqnorm(_bits(a, "bf16"), "bf16") + O.grad_sqnorm(_bits(b, "bf16"), "bf16")
        print(f"gathered norm replay, scale {scale}", flush=True)
        # the float64 sum is within 1e-12, so the fp32 norm is within one rounding of its last place
        assert abs(norm.item() - sq ** 0.5) <= 2.0 ** -23 * sq ** 0.5
        assert coef.item() == np.float32(O.clip_coef(float(norm.item()) ** 2, 1.0)[0])


def test_sqnorm_is_the_running_sum_itself(hip_device):
    """acc.sqnorm is one tensor for the accumulator's life: taken before the adds it holds each of them as its
    stream gets there, changed in place (an all-reduce over ranks) it is what finish takes, and reading the
    attribute launches nothing, so it needs no order with adds that still run on another stream."""
    from slideformer_amd import LayerAdam

    grads = [(torch.randn(n, device=hip_device) * 1e-2).bfloat16() for n in (300_001, 5, ONE + 1)]
    sums = [O.grad_sqnorm(_bits(g, "bf16"), "bf16") for g in grads]
    acc = LayerAdam().grad_norm_begin(hip_device)
    held = acc.sqnorm
    torch.cuda.synchronize()
    acc.add(grads[0])
    assert abs(held.item() - sums[0]) <= 1e-12 * sums[0]
    side = torch.cuda.Stream()
    acc.add(grads[1:], stream=side)
    assert acc.sqnorm is held
    side.synchronize()
    want = sum(sums)
    assert abs(held.item() - want) <= 1e-12 * want
    held.mul_(9.0)
    coef, norm = acc.finish(0.25)
    c_ref, n_ref = O.clip_coef(held.item(), 0.25)
    assert abs(held.item() - 9.0 * want) <= 9e-12 * want
    assert coef.item() == np.float32(c_ref) and norm.item() == np.float32(n_ref)


TRIP = 32_768     # elements that the small-grid build's two workgroups read in one trip


@pytest.mark.parametrize("kind", ["bf16", "f32", "f16"])
@pytest.mark.parametrize("sizes,off", [((TRIP, TRIP), 0), ((2 * TRIP, 0, TRIP, 3 * TRIP, 0), 0), ((0, TRIP), 0),
                                       ((TRIP, TRIP - 256, TRIP), 0), ((TRIP + 256, TRIP), 0),
                                       ((TRIP + 4, TRIP - 4), 0), ((3 * TRIP + 3, 2 * TRIP + 1), 1)])
def test_norm_over_buffers_of_whole_trips(sizes, off, kind, hip_device):
    """Buffers that are whole trips of the grid, alone, with empty ones among them, and beside one whose last run or
    last trip is not whole; also whole but for the elements before and after the aligned groups."""
    L = H.load_small_grid()
    bufs = [(torch.randn(n + 8, device=hip_device) * 1e-2).to(H.TD[kind])[off:off + n] for n in sizes]
    exact = sum(O.grad_sqnorm(_bits(g, kind), None if kind == "f32" else kind) for g in bufs if g.numel())
    for order in (bufs, bufs[::-1]):
        ws = torch.full((2,), float("nan"), dtype=torch.float64, device=hip_device)
        sq = torch.full((1,), float("nan"), dtype=torch.float64, device=hip_device)
        flat = [x for g in order for x in (g.data_ptr(), g.numel())]
        arr = ctypes.cast((ctypes.c_uint64 * len(flat))(*flat), ctypes.POINTER(_lib.LaGradBuffer))
        print(f"whole trips {sizes} {off} {kind}", flush=True)
        assert L.la_grad_norm_multi(H.CODE[kind], arr, len(order), ws.data_ptr(), 16, sq.data_ptr(), 0, 0.0, None,
                                    None, torch.cuda.current_stream().cuda_stream) == 0
        assert abs(sq.item() - exact) <= 1e-12 * exact
