"""Sinkhorn calls under graph capture.  A shape that ordinarily runs in one
cooperative launch (which cannot be recorded) takes the streaming steps there,
with their bits; K is built once, by whichever call knows that nobody has yet.

Graphs are replayed several times, with new costs and eager work between the
replays, and every replay is compared with the eager streaming steps.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

import torchmatch_amd  # noqa: F401
import workloads
from torchmatch_amd import _native
from torchmatch_amd.transport.matrix import _sinkhorn

pytestmark = pytest.mark.gpu

SHAPES = [(2, 64, 80), (3, 300, 256), (1, 260, 1025)]
OPS = torch.ops.torchmatch_amd


def _inputs(shape, device, seed=0):
    B, N, M = shape
    return (workloads.sinkhorn_points(B, N, M, 8, seed=seed).to(device),
            workloads.dirichlet(B, N, seed=seed + 1).to(device),
            workloads.dirichlet(B, M, seed=seed + 2).to(device))


def _eager_steps(monkeypatch, fn):
    monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", "0")
    out = fn()
    torch.cuda.synchronize()
    monkeypatch.delenv("TORCHMATCH_AMD_SINKHORN_RESIDENT")
    return out


def _replays_match(graph, cost, outs, shape, device, monkeypatch, eager):
    for seed in (3, 4, 5):
        cost.copy_(_inputs(shape, device, seed)[0])
        want = _eager_steps(monkeypatch, eager)
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(outs, want):
            assert torch.equal(x, y), (shape, seed)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("potentials", [False, True])
def test_whole_call(shape, potentials, device, monkeypatch):
    cost, a, b = _inputs(shape, device)

    def call():
        out = _sinkhorn.log_sinkhorn_plan(cost, eps=0.05, n_iter=7, a=a, b=b,
                                          return_potentials=potentials)
        return out if potentials else (out,)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = call()
    _replays_match(graph, cost, outs, shape, device, monkeypatch, call)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_prepared_outside(shape, device, monkeypatch):
    """The preparation runs eagerly and leaves K to the iteration, which is
    recorded, twice: at the epsilon it was prepared for and from another."""
    cost, a, b = _inputs(shape, device)
    form = _sinkhorn.FORM_PLAN

    def prepare():
        return OPS.sinkhorn_prepare.form(cost, None, a, b, 0.05, False, form)[0]

    def iterate(ws):
        first = OPS.sinkhorn_iterate.form(cost, None, ws, [0.05] * 5, 0.0, 0.05, True, form)
        moved = OPS.sinkhorn_iterate.form(cost, None, ws, [0.2] * 2 + [0.05] * 3, 0.0, 0.05, True,
                                          form)
        again = OPS.sinkhorn_iterate.form(cost, None, ws, [0.2] * 2 + [0.1] * 3, 0.0, 0.2, True,
                                          form)
        return (*first, *moved, *again)

    ws = prepare()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = iterate(ws)

    def eager():
        # each solve on a workspace of its own
        res = []
        for sched, k in (([0.05] * 5, 0.05), ([0.2] * 2 + [0.05] * 3, 0.0),
                         ([0.2] * 2 + [0.1] * 3, 0.0)):
            w = OPS.sinkhorn_prepare.form(cost, None, a, b, k, False, form)[0]
            res += OPS.sinkhorn_iterate.form(cost, None, w, sched, 0.0, k, True, form)
        return res

    for seed in (3, 4, 5):
        cost.copy_(_inputs(shape, device, seed)[0])
        want = _eager_steps(monkeypatch, eager)
        prepare_into(ws, cost, a, b, shape, form)
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(outs, want):
            assert torch.equal(x, y), (shape, seed)


def prepare_into(ws, cost, a, b, shape, form, k_eps=0.05, offset=0):
    rc = _native.lib().tm_sinkhorn_prepare_form_f32(
        cost.data_ptr(), None, a.data_ptr(), b.data_ptr(), *shape, ctypes.c_float(k_eps), form,
        ws.data_ptr() + offset, ws.numel() - offset,
        torch.cuda.current_stream().cuda_stream)
    assert rc == _native.TM_OK


@pytest.mark.parametrize("shape", [(2, 63, 79), (1, 260, 1025)], ids=str)
def test_k_is_built_once(shape, device):
    """Where the preparation pass has written K (here: a workspace that is not
    16-byte aligned, so that neither call runs resident), the iteration does not
    write it again: it shows what was changed there in between."""
    B, N, M = shape
    cost, a, b = _inputs(shape, device)
    form = _sinkhorn.FORM_PLAN
    nbytes = _native.lib().tm_sinkhorn_workspace_bytes(B, N, M)
    eps, plans = 0.0625, []  # a power of two: K is exact
    for shift in (0.0, 0.5):
        ws = torch.zeros(nbytes + 16, dtype=torch.uint8, device=device)
        prepare_into(ws, cost, a, b, shape, form, k_eps=eps, offset=8)
        K = ws[8:8 + 4 * B * N * M].view(torch.float32)
        assert torch.equal(K, (-cost / eps).flatten())
        K += shift
        plan, lu, lv = torch.empty_like(cost), torch.empty_like(a), torch.empty_like(b)
        rc = _native.lib().tm_sinkhorn_iterate_form_f32(
            cost.data_ptr(), None, B, N, M, (ctypes.c_double * 1)(eps), 1, 0.0,
            ctypes.c_float(eps), form, plan.data_ptr(), lu.data_ptr(), lv.data_ptr(),
            ws.data_ptr() + 8, nbytes + 8, torch.cuda.current_stream().cuda_stream)
        assert rc == _native.TM_OK
        torch.cuda.synchronize()
        assert torch.equal(K, (-cost / eps).flatten() + shift)
        plans.append(lu)
    # log_u = log a - LSE(K) moves by the shift
    assert (plans[0] - plans[1] - 0.5).abs().max().item() < 1e-4
