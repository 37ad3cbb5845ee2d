"""The resident Sinkhorn solve (csrc/sk_resident_kernel.h): the whole iteration
in one launch.  Sizes at the edges of its tiles, one workgroup per problem and
several (merged by every workgroup, and by column owners), steps it refuses
and redoes from the cost, degenerate marginals, and a schedule longer than a
launch takes (which the streaming steps serve).

The oracle is run in float64.  A log-plan entry is one float32 rounding of a
value up to 2^7 (4e-6) plus the potentials' error; every quantity is held to
the 1e-5 the parity tests use.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import torchmatch_amd  # noqa: F401
from oracle import sinkhorn as sk
import sk_parity
import workloads
from torchmatch_amd.transport.matrix import Backend, solve

pytestmark = pytest.mark.gpu

# (B, N, M): one row, one column, tile edges and remainders of each layout
SHAPES = [
    (3, 1, 1), (2, 1, 70), (2, 70, 1), (2, 33, 64), (2, 64, 65), (3, 127, 96), (2, 130, 128),
    (1, 260, 129), (2, 97, 193), (1, 500, 256), (2, 65, 257), (1, 129, 385), (1, 300, 513),
    (1, 70, 769), (2, 40, 1024), (1, 130, 1025), (1, 34, 1537), (1, 150, 2048), (1, 20, 2049),
    (1, 70, 4096), (300, 20, 24),
]


def _check(label, cost, a, b, eps, n_iter, device, rho=None, scaling=None, mask=None):
    c = cost if mask is None else cost.masked_fill(~mask, float("inf"))
    dev = {"a": a.to(device), "b": b.to(device), "reg": eps, "n_iter": n_iter,
           "scaling": scaling, "mask": None if mask is None else mask.to(device)}
    if rho is None:
        ref = dict(zip(("plan", "f", "g"), sk.log_sinkhorn_plan(
            c, eps=eps, n_iter=n_iter, a=a, b=b, scaling=scaling, dtype=torch.float64)))
        # the resident plan, and the call that reads the potentials too
        got = dict(zip(("plan", "f", "g"), solve(cost.to(device), unpack=True, **dev)))
        ref["resident plan"], got["resident plan"] = ref["plan"], solve(cost.to(device), **dev)
    else:
        ref = {"plan": sk.unbalanced_sinkhorn_plan(
            c, eps=eps, n_iter=n_iter, rho=rho, a=a, b=b, scaling=scaling,
            dtype=torch.float64)[0]}
        got = {"plan": solve(cost.to(device), backend=Backend.UNBALANCED_SINKHORN, rho=rho,
                             **dev)}
    torch.cuda.synchronize()
    for name, x in got.items():
        err = sk_parity.logp_err(x, ref[name])
        print(f"{label} {name}: {err:.2e}", flush=True)
        assert err <= sk_parity.ELEM_BOUND, (label, name, err)


@pytest.mark.parametrize("mode", [None, "exact"])
@pytest.mark.parametrize("rho", [None, 0.7])
def test_tile_edges(mode, rho, device, monkeypatch):
    """Every step from P, and (``exact``) every step from the cost."""
    if mode:
        monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", mode)
    for B, N, M in SHAPES:
        cost = workloads.sinkhorn_points(B, N, M, 8, seed=N + M)
        if N > 4 and M > 8:
            cost[0, 2, :] = float("inf")      # an empty row and column
            cost[B - 1, :, 5] = float("inf")
        _check(f"{(B, N, M)} rho {rho} {mode}", cost, workloads.dirichlet(B, N, seed=1),
               workloads.dirichlet(B, M, seed=2), 0.05, 12, device, rho=rho)


@pytest.mark.parametrize(("B", "N", "M"), [(2, 60, 90), (2, 700, 300), (1, 400, 1200)])
def test_masked_and_scaled(B, N, M, device):
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N)
    mask = torch.rand(B, N, M, generator=torch.Generator().manual_seed(3)) < 0.7
    a, b = workloads.dirichlet(B, N, seed=4), workloads.dirichlet(B, M, seed=5)
    _check("scaled", cost, a, b, 0.03, 40, device, scaling=0.8, mask=mask)
    # 200 epsilons: more runs than one launch takes
    _check("long schedule", cost, a, b, 0.03, 200, device, scaling=0.985, mask=mask)


@pytest.mark.parametrize(("B", "N", "M"), [(2, 60, 90), (2, 500, 300), (1, 300, 1200)])
def test_degenerate_marginals(B, N, M, device):
    """Zero and tiny masses, rows whose only partners carry none, and an epsilon
    at which the row-maximum start underflows (the step is refused and redone)."""
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=M)
    a, b = workloads.dirichlet(B, N, seed=6), workloads.dirichlet(B, M, seed=7)
    a[:, 3] = 0.0
    b[:, 4:9] = 0.0
    a[:, 5] = 1e-30
    b[0, 11] = 1e-25
    cost[0, 7, :] = float("inf")
    cost[0, 7, 4:9] = 0.25                    # allowed only where b is zero
    _check("degenerate", cost, a, b, 0.05, 20, device)
    _check("degenerate, unbalanced", cost, a, b, 0.05, 20, device, rho=0.3)
    # |C| / eps up to 2000: float32 itself resolves the log plan to 1e-4 there,
    # so the potentials (in units of the cost) are what is compared
    args = {"reg": 5e-4, "n_iter": 15, "a": a.to(device), "b": b.to(device)}
    ref = sk.log_sinkhorn_plan(cost, eps=5e-4, n_iter=15, a=a, b=b, dtype=torch.float64)
    got = solve(cost.to(device), unpack=True, **args)
    for x, r in zip(got[1:], ref[1:]):
        # the float32 step epsilon of the solve: 3e-8 of potentials below 2
        assert sk_parity.pot_err(x, r) <= 1e-6


@pytest.mark.parametrize(("B", "N", "M", "rho"), [
    (2, 1, 3, None), (2, 65, 64, 0.5), (3, 120, 250, None), (1, 300, 513, None),
    (1, 260, 1000, 0.5),
])
def test_float64(B, N, M, rho, device):
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N + 1).double()
    a = workloads.dirichlet(B, N, seed=8).double()
    b = workloads.dirichlet(B, M, seed=9).double()
    if rho is None:
        ref = sk.log_sinkhorn_plan(cost, eps=0.05, n_iter=40, a=a, b=b, dtype=torch.float64)[0]
        got = solve(cost.to(device), a=a.to(device), b=b.to(device), reg=0.05, n_iter=40)
    else:
        ref = sk.unbalanced_sinkhorn_plan(cost, eps=0.05, n_iter=40, rho=rho, a=a, b=b,
                                          dtype=torch.float64)[0]
        got = solve(cost.to(device), backend=Backend.UNBALANCED_SINKHORN, rho=rho,
                    a=a.to(device), b=b.to(device), reg=0.05, n_iter=40)
    # values below 2^6, ulp 7e-15, a few roundings a step that do not add up
    assert sk_parity.logp_err(got, ref) <= 2e-13


@pytest.mark.parametrize("mode", [None, "exact"])
@pytest.mark.parametrize("where", ["row", "column", "both"])
@pytest.mark.parametrize(("B", "N", "M", "dtype", "far"), [
    (2, 60, 90, "float64", 1e9), (2, 60, 90, "float64", 1e13), (1, 400, 300, "float64", 1e11),
    (1, 200, 1000, "float64", 1e9), (2, 60, 90, "float32", 1e8), (1, 400, 1200, "float32", 1e8)])
def test_far_row_and_column(B, N, M, dtype, far, where, mode, device, monkeypatch):
    """A row and a column of finite costs so large (|C| / eps of 3e9 and more)
    that a maximum held in float32 misses the sum by more than exp's range.
    Epsilon is a power of two, the same in both types."""
    if mode:
        monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", mode)
    eps, dt = 2.0 ** -5, getattr(torch, dtype)
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=M).to(dt)
    if where != "column":
        cost[:, 3, :] = far
    if where != "row":
        cost[:, :, 7] = far
    a, b = workloads.dirichlet(B, N, seed=1).to(dt), workloads.dirichlet(B, M, seed=2).to(dt)
    ref = sk.log_sinkhorn_plan(cost.double(), eps=eps, n_iter=10, a=a.double(), b=b.double(),
                               dtype=torch.float64)[0]
    got = solve(cost.to(device), a=a.to(device), b=b.to(device), reg=eps, n_iter=10)
    if dtype == "float32":  # entries of a far row or column that carry no mass
        got = got.double().cpu()
        none = ref < -1e6
        assert ((got - ref).abs()[none] <= 2.0 ** -23 * ref.abs()[none]).all()
        got[none] = ref[none]
    err = sk_parity.logp_err(got, ref)
    # a few float64 roundings of |C| / eps in each of the two, over the float32
    # tests' bound or test_float64's
    bound = 16 * 2.0 ** -52 * far / eps + (sk_parity.ELEM_BOUND if dtype == "float32" else 2e-13)
    print(f"far {(B, N, M)} {dtype} {far:.0e} {where} {mode}: {err:.2e}, bound {bound:.2e}",
          flush=True)
    assert err <= bound


@pytest.mark.parametrize("mode", [None, "exact"])
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize(("B", "N", "M"), [(3, 64, 80), (1, 400, 300), (1, 300, 1200)])
def test_unbalanced_large_costs(B, N, M, dtype, mode, device, monkeypatch):
    """Costs far above rho: the plan's mass, and with it every multiplier, is
    e^-(cost / 2 rho) or less, below any float, while the log plan is an ordinary
    number.  A constant added to every cost; an isolated pair (a row and a
    column far from all others and close to each other) and an isolated row;
    two blocks whose masses differ by e^-150; a far column of finite costs.
    Epsilon and rho are powers of two, the same in both types."""
    if mode:
        monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", mode)
    dt = getattr(torch, dtype)
    base = workloads.sinkhorn_points(B, N, M, 8, seed=M).to(dt)
    a, b = workloads.dirichlet(B, N, seed=1).to(dt), workloads.dirichlet(B, M, seed=2).to(dt)
    cases = {f"offset {x}": base + x for x in (200.0, 500.0, 3000.0)}
    c = base.clone()
    c[:, 3, :] = c[:, :, 7] = 400.0
    c[:, 3, 7] = 0.5
    c[:, 9, :] = 700.0
    cases["isolated"] = c
    c = base + 300.0
    c[:, : N // 2, : M // 2] -= 300.0
    c[:, : N // 2, M // 2 :] = c[:, N // 2 :, : M // 2] = 9000.0
    cases["blocks"] = c
    c = base.clone()
    c[:, :, 7] = 1e9
    cases["far column"] = c
    for name, cost in cases.items():
        kw = {"rho": 1.0, "n_iter": 30 if name != "offset 500.0" else 100}
        ref = sk.unbalanced_sinkhorn_plan(cost.double(), eps=0.125, a=a.double(), b=b.double(),
                                          dtype=torch.float64, **kw)[0]
        got = solve(cost.to(device), backend=Backend.UNBALANCED_SINKHORN, reg=0.125,
                    a=a.to(device), b=b.to(device), **kw)
        scale = 1.0 + ref[torch.isfinite(ref)].abs()
        sk_parity.logp_err(got, ref)  # the same entries finite
        err = ((got.cpu().double() - ref).abs()[torch.isfinite(ref)] / scale).max().item()
        # float32: the parity bound, and the output's and K's rounding (2^-24 of
        # an entry each); float64: a few roundings of the same size
        bound = 1e-5 if dtype == "float32" else 64 * 2.0 ** -52
        print(f"unbalanced {name} {(B, N, M)} {dtype} {mode}: {err:.2e}", flush=True)
        assert err <= bound, (name, err)


@pytest.mark.parametrize("rho", [None, 0.3])
@pytest.mark.parametrize(("B", "N", "M"), [(2, 60, 90), (1, 400, 300)])
def test_denormal_marginals(B, N, M, rho, device):
    """Masses below float32's normal range: their multipliers' reciprocals are
    not float32 numbers."""
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N)
    a, b = workloads.dirichlet(B, N, seed=6), workloads.dirichlet(B, M, seed=7)
    a[:, 5], b[:, 11], b[:, 20] = 1e-40, 3e-39, 1e-44
    kw = {"a": a.to(device), "b": b.to(device), "reg": 0.05, "n_iter": 20}
    if rho is None:
        ref = sk.log_sinkhorn_plan(cost, eps=0.05, n_iter=20, a=a, b=b, dtype=torch.float64)[0]
        got = solve(cost.to(device), **kw)
    else:
        ref = sk.unbalanced_sinkhorn_plan(cost, eps=0.05, n_iter=20, rho=rho, a=a, b=b,
                                          dtype=torch.float64)[0]
        got = solve(cost.to(device), backend=Backend.UNBALANCED_SINKHORN, rho=rho, **kw)
    err = sk_parity.logp_err(got, ref)
    # log masses down to -101: one float32 rounding of that (4e-6) more
    assert err <= sk_parity.ELEM_BOUND + 4e-6, err


@pytest.mark.parametrize(("B", "N", "M", "dtype", "rho"), [
    (2, 400, 300, "float32", None), (70, 300, 200, "float32", 0.7), (1, 300, 1200, "float32", None),
    (1, 1810, 43, "float32", None), (2, 700, 300, "float64", None), (2, 300, 256, "float64", 0.7)])
def test_given_up(B, N, M, dtype, rho, device, monkeypatch):
    """Workgroups that do not wait for the others of their problem at all (the
    limit of every wait is 0): the problems they give up are solved behind the
    launch, whatever is left of the others' results."""
    dt = getattr(torch, dtype)
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N + M)
    mask = None
    if dtype == "float32":
        mask = torch.rand(B, N, M, generator=torch.Generator().manual_seed(3)) < 0.8
        mask[0, 2, :] = False
        mask[0, :, 5] = False
    a, b = workloads.dirichlet(B, N, seed=1), workloads.dirichlet(B, M, seed=2)
    a[:, 4] = b[:, 9] = 0.0
    c = cost.to(dt) if mask is None else cost.masked_fill(~mask, float("inf"))
    kw = {"a": a.to(device, dt), "b": b.to(device, dt), "reg": 0.05, "n_iter": 12, "scaling": 0.7,
          "mask": None if mask is None else mask.to(device)}
    if rho is None:
        ref = sk.log_sinkhorn_plan(c, eps=0.05, n_iter=12, a=a.to(dt), b=b.to(dt), scaling=0.7,
                                   dtype=torch.float64)[0]
    else:
        kw |= {"backend": Backend.UNBALANCED_SINKHORN, "rho": rho}
        ref = sk.unbalanced_sinkhorn_plan(c, eps=0.05, n_iter=12, rho=rho, a=a.to(dt), b=b.to(dt),
                                          scaling=0.7, dtype=torch.float64)[0]
    monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", "late")
    for _ in range(2):
        err = sk_parity.logp_err(solve(cost.to(device, dt), **kw), ref)
        print(f"given up {(B, N, M)} {dtype} rho {rho}: {err:.2e}", flush=True)
        assert err <= (sk_parity.ELEM_BOUND if dtype == "float32" else 2e-13)


@pytest.mark.parametrize("n", [2, 40, 600])
def test_tiny_masses_that_drift(n, device):
    """A row and a column of tiny mass that only have each other, in a problem
    without a solution (row 0 alone cannot fill column 0), so that the potentials
    drift by a factor a step: their multipliers become denormal while they are
    all that some sums have."""
    cost = torch.full((1, n, n), float("inf"))
    k = n // 2  # k independent 2 x 2 problems
    for i in range(k):
        cost[0, 2 * i: 2 * i + 2, 2 * i: 2 * i + 2] = torch.tensor(
            [[-19.32 + 0.01 * i, float("inf")], [-19.74, -19.30]])
    a = torch.tensor([0.215, 7.85e-26]).repeat(k)[None] / k
    b = torch.tensor([0.749, 2.51e-21]).repeat(k)[None] / k
    ref = sk.log_sinkhorn_plan(cost, eps=2.0 ** -5, n_iter=50, a=a, b=b, dtype=torch.float64)[0]
    got = solve(cost.to(device), reg=2.0 ** -5, n_iter=50, a=a.to(device), b=b.to(device))
    sk_parity.logp_err(got, ref)  # the same entries finite
    fin = torch.isfinite(ref)
    d = (got.cpu().double() - ref).abs()[fin] / (1.0 + ref[fin].abs())
    print(f"tiny masses {n}: {d.max().item():.2e}", flush=True)
    # log plans down to -500, each rounded to 2^-24 of that, over potentials of 600
    assert d.max().item() <= 1e-6


@pytest.mark.skipif(np.finfo(np.longdouble).nmant < 63, reason="needs an 80-bit long double")
@pytest.mark.parametrize(("N", "M", "eps", "n_iter", "rho"), [
    (300, 200, 0.05, 100, None), (64, 300, 0.1, 100, None), (300, 200, 0.05, 100, 1.0),
    (120, 90, 0.02, 60, 0.5)])
def test_float64_plan_is_no_further_from_80_bits(N, M, eps, n_iter, rho, device, monkeypatch):
    """A float64 resident plan against the same recurrence in 80 bits, and the
    streaming steps' plan: the resident one is no further off (2-norm; one
    rounding of every entry is about 6e-17 of it)."""
    cost = workloads.sinkhorn_points(1, N, M, 8, seed=N + 1).double()
    a, b = (workloads.dirichlet(1, k, seed=s).double() for k, s in ((N, 1), (M, 2)))
    L = np.longdouble
    K = (-(cost[0].numpy() / eps)).astype(L)  # K as float64 has it, on both sides
    la, lb = np.log(a[0].numpy().astype(L)), np.log(b[0].numpy().astype(L))
    lu, lv = np.zeros(N, L), np.zeros(M, L)
    damp = L(1.0 if rho is None else 1.0 / (1.0 + eps / rho))

    def lse(x, axis):
        m = x.max(axis)
        return np.log(np.exp(x - np.expand_dims(m, axis)).sum(axis)) + m

    for _ in range(n_iter):
        lu = damp * (la - lse(K + lv[None, :], 1))
        lv = damp * (lb - lse(K + lu[:, None], 0))
    true = lu[:, None] + K + lv[None, :]
    kw = {"a": a.to(device), "b": b.to(device), "reg": eps, "n_iter": n_iter}
    if rho is not None:
        kw |= {"backend": Backend.UNBALANCED_SINKHORN, "rho": rho}
    err = []
    for mode in (None, "0"):
        if mode:
            monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", mode)
        d = solve(cost.to(device), **kw)[0].cpu().numpy().astype(L) - true
        err.append(float(np.sqrt((d * d).sum() / (true * true).sum())))
    print(f"80 bits {(N, M)} rho {rho}: resident {err[0]:.2e}, steps {err[1]:.2e}", flush=True)
    assert err[0] <= err[1] and err[0] <= 1e-16


@pytest.mark.parametrize(("B", "N", "M"), [
    (1, 1810, 43), (51, 634, 42), (1, 2000, 17), (2, 700, 5), (1, 1500, 1), (1, 700, 100)])
def test_fewer_workgroups_than_merge_groups(B, N, M, device):
    """Narrow and tall: the threads that merge a column are more than the
    workgroups that have a partial of it (all but the last shape)."""
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N + M)
    _check(f"{(B, N, M)}", cost, workloads.dirichlet(B, N, seed=1),
           workloads.dirichlet(B, M, seed=2), 0.05, 20, device)


@pytest.mark.parametrize(("B", "N", "M"), [(2, 900, 7), (1, 1200, 40), (1, 600, 60)])
def test_fewer_workgroups_than_merge_groups_float64(B, N, M, device):
    test_float64(B, N, M, None, device)


@pytest.mark.parametrize(("B", "N", "M", "dtype", "rho"), [
    (4, 604, 174, "float32", None), (2, 63, 73, "float32", None),
    (2, 60, 120, "float32", None), (5, 191, 55, "float64", None),
    (2, 300, 256, "float32", 0.7), (3, 38, 43, "float32", 0.7), (2, 90, 73, "float64", 0.7)])
def test_potentials_keep_the_steps_bits(B, N, M, dtype, rho, device, monkeypatch):
    """Potentials show the neutral mode's rounding: a call that reads them gets
    the streaming steps' bits, except on the shapes whose steps carry float64
    potentials."""
    dt = getattr(torch, dtype)
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=N).to(device, dt)
    args = {"a": workloads.dirichlet(B, N, seed=1).to(device, dt),
            "b": workloads.dirichlet(B, M, seed=2).to(device, dt), "reg": 0.05, "n_iter": 60,
            "unpack": True}
    if rho is not None:
        args |= {"backend": Backend.UNBALANCED_SINKHORN, "rho": rho}
    got = solve(cost, **args)
    monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", "0")
    for x, y in zip(got, solve(cost, **args)):
        assert torch.equal(x, y)


@pytest.mark.parametrize(("B", "N", "M"), [(5, 120, 1028), (2, 300, 200)])
def test_streaming_groups_same_bits(B, N, M, device, monkeypatch):
    """The streaming step (which serves captures and matrices too large for the
    chip) on shapes the resident solve takes by default: every batch-group
    split gives the same bits, within the bound of the resident plan."""
    cost = workloads.sinkhorn_points(B, N, M, 8, seed=31).to(device)
    args = {"a": workloads.dirichlet(B, N, seed=1).to(device),
            "b": workloads.dirichlet(B, M, seed=2).to(device), "reg": 0.05, "n_iter": 30}
    resident = solve(cost, **args)
    monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_FUSED", "1")
    plans = []
    for groups in ("1", "2", "4"):
        monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_GROUPS", groups)
        plans.append(solve(cost, **args))
    assert torch.equal(plans[0], plans[1]) and torch.equal(plans[0], plans[2])
    assert sk_parity.logp_err(plans[0], resident.cpu()) <= sk_parity.ELEM_BOUND


def test_streaming_steps_still_match_oracle(device, monkeypatch):
    """What other files hold to the oracle through calls that now run resident,
    once more on the streaming steps."""
    import test_sinkhorn_f64_gpu as f64
    import test_sinkhorn_fullsize_gpu as full
    import test_sinkhorn_gpu as f32

    monkeypatch.setenv("TORCHMATCH_AMD_SINKHORN_RESIDENT", "0")
    f64.test_unbalanced_f64_matches_oracle(device)
    f64.test_f64_scaling_and_mask(device)
    f32.test_step_shapes_match_oracle(None, (2, 150, 1500), device, monkeypatch)
    f32.test_unbalanced_matches_oracle(1, 500, 300, 0.02, 100, 1.0, device)
    f32.test_forbidden_cells_rows_and_columns(device)
    case = full.INDEX["c4"]
    cost, a, b = full._inputs(case)
    full._check("C4 streaming", case, *full._run_device(case, cost, a, b, device), cost,
                full._fixture(case))
