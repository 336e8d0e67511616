"""Merged couplings and their entries against the oracle on dense systems.

A dense complex Hamiltonian makes every kind of entry: complex factors, two
coefficients on one coupling, a term and its conjugate on a diagonal output,
conjugated inputs.  The sizes are the edges of the tables: one block with few
rows, with as many as the paired forms hold, and several blocks.  A chain
whose every term has a factor of its own has more entries than a workgroup
holds, and takes the gather tables.  Plans of several blocks give bitwise the
right-hand side of the gather tables."""

from __future__ import annotations

import numpy as np
import pytest
import sympy as smp

from centrex_tlf_amd.lindblad import normalize_stop_event, population, prepare_lindblad_problem
from centrex_tlf_amd.lindblad._driver import build_save_plan
from centrex_tlf_amd.lindblad.native import DevicePlan
from centrex_tlf_amd.lindblad.systems import OBESystem
from oracle.lb_oracle import Oracle

from ._dense import CHAIN_PARAMETERS, chain_system, random_density
from ._gpu import require_gpu
from .systems import tlf_n39

pytestmark = pytest.mark.gpu


def dense_system(n: int, seed: int = 3):
    """H = H0 + w f(t) (A + A^T) / 2 + c B + conj(c) B^T, H0 dense Hermitian, one decay."""
    rng = np.random.default_rng(seed)
    h0 = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    h0 = h0 + h0.conj().T
    w, c = smp.Symbol("w", real=True), smp.Symbol("c", complex=True)
    H = smp.zeros(n, n)
    for i in range(n):
        for j in range(n):
            H[i, j] = complex(h0[i, j]) if i != j else float(h0[i, i].real)
            if abs(i - j) == 1:
                H[i, j] += w / 2 + (c * 0.75 if i < j else smp.conjugate(c) * 0.75)
    C = np.zeros((1, n, n), dtype=np.complex128)
    C[0, 0, n - 1] = 0.6
    return OBESystem(H_symbolic=H, C_array=C), {"amp": 0.7, "c0": 0.3 - 0.4j, "w": "amp*cos(3*t)", "c": "c0*exp(2*I*t)"}


@pytest.mark.parametrize("n", [2, 4, 7, 12])
def test_dense_rhs_matches_oracle(n):
    torch = require_gpu()
    system, params = dense_system(n)
    prepared = prepare_lindblad_problem(system, params, backend="host")
    plan, oracle = prepared.device_plan(), Oracle(prepared)
    ys = np.stack([prepared.layout.pack(random_density(n, seed=s)) for s in range(2)])
    ts = np.asarray([0.3, 1.7])
    got = plan.rhs(torch.as_tensor(ys, device="cuda"), torch.as_tensor(ts, device="cuda")).cpu().numpy()
    for b in range(2):
        want = oracle.rhs(ys[b], ts[b])
        # 2 n + 4 products per output, each within an ulp of the largest
        np.testing.assert_allclose(got[b], want, rtol=0, atol=4 * n * 2.3e-16 * np.abs(want).max() * 4)
    kw = dict(abstol=1e-9, reltol=1e-7, dt=1e-3)
    values, stats, _ = plan.solve(ys[0], 0.0, 0.05, output_kind="populations", n_traj=1, **kw)
    ref = oracle.solve_batch(ys[0], (0.0, 0.05), output="populations", output_when="final", **kw)
    assert int(stats[0, 3]) == 0 and int(stats[0, 0]) == int(np.ravel(ref["accepted"])[0])
    np.testing.assert_allclose(values.cpu().numpy()[0], np.ravel(ref["final"]), rtol=0, atol=1e-12)


def test_more_entries_than_fit_take_the_gather_tables():
    torch = require_gpu()
    n = 60
    prepared = prepare_lindblad_problem(chain_system(n), dict(CHAIN_PARAMETERS), backend="host")
    flat = prepared.flat_plan
    terms = len(flat["factors_re"])
    assert terms > 2 * 4095  # a value of its own for every term: more than the entry index holds
    for k in ("factors_re", "factors_im"):
        flat[k] = np.ascontiguousarray(np.asarray(flat[k]) * (1.0 + 1e-3 * np.arange(terms) / terms))
    plan, oracle = prepared.device_plan(), Oracle(prepared)
    y = prepared.layout.pack(random_density(n, seed=1))
    got = plan.rhs(torch.as_tensor(y, device="cuda"), torch.as_tensor(np.asarray([0.41]), device="cuda")).cpu().numpy()[0]
    want = oracle.rhs(y, 0.41)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-12 * np.abs(want).max())


@pytest.mark.parametrize("solver", ["dopri5", "tsit5"])
@pytest.mark.parametrize("variant", [1, 2, 3, 4])
def test_lean_form_is_bitwise_the_general_form(solver, variant):
    """Final outputs and the step integral (lean multi-wave form) against the
    last row and the integral of a trace of the accepted steps (general form),
    one, two and three slots a lane."""
    require_gpu()
    system, params, rho0, t_span, weights = tlf_n39()
    prepared = prepare_lindblad_problem(system, params, backend="host")
    plan, y0 = DevicePlan(prepared.flat_plan), prepared.layout.pack(rho0)
    t1 = np.asarray([0.02, 0.3, 0.11]) * t_span[1]
    kw = dict(abstol=1e-9, reltol=1e-7, dt=1e-8, solver=solver, variant=variant, restrict_support=False,
              weights=weights, with_integral=True, output_kind="full", n_traj=3)
    rows, stats, _, integral, counts, _ = plan.solve(y0, t_span[0], t1, trace=True, capacity=400, **kw)
    final, lean_stats, *_, lean_integral = plan.solve(y0, t_span[0], t1, **kw)
    assert bool((stats == lean_stats).all()) and int(stats[:, 3].max()) == 0
    for b, n in enumerate(counts.cpu().numpy()):
        assert n == int(stats[b, 0]) + 1 and bool((rows[b, n - 1] == final[b]).all())
    assert bool((integral == lean_integral).all())


def in_gather_form(flat: dict) -> dict:
    """The plan with further terms on every output, each of a value and an input
    of its own: too many values for the coupling tables, and at 1e-300 too small
    to change a rounded sum."""
    ptrs = np.asarray(flat["output_ptrs"])
    outputs = len(ptrs) - 1
    each = -(-4200 // outputs)
    at = np.repeat(ptrs[1:], each)
    value = 1e-300 * (1.0 + np.arange(at.size) / at.size)
    inputs = (np.repeat(np.arange(outputs), each) + np.tile(np.arange(each), outputs)) % outputs
    extra = dict(input_indices=inputs, coeff_indices=-1, factors_re=value,
                 factors_im=-value, input_conj=1, coeff_conj=0)
    out = dict(flat, output_ptrs=ptrs + (each * np.arange(outputs + 1)).astype(ptrs.dtype))
    for name, v in extra.items():
        old = np.asarray(flat[name])
        out[name] = np.ascontiguousarray(np.insert(old, at, np.asarray(v).astype(old.dtype)))
    return out


@pytest.mark.parametrize("case", ["n39", "dense 12"])
def test_several_blocks_round_as_the_gather_tables(case):
    torch = require_gpu()
    system, params = tlf_n39()[:2] if case == "n39" else dense_system(12)
    prepared = prepare_lindblad_problem(system, params, backend="host")
    plans = [DevicePlan(prepared.flat_plan), DevicePlan(in_gather_form(prepared.flat_plan))]
    n = 39 if case == "n39" else 12
    ys = torch.as_tensor(np.stack([prepared.layout.pack(random_density(n, seed=s)) for s in range(3)]), device="cuda")
    ts = torch.as_tensor(np.asarray([0.0, 0.3, 1.7]) * (1e-6 if case == "n39" else 1.0), device="cuda")
    got, want = (plan.rhs(ys, ts) for plan in plans)
    assert float(want.abs().max()) > 0.1 and int(((got - want).abs() >= 1e-290).sum()) == 0


@pytest.mark.parametrize("solver", ["dopri5", "tsit5", "fixed_rk2", "fixed_rk4", "fixed_dopri5"])
@pytest.mark.parametrize("n", [7, 12])
def test_every_kernel_in_gather_form(n, solver):
    """Final outputs, traces, save plans and stop events of the same system over
    couplings and over gather tables: 78 elements (two blocks) bitwise, 28 (one
    block, whose couplings are merged) to rounding."""
    require_gpu()
    system, params = dense_system(n)
    prepared = prepare_lindblad_problem(system, params, backend="host")
    plans = [DevicePlan(prepared.flat_plan), DevicePlan(in_gather_form(prepared.flat_plan))]
    y0 = prepared.layout.pack(random_density(n, seed=4)) / n
    save = build_save_plan(np.linspace(0.0, 0.3, 7), 0.0, 0.3, True)
    event = normalize_stop_event(population([0, 1], threshold=float(np.real(y0[0] + y0[1])) + 0.02), prepared)
    kw = dict(solver=solver, n_traj=2, restrict_support=False, abstol=1e-9, reltol=1e-7,
              dt=0.013 if solver.startswith("fixed") else 1e-3)
    fired = []
    for call in (dict(output_kind="full"), dict(output_kind="integral", weights=[(0, 0.7), (n - 1, 0.2)]),
                 dict(output_kind="populations", trace=True, save_plan=save, capacity=save.size),
                 dict(output_kind="full", trace=True, capacity=400), dict(output_kind="populations", stop_event=event)):
        if n == 7 and call.get("capacity") == 400:
            continue  # rows at steps whose sizes are rounded apart
        want, got = (plan.solve(y0, 0.0, 0.3, **kw, **call) for plan in plans)
        assert int(want[1][:, 3].max()) == 0 and bool((got[1] == want[1]).all())
        # one block: fixed steps are rounded to a few ulps of |H| h ~ 1 each; adaptive
        # ones follow the rounding of an error estimate of size abstol (1e-6 of it), and
        # the results stay within the solve's own error
        bound = 1e-290 if n == 12 else 1e-12 if solver.startswith("fixed") else 1e-9
        for a, b in zip(got, want):
            if a is not None and a.dtype.is_floating_point:
                off = float((a.nan_to_num(7.0) - b.nan_to_num(7.0)).abs().max())
                assert off <= bound, (call["output_kind"], off)
        if "stop_event" in call:
            fired.append(bool(got[-1].isfinite().all()))
    assert fired == [True]
