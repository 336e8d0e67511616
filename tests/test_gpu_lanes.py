"""The plan-specialised one-wave kernels give bitwise the results of the
precompiled kernels in every form: save plans, traces of accepted steps, rates,
stop events, fixed steps and the adjoint's tape, with two trajectories per wave
(23 elements) and one (41 elements), odd batches and end times of their own."""

from __future__ import annotations

import numpy as np
import pytest
import sympy as smp

from centrex_tlf_amd.lindblad import normalize_stop_event, population, prepare_lindblad_problem
from centrex_tlf_amd.lindblad._driver import build_save_plan
from centrex_tlf_amd.lindblad.native import DevicePlan, Tape

from ._gpu import require_gpu
from .systems import GAMMA, coherent_ground, tlf_n39, tlf_n39_xy

pytestmark = pytest.mark.gpu

TOL = dict(abstol=1e-9, reltol=1e-7, dt=1e-8)


@pytest.fixture(scope="module", params=["two per wave", "one per wave"])
def plans(request):
    require_gpu()
    system, params, rho0, t_span, weights = tlf_n39() if request.param == "two per wave" else tlf_n39_xy()
    if request.param == "one per wave":
        rho0 = coherent_ground(system)
    prepared = prepare_lindblad_problem(system, params, backend="host")
    base, spec = DevicePlan(prepared.flat_plan), DevicePlan(prepared.flat_plan).specialize()
    rng = np.random.default_rng(17)
    B = 37
    slots = [prepared.slot_names.index("delta0"), prepared.slot_names.index("Omega0")]
    pb = np.stack([rng.uniform(-5, 5, B), rng.uniform(0.1, 10, B)], axis=1).astype(complex) * GAMMA
    t1 = rng.uniform(0.3, 1.0, B) * t_span[1]
    t1[5], t1[17] = t_span[0], -1.0e-9
    call = dict(override_slots=slots, override_values=pb, weights=weights)
    return prepared, base, spec, prepared.layout.pack(rho0), t_span, t1, call


def _equal(base, spec, y0, t0, t1, **kw):
    want, got = base.solve(y0, t0, t1, **kw), spec.solve(y0, t0, t1, **kw)
    for a, b in zip(want, got):
        if a is None:
            assert b is None
            continue
        assert a.shape == b.shape and bool((a.nan_to_num(7.0) == b.nan_to_num(7.0)).all())
    assert spec.specialize_failure() is None
    return got


@pytest.mark.parametrize("solver", ["dopri5", "tsit5"])
@pytest.mark.parametrize("output", ["populations", "full", "rate", "integral"])
def test_save_plans_and_traces(plans, solver, output):
    prepared, base, spec, y0, t_span, t1, call = plans
    save = build_save_plan(np.linspace(*t_span, 23), *t_span, True)
    kw = dict(call, solver=solver, output_kind=output, trace=True, **TOL)
    out = _equal(base, spec, y0, *t_span, save_plan=save, capacity=save.size, with_times=True, with_integral=True, **kw)
    assert int(out[4].min()) == save.size
    # a row per accepted step, too few rows for the longest (status 7), own end times
    out = _equal(base, spec, y0, t_span[0], t1, capacity=60, with_times=True, **kw)
    assert int(out[1][17, 3]) == 4 and {0, 7} >= set(np.unique(out[1][:, 3].cpu().numpy())) - {4}
    # save points past an end time: "ended before all saveat"
    out = _equal(base, spec, y0, t_span[0], t1, save_plan=save, capacity=save.size, **kw)
    assert (out[1][:, 3] == 6).any()


@pytest.mark.parametrize("solver", ["dopri5", "tsit5"])
@pytest.mark.parametrize("kind", ["population", "expression"])
def test_stop_events(plans, solver, kind):
    prepared, base, spec, y0, t_span, t1, call = plans
    envelope = smp.Symbol("Ω0", real=True) / smp.Symbol("Omega0", real=True) - 0.5
    event = population([36, 37, 38], threshold=0.02) if kind == "population" else envelope
    event = normalize_stop_event(event, prepared)
    kw = dict(call, solver=solver, stop_event=event, **TOL)
    out = _equal(base, spec, y0, *t_span, output_kind="full", with_integral=True, **kw)
    assert 0 < int((~out[-1].isnan()).sum())
    _equal(base, spec, y0, t_span[0], t1, output_kind="populations", **kw)
    save = build_save_plan(np.linspace(*t_span, 9), *t_span, True)
    _equal(base, spec, y0, *t_span, output_kind="populations", trace=True, save_plan=save, capacity=save.size + 1, **kw)


@pytest.mark.parametrize("solver", ["fixed_rk2", "fixed_rk4", "fixed_dopri5"])
def test_fixed_steps(plans, solver):
    prepared, base, spec, y0, t_span, t1, call = plans
    kw = dict(call, solver=solver, dt=2.3e-8)
    _equal(base, spec, y0, t_span[0], t1, output_kind="populations", with_integral=True, **kw)
    save = build_save_plan(np.linspace(*t_span, 7), *t_span, True)
    _equal(base, spec, y0, *t_span, output_kind="rate", trace=True, save_plan=save, capacity=save.size, **kw)
    out = _equal(base, spec, y0, *t_span, output_kind="populations", maxiters=5, **kw)
    assert (out[1][:, 3] == 1).all()


def test_tape(plans):
    prepared, base, spec, y0, t_span, t1, call = plans
    support = base.support_of(y0)
    slots = base.support_info(support)["slot_count"]
    tapes = [Tape(len(t1), slots, 400) for _ in range(2)]
    for plan, tape in zip((base, spec), tapes):
        plan.solve(y0, t_span[0], t1, output_kind="integral", support=support, tape=tape, **call, **TOL)
    for name in ("t", "h", "c", "f", "y", "n"):
        assert bool((getattr(tapes[0], name) == getattr(tapes[1], name)).all()), name
