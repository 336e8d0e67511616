"""Time-dependent programs as steps of independent operations over one wave (the
multi-wave kernels) against the same programs interpreted one by one.

A second system adds z times a long sum to the drive, z = 0: its programs are too
long for steps, its values are the same.  The expressions use every kind of
operation: products, quotients and differences, a power with a parameter as its
exponent, constant real powers of negative bases, a builtin, helpers with several
arguments, comparisons and a conjugate."""

from __future__ import annotations

import numpy as np
import pytest

from centrex_tlf_amd.lindblad import (
    LindbladParameters,
    Time,
    gaussian,
    normalize_stop_event,
    phase_modulation,
    population,
    prepare_lindblad_problem,
    sine,
    square_wave_profile,
)
from centrex_tlf_amd.lindblad._driver import build_save_plan
from centrex_tlf_amd.lindblad.native import DevicePlan

from ._dense import chain_system, random_density
from ._gpu import require_gpu

pytestmark = pytest.mark.gpu


def problem(long: bool):
    p = LindbladParameters()
    a = p.complex("a", 0.6 + 0.25j)
    w = p.real("w", 1.3)
    z = p.real("z", 0.0)
    t = Time()
    drive = (a * sine(t, angular_frequency=w) + phase_modulation(t, 0.5, w) / (1.0 + t) ** w
             + square_wave_profile(t, low=0.1, high=0.4, period=0.2) - (0.3 - t) ** 3.0 * 0.2)
    if long:
        total = sine(t, angular_frequency=w)
        for k in range(2, 60):
            total = total + sine(t, angular_frequency=w * float(k)) * float(k)
        drive = drive + z * total
    p.bind("Omega", drive, finalize=False)
    p.bind("delta", -((w * t + 0.01) ** 0.5) * 0.1 + gaussian(t, center=0.2, sigma=0.07, amplitude=0.3), finalize=False)
    p._finalize()
    return prepare_lindblad_problem(chain_system(14), p, backend="host")


@pytest.mark.parametrize("solver", ["dopri5", "tsit5", "fixed_rk4", "fixed_dopri5"])
def test_steps_are_bitwise_the_interpreter(solver):
    require_gpu()
    problems = [problem(long) for long in (False, True)]
    plans = [DevicePlan(q.flat_plan) for q in problems]
    assert plans[0].info["slot_count"] == 128
    # the steps and their 8 copies of the slots lie in LDS; the long program has none
    assert plans[0].info["lds_bytes"] > plans[1].info["lds_bytes"]
    y0 = problems[0].layout.pack(random_density(14, seed=3)) / 14
    slots = [q.slot_names.index("w") for q in problems]
    rows = np.linspace(0.5, 2.5, 5)[:, None].astype(complex)
    save = build_save_plan(np.linspace(0.0, 0.5, 6), 0.0, 0.5, True)
    event = [normalize_stop_event(population([0], threshold=float(y0[0]) + 0.05), q) for q in problems]
    kw = dict(solver=solver, restrict_support=False, abstol=1e-9, reltol=1e-7,
              dt=0.011 if solver.startswith("fixed") else 1e-3)
    for call in (dict(output_kind="full"), dict(output_kind="populations", trace=True, save_plan=save, capacity=save.size),
                 dict(output_kind="populations", stop_event=True)):
        got, want = (plan.solve(y0, 0.0, 0.5, override_slots=[s], override_values=rows, **kw,
                                **{k: event[i] if k == "stop_event" else v for k, v in call.items()})
                     for i, (plan, s) in enumerate(zip(plans, slots)))
        assert int(want[1][:, 3].max()) == 0 and int(want[1][:, 0].min()) > 10
        for x, y in zip(got, want):
            assert x is None or bool((x.nan_to_num(7.0) == y.nan_to_num(7.0)).all())
