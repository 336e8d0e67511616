"""Plans and calls near a workgroup's 160 KB of LDS.

A 76-level chain fills the publication buffers and self coefficients of 46
blocks (147 KB with its programs interpreted).  The programs in steps need 8
copies of their slots more: with 18 cosines they fit, with 22 and 26 they do
not and the programs are interpreted, with 30 they are too long for steps at
all.  A stop event whose expression is some 900 deep leaves a plan of 820
elements no room for its couplings' entries, so it runs on the gather tables."""

from __future__ import annotations

import numpy as np
import pytest

from centrex_tlf_amd.lindblad import prepare_lindblad_problem
from centrex_tlf_amd.lindblad.ir import CompiledExpression, InstructionOp
from centrex_tlf_amd.lindblad.native import DevicePlan
from oracle.lb_oracle import Oracle

from ._dense import CHAIN_PARAMETERS, chain_system, random_density
from ._gpu import require_gpu

pytestmark = pytest.mark.gpu

LIMIT = 160 * 1024


@pytest.mark.parametrize("cosines", [18, 22, 26, 30])
def test_long_programs_of_large_plans(cosines):
    torch = require_gpu()
    n = 76
    drive = " + ".join(["1"] + [f"0.01*cos({1 + 0.1 * k:.1f}*t)" for k in range(cosines)])
    params = {"omega0": 1.0, "delta": 0.2, "Omega": f"omega0*({drive})"}
    prepared = prepare_lindblad_problem(chain_system(n), params, backend="host")
    plan, oracle = DevicePlan(prepared.flat_plan), Oracle(prepared)
    assert plan.info["slot_count"] == 2944 and 140_000 < plan.info["lds_bytes"] <= LIMIT
    ys = np.stack([prepared.layout.pack(random_density(n, seed=s)) for s in range(2)])
    ts = np.asarray([0.3, 1.7])
    got = plan.rhs(torch.as_tensor(ys, device="cuda"), torch.as_tensor(ts, device="cuda")).cpu().numpy()
    for b in range(2):
        want = oracle.rhs(ys[b], ts[b])
        # 8 products per output, each within an ulp of the largest
        np.testing.assert_allclose(got[b], want, rtol=0, atol=40 * 2.3e-16 * np.abs(want).max())
    y0, span = ys[0] / n, (0.0, 0.4)
    for solver in ("dopri5", "tsit5"):
        kw = dict(abstol=1e-9, reltol=1e-7, dt=1e-3)
        values, stats, _ = plan.solve(y0, *span, solver=solver, output_kind="populations", n_traj=1,
                                      restrict_support=False, **kw)
        ref = oracle.solve_batch(y0, span, solver=solver, output="populations", output_when="final", **kw)
        assert int(stats[0, 3]) == 0 and int(stats[0, 0]) == int(np.ravel(ref["accepted"])[0])
        np.testing.assert_allclose(values.cpu().numpy()[0], np.ravel(ref["final"]), rtol=0, atol=1e-12)


def chain_of_many_values(n: int):
    """A chain whose terms take 60 values each in turn, some 10 KB of entries."""
    prepared = prepare_lindblad_problem(chain_system(n), dict(CHAIN_PARAMETERS), backend="host")
    flat = prepared.flat_plan
    scale = 1.0 + 1e-3 * (np.arange(len(flat["factors_re"])) % 60)
    for k in ("factors_re", "factors_im"):
        flat[k] = np.ascontiguousarray(np.asarray(flat[k]) * scale)
    return prepared


@pytest.mark.parametrize("solver, kw", [("dopri5", dict(abstol=1e-9, reltol=1e-7, dt=1e-3)),
                                        ("fixed_rk4", dict(dt=0.01))])
def test_deep_stop_event_takes_the_gather_tables(solver, kw):
    require_gpu()
    n, t_stop = 40, 0.137
    prepared = chain_of_many_values(n)
    plan = DevicePlan(prepared.flat_plan)
    info = plan.info
    # the gather form's LDS but the expression stacks: two publication buffers,
    # self coefficients, eight coefficient rows and slot copies, 2 KB parked,
    # weights, event populations, block sums
    rest = (32 * info["n_published"] + 16 * info["slot_count"] + 128 * (info["n_coefficients"] + 1)
            + 128 * int(prepared.flat_plan["n_slots"]) + 2048 + 8 * ((n + 1) & ~1) + 8 * ((n + 3) & ~1)
            + 32 * (info["slot_count"] // 64) + 32)
    depth = (LIMIT - rest) // 128
    assert 800 < depth <= 1024
    op = InstructionOp
    row = lambda code, re=0.0: (int(code), 0, 0, 0, re, 0.0)  # noqa: E731
    deep = (row(op.TIME),) + (row(op.CONST),) * (depth - 2) + (row(op.CONST, -t_stop),) + (row(op.ADD),) * (depth - 1)
    flat = (row(op.TIME), row(op.CONST, -t_stop), row(op.ADD))
    y0 = prepared.layout.pack(random_density(n, seed=1)) / n
    got, want = (plan.solve(y0, 0.0, 0.3, solver=solver, output_kind="populations", n_traj=3, restrict_support=False,
                            stop_event=dict(kind="runtime_expression", expression=CompiledExpression(instructions=e),
                                            name="t - t_stop"), **kw) for e in (deep, flat))
    # the root of an adaptive step is found to rounding, a fixed one ends at the step after it
    near = 1e-12 if solver == "dopri5" else kw["dt"]
    assert int(got[1][:, 3].max()) == 0 and bool(((got[-1] - t_stop).abs() < near).all())
    for a, b in zip(got, want):  # both forms round alike (several blocks)
        assert bool((a.nan_to_num(7.0) == b.nan_to_num(7.0)).all())
