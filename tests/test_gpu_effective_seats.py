"""Effective-Hamiltonian trajectories that share a workgroup give bitwise the
results of a workgroup each: batches of one, two and four seats per workgroup
(by the trajectories for each of a given number of workgroups), fields in
different grid intervals and off the grid, odd batches, every output kind and
both ways to take the first step.  Rows are sorted by length only where that
does not pad the tables more."""

from __future__ import annotations

import numpy as np
import pytest

from centrex_tlf_amd.lindblad.effective import (
    debug_effective_lindblad_rhs,
    effective_operator_payload,
    prepare_effective_lindblad_plan,
    split_real_rho,
)

from ._effective import random_plan_dict
from ._gpu import require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver, dt", [("dopri5", 1e-3), ("tsit5", float("nan"))])
@pytest.mark.parametrize("n, density", [(3, 0.05), (9, 0.1)])
def test_seats_are_bitwise_a_workgroup_each(n, density, solver, dt):
    torch = require_gpu()
    plan = prepare_effective_lindblad_plan(random_plan_dict(n=n, seed=n, density=density))
    dev, cus = plan.device, torch.cuda.get_device_properties(0).multi_processor_count
    rho0 = np.zeros((n, n), dtype=complex)
    rho0[0, 0] = rho0[1, 1] = 0.5
    y0 = split_real_rho(rho0)
    B = 3 * cus + 5  # four seats a workgroup
    rng = np.random.default_rng(3)
    # x(1) = x0 + 0.35: the whole grid, and some trajectories that leave it
    ov = np.stack([rng.uniform(0.3, 2.0, B), rng.uniform(-0.99, 0.75, B)], axis=1)
    slots = [plan.slot_names.index("Omega_amp"), plan.slot_names.index("x0")]
    kw = dict(solver=solver, dt=dt, abstol=1e-8, reltol=1e-6, override_slots=slots, workgroups=cus)
    save = np.asarray([0.0, 0.31, 0.77, 1.0])
    calls = [dict(output_kind="populations", save_plan=[1.0], save_start=False),
             dict(output_kind="full", save_plan=save, capacity=4),
             dict(output_kind="selected", selected=[(0, 0), (1, 0)], capacity=200),
             dict(output_kind="integral", weights=[(0, 0.7), (n + 1, 0.2)])]
    for call in calls:
        want = [dev.solve(y0, 0.0, 1.0, n_traj=len(ov[i:i + cus]), override_values=ov[i:i + cus], **kw, **call)
                for i in range(0, B, cus)]
        for rows in (B, cus + 7):  # four seats, two seats
            got = dev.solve(y0, 0.0, 1.0, n_traj=rows, override_values=ov[:rows], **kw, **call)
            for k in range(5):
                ref = torch.cat([w[k] for w in want])[:rows]
                assert bool((got[k].nan_to_num(7.0) == ref.nan_to_num(7.0)).all()), (call["output_kind"], rows, k)
    status = got[1][:, 3].cpu().numpy()
    assert 0 < (status != 0).sum() < len(status)  # a field above the grid ends its own trajectory only


def test_rows_keep_their_order_where_sorting_pads_more():
    """Rows 0..63 hold 1..64 entries of one operator, rows 64..127 of another:
    in their own order 64 + 64 cells a lane, sorted by length 64 + 64 + 32 + 32."""
    torch = require_gpu()
    n, grid = 8, np.linspace(-1.0, 1.0, 400)
    plan = random_plan_dict(n=n, n_grid=2, seed=1)
    rng = np.random.default_rng(2)
    first, second = np.zeros((128, 128)), np.zeros((128, 128))
    for r in range(64):
        first[r, : r + 1] = rng.normal(size=r + 1)
        second[64 + r, 127 - r:] = rng.normal(size=r + 1)
    for key, m in (("sparse_combined", first), ("sparse_opt", second), ("sparse_det", 0 * first)):
        plan[key] = effective_operator_payload([m] * grid.size, grid)
    plan.update(n_grid=grid.size, field_grid=grid)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan = prepare_effective_lindblad_plan(plan)
    used = free - torch.cuda.mem_get_info()[0]
    cells = 32 * 399 * 64 * 128  # 32 bytes a cell and grid interval
    assert used < 1.25 * cells, (used, cells)
    y = rng.normal(size=128)
    got = np.asarray(debug_effective_lindblad_rhs(plan, y, 2.5)["dy"])
    want = first @ y + 0.5 * second @ y  # the pulse's top, Omega = 1
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-13 * np.abs(want).max())
