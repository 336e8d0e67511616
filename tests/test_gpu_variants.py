"""Kernel variants by name: ids that stored tunings and calls hold keep their
meaning, and the single-wave names are one kernel without a limit on a plan's
rows."""

from __future__ import annotations

import numpy as np
import pytest

from centrex_tlf_amd.lindblad import prepare_lindblad_problem, two_level_system
from centrex_tlf_amd.lindblad.native import DevicePlan, NativeError, kernel_variants

from ._dense import random_density
from ._gpu import require_gpu
from .systems import tlf_n39
from .test_gpu_couplings import dense_system

pytestmark = pytest.mark.gpu


def test_paired_ids_keep_their_meaning():
    """Variants 16 and 17 take plans of up to 8 and 12 rows, as they always did,
    and there is no other: systems of 2, 4 and 8 rows."""
    require_gpu()
    system, params, rho0, *_ = tlf_n39()
    tlf = prepare_lindblad_problem(system, params, backend="host")
    two = prepare_lindblad_problem(two_level_system(omega_name="Omega", delta_name="delta"),
                                   {"Omega": 0.7, "delta": 0.2}, backend="host")
    system, params = dense_system(5)
    five = prepare_lindblad_problem(system, params, backend="host")
    rows = []
    for prepared, rho in ((two, np.diag([1.0, 0.0])), (tlf, rho0), (five, random_density(5, seed=2) / 5)):
        plan, y0 = DevicePlan(prepared.flat_plan), prepared.layout.pack(np.asarray(rho, dtype=complex))
        support = plan.support_of(y0)
        rows.append(plan.support_info(support)["gather_rows"])
        assert [plan.launch_info(support, variant=v)["variant"] for v in (0, 16, 17)] == [16, 16, 17]
        with pytest.raises(NativeError, match="unknown kernel variant"):
            plan.launch_info(support, variant=18)
        kw = dict(output_kind="populations", n_traj=5, abstol=1e-9, reltol=1e-7, dt=1e-8)
        t1 = 1e-6 if prepared is tlf else 0.3
        want = plan.solve(y0, 0.0, t1, variant=13, **kw)  # one trajectory a wave
        for v in (16, 17):
            got = plan.solve(y0, 0.0, t1, variant=v, **kw)
            assert all(bool((a == b).all()) for a, b in zip(got[:2], want[:2]))
    assert len(kernel_variants()) == 17
    assert rows[0] <= 4 and rows[1] <= 4 and 4 < rows[2] <= 8, rows


@pytest.mark.parametrize("n", [7, 10])
def test_single_wave_names_are_one_kernel(n):
    """28 and 55 elements, some 13 and 19 coupling rows."""
    torch = require_gpu()
    system, params = dense_system(n)
    prepared = prepare_lindblad_problem(system, params, backend="host")
    plan = DevicePlan(prepared.flat_plan)
    assert (plan.info["gather_rows"] > 16) == (n == 10)
    assert [plan.launch_info(variant=v)["variant"] for v in (12, 13, 14, 15)] == [12, 13, 13, 13]
    y0 = prepared.layout.pack(random_density(n, seed=1)) / n
    kw = dict(output_kind="populations", n_traj=3, abstol=1e-9, reltol=1e-7, dt=1e-3)
    want = plan.solve(y0, 0.0, 0.3, variant=1, **kw)  # the multi-wave form
    assert int(want[1][:, 3].max()) == 0
    for v in (0, 12, 13, 14, 15):
        got = plan.solve(y0, 0.0, 0.3, variant=v, **kw)
        assert all(bool((a == b).all()) for a, b in zip(got[:2], want[:2])), v
    assert torch.isfinite(want[0]).all()

