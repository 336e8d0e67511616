"""The digits of long 72-level flights.

Over the 12,000 to 19,000 steps of these flights, whose drive jumps every
microsecond, a rounding in the right-hand side or the step-size control reaches
the populations some 10,000 times as large: an input moved by one rounding, the
same controller from a log and an exp, or an output's terms summed in another
order move them by 3e-12 to 1.3e-11 here (2-norm over the levels).  The recorded
results are those of the term-by-term right-hand side in the plan's order with
the reference's controller (two powers, common.rs:32-70), as the general form
computed them; the kernels that run such batches are to give the same digits.
1e-13 is a thirtieth of what any other order of operations shows on these six
trajectories."""

from __future__ import annotations

import json
from pathlib import Path

import numpy as np
import pytest

from centrex_tlf_amd.lindblad import UnevenGroup, prepare_lindblad_problem, solve_uneven_batch

from ._gpu import require_gpu
from .systems import tlf_n72

pytestmark = pytest.mark.gpu

RECORDED = json.loads((Path(__file__).parent / "golden" / "tlf_n72_digits.json").read_text())


def _floats(v):
    return np.asarray([_floats(x) for x in v] if isinstance(v, list) else float.fromhex(v))


@pytest.mark.parametrize("solver", ["dopri5", "tsit5"])
def test_long_flights_keep_their_digits(solver):
    require_gpu()
    system, params, rho0, _, weights = tlf_n72()
    prepared = prepare_lindblad_problem(system, params, backend="gpu")
    sigma, delta = _floats(RECORDED["sigma"]), _floats(RECORDED["delta0"])
    rows = np.stack([sigma, sigma, delta], axis=1).astype(complex)
    group = UnevenGroup(prepared, rho0, 2.0 * sigma, ["sigma", "t_center", "delta0"], rows, weights)
    (res,) = solve_uneven_batch([group], solver=solver, tuning=None, abstol=1e-10, reltol=1e-8, dt=1e-8)
    want = RECORDED[solver]
    np.testing.assert_array_equal(res.stats[:, 0], want["accepted"])
    off = np.linalg.norm(res.populations - _floats(want["populations"]), axis=1)
    print(f"{solver}: largest 2-norm of a trajectory's difference {off.max():.2e}")
    assert off.max() <= 1e-13
    np.testing.assert_allclose(res.photons, _floats(want["photons"]), rtol=1e-13)
