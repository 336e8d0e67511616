"""The multi-wave adjoint over couplings: dense systems with every kind of
entry (time-independent and time-dependent parameters, complex factors, two
coefficients on one coupling), one to four slots a lane, and a plan whose
entries do not fit, which takes the gather form.  Every shape of both forms that
covers a plan gives the same gradient of one tape."""

from __future__ import annotations

import numpy as np
import pytest
import sympy as smp

from centrex_tlf_amd.lindblad import prepare_lindblad_problem
from centrex_tlf_amd.lindblad.adjoint import DifferentiablePhotonCount
from centrex_tlf_amd.lindblad.native import NativeError
from centrex_tlf_amd.lindblad.systems import OBESystem

from ._dense import chain_system, random_density
from ._gpu import require_gpu

pytestmark = pytest.mark.gpu

# The error estimate is a difference of terms of |k| h ~ 5 (|H| ~ 10, elements of
# rho ~ 3, h ~ 0.1): rounding changes the error norm by about NOISE = eps 5 /
# abstol = 1e-8 of itself, and with it the step sizes' share of the derivative
# (adaptive - frozen).  Two kernels differ by that; +-D differences of the
# adaptive map see NOISE / D on each side.
NOISE, D = 1e-8, 1e-6
TOL = dict(abstol=1e-7, reltol=1e-5, dt=1e-3)


def dense_problem(n: int):
    rng = np.random.default_rng(5)
    h0 = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    h0 = h0 + h0.conj().T
    s, w, c = smp.Symbol("s", real=True), smp.Symbol("w", real=True), smp.Symbol("c", complex=True)
    H = smp.zeros(n, n)
    for i in range(n):
        for j in range(n):
            H[i, j] = complex(h0[i, j]) if i != j else float(h0[i, i].real) + s * i
            if abs(i - j) == 1:
                H[i, j] += w / 2 + (c * 0.75 if i < j else smp.conjugate(c) * 0.75)
            if abs(i - j) == 2:
                H[i, j] += s * (0.4j if i < j else -0.4j)
    C = np.zeros((1, n, n), dtype=np.complex128)
    C[0, 0, n - 1] = 0.6
    params = {"amp": 0.7, "phi": 0.3, "s": 0.9, "w": "amp*cos(3*t)", "c": "0.5*exp(I*(2*t + phi))"}
    return prepare_lindblad_problem(OBESystem(H_symbolic=H, C_array=C), params, backend="host"), ["amp", "phi", "s"], 1.0


def chain_problem(n: int, unique_factors: bool):
    params = {"omega0": 1.0, "delta": 0.2, "frequency": 1.9, "Omega": "omega0*(1 + 0.4*cos(frequency*t))"}
    prepared = prepare_lindblad_problem(chain_system(n), params, backend="host")
    if unique_factors:  # a value of its own for every term: more than the entry index holds
        flat = prepared.flat_plan
        terms = len(flat["factors_re"])
        for k in ("factors_re", "factors_im"):
            flat[k] = np.ascontiguousarray(np.asarray(flat[k]) * (1.0 + 1e-3 * np.arange(terms) / terms))
    return prepared, ["omega0", "delta", "frequency"], 0.6


# the shapes (1-based variants) over couplings and over gather tables that cover
# 64, 128, 832 and 1,856 slots
SHAPES = {"dense 4": ((7, 8, 9), (1, 2, 3, 4)), "dense 12": ((7, 8, 9), (1, 2, 3, 4)),
          "chain 40": ((8, 9), (1, 2, 3, 4)), "chain 60": ((9,), (4,)), "chain 60 unique": ((), (4,))}


@pytest.mark.parametrize("solver", ["dopri5", "tsit5"])
@pytest.mark.parametrize("case", ["dense 4", "dense 12", "chain 40", "chain 60", "chain 60 unique"])
def test_matches_finite_differences_of_the_replayed_steps(case, solver):
    require_gpu()
    kind, n = case.split()[0], int(case.split()[1])
    prepared, names, t1 = dense_problem(n) if kind == "dense" else chain_problem(n, case.endswith("unique"))
    engine = DifferentiablePhotonCount(prepared, names, [(n - 1, 0.8), (0, -0.3)], (0.0, t1), solver=solver,
                                       tape_capacity=512, **TOL)
    y0 = prepared.layout.pack(random_density(n, seed=2))
    base = np.asarray([complex(prepared.parameters.base_parameters[k]).real for k in names])
    p = base * (1.0 + np.asarray([[0.0], [0.1], [-0.2]]))
    counts, tape = engine.forward(p, y0)
    block, gather = SHAPES[case]
    variant = block[0] if n == 4 else 0  # a plan of one block takes the single-block form by itself
    frozen = engine.gradient(p, y0, tape, mode="frozen", variant=variant).cpu().numpy()
    adaptive = engine.gradient(p, y0, tape, variant=variant).cpu().numpy()
    fd, fd_adaptive, same = np.zeros_like(p), np.zeros_like(p), np.ones(len(p), dtype=bool)
    for m in range(p.shape[1]):
        hi, lo = p.copy(), p.copy()
        hi[:, m] *= 1 + D
        lo[:, m] *= 1 - D
        step = (hi - lo)[:, m]
        fd[:, m] = (engine.replay(hi, y0, tape) - engine.replay(lo, y0, tape)).cpu().numpy() / step
        (vh, th), (vl, tl) = engine.forward(hi, y0), engine.forward(lo, y0)
        fd_adaptive[:, m] = (vh - vl).cpu().numpy() / step
        same &= ((th.n == tape.n) & (tl.n == tape.n)).cpu().numpy()
    scale, share = np.abs(fd).max(), np.abs(adaptive - frozen).max()
    # central differences: rounding eps |I| / (D |p|), truncation D^2
    bound = 1e-8 * scale + 20 * 2.3e-16 * np.abs(counts.cpu().numpy()).max() / (D * np.abs(p).min())
    np.testing.assert_allclose(frozen, fd, rtol=0, atol=bound)
    # an attempt count that changes under +-D is a jump of the adaptive map
    assert same.any()
    np.testing.assert_allclose(adaptive[same], fd_adaptive[same], rtol=0, atol=bound + 2 * NOISE / D * share)
    # 0: the single-block form for n = 4, the form above for the others; 5 and 6
    # are the single-block shapes of 12 and 16 gather rows
    for v in (0, 1, 2, 3, 4, 7, 8, 9) if n == 4 else range(10):
        if v not in (0,) + block + gather:
            with pytest.raises(NativeError, match="does not cover"):
                engine.gradient(p, y0, tape, variant=v)
            continue
        for mode, got in (("frozen", frozen), ("adaptive", adaptive)):
            other = engine.gradient(p, y0, tape, mode=mode, variant=v).cpu().numpy()
            np.testing.assert_allclose(got, other, rtol=0, atol=1e-12 * scale + 2 * NOISE * share,
                                       err_msg=f"{mode}, variant {v}")
