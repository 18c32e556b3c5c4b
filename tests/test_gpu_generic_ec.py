"""The general entropy-conservative time derivative (runtime-sized elements) at the edges of its
work split, against the CPU oracle: more nodes than a 256-thread workgroup has threads (one
thread per node, 512 threads), few nodes (workgroups of 64, and of 128 on many elements), even and odd counts (the
half-way cyclic offset), sparse and dense operators, the atomic and the deterministic variant,
and the Runge-Kutta stage combination in its epilogue for one, two and three stages.

Bars as in test_gpu_parity.py: 1e-12 for a residual, 1e-10 after Runge-Kutta steps; where the
derivative itself amplifies rounding (257 nodes on a line) 8 eps times the largest row sum of
|D| times the largest state, over the largest residual."""

import numpy as np
import pytest

from oracle import oracle as O
from sse import FluxDifferencingForm
from sse.conservation_laws import (EntropyConservativeNumericalFlux, EulerEquations,
                                   LaxFriedrichsNumericalFlux)
from sse.geometry import make_spatial_discretization
from sse.mesh import uniform_periodic_mesh
from sse.reference_approximation import (ModalMulti, NodalMulti, NodalTensor,
                                         ReferenceApproximationLine)
from sse.solvers import MI355X, Solver, semidiscretize
from sse.workloads import density_wave_3d_config, euler_3d_hex, euler_vortex_2d_modal

pytestmark = pytest.mark.gpu


def _line(approx, M):
    law = EulerEquations(1, 1.4)

    def ic(x, t=0.0):
        rho = 1.0 + 0.3 * np.sin(np.pi * x[0])
        return np.stack([rho, 0.4 * rho, 2.5 + 0.08 * rho], -1)

    ref = ReferenceApproximationLine(approx)
    sd = make_spatial_discretization(uniform_periodic_mesh(ref, (0.0, 2.0), M), ref)
    form = FluxDifferencingForm(inviscid_numerical_flux=LaxFriedrichsNumericalFlux())
    return law, sd, ic, form, semidiscretize(law, sd, ic, form, (0.0, 1.0))


CASES = {
    "line_257_nodes": lambda: _line(NodalTensor(256), 2),       # one thread per node, 512 threads
    "line_modal_p2": lambda: _line(ModalMulti(2), 5),           # 3 modes: 85 threads per node
    "tri_modal_p2": lambda: euler_vortex_2d_modal(M=3, p=2, approx=ModalMulti)[:5],
    "tri_nodal_p4": lambda: euler_vortex_2d_modal(M=2, p=4, approx=NodalMulti)[:5],  # 40 nodes: 256 threads
    "tri_nodal_p5": lambda: euler_vortex_2d_modal(M=2, p=5, approx=NodalMulti)[:5],
    "tet_modal_p2": lambda: density_wave_3d_config(M=1, p=2, approx=ModalMulti, ic_strength=0.2)[:5],
    "tet_modal_p4": lambda: density_wave_3d_config(M=1, p=4, approx=ModalMulti, ic_strength=0.2)[:5],
    "hex_p2": lambda: euler_3d_hex(M=2, p=2)[:5],
    "hex_p4": lambda: euler_3d_hex(M=2, p=4)[:5],               # 275 nodes: 512 threads
}


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("det", [False, True], ids=["atomic", "deterministic"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_residual_at_the_edges_of_the_work_split(name, det):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    law, sd, _, form, ode = CASES[name]()
    solver = Solver(law, sd, form, parallelism=MI355X(deterministic=det))
    rng = np.random.default_rng(7)
    u0 = np.asfortranarray(ode.u0 * (1.0 + 1e-3 * rng.standard_normal(ode.u0.shape)))
    u = to_device(u0)
    du = torch.empty_like(u)
    semi_discrete_residual(du, u, solver)
    torch.cuda.synchronize()
    assert solver.describe().startswith("generic"), solver.describe()
    expected = O.residual(solver.arrays, u0)
    ref = sd.reference_approximation
    rows = max(np.abs(np.asarray(Dm)).sum(1).max() for Dm in ref.D) / sd.geometric_factors.J_q.min()
    bar = max(1e-12, 8 * np.finfo(float).eps * rows * np.abs(u0).max() / np.abs(expected).max())
    if not name.startswith("line_257"):
        bar = 1e-12
    assert _rel(to_host(du), expected) <= bar


@pytest.mark.parametrize("stages", [1, 2, 3])
def test_stage_combination_in_the_epilogue(stages):
    from types import SimpleNamespace

    from sse.time_integration import erk_steps, to_device, to_host
    # forward Euler, Heun, and a third-order tableau whose second row skips the first stage
    A = {1: [[0.0]], 2: [[0, 0], [1, 0]], 3: [[0, 0, 0], [0.5, 0, 0], [0, 0.75, 0]]}[stages]
    b = {1: [1.0], 2: [0.5, 0.5], 3: [2 / 9, 3 / 9, 4 / 9]}[stages]
    alg = SimpleNamespace(A=np.array(A, dtype=float), b=np.array(b))
    law, sd, _, form, ode = euler_3d_hex(M=2, p=2)[:5]
    solver = Solver(law, sd, FluxDifferencingForm(inviscid_numerical_flux=EntropyConservativeNumericalFlux()))
    u = to_device(ode.u0)
    erk_steps(solver, u, 1e-3, 3, alg)
    ref = O.erk_steps(solver.arrays, ode.u0, 1e-3, 3, alg.A, alg.b)
    assert _rel(to_host(u), ref) <= 1e-10


UNITS = [(17, 8), (-20, 8), (0, -9), (-300, 150), (300, -90)]  # powers of two of density and of velocity


@pytest.mark.parametrize("a,c", UNITS)
@pytest.mark.parametrize("name", ["hex_p2", "hex_p4", "line"])
def test_residual_does_not_depend_on_the_units(name, a, c):
    """A state in units of 2^a for density and 2^c for velocity (pressures from 2^-63 to 2^316; the
    first ones are near those of air in kg, m and s, p / rho = 6e4): such a change of units is exact, so
    the deterministic residual of a nodal scheme is that of the state near one, bit by bit. (The tests
    above compare states near one with the oracle.)"""
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    law, sd, _, _, ode = _line(NodalTensor(5), 7) if name == "line" else CASES[name]()
    form = FluxDifferencingForm(inviscid_numerical_flux=LaxFriedrichsNumericalFlux())
    solver = Solver(law, sd, form, parallelism=MI355X(deterministic=True))
    d = law.d
    state = np.ldexp(1.0, [a] + [a + c] * d + [a + 2 * c]).reshape(1, -1, 1)
    flux = np.ldexp(1.0, [a + c] + [a + 2 * c] * d + [a + 3 * c]).reshape(1, -1, 1)

    def residual(u0):
        u = to_device(np.asfortranarray(u0))
        du = torch.empty_like(u)
        semi_discrete_residual(du, u, solver)
        torch.cuda.synchronize()
        return to_host(du)

    got = residual(ode.u0)
    assert solver.describe().startswith("generic"), solver.describe()
    assert np.isfinite(got).all() and np.abs(got).max() > 0.0
    assert np.array_equal(residual(ode.u0 * state), got * flux)


@pytest.mark.parametrize("det", [False, True], ids=["atomic", "deterministic"])
@pytest.mark.parametrize("make,problems", [
    (lambda: euler_vortex_2d_modal(M=4, p=4, approx=ModalMulti), 25),                      # 40 nodes, 800 elements
    (lambda: density_wave_3d_config(M=2, p=2, approx=ModalMulti, ic_strength=0.2), 65),    # 63 nodes, 3,120
], ids=["tri_p4", "tet_p2"])
def test_workgroups_of_128_on_many_elements(make, problems, det):
    """Many small problems in one batch are one mesh of enough elements for smaller workgroups."""
    from sse.batch import BatchedSolver
    from sse.time_integration import to_device, to_host
    law, sd, _, form, ode = make()[:5]
    solver = Solver(law, sd, form, parallelism=MI355X(deterministic=det))
    batch = BatchedSolver([solver] * problems)
    assert f"N_e={problems * sd.N_e}" in batch.describe(), batch.describe()
    starts = [np.asfortranarray(ode.u0 * (1.0 + 1e-3 * np.random.default_rng(r).standard_normal(ode.u0.shape)))
              for r in range(3)]
    u = [to_device(starts[i % 3]) for i in range(problems)]
    batch.rk_steps(u, [1e-3] * problems, 2)
    refs = [O.rk_steps(solver.arrays, x, 1e-3, 2) for x in starts]
    worst = max(_rel(to_host(x), refs[i % 3]) for i, x in enumerate(u))
    assert worst <= 1e-10
