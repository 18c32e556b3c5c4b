"""The line-by-line StandardForm kernels of scalar laws at the edges of their slots and of their
face operators, against the CPU oracle: workgroups whose last slots are past the mesh, ensembles
with fewer and with more members than a workgroup has slots, both mapping forms, advection alone,
and facet quadratures whose nodes do not lie on the volume lines (general face rows).

Bars as in test_gpu_parity.py: 1e-12 for a residual, 1e-10 after Runge-Kutta steps."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.batch import BatchedSolver
from sse.conservation_laws import (BR1, LaxFriedrichsNumericalFlux,
                                   LinearAdvectionDiffusionEquation, LinearAdvectionEquation)
from sse.geometry import ChanWilcoxMetrics, make_spatial_discretization
from sse.mesh import UniformWarping, uniform_periodic_mesh, warp_mesh
from sse.reference_approximation import (GaussQuadrature, LGLQuadrature, ModalTensor,
                                         ReferenceApproximationTet, ReferenceApproximationTri)
from sse.solvers import (PhysicalOperator, SkewSymmetricMapping, Solver, StandardForm,
                         StandardMapping)

pytestmark = pytest.mark.gpu

VELOCITY = (1.0, 0.5, 0.25)


@pytest.fixture(autouse=True)
def _default_kernels(monkeypatch):
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels


def _solver(elem, p, M, b=0.01, skew=True, lgl_facets=False):
    d = 2 if elem == "tri" else 3
    make = ReferenceApproximationTri if d == 2 else ReferenceApproximationTet
    rule = None
    if lgl_facets:
        rule = LGLQuadrature(p) if d == 2 else (LGLQuadrature(p), GaussQuadrature(p, 1, 0))
    ref = make(ModalTensor(p), mapping_degree=p, facet_quadrature_rule=rule)
    mesh = uniform_periodic_mesh(ref, ((0.0, 1.0),) * d, (M,) * d)
    mesh = warp_mesh(mesh, ref, UniformWarping(0.04, (1.0,) * d)) if d == 3 else warp_mesh(mesh, ref, 0.1)
    sd = make_spatial_discretization(mesh, ref, ChanWilcoxMetrics())
    a = VELOCITY[:d]
    law = LinearAdvectionEquation(a) if b is None else LinearAdvectionDiffusionEquation(a, b)
    form = StandardForm(mapping_form=SkewSymmetricMapping() if skew else StandardMapping(),
                        inviscid_numerical_flux=LaxFriedrichsNumericalFlux(), viscous_numerical_flux=BR1())
    return Solver(law, sd, form, PhysicalOperator())


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def _state(solver, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal(solver.size()))


@pytest.mark.parametrize("elem,p,M,b,skew,lgl", [
    ("tri", 2, 3, 0.01, True, False), ("tri", 3, 3, 0.01, False, False), ("tri", 4, 5, None, True, False),
    ("tri", 4, 3, 0.01, True, True), ("tri", 6, 3, 0.01, True, False),
    ("tet", 2, 1, 0.01, True, False), ("tet", 3, 1, 0.01, True, False), ("tet", 3, 1, 0.01, True, True),
    ("tet", 4, 1, 0.01, False, False), ("tet", 4, 1, None, True, False), ("tet", 5, 1, 0.01, True, False),
    ("tet", 5, 1, 0.01, False, True),
])
def test_residual(elem, p, M, b, skew, lgl):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    s = _solver(elem, p, M, b, skew, lgl)
    u0 = _state(s, 3)
    u = to_device(u0)
    du = torch.empty_like(u)
    semi_discrete_residual(du, u, s)
    torch.cuda.synchronize()
    assert s.describe().startswith("standard tensor"), s.describe()
    assert s.describe().endswith("faces=general" if lgl else "faces=lines"), s.describe()
    assert _rel(to_host(du), O.residual(s.arrays, u0)) <= 1e-12


@pytest.mark.parametrize("elem,p,members", [("tet", 3, 2), ("tet", 3, 3), ("tet", 3, 7), ("tri", 4, 4), ("tri", 4, 13)])
def test_ensemble(elem, p, members):
    from sse.time_integration import to_device, to_host
    base = _solver(elem, p, 1 if elem == "tet" else 3)
    law = base.conservation_law
    solvers = [base.with_law(LinearAdvectionDiffusionEquation(law.a, 0.002 * (r + 1))) for r in range(members)]
    u0 = [_state(base, 11 + r) for r in range(members)]
    dts = [1e-4 * (1 + 0.1 * r) for r in range(members)]
    u = [to_device(x) for x in u0]
    BatchedSolver(solvers).rk_steps(u, dts, 3)
    for s, x, y, dt in zip(solvers, u, u0, dts):
        assert _rel(to_host(x), O.rk_steps(s.arrays, y, dt, 3)) <= 1e-10
