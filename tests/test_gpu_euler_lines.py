"""The line-by-line projection of the Euler kernels at the edges of its element groups (meshes that
do not fill the last workgroup) and with facet quadratures whose nodes do not lie on the volume
lines (general face rows), against the CPU oracle: the residual, and the pull-back against the
oracle's forward mode. The states are perturbed node by node, so many pairs are just past the
log-mean's series (|y - x| >= 1e-2 (x + y)), where log y - log x carries a relative error of
eps / 2e-2 in the device's flux and in the oracle's; a residual sums such fluxes with the weights of
the rows of D. Bar: 4 (eps / 2e-2) times the largest row sum of |D| / J times the largest state; and
1e-11 of the summed magnitudes for the pull-back, as in test_gpu_parity.py."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.conservation_laws import EulerEquations, EulerPeriodicTest, LaxFriedrichsNumericalFlux
from sse.geometry import ChanWilcoxMetrics, make_spatial_discretization
from sse.mesh import UniformWarping, uniform_periodic_mesh, warp_mesh
from sse.reference_approximation import (GaussQuadrature, LGLQuadrature, ModalTensor,
                                         ReferenceApproximationTet, ReferenceApproximationTri)
from sse.solvers import FluxDifferencingForm, project_function, Solver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _default_kernels(monkeypatch):
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels


def _problem(elem, p, M, lgl=False):
    d = 2 if elem == "tri" else 3
    make = ReferenceApproximationTri if d == 2 else ReferenceApproximationTet
    rule = None
    if lgl:
        rule = LGLQuadrature(p) if d == 2 else (LGLQuadrature(p), GaussQuadrature(p, 1, 0))
    ref = make(ModalTensor(p), mapping_degree=p, facet_quadrature_rule=rule)
    mesh = uniform_periodic_mesh(ref, ((0.0, 2.0),) * d, (M,) * d)
    mesh = warp_mesh(mesh, ref, UniformWarping(0.04, (2.0,) * d)) if d == 3 else warp_mesh(mesh, ref, 0.1)
    sd = make_spatial_discretization(mesh, ref, ChanWilcoxMetrics())
    law = EulerEquations(d, 1.4)
    s = Solver(law, sd, FluxDifferencingForm(inviscid_numerical_flux=LaxFriedrichsNumericalFlux()))
    u0 = project_function(EulerPeriodicTest(d, 1.4, 0.1, 2.0), sd)
    rng = np.random.default_rng(5)
    return s, np.asfortranarray(u0 * (1.0 + 1e-3 * rng.standard_normal(u0.shape)))


CASES = [("tri", 2, 3, False), ("tri", 3, 3, False), ("tri", 4, 2, False), ("tri", 5, 3, False), ("tri", 6, 1, False),
         ("tri", 2, 3, True), ("tri", 4, 2, True), ("tet", 2, 1, False), ("tet", 3, 1, False), ("tet", 4, 1, False), ("tet", 5, 1, False),
         ("tet", 3, 1, True)]


def _check_family(s, elem, p, lgl):
    """The line kernels, with general face rows for LGL facets of Tri p = 2. Where a volume node meets
    more than ten facet nodes (LGL from p = 3 on) the general kernels run."""
    if not lgl:
        assert s.describe().startswith("struct") and "faces=lines" in s.describe(), s.describe()
    elif (elem, p) == ("tri", 2):
        assert s.describe().startswith("struct") and "faces=general" in s.describe(), s.describe()
    else:
        assert s.describe().startswith("generic"), s.describe()


@pytest.mark.parametrize("elem,p,M,lgl", CASES)
def test_residual(elem, p, M, lgl):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    s, u0 = _problem(elem, p, M, lgl)
    u = to_device(u0)
    du = torch.empty_like(u)
    semi_discrete_residual(du, u, s)
    torch.cuda.synchronize()
    _check_family(s, elem, p, lgl)
    sd = s.spatial_discretization
    rows = max(np.abs(np.asarray(Dm)).sum(1).max() for Dm in sd.reference_approximation.D)
    bar = 4 * np.finfo(float).eps / 2e-2 * rows / sd.geometric_factors.J_q.min() * np.abs(u0).max()
    assert np.abs(to_host(du) - O.residual(s.arrays, u0)).max() <= bar, s.describe()


@pytest.mark.parametrize("elem,p,M,lgl", CASES)
def test_pull_back(elem, p, M, lgl):
    from sse.adjoint import residual_vjp
    s, u0 = _problem(elem, p, M, lgl)
    rng = np.random.default_rng(6)
    du, y = (np.asfortranarray(rng.standard_normal(u0.shape)) for _ in range(2))
    ubar, lam = residual_vjp(s, u0, y)
    _check_family(s, elem, p, lgl)
    _, jv = O.residual_jvp(s.arrays, u0, du, 0.7)
    a, b = float((ubar * du).sum()) + 0.7 * lam, float((y * jv).sum())
    assert abs(a - b) <= 1e-11 * float(np.abs(y * jv).sum())
