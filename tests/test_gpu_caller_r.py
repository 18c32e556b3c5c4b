"""The extrapolation R is the caller's: one that factorises along the lines of the grid (to the rounding of
its entries) runs the line kernels, any other one the general kernels, and both give its residual. R is
the package's with every entry off by up to 5e-13 of itself, against the CPU oracle with the same R.

Bars as in test_gpu_parity.py: 1e-12 for a residual, 1e-10 after Runge-Kutta steps."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.batch import BatchedSolver
from sse.conservation_laws import LinearAdvectionDiffusionEquation
from sse.solvers import _fptr
from sse.workloads import advection_diffusion_3d_config, density_wave_3d_config, vortex_2d_config

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _default_kernels(monkeypatch):
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels


CASES = {
    "tri": (lambda: vortex_2d_config(M=4, p=4)[:5], "struct", "generic"),
    "tet": (lambda: density_wave_3d_config(M=1, p=3, ic_strength=0.2)[:5], "struct", "generic"),
    "advdiff": (lambda: advection_diffusion_3d_config(M=1, p=3)[:5], "standard tensor", "standard d=3"),
}


def _with_r(s, off):
    """The solver with every entry of R off by up to `off` of itself."""
    A = s.arrays
    noise = np.random.default_rng(4).uniform(-1.0, 1.0, A.R.shape)
    A.R = np.asfortranarray(A.R * (1.0 + off * noise))
    A.desc.R = _fptr(A.R)
    return s


@pytest.mark.parametrize("off", [0.0, 1e-16, 1e-14, 5e-13])
@pytest.mark.parametrize("name", list(CASES))
def test_residual(name, off):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    make, lines, general = CASES[name]
    s = _with_r(make()[4].p, off)
    u0 = np.random.default_rng(3).standard_normal(s.size()) if name == "advdiff" else make()[4].u0
    u0 = np.asfortranarray(u0)
    u = to_device(u0)
    du = torch.empty_like(u)
    semi_discrete_residual(du, u, s)
    torch.cuda.synchronize()
    assert s.describe().startswith(lines if off <= 1e-16 else general), s.describe()
    ref = O.residual(s.arrays, u0)
    assert np.abs(to_host(du) - ref).max() <= 1e-12 * np.abs(ref).max()


def test_ensemble():
    from sse.time_integration import to_device, to_host
    s = _with_r(CASES["advdiff"][0]()[4].p, 5e-13)
    law = s.conservation_law
    solvers = [s.with_law(LinearAdvectionDiffusionEquation(law.a, 0.002 * (r + 1))) for r in range(3)]
    u0 = [np.asfortranarray(np.random.default_rng(r).standard_normal(s.size())) for r in range(3)]
    u = [to_device(x) for x in u0]
    BatchedSolver(solvers).rk_steps(u, [1e-4] * 3, 3)
    for q, x, y in zip(solvers, u, u0):
        ref = O.rk_steps(q.arrays, y, 1e-4, 3)
        assert np.abs(to_host(x) - ref).max() <= 1e-10 * np.abs(ref).max()
