"""The matrix-core nodal values at the edges of its tiles (6 to 35 modes, fewer and more than 16
rows of modal data, element counts that do not fill a workgroup of 16), against the CPU oracle. The
states are perturbed node by node; bar as in test_gpu_euler_lines.py: 4 (eps / 2e-2) times the
largest row sum of |D| / J times the largest state."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.reference_approximation import ModalMulti
from sse.solvers import Solver
from sse.workloads import density_wave_3d_config, euler_vortex_2d_modal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,p,M", [(2, 2, 3), (2, 5, 2), (3, 2, 1), (3, 3, 2), (3, 4, 1)])
def test_residual(d, p, M, monkeypatch):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels
    monkeypatch.setenv("SSE_NODAL_MFMA", "1")
    if d == 2:
        law, sd, _, form, ode = euler_vortex_2d_modal(M=M, p=p, approx=ModalMulti)[:5]
    else:
        law, sd, _, form, ode = density_wave_3d_config(M=M, p=p, approx=ModalMulti, ic_strength=0.2)[:5]
    solver = Solver(law, sd, form)
    rng = np.random.default_rng(8)
    u0 = np.asfortranarray(ode.u0 * (1.0 + 1e-3 * rng.standard_normal(ode.u0.shape)))
    u = to_device(u0)
    du = torch.empty_like(u)
    semi_discrete_residual(du, u, solver)
    torch.cuda.synchronize()
    assert "nodal_values=mfma" in solver.describe(), solver.describe()
    rows = max(np.abs(np.asarray(Dm)).sum(1).max() for Dm in sd.reference_approximation.D)
    bar = 4 * np.finfo(float).eps / 2e-2 * rows / sd.geometric_factors.J_q.min() * np.abs(u0).max()
    assert np.abs(to_host(du) - O.residual(solver.arrays, u0)).max() <= bar
