"""Residuals whose result goes where the state is: dudt the memory of u itself, or shifted by one
element, by less and by half the state, in every kernel family, against the CPU oracle. The result is
that of u before the call. Bar as in test_gpu_parity.py: 1e-12 of the largest entry."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.reference_approximation import ModalMulti
from sse.solvers import Solver
from sse.workloads import (advection_diffusion_3d_config, density_wave_3d_config, euler_1d_gauss, euler_3d_hex,
                           euler_vortex_2d_modal, vortex_2d_config)

pytestmark = pytest.mark.gpu

CASES = {
    "hex_nodal": (lambda: euler_3d_hex(M=5, p=3)[:5], "generic"),  # 125 elements read their neighbours' u
    "line_gauss": (lambda: euler_1d_gauss()[:5], "generic"),
    "tri_multi": (lambda: euler_vortex_2d_modal(M=3, p=3, approx=ModalMulti)[:5], "generic"),
    "tri_tensor": (lambda: vortex_2d_config(M=6, p=4)[:5], "struct"),
    "tet_tensor": (lambda: density_wave_3d_config(M=2, p=3, ic_strength=0.2)[:5], "struct"),
    "advdiff_tet": (lambda: advection_diffusion_3d_config(M=2, p=3)[:5], "standard tensor"),
}


@pytest.mark.parametrize("part", ["same", "one element", "three values", "half"])
@pytest.mark.parametrize("name", list(CASES))
def test_residual_into_the_state(name, part, monkeypatch):
    import torch
    from sse import semi_discrete_residual
    from sse.time_integration import to_device, to_host
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels
    make, family = CASES[name]
    law, sd, _, form, ode = make()
    s = ode.p
    assert s.describe().startswith(family), s.describe()
    u0 = to_device(ode.u0)
    n = u0.numel()
    shift = {"same": 0, "one element": n // u0.shape[0], "three values": 3, "half": n // 2}[part]
    for back in (False, True):  # dudt after u in memory, and before it
        buf = torch.empty(n + shift, dtype=torch.float64, device="cuda")
        u = (buf[shift:] if back else buf[:n]).view(u0.shape)
        dudt = (buf[:n] if back else buf[shift:]).view(u0.shape)
        u.copy_(u0)
        semi_discrete_residual(dudt, u, s)
        torch.cuda.synchronize()
        got, ref = to_host(dudt.clone()), O.residual(s.arrays, ode.u0)
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
