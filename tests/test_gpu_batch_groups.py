"""Triangle problems of different degrees advanced by shared launches: the smallest meshes and odd
element counts, next to groups that keep their own launches (a second flux of one degree, a
deterministic solver, tetrahedra), eagerly and from the captured graph, against the CPU oracle's RK
steps. Bar: 1e-10 of the largest state entry, as for the batch of 256 problems in
test_gpu_configs.py."""

import numpy as np
import pytest

from oracle import oracle as O
from sse.conservation_laws import (EntropyConservativeNumericalFlux, EulerEquations, EulerPeriodicTest,
                                   LaxFriedrichsNumericalFlux)
from sse.geometry import ChanWilcoxMetrics, make_spatial_discretization
from sse.mesh import UniformWarping, uniform_periodic_mesh, warp_mesh
from sse.reference_approximation import (ModalTensor, ReferenceApproximationTet, ReferenceApproximationTri)
from sse.solvers import FluxDifferencingForm, MI355X, Solver, project_function

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _default_kernels(monkeypatch):
    monkeypatch.delenv("SSE_KERNELS", raising=False)  # another test's choice of kernels
    monkeypatch.delenv("SSE_BATCH_BRANCHES", raising=False)


def _problem(elem, p, M, flux="lf", det=False):
    d = 2 if elem == "tri" else 3
    ref = (ReferenceApproximationTri if d == 2 else ReferenceApproximationTet)(ModalTensor(p), mapping_degree=p)
    mesh = uniform_periodic_mesh(ref, ((0.0, 2.0),) * d, (M,) * d)
    mesh = warp_mesh(mesh, ref, UniformWarping(0.04, (2.0,) * d)) if d == 3 else warp_mesh(mesh, ref, 0.1)
    sd = make_spatial_discretization(mesh, ref, ChanWilcoxMetrics())
    nf = LaxFriedrichsNumericalFlux() if flux == "lf" else EntropyConservativeNumericalFlux()
    s = Solver(EulerEquations(d, 1.4), sd, FluxDifferencingForm(inviscid_numerical_flux=nf),
               parallelism=MI355X(deterministic=det))
    u0 = project_function(EulerPeriodicTest(d, 1.4, 0.1, 2.0), sd)
    return s, u0, 0.05 * (2.0 / M) / ((2 * p + 1) * 3.0)


# problems, and how many groups of them share their launches
SHARED = {"every degree": 5, "two degrees": 2, "one degree": 0, "with others": 3}
BATCHES = {
    "every degree": [("tri", p, M) for p, M in ((2, 3), (3, 1), (4, 3), (5, 1), (6, 3), (3, 5))],
    "two degrees": [("tri", 6, 1), ("tri", 2, 1)],
    "one degree": [("tri", 5, 3), ("tri", 5, 1)],
    "with others": [("tet", 2, 1), ("tri", 3, 3), ("tri", 3, 3, "ec"), ("tri", 5, 3, "lf", True), ("tri", 4, 1),
                    ("tri", 6, 3)],
}


@pytest.mark.parametrize("name", list(BATCHES))
@pytest.mark.parametrize("graph", [True, False])
def test_rk_steps(name, graph):
    import torch
    from sse.batch import BatchedSolver
    from sse.time_integration import to_device, to_host
    probs = [_problem(*c) for c in BATCHES[name]]
    batch = BatchedSolver([s for s, _, _ in probs])
    assert batch.describe().count("shared launches") == SHARED[name], batch.describe()
    states = [to_device(u0) for _, u0, _ in probs]
    for n in (3, 1, 2):  # captured in the first call and replayed in the third
        batch.rk_steps(states, [dt for _, _, dt in probs], n, use_graph=graph)
        torch.cuda.synchronize()
    for c, (s, u0, dt), u in zip(BATCHES[name], probs, states):
        want = O.rk_steps(s.arrays, u0, dt, 6)
        assert np.abs(to_host(u) - want).max() <= 1e-10 * np.abs(want).max(), (c, batch.describe())


@pytest.mark.parametrize("host", [False, True], ids=["device", "host"])
def test_more_problems_than_one_move(host):
    """33 problems (one more than the states moved by a launch), and a state that is not physical
    in the last of them: reported, and gone with the next call."""
    from sse.batch import BatchError, BatchedSolver
    from sse.time_integration import to_device, to_host
    probs = [_problem("tri", 2 + i % 3, 1 + i % 2) for i in range(33)]
    batch = BatchedSolver([s for s, _, _ in probs])
    fresh = lambda: [np.array(u0, order="F") if host else to_device(u0) for _, u0, _ in probs]
    dts = [dt for _, _, dt in probs]
    bad = fresh()
    bad[-1][...] = -1.0
    with pytest.raises(BatchError, match="non-physical"):
        batch.rk_steps(bad, dts, 1)
    states = fresh()
    batch.rk_steps(states, dts, 3)
    for (s, u0, dt), u in zip(probs, states):
        want = O.rk_steps(s.arrays, u0, dt, 3)
        assert np.abs((u if host else to_host(u)) - want).max() <= 1e-10 * np.abs(want).max()


def test_states_in_memory_of_other_kinds():
    """States passed as device memory that the batch's kernels do not move: pinned and pageable host
    memory (as a copy by the runtime takes it), beside states on the device."""
    import ctypes as C

    import torch
    from sse import abi
    from sse.batch import BatchedSolver
    from sse.time_integration import to_device, to_host
    probs = [_problem("tri", 2 + i % 3, 1 + i % 2) for i in range(5)]
    batch = BatchedSolver([s for s, _, _ in probs])
    on_device = [to_device(u0) for _, u0, _ in probs]
    states = list(on_device)
    states[1] = torch.empty(on_device[1].shape, dtype=torch.float64, pin_memory=True).copy_(on_device[1])
    states[2] = on_device[2].cpu()
    torch.cuda.synchronize()
    ptrs = (C.c_void_p * 5)(*[x.data_ptr() for x in states])
    dt = np.array([dt for _, _, dt in probs])
    for n in (1, 2):
        code = batch.lib.sse_batch_rk_steps(batch.handle, ptrs, dt.ctypes.data_as(C.POINTER(C.c_double)), n,
                                            abi.SSE_DEVICE, 1)
        assert code == 0, batch.lib.sse_batch_last_error(batch.handle)
    for (s, u0, dt_), x in zip(probs, states):
        want = O.rk_steps(s.arrays, u0, dt_, 3)
        assert np.abs(to_host(x.cuda()) - want).max() <= 1e-10 * np.abs(want).max()
