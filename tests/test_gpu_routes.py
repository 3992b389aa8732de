"""Calls whose kernels depend on the mesh: what a run gives must not depend on
which of the paired (pair.hpp) and the general kernels it gets."""
import numpy as np
import pytest

import miniaero_amd as M

pytestmark = pytest.mark.gpu

RAMP = dict(problem_type=2, angle=20.0)


def _case(shape, scheme=(1, 1, 0), **more):
    nx, ny, nz = shape
    o = M.Options(**dict(dict(problem_type=1, lx=nx / 64, ly=ny / 128, lz=nz / 128, nx=nx, ny=ny, nz=nz, dt=1e-6,
                              ntimesteps=4, second_order_space=scheme[0], viscous=scheme[1], limiter=scheme[2],
                              ic_kind=2, perturb=0.02, seed=5, bc_kind=(1, 1, 3, 2, 4, 1)), **more))
    return M.Parallel3DMesh(o.nx, o.ny, o.nz, o.lx, o.ly, o.lz, o.problem_type, o.angle,
                            options=o).fillMeshData(), o


@pytest.mark.parametrize("graph", [0, 2])
@pytest.mark.parametrize("precision", [0, 1])
def test_time_of_fixed_steps(precision, graph):
    """A box (paired), a FP32 ramp (general kernels) and both as one batch of
    different time steps: the time is the sum of the steps in step order."""
    cases = [_case((9, 7, 5), precision=precision, dt=1e-6),
             _case((6, 5, 4), precision=precision, dt=3e-7, **RAMP)]
    runs = [M.TimeSolverExplicitRK4(*c) for c in cases] + [M.BatchSolver(cases)]
    try:
        for s in runs:
            if graph:
                s.set_graph(graph)
            s.initialize()
            s.step(5)
        for k, (_, o) in enumerate(cases):
            t = 0.0
            for _ in range(5):
                t += o.dt
            assert runs[k].time() == (t, o.dt)
            assert runs[2].case_time(k) == (t, o.dt)
    finally:
        for s in runs:
            s.close()
