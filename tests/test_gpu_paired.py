"""The paired-mesh kernels (boxes: every face along an axis; ramps: the form for
skew meshes) where they can go wrong: dimensions of one cell, tiles and 64-cell
chunks with remainders, every boundary kind on every scheme, values outside the
range of the short quotients.

FP64 equals the oracle bit for bit.  A batch of boxes and ramps together runs
the general kernels for all its cases, so it gives the general kernels' bits
for the meshes, in FP32 too: results are equal.
"""
import numpy as np
import pytest

import miniaero_amd as M
from test_gpu_parity import Pair, _log

pytestmark = pytest.mark.gpu

SHAPES = [(65, 1, 1), (1, 2, 67), (5, 9, 13), (33, 16, 9)]
SCHEMES = [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)]  # second order, viscous, limiter
WALLS = [(1, 1, 3, 2, 4, 1), (4, 1, 2, 3, 3, 2)]


RAMP = dict(problem_type=2, angle=20.0)


def _kw(shape, scheme, walls=0, **more):
    nx, ny, nz = shape  # spacings that are powers of two: every area vector exactly along its axis
    return dict(dict(problem_type=1, lx=nx / 64, ly=ny / 128, lz=nz / 128, nx=nx, ny=ny, nz=nz, dt=1e-6,
                     ntimesteps=4, second_order_space=scheme[0], viscous=scheme[1], limiter=scheme[2], ic_kind=2,
                     perturb=0.02, seed=5, bc_kind=WALLS[walls]), **more)


def _same_as_oracle(p, n):
    G, R = p.step(n)
    _log(f"  {n} steps: bitwise={np.array_equal(G, R, equal_nan=True)}, nan {np.isnan(R).sum()}")
    assert np.array_equal(G, R, equal_nan=True)
    if p.opts.second_order_space or p.opts.viscous:
        (g, lim), (og, olim) = p.gpu.gradients(), p.cpu.gradients()
        assert np.array_equal(g, og, equal_nan=True)
        if p.opts.second_order_space:
            assert np.array_equal(lim, olim, equal_nan=True)


@pytest.mark.parametrize("mesh", [{}, RAMP], ids=["box", "ramp"])
@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("shape", SHAPES)
def test_equal_to_the_oracle(shape, scheme, mesh):
    for k, more in enumerate(({}, dict(workgroups_per_cu=1))):
        p = Pair(_kw(shape, scheme, k, **mesh, **more))
        try:
            _same_as_oracle(p, 1)
            _same_as_oracle(p, 3)
        finally:
            p.close()


@pytest.mark.parametrize("what", ["tiny", "huge", "nan"])
@pytest.mark.parametrize("mesh", [{}, RAMP], ids=["box", "ramp"])
@pytest.mark.parametrize("scheme", SCHEMES)
def test_values_outside_the_short_quotients_range(scheme, mesh, what):
    p = Pair(_kw((17, 9, 8), scheme, **mesh))
    try:
        U = p.gpu.state().copy()
        c = np.arange(3, U.shape[0], 97)
        if what == "tiny":
            U[:, 2:4] = 0.0
            U[c, 2] = U[c, 0] * 1e-290
            U[c[::2], 3] = U[c[::2], 0] * -3e-312
        elif what == "huge":
            U[c, 1] = U[c, 0] * 1e140
            U[c, 4] = U[c, 1] ** 2 / U[c, 0]
        else:
            U[c, 1 + scheme[1]] = np.nan
        p.gpu.set_state(U)
        p.cpu.set_state(U)
        _same_as_oracle(p, 1)
        _same_as_oracle(p, 1)
    finally:
        p.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", SCHEMES)
def test_equal_to_the_general_kernels(scheme, precision):
    for k, shape in enumerate(SHAPES):
        cases = []
        for mesh in ({}, RAMP):
            o = M.Options(**_kw(shape, scheme, k % 2, precision=precision, **mesh))
            cases.append((M.Parallel3DMesh(o.nx, o.ny, o.nz, o.lx, o.ly, o.lz, o.problem_type, o.angle,
                                           options=o).fillMeshData(), o))
        _log(f"[gpu-paired] {shape} {scheme} precision {precision}")
        runs = [M.BatchSolver(cases)] + [M.TimeSolverExplicitRK4(*c) for c in cases]
        try:
            for s in runs:
                s.initialize()
                s.step(4)
            U, off = runs[0].state(), runs[0].offsets
            assert np.isfinite(U).all()
            for j in range(2):
                assert np.array_equal(runs[1 + j].state(), U[off[j]:off[j + 1]]), ("box", "ramp")[j]
        finally:
            for s in runs:
                s.close()
