"""Calls whose kernels depend on the mesh: what a run gives must not depend on
which of the paired (pair.hpp) and the general kernels it gets."""
import numpy as np
import pytest

import miniaero_amd as M
from test_skew_plan import rotated_mesh

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


def _solo_equals_batched(case, other, steps=4, **solo):
    """The case alone and in a batch with `other`, a box, which keeps both on the
    general kernels: the same bits."""
    md, o = case
    runs = [M.TimeSolverExplicitRK4(md, o.replace(**solo)), M.BatchSolver([case, other])]
    try:
        for s in runs:
            s.initialize()
            s.step(steps)
        n = runs[1].offsets[1]
        U = runs[1].state()[:n]
        assert np.isfinite(U).all()
        assert np.array_equal(runs[0].state(), U)
        assert np.array_equal(runs[0].residual(), runs[1].residual()[:n])
        if o.second_order_space or o.viscous:
            for a, b in zip(runs[0].gradients(), runs[1].gradients()):
                assert np.array_equal(a, b[:n])
    finally:
        for s in runs:
            s.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)])
@pytest.mark.parametrize("tile", [(0, 0, 0), (4, 8, 8), (3, 7, 9), (-1, 0, 0)])
def test_rotated_boxes(scheme, precision, tile):
    """Meshes with no face along an axis: up to three chunks of a block's faces."""
    box, o = _case((21, 13, 10), scheme, precision=precision, tile_shape=tile)
    _solo_equals_batched((rotated_mesh(o), o), _case((6, 5, 4), scheme, precision=precision, tile_shape=tile))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)])
def test_batch_of_skew_meshes(scheme, precision):
    """Meshes of different sizes merged in the skew form, their tables' side and
    slot bits above cell and record numbers that follow another mesh's: the bits
    of each one alone."""
    cases = []
    for shape, angles in (((21, 13, 10), (0.4, 0.3, 0.2)), ((1, 3, 17), (0.1, 0.7, 0.3)), ((9, 8, 7), (0.2, 0.2, 1.0))):
        o = _case(shape, scheme, precision=precision)[1]
        cases.append((rotated_mesh(o, angles), o))
    if not precision:  # (a ramp's area vectors carry noise too small for the FP32 form)
        cases.append(_case((17, 9, 8), scheme, **RAMP))
    runs = [M.BatchSolver(cases)] + [M.TimeSolverExplicitRK4(*c) for c in cases]
    try:
        for s in runs:
            s.initialize()
            s.step(4)
        for k in range(len(cases)):
            assert np.array_equal(runs[0].case_state(k), runs[1 + k].state())
    finally:
        for s in runs:
            s.close()


@pytest.mark.parametrize("scheme", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)])
@pytest.mark.parametrize("tile", [(1, 1, 1), (2, 2, 2), (1, 4, 4), (4, 8, 1), (1, 1, 21), (1, 1, 22)])
def test_tiles_of_few_cells(scheme, tile):
    """Tiles whose faces of a class fill one chunk of 64, and (1 x 1 x 22: 67
    faces across) tiles where one class does not."""
    box = _case((13, 11, 23), scheme, tile_shape=tile)
    other = _case((6, 5, 4), scheme, tile_shape=tile, **RAMP)
    _solo_equals_batched(box, other)
    _solo_equals_batched((rotated_mesh(box[1]), box[1]), _case((6, 5, 4), scheme, tile_shape=tile))


def test_lists_of_mostly_padding_are_not_made():
    """373k tiles of one cell: 72 million list entries for the paired kernels."""
    md, o = _case((72, 72, 72))
    U = []
    for tile in ((1, 1, 1), (0, 0, 0)):
        s = M.TimeSolverExplicitRK4(md, o.replace(tile_shape=tile))
        try:
            s.initialize()
            s.step(2)
            U.append(s.state())
            if tile[0]:
                assert s.sizes()["device_bytes"] < 1500 * 72 ** 3
        finally:
            s.close()
    assert np.array_equal(*U)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 1), (1, 2, 2), (7, 1, 1), (13, 11, 7)])
def test_gradients_read_in_parts(shape, precision):
    """Gradients come back a third of the cells at a time: meshes of one to a few
    cells and counts that three does not divide, together and one at a time."""
    from miniaero_amd import _lib
    case = _case(shape, precision=precision)
    _solo_equals_batched(case, _case((3, 2, 2), precision=precision, **RAMP))
    s = M.TimeSolverExplicitRK4(*case)
    try:
        s.initialize()
        s.step(2)
        U, (g, lim) = s.state(), s.gradients()
        assert np.isfinite(g).all() and np.isfinite(lim).all()
        g1, l1 = np.empty_like(g), np.empty_like(lim)
        _lib.check(s._L.ma_solver_get_gradients(s._h, g1.ctypes.data_as(_lib._D), None))
        _lib.check(s._L.ma_solver_get_gradients(s._h, None, l1.ctypes.data_as(_lib._D)))
        assert np.array_equal(g, g1) and np.array_equal(lim, l1)
        assert np.array_equal(s.state(), U)
        s.step(2)
        t = M.TimeSolverExplicitRK4(*case)
        try:
            t.initialize()
            t.step(4)
            assert np.array_equal(s.state(), t.state())
        finally:
            t.close()
    finally:
        s.close()


@pytest.mark.parametrize("precision,shape", [(0, (16, 16, 8)), (0, (23, 10, 9)), (0, (32, 16, 16)), (0, (27, 19, 16)),
                                             (1, (64, 32, 32)), (1, (41, 40, 40))])
def test_reads_ordered_by_the_host_and_on_the_device(precision, shape):
    """State, residual, gradients and limiters on both sides of the sizes up to
    which the host puts them into order: 2048 and 8192 cells, 65536 in FP32."""
    from miniaero_amd import _lib
    case = _case(shape, precision=precision)
    small = _case((3, 2, 2), precision=precision, **RAMP)
    _solo_equals_batched(case, small)
    s = M.TimeSolverExplicitRK4(*case)
    try:
        s.initialize()
        s.step(2)
        g, lim = s.gradients()
        g1, l1 = np.empty_like(g), np.empty_like(lim)
        _lib.check(s._L.ma_solver_get_gradients(s._h, g1.ctypes.data_as(_lib._D), None))
        _lib.check(s._L.ma_solver_get_gradients(s._h, None, l1.ctypes.data_as(_lib._D)))
        assert np.array_equal(g, g1) and np.array_equal(lim, l1)
    finally:
        s.close()


def test_default_tiles():
    """4x4x4 up to 128 cells per CU, 4x4x8 above for runs on the paired kernels
    (4x4x4 for others: stretched beyond their bounds, a FP32 ramp whose area
    vectors carry noise, a box and a ramp as one batch), 4x8x8 from 256 on; the same bits with each."""
    cus = 256
    kw = dict(lx=1.0, ly=0.05, lz=0.025, dt=1e-14)
    small, medium, large = (4, 4, 4), (4, 4, 8), (4, 8, 8)
    cases = [((cus // 2, 16, 16), {}, small), ((cus // 2 + 1, 16, 16), {}, medium), ((cus, 16, 16), {}, large),
             ((cus // 2 + 1, 16, 16), dict(precision=1), medium),
             ((64, 40, 16), dict(precision=1, lx=2.0, ly=2.0, lz=1.0, problem_type=2, angle=30.0), small),
             ((65, 40, 16), dict(y_stretch=1.45), small), ((65, 40, 16), dict(y_stretch=1.05), medium)]
    for shape, more, tile in cases:
        md, o = _case(shape, **dict(kw, **more))
        U = []
        for t in ((0, 0, 0), (4, 4, 4), (4, 4, 8), (4, 8, 8)):
            s = M.TimeSolverExplicitRK4(md, o.replace(tile_shape=t))
            try:
                assert s.tile_shape()[0] == (t if t[0] else tile), (shape, more)
                s.initialize()
                s.step(1)
                U.append(s.state())
            finally:
                s.close()
        assert all(np.array_equal(U[0], x, equal_nan=True) for x in U[1:])
    n = cus * 128 // 2 // 256 + 1
    both = M.BatchSolver([_case((n, 16, 16)), _case((n, 16, 16), ly=1.0, lz=1.0, **RAMP)])
    try:
        assert both.tile_shape()[0] == small
    finally:
        both.close()


@pytest.mark.parametrize("graph", [0, 2])
def test_state_read_while_another_thread_steps(graph):
    """A monitor thread's reads go through the buffer that a step accumulates in:
    they come between steps, and the run ends with an undisturbed run's bits."""
    import threading
    case = _case((24, 20, 16))
    states = []
    for watch in (False, True):
        s = M.TimeSolverExplicitRK4(*case)
        try:
            s.set_graph(graph)
            s.initialize()
            done = threading.Event()
            seen = []

            def read():
                while not done.is_set():
                    seen.append(np.isfinite(s.state()).all() and np.isfinite(s.residual()).all())

            t = threading.Thread(target=read)
            if watch:
                t.start()
            for _ in range(60):
                s.step(3 if not graph else 4)
            done.set()
            if watch:
                t.join()
                assert seen and all(seen)
            states.append(s.state())
        finally:
            done.set()
            s.close()
    assert np.array_equal(*states)


def _states(case, variants, steps):
    out = []
    for v in variants:
        s = M.TimeSolverExplicitRK4(case[0], case[1].replace(**v.get("options", {})))
        try:
            if v.get("persistent"):
                s.set_persistent(True)
            s.initialize()
            s.step(steps)
            out.append([s.state(), s.residual()])
            if case[1].second_order_space or case[1].viscous:
                out[-1] += list(s.gradients())
        finally:
            s.close()
    return out


def _same(states):
    assert np.isfinite(states[0][0]).all()
    for other in states[1:]:
        for a, b in zip(states[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(33, 17, 9), (21, 19, 11)])
def test_own_side_form_with_partial_blocks(shape, precision):
    """Viscous second order in tiles of more than 128 cells, where a cell's three
    high faces are one wavefront's (pair.hpp, own_faces), and tiles of a last
    block with fewer than 64 cells: inactive lanes, neighbours behind the block's
    end, padded chunks.  FP64 equals the oracle; FP32 the small default tiles."""
    from test_gpu_parity import Pair
    tiles = [(4, 8, 8), (3, 7, 9), (5, 5, 10), (-1, 0, 0)]
    cells = [256 if t[0] < 0 else t[0] * t[1] * t[2] for t in tiles]
    n = shape[0] * shape[1] * shape[2]
    assert all(c > 128 for c in cells) and cells[1] % 64 and cells[2] % 64 and n % 256 % 64
    _same(_states(_case(shape, precision=precision),
                  [dict(options=dict(tile_shape=t)) for t in [(0, 0, 0)] + tiles], 4))
    if not precision:
        for t in tiles[:3]:
            o = _case(shape)[1]
            p = Pair(dict({k: getattr(o, k) for k in ("problem_type", "lx", "ly", "lz", "nx", "ny", "nz", "dt", "ntimesteps",
                                                      "second_order_space", "viscous", "limiter", "ic_kind", "perturb",
                                                      "seed", "bc_kind")}, tile_shape=t))
            try:
                G, R = p.step(3)
                assert np.array_equal(G, R)
            finally:
                p.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", [(1, 0, 1), (1, 1, 0), (0, 1, 0)])
def test_skew_tiles_walked_and_long(scheme, precision):
    """Skew meshes of 93k cells: workgroups that walk several tiles each, lists of
    more entries than a workgroup has threads; the default layout's bits."""
    o = _case((101, 33, 28), scheme, precision=precision)[1]
    _same(_states((rotated_mesh(o), o),
                  [dict(options=x) for x in ({}, dict(tile_shape=(3, 5, 7), workgroups_per_cu=1),
                                             dict(tile_shape=(4, 8, 8)),
                                             dict(tile_shape=(4, 8, 8), workgroups_per_cu=1))], 2))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)])
def test_persistent_steps_on_skew_meshes(scheme, precision):
    o = _case((19, 12, 9), scheme, precision=precision)[1]
    _same(_states((rotated_mesh(o), o), [dict(), dict(persistent=True)], 3))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("scheme", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (1, 1, 0)])
def test_internal_faces_pointing_down_their_axis(scheme, precision):
    """A box some of whose internal faces have their cells the other way round:
    along an axis, but of the class of faces along none."""
    from test_skew_plan import _frames
    md, o = _case((13, 11, 10), scheme, precision=precision)
    f = md.internal_faces
    turn = np.arange(f.nfaces_) % 3 == 1
    f.face_cell_conn = np.where(turn[:, None], f.face_cell_conn[:, ::-1], f.face_cell_conn)
    f.face_normal = np.where(turn[:, None], -f.face_normal, f.face_normal) + 0.0  # (no -0)
    f.face_tangent, f.face_binormal = _frames(f.face_normal)
    f.cell_flux_index = f.permute_vector = None
    assert md.plan()["derived_frames"]
    _solo_equals_batched((md, o), _case((6, 5, 4), scheme, precision=precision))


@pytest.mark.parametrize("scheme", [(1, 0, 0), (1, 1, 0)])
@pytest.mark.parametrize("stretch", [1.22, 1.28])
def test_plates_on_both_sides_of_the_bounds(stretch, scheme):
    """Stretched plates just inside the paired kernels' largest ratio of area times
    displacement to volume, 2^14, and just beyond it, as the default tiles of runs
    of this size tell: the oracle's bits."""
    from test_gpu_parity import Pair
    p = Pair(dict(problem_type=1, lx=1.0, ly=0.05, lz=0.025, nx=48, ny=48, nz=16, y_stretch=stretch, dt=1e-12,
                  ntimesteps=2, second_order_space=scheme[0], viscous=scheme[1], limiter=scheme[2], ic_kind=2,
                  perturb=0.01, seed=5))
    try:
        ratio = (1 / 48) / (2 * 0.05 * (stretch - 1) / (stretch ** 48 - 1))
        assert p.gpu.tile_shape()[0] == ((4, 4, 8) if ratio < 2 ** 14 else (4, 4, 4))
        G, R = p.step(2)
        assert np.isfinite(R).all() and np.array_equal(G, R)
    finally:
        p.close()


FIRST_CAPTURE = """
import sys
sys.path[:0] = %r
import numpy as np
import miniaero_amd as M
from test_gpu_routes import _case
md, o = _case((33, 17, 9), workgroups_per_cu=1)
states = []
for graph in (2, 0):
    s = M.TimeSolverExplicitRK4(md, o)
    if graph:
        s.set_graph(graph)
    s.initialize()
    s.step(4)
    states.append(s.state())
    s.close()
assert np.isfinite(states[0]).all() and np.array_equal(*states)
"""


def test_first_use_of_the_walking_kernels_in_a_capture():
    """A process whose first launch of these kernels, in a code object that nothing
    else of the run has loaded, is recorded into a graph."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", FIRST_CAPTURE % [here, os.path.dirname(here)]], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
