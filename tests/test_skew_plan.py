"""Planning meshes whose faces are along no axis at all (host only)."""
import resource
import subprocess
import sys

import numpy as np
import pytest

import miniaero_amd as M


def _frames(n):
    """Tangent and binormal of area vectors by Face.C:37-98's rule, operation
    for operation, so that the plan recognises them."""
    m = np.abs(n)
    i1 = np.where(m[:, 1] > m[:, 0], 1, 0)
    i1 = np.where(m[:, 2] > np.where(i1 == 0, m[:, 0], m[:, 1]), 2, i1)
    r = np.arange(len(n))
    p, q = n[r, i1], n[r, (i1 + 2) % 3]
    den = np.sqrt(p * p + q * q)
    t = np.zeros_like(n)
    t[r, i1], t[r, (i1 + 2) % 3] = q / den, -p / den
    b = np.stack([n[:, 1] * t[:, 2] - t[:, 1] * n[:, 2], -n[:, 0] * t[:, 2] + t[:, 0] * n[:, 2],
                  n[:, 0] * t[:, 1] - t[:, 0] * n[:, 1]], 1)
    return t, b


def rotated_mesh(options, angles=(0.4, 0.3, 0.2)):
    """The options' box turned about x, then y, then z: every face is along no axis."""
    R = np.eye(3)
    for a, (i, j) in zip(angles, ((1, 2), (0, 2), (0, 1))):
        Q = np.eye(3)
        Q[i, i] = Q[j, j] = np.cos(a)
        Q[i, j], Q[j, i] = -np.sin(a), np.sin(a)
        R = Q @ R
    o = options
    md = M.Parallel3DMesh(o.nx, o.ny, o.nz, o.lx, o.ly, o.lz, o.problem_type, o.angle, options=o).fillMeshData()
    md.cell_coordinates = md.cell_coordinates @ R.T
    for f in [md.internal_faces] + [g for _, g in md.boundary_faces]:
        f.coordinates = f.coordinates @ R.T
        f.face_normal = f.face_normal @ R.T
        f.face_tangent, f.face_binormal = _frames(f.face_normal)
    return md


@pytest.mark.parametrize("shape", [(4, 8, 8), (9, 8, 7), (33, 17, 9), (1, 1, 70)])
def test_plan_of_a_rotated_box(shape):
    """A block of 64 cells holds up to 192 faces of the one class, three chunks
    of a tile's list.  In a process of its own, bounded in time and memory."""
    code = ("import sys; sys.path[:0] = {!r}\n"
            "import miniaero_amd as M; from test_skew_plan import rotated_mesh\n"
            "o = M.Options(problem_type=1, lx=1.0, ly=0.5, lz=0.5, nx={}, ny={}, nz={})\n"
            "p = rotated_mesh(o).plan()\n"
            "print(p); assert all(p.values()), p\n").format(sys.path, *shape)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=60,
                       preexec_fn=lambda: resource.setrlimit(resource.RLIMIT_DATA, (8 << 30, 8 << 30)))
    assert r.returncode == 0, r.stderr[-2000:]
