import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")


# ---------------------------------------------------------------- shared workloads
# 2D lid-driven cavity: 100x100 lattice on [0,1]^2, interior jitter +-0.25h,
# PHS r^3 + degree-3 polynomial, 30-node stencils (the 10k-node cavity case).
CAVITY2D = dict(dim=2, n=100, jitter=0.25, seed=20240601, k_interior=30)
# Small 3D cube with the 1M-node case's stencil rule: 40 interior nodes,
# 60/55/50 on lattice layers 0/1/2 (faces and the two layers under them).
CUBE3D_SMALL = dict(dim=3, n=16, jitter=0.3, seed=7, k_interior=40, k_layers=(60, 55, 50))


@pytest.fixture(scope="session")
def cavity2d():
    import memphys_amd as M
    return M.box_cloud(**CAVITY2D)


@pytest.fixture(scope="session")
def cube3d_small():
    import memphys_amd as M
    return M.box_cloud(**CUBE3D_SMALL)


def lid_bc(cloud, lid_axis):
    """Cavity boundary conditions: velocity Dirichlet on every wall (u = 1 on
    the lid face x[lid_axis] = 1), pressure Neumann everywhere."""
    nv, dim = cloud.nv, cloud.dim
    u_dir = np.ones(nv, dtype=np.uint8)
    p_dir = np.zeros(nv, dtype=np.uint8)
    u0 = np.zeros(nv)
    lid = (cloud.boundary == 1) & (np.abs(cloud.xyz[:, lid_axis] - 1.0) < 1e-12)
    u0[lid] = 1.0
    return u_dir, p_dir, u0


def rel_err(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    den = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (den if den > 0 else 1.0)


def row_block_columns(cloud):
    """Distinct columns per block of 256 device rows, as the upload lists them: rows in
    Morton order of the coordinates, then by decreasing stencil length inside windows
    of 4096; a padding slot holds its own row."""
    dim, nv = cloud.dim, cloud.nv
    bits = 10 if dim == 3 else 16
    lo, hi = cloud.xyz.min(axis=0), cloud.xyz.max(axis=0)
    span = np.where(hi > lo, hi - lo, 1.0)
    g = np.minimum(2.0 ** bits - 1, np.floor((cloud.xyz - lo) / span * 2.0 ** bits))
    g = g.astype(np.uint64)
    key = np.zeros(nv, np.uint64)
    for b in range(bits):
        for a in range(dim):
            bit = (g[:, a] >> np.uint64(b)) & np.uint64(1)
            key |= bit << np.uint64(b * dim + a)
    order = np.argsort(key, kind="stable")
    length = np.diff(cloud.row_ptr)
    for w in range(0, nv, 4096):
        part = order[w:w + 4096]
        order[w:w + 4096] = part[np.argsort(-length[part], kind="stable")]
    out = []
    for b in range(0, nv + 1, 256):  # (nv + 1: the border unknown's row)
        rows = order[b:b + 256]
        cols = [cloud.col[cloud.row_ptr[r]:cloud.row_ptr[r + 1]] for r in rows]
        n = len(np.unique(np.concatenate(cols))) if len(rows) else 0
        out.append(n + (-len(rows)) % 64)  # padding rows of the last row's slice
    return np.array(out)
