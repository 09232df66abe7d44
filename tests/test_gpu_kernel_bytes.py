"""The bytes per launch that mp_kernel_timing_get reports are those of the kernels that
ran: staged entries or gathers in the step kernels, and on small systems the work
fused with the product."""
import numpy as np
import pytest
from conftest import row_block_columns

pytestmark = pytest.mark.gpu


def _print(*a):
    print(*a, flush=True)


def step_bytes(cloud, staged, nuniq):
    """Predictor, right-hand side, corrector: weights, columns (staged: two bytes an
    entry and four per distinct column of a row block), row lengths, and each
    vector once (gathering: the velocities in packed rows of 2 or 4)."""
    W, N, D = cloud.nnz, cloud.nv, cloud.dim
    cols = 2 * W + 4 * nuniq if staged else 4 * W
    V = D if staged else (4 if D == 3 else 2)
    hat = D + (0 if staged else V)
    return [cols + 8 * W * (D + 1) + N * (4 + 8 * (V + hat + D + D)),
            cols + 8 * W * D + N * (4 + 8 * (V + 1)),
            cols + 8 * W * D + N * (4 + 8 * (1 + D + D))]


def _steps(ctx, cloud, krylov=0, precision=0, precond=0, steps=2, restart=0, tol=1e-8):
    import memphys_amd as M
    u_dir, p_dir, u0 = M.lid_conditions(cloud)
    ctx.upload(cloud)
    ctx.weights(3, 3, download=False)
    ctx.fs_create(1.0, 0.01, 1e-5, 2, tol, 3000, u_dir, u_dir,
                  u_dir if cloud.dim == 3 else None, p_dir, krylov=krylov, precision=precision,
                  precond=precond, restart=restart)
    ctx.set_field(M.MP_U, u0)
    for f in range(1, cloud.dim):
        ctx.set_field(f, np.zeros(cloud.nv))
    ctx.set_field(M.MP_P, np.zeros(ctx.n_sys))
    ctx.step(1, 0)  # (the kernels' first launches load them, which would set the cut)
    ctx.kernel_timing(True)
    ctx.step(steps, 1)


@pytest.mark.parametrize("dim,n,k", [(2, 40, 20), (2, 411, 20), (3, 16, 40), (3, 56, 40)])
def test_step_kernel_bytes(dim, n, k):
    import memphys_amd as M
    cloud = M.box_cloud(dim=dim, n=n, jitter=0.25, seed=5, k_interior=k)
    u = row_block_columns(cloud)
    staged = len(u) > 640
    with M.Context(0) as ctx:
        _steps(ctx, cloud, krylov=1, precision=1, precond=1, steps=1)
        got = [ctx.kernel_timing_get(q)[2] for q in (1, 2, 3)]
    _print("dim", dim, "n", n, "blocks", len(u), "max", u.max(), "staged", staged, got)
    assert got == step_bytes(cloud, staged, int(u.sum()))


@pytest.mark.parametrize("length,staged", [(12, False), (20, True)])
def test_staging_needs_reuse(length, staged):
    """170k rows in two dimensions.  Rows of 12 whose columns lie anywhere: a row block's
    3,000 distinct columns would fit, but each serves one entry, so the step kernels
    gather.  Rows of 20 with their columns within 1,000 rows: 2,000 distinct columns,
    each serving more than two."""
    import memphys_amd as M
    rng = np.random.default_rng(3)
    nv = 170_011
    row = np.repeat(np.arange(nv), length)
    off = rng.integers(1, 1000 if staged else nv, nv * length)
    col = ((row + off) % nv).astype(np.int32)
    col[::length] = np.arange(nv)
    cloud = M.Cloud(dim=2, xyz=np.c_[np.linspace(0, 1, nv), np.zeros(nv)],
                    boundary=np.zeros(nv, np.uint8), normal=np.zeros((nv, 2)),
                    row_ptr=(np.arange(nv + 1) * length).astype(np.int32), col=col,
                    ksize=np.full(nv, length, np.int32), layer=np.zeros(nv, np.int32))
    u = row_block_columns(cloud)
    _print("max", u.max(), "reuse", cloud.nnz / u.sum())
    assert 2 * u.max() <= 8192 and (cloud.nnz / u.sum() > 2 if staged else
                                    cloud.nnz / u.sum() < 1.1)
    w = 0.1 * rng.uniform(-1, 1, cloud.nnz)
    u_dir = np.zeros(nv, np.uint8)
    u_dir[0] = 1
    with M.Context(0) as ctx:
        ctx.upload(cloud)
        ctx.set_weights(w, w, None, w)
        ctx.fs_create(1.0, 0.01, 1e-5, 2, 1e-8, 100, u_dir, u_dir, None, np.zeros(nv, np.uint8))
        got = [ctx.kernel_timing_get(q)[2] for q in (1, 2, 3)]
    assert got == step_bytes(cloud, staged, int(u.sum()))


@pytest.mark.parametrize("n,lo,hi", [(40, 44, 60), (170, 28, 36), (420, 28, 36)])
def test_bicgstab_product_bytes(n, lo, hi):
    """FP64 BiCGSTAB, per row and beside the matrix.  Up to 96 row blocks the two
    products gather r, p, v and r, v, write p, v and s, t and read r0: 60 and 44
    bytes with D^-1 and the length.  In the other forms x, the product, r0: 36 and
    28.  The reported mean lies between."""
    import memphys_amd as M
    cloud = M.box_cloud(dim=2, n=n, jitter=0.25, seed=5, k_interior=20)
    u = row_block_columns(cloud)
    with M.Context(0) as ctx:
        _steps(ctx, cloud, tol=1e-3)
        launches, _, got, _ = ctx.kernel_timing_get(0)
    matrix = 10 * cloud.nnz + 4 * int(u.sum()) if len(u) > 640 else 12 * cloud.nnz
    rows = (got - matrix) / cloud.nv
    _print("n", n, "blocks", len(u), "launches", launches, "bytes per row", rows)
    assert launches >= 1
    assert lo <= rows <= hi


@pytest.mark.parametrize("n,fused", [(40, True), (420, False)])
def test_gmres_product_bytes(n, fused):
    """FP64 GMRES(30) with the multigrid (it would stall with Jacobi or short cycles, and
    BiCGSTAB end the solve): the V-cycle's FP32 output, the product, D^-1 and the
    length, 24 bytes a row; on small systems the launch of iteration k also reads
    the k + 1 basis vectors."""
    import memphys_amd as M
    cloud = M.box_cloud(dim=2, n=n, jitter=0.25, seed=5, k_interior=20)
    u = row_block_columns(cloud)
    with M.Context(0) as ctx:
        _steps(ctx, cloud, krylov=1, restart=30, precond=1, steps=1)
        launches, _, got, _ = ctx.kernel_timing_get(0)
    matrix = 12 * cloud.nnz if fused else 10 * cloud.nnz + 4 * int(u.sum())
    rows = (got - matrix) / cloud.nv
    _print("n", n, "blocks", len(u), "launches", launches, "bytes per row", rows)
    assert launches >= 1
    if fused:
        assert 24 + 8 <= rows <= 24 + 240
    else:
        assert abs(rows - 24) < 1e-6
