"""Krylov solves around the sizes where the small-system kernels take over: 64
rows per block with a wavefront per chain, BiCGSTAB iterations of three, five or
eight launches, GMRES with its Hessenberg column in the update.  A system's
iterates do not depend on which of them runs, so a cavity inside a batch large
enough for the general kernels equals its stand-alone run bit for bit, and
every size meets the oracle's operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _print(*a):
    print(*a, flush=True)


def _run(ctx, cloud, krylov, precision, steps=2):
    import memphys_amd as M
    u_dir, p_dir, u0 = M.lid_conditions(cloud)
    ctx.weights(3, 3, download=False)
    ctx.fs_create(1.0, 0.01, 1e-5, 2, 1e-10, 4000, u_dir, u_dir, None, p_dir, krylov=krylov,
                  precision=precision, restart=30)
    ctx.set_field(M.MP_U, u0)
    ctx.set_field(M.MP_V, np.zeros(cloud.nv))
    ctx.set_field(M.MP_P, np.zeros(ctx.n_sys))
    ctx.step(steps, 0)
    return [ctx.get_field(f) for f in (M.MP_U, M.MP_V, M.MP_P)]


@pytest.mark.parametrize("krylov", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_small_cavity_in_large_batch_is_bit_identical(krylov, precision):
    """Cavities of 1, 3, 96, 97 and 128 row blocks alone (three- and five-launch
    BiCGSTAB, both GMRES updates) and in one batch of more than 640 blocks
    (the general kernels)."""
    import memphys_amd as M
    sizes = [15, 27, 156, 157, 181, 460]
    clouds = [M.box_cloud(dim=2, n=n, jitter=0.25, seed=n, k_interior=30) for n in sizes]
    rows = [-(-(c.nv + 1) // 256) for c in clouds]
    _print("row blocks", rows)
    assert rows[:5] == [1, 3, 96, 97, 128] and sum(rows) > 640
    with M.Context(0) as ctx:
        cat = ctx.upload_batch(clouds)
        batch = _run(ctx, cat, krylov, precision)
        iters = [ctx.batch_stats(q).iterations for q in range(len(clouds))]
    off = 0
    for q, c in enumerate(clouds[:5]):
        with M.Context(0) as ctx:
            ctx.upload(c)
            alone = _run(ctx, c, krylov, precision)
            st = ctx.stats()
        _print("n", sizes[q], "blocks", rows[q], "iterations", st.iterations, iters[q])
        assert st.iterations == iters[q]
        for a, b in zip(alone, batch):
            assert np.array_equal(a[:c.nv], b[off:off + c.nv])
        assert alone[2][c.nv] == batch[2][cat.nv + q]  # border unknown
        off += c.nv


@pytest.mark.parametrize("n,k", [(8, 12), (15, 30), (17, 65), (64, 20)])
def test_small_system_solves_its_operator(n, k):
    """Stencils of 12 to 65 entries (one to seventeen groups of four: chains of
    unequal length, tails past the prefetched groups)."""
    import memphys_amd as M
    import oracle as O
    import scipy.sparse as sp
    cloud = M.box_cloud(dim=2, n=n, jitter=0.25, seed=3, k_interior=k)
    w = O.stencil_weights(cloud, 3, 3)[:4]
    p_dir = np.zeros(cloud.nv, dtype=np.uint8)
    ones = np.ones(cloud.nv, dtype=np.uint8)
    fs = O.FractionalStep(cloud, w, ones, ones, None, p_dir, 1.0, 0.01, 1e-3, 2, solver_kind=0,
                          precond=2, tol=1e-14)
    rp, ci, v = fs.ppe_csr()
    rng = np.random.default_rng(n)
    for prec in (0, 1):
        with M.Context(0) as ctx:
            ctx.upload(cloud)
            ctx.set_weights(*w)
            m = ctx.solver_init(p_dir, 0.0, 0.0, 1.0, tol=1e-10, n_iter=20000, precision=prec)
            A = sp.csr_matrix((v, ci, rp), shape=(m, m))
            b = rng.standard_normal(m)
            b[-1] = 0.0
            x, _ = ctx.solve(b, np.zeros(m))
            res = np.linalg.norm(A @ x - b) / np.linalg.norm(b)
            _print("n", n, "k", k, "prec", prec, "iterations", ctx.stats().iterations, "res", res)
            # the solver's own FP64 test, plus the rounding of A x on this host
            assert res <= 1.1e-10


@pytest.mark.parametrize("spread", [40, 10 ** 9])
@pytest.mark.parametrize("prec", [0, 1])
def test_large_system_with_local_and_scattered_columns(spread, prec):
    """170k rows (above the small systems' sizes) whose columns lie near their
    row (each row block's distinct entries staged in LDS) or anywhere (more
    distinct entries than are staged: gathered directly), with rows of 3 to 35
    entries and a block of padding rows."""
    import memphys_amd as M
    import scipy.sparse as sp
    rng = np.random.default_rng(8)
    nv = 170_011
    x = np.sort(rng.random(nv))
    length = rng.integers(3, 36, nv)
    length[:4096] = 35
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    row = np.repeat(np.arange(nv), length)
    off = rng.integers(1, min(spread, nv // 2), rp[-1]) * rng.choice([-1, 1], rp[-1])
    col = ((row + off) % nv).astype(np.int32)
    col[rp[:-1]] = np.arange(nv)
    cloud = M.Cloud(dim=2, xyz=np.c_[x, np.zeros(nv)], boundary=np.zeros(nv, np.uint8),
                    normal=np.zeros((nv, 2)), row_ptr=rp, col=col, ksize=length.astype(np.int32),
                    layer=np.zeros(nv, np.int32))
    lap = 0.4 * rng.uniform(-1, 1, rp[-1]) / length[row]
    with M.Context(0) as ctx:
        ctx.upload(cloud)
        ctx.set_weights(lap, lap, None, lap)
        n = ctx.solver_init(np.zeros(nv, np.uint8), 1.0, 0.0, 1.0, tol=1e-11, n_iter=500,
                            precision=prec)
        assert n == nv + 1
        A = sp.csr_matrix((lap, col, rp), shape=(nv, nv)) + sp.identity(nv)
        b = rng.standard_normal(n)
        sol, _ = ctx.solve(b, np.zeros(n))
        r = np.r_[A @ sol[:nv] + sol[nv], sol[:nv].sum()] - b
        res = np.linalg.norm(r) / np.linalg.norm(b)
        _print("spread", spread, "prec", prec, "iterations", ctx.stats().iterations, "res", res)
        assert res <= 1.1e-11  # the solver's FP64 test, plus this host's rounding


def _with_far_columns(cloud, weights, rows, extra, rng):
    """The cloud with `extra` columns from anywhere appended to the stencils of `rows`, and
    its weights with small ones (1e-3 of the stencil's own) there."""
    import memphys_amd as M
    nv = cloud.nv
    add = np.zeros(nv, np.int64)
    add[rows] = extra
    length = np.diff(cloud.row_ptr)
    rp = np.concatenate([[0], np.cumsum(length + add)]).astype(np.int32)
    old = np.arange(cloud.nnz) + np.repeat(rp[:-1] - cloud.row_ptr[:-1], length)
    new = (rp[rows] + length[rows])[:, None] + np.arange(extra)
    col = np.empty(rp[-1], np.int32)
    col[old] = cloud.col
    col[new] = rng.integers(0, nv, new.shape)
    out = []
    for w in weights:
        if w is None:
            out.append(None)
            continue
        x = np.empty(rp[-1])
        x[old] = w
        x[new] = rng.uniform(-1, 1, new.shape) * 1e-3 * np.abs(w[cloud.row_ptr[rows]])[:, None]
        out.append(x)
    c = M.Cloud(dim=cloud.dim, xyz=cloud.xyz, boundary=cloud.boundary, normal=cloud.normal,
                row_ptr=rp, col=col, ksize=(length + add).astype(np.int32), layer=cloud.layer)
    return c, out


@pytest.mark.parametrize("dim,n,k,extra,form", [
    (2, 411, 30, 0, "staged"), (3, 56, 40, 0, "staged"), (3, 56, 150, 0, "staged"),
    (2, 411, 30, 19, "steps gather"), (3, 56, 40, 14, "steps gather"),
    (2, 411, 30, 32, "all gather"), (3, 56, 40, 32, "all gather")])
def test_large_cloud_step_matches_its_operators(dim, n, k, extra, form):
    """One Euler step of a cloud above 640 row blocks against the operator products,
    which gather: the predictor's source and the corrected velocity bit for bit, the
    pressure by its residual.  The predictor, right-hand side and corrector read
    staged entries, unless one row block has too many distinct columns for `dim`
    vectors in 64 KB (256 rows with columns from anywhere), or for the products too."""
    import memphys_amd as M
    from conftest import row_block_columns
    from test_gpu_kernel_bytes import step_bytes
    kw = dict(k_layers=(60, 55, 50)) if k == 40 else {}
    cloud = M.box_cloud(dim=dim, n=n, jitter=0.25, seed=5, k_interior=k, **kw)
    rng = np.random.default_rng(1)
    u_dir, p_dir, _ = M.lid_conditions(cloud)
    wall = cloud.boundary == 1
    weights = None
    if extra:
        inner = np.flatnonzero(~wall)
        near = inner[np.argsort(np.linalg.norm(cloud.xyz[inner] - 0.3, axis=1))[:256]]
        with M.Context(0) as ctx:
            ctx.upload(cloud)
            weights, _ = ctx.weights(3, 3)
        cloud, weights = _with_far_columns(cloud, weights, near, extra, rng)
    blocks = row_block_columns(cloud)
    _print("dim", dim, "extra", extra, "distinct columns", blocks.max())
    assert len(blocks) > 640
    assert {"staged": blocks.max() <= 8192 // dim, "all gather": blocks.max() > 6144,
            "steps gather": 8192 // dim < blocks.max() <= 6144}[form]
    rho, mu, dt, tol = 1.0, 0.01, 1e-5, 1e-9
    with M.Context(0) as ctx:
        ctx.upload(cloud)
        if weights:
            ctx.set_weights(*weights)
        else:
            ctx.weights(3, 3, download=False)
        ctx.fs_create(rho, mu, dt, 2, tol, 4000, u_dir, u_dir, u_dir if dim == 3 else None, p_dir,
                      precision=M.MP_PREC_MIXED, precond=M.MP_PRECOND_AMG,
                      krylov=M.MP_KRYLOV_GMRES)
        assert ctx.kernel_timing_get(1)[2] == step_bytes(cloud, form == "staged",
                                                         int(blocks.sum()))[0]
        u = [np.where(wall, 0.0, rng.standard_normal(cloud.nv)) for _ in range(dim)]
        for q in range(dim):
            ctx.set_field(q, u[q])
        ctx.set_field(M.MP_P, np.zeros(ctx.n_sys))
        ctx.step(1, 0)
        src = [ctx.get_field(M.MP_SU + q) for q in range(dim)]
        new = [ctx.get_field(q) for q in range(dim)]
        p = ctx.get_field(M.MP_P)
        grad = lambda f: [ctx.apply(o, f) for o in range(dim)]
        hat = []
        for q in range(dim):
            g = grad(u[q])
            conv = -(u[0] * g[0]) - u[1] * g[1]
            if dim == 3:
                conv = conv - u[2] * g[2]
            s = rho * conv + mu * ctx.apply(M.MP_LAP, u[q])
            assert np.array_equal(s, src[q])
            hat.append(u[q] + (dt / rho) * s)
        gp = grad(p[:cloud.nv])
        for q in range(dim):
            assert np.array_equal(np.where(wall, u[q], hat[q] - (dt * gp[q]) / rho), new[q])
        div = sum(ctx.apply(o, hat[o]) for o in range(dim))
        flux = sum((u[a] - hat[a]) * cloud.normal[:, a] for a in range(dim))
        b = np.where(wall, -rho * flux / dt, div * rho / dt)
        ap = np.where(wall, sum(cloud.normal[:, a] * gp[a] for a in range(dim)),
                      ctx.apply(M.MP_LAP, p[:cloud.nv])) + p[cloud.nv]
        res = np.linalg.norm(ap - b) / np.linalg.norm(b)
        _print("dim", dim, "k", k, "residual", res, ctx.stats().rel_res)
        assert res <= 1.5 * tol  # the solver's FP64 test, and the sums' own rounding


def _chain_system(nv, m=12):
    """A cloud whose operator is the identity plus x_{i-1} in row i for the m nodes 2 .. m+1.
    With b = e_1, one BiCGSTAB iteration from x = 0 leaves a residual exactly
    orthogonal to the first one (alpha = 1, omega = 1/2, r = (e_3 - e_2) / 2): the
    solver has to restart.  The solution is 1, -1, 1, ... along the chain."""
    import memphys_amd as M
    length = np.ones(nv, np.int32)
    length[2:2 + m] = 2
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    col = np.empty(rp[-1], np.int32)
    col[rp[:-1]] = np.arange(nv)
    col[rp[2:2 + m] + 1] = np.arange(1, 1 + m)
    lap = np.zeros(rp[-1])
    lap[rp[2:2 + m] + 1] = 1.0
    boundary = np.zeros(nv, np.uint8)
    boundary[0] = 1  # (Dirichlet: no border unknown)
    cloud = M.Cloud(dim=2, xyz=np.c_[np.linspace(0, 1, nv), np.zeros(nv)], boundary=boundary,
                    normal=np.tile([1.0, 0.0], (nv, 1)), row_ptr=rp, col=col, ksize=length,
                    layer=np.zeros(nv, np.int32))
    b, x = np.zeros(nv), np.zeros(nv)
    b[1] = 1.0
    x[1:2 + m] = (-1.0) ** np.arange(m + 1)
    return cloud, lap, b, x


@pytest.mark.parametrize("prec", [0, 1])
def test_bicgstab_restart_is_the_same_in_every_form(prec):
    """The breakdown of r0.r and its restart in iterations of three, five and eight
    launches, alone and in batches beside a system that runs on and one that is done
    from the start: the solution, and the same bits in every form (the rest of each
    system is zero, so its size does not enter the sums)."""
    import memphys_amd as M
    rng = np.random.default_rng(6)
    first = None

    def solve(parts):
        """Solutions of [(cloud, lap, b)] as one context's systems, and the restarts."""
        with M.Context(0) as ctx:
            cat = parts[0][0] if len(parts) == 1 else ctx.upload_batch([p[0] for p in parts])
            if len(parts) == 1:
                ctx.upload(cat)
            lap = np.concatenate([p[1] for p in parts])
            zero = np.zeros_like(lap)
            ctx.set_weights(zero, zero, None, lap)
            n = ctx.solver_init(cat.boundary, 1.0, 0.0, 1.0, tol=1e-13, n_iter=300,
                                precision=prec)
            assert n == cat.nv
            x, _ = ctx.solve(np.concatenate([p[2] for p in parts]), np.zeros(n))
            at = np.cumsum([0] + [p[0].nv for p in parts])
            return [x[a:e] for a, e in zip(at[:-1], at[1:])], ctx.stats().restarts

    for nv in (200, 25_100, 170_011):  # 1, 99 and 665 row blocks
        cloud, lap, b, x = _chain_system(nv)
        (got,), restarts = solve([(cloud, lap, b)])
        _print("nv", nv, "restarts", restarts, "error", np.abs(got - x).max())
        assert restarts >= 1
        assert np.abs(got - x).max() <= 1e-11
        first = got[:14] if first is None else first
        assert np.array_equal(got[:14], first)
    small = _chain_system(200)
    for nv in (3_000, 170_011):  # a batch of fused iterations, and one of eight launches
        cloud = _chain_system(nv, m=nv - 2)[0]
        lap = 0.3 * rng.uniform(-1, 1, cloud.nnz)
        lap[cloud.row_ptr[:-1]] = 0.0
        other = (cloud, lap, rng.standard_normal(nv))
        idle = (small[0], small[1], np.zeros(200))
        (a, o, z, c), _ = solve([small[:3], other, idle, small[:3]])
        assert np.array_equal(a[:14], first) and np.array_equal(c[:14], first)
        assert not z.any()
        r = o.copy()
        r[2:] += lap[cloud.row_ptr[2:-1] + 1] * o[1:-1]
        assert np.linalg.norm(r - other[2]) <= 1.1e-13 * np.linalg.norm(other[2])


def test_middle_size_in_large_batch_is_bit_identical():
    """A cavity of 352 row blocks, between the sizes that the Hessenberg column runs in the
    update (128) and those of the general kernels (640): alone and in a batch."""
    import memphys_amd as M
    clouds = [M.box_cloud(dim=2, n=n, jitter=0.25, seed=n, k_interior=30) for n in (300, 290)]
    assert [-(-(c.nv + 1) // 256) for c in clouds] == [352, 329]
    for krylov in (0, 1):
        with M.Context(0) as ctx:
            cat = ctx.upload_batch(clouds)
            batch = _run(ctx, cat, krylov, 1, steps=1)
            iters = ctx.batch_stats(0).iterations
        with M.Context(0) as ctx:
            ctx.upload(clouds[0])
            alone = _run(ctx, clouds[0], krylov, 1, steps=1)
            assert ctx.stats().iterations == iters
        for a, b in zip(alone, batch):
            assert np.array_equal(a[:clouds[0].nv], b[:clouds[0].nv])


@pytest.mark.parametrize("krylov,precision", [(0, 1), (1, 0), (1, 1)])
def test_large_batch_with_multigrid(krylov, precision):
    """Cavities of 1 to 513 row blocks in a batch of 650: staged V-cycle products over
    several systems and their padding rows, several norm steps beside one product, and
    systems that stop before the others.  The fields match the stand-alone runs to the
    solver's accuracy (the solves run to 1e-12, which fixes a full-Neumann pressure to
    about 1e-10; the hierarchies of a batch share one depth, so not bit for bit)."""
    import memphys_amd as M
    from conftest import rel_err
    sizes = [15, 362, 40, 150, 100]
    clouds = [M.box_cloud(dim=2, n=n, jitter=0.25, seed=n, k_interior=30) for n in sizes]
    assert sum(-(-(c.nv + 1) // 256) for c in clouds) > 640

    def run(ctx, cloud):
        u_dir, p_dir, u0 = M.lid_conditions(cloud)
        ctx.weights(3, 3, download=False)
        ctx.fs_create(1.0, 0.01, 1e-5, 2, 1e-12, 4000, u_dir, u_dir, None, p_dir,
                      krylov=krylov, precision=precision, precond=M.MP_PRECOND_AMG)
        ctx.set_field(M.MP_U, u0)
        ctx.set_field(M.MP_V, np.zeros(cloud.nv))
        ctx.set_field(M.MP_P, np.zeros(ctx.n_sys))
        ctx.step(2, 0)
        return [ctx.get_field(f) for f in (M.MP_U, M.MP_V, M.MP_P)]

    with M.Context(0) as ctx:
        cat = ctx.upload_batch(clouds)
        batch = run(ctx, cat)
        stats = [ctx.batch_stats(q) for q in range(len(clouds))]
    at = 0
    for q, c in enumerate(clouds):
        with M.Context(0) as ctx:
            ctx.upload(c)
            alone = run(ctx, c)
            its = ctx.stats().iterations
        err = [rel_err(b[at:at + c.nv], a[:c.nv]) for a, b in zip(alone, batch)]
        _print("n", sizes[q], "iterations", its, stats[q].iterations, "err", err)
        assert stats[q].converged and max(err) <= 1e-8
        at += c.nv
