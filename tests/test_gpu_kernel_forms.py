"""Forms that kernels take by size or by the matrix's entries, at the sizes
where they can go wrong, against the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

from hazmath_amd import capi, problems
from test_gpu_parity import _hierarchies, _set_precision, _solve_both

pytestmark = pytest.mark.gpu


def _with_stored_zeros(ia, ja, va, per_row, seed):
    """The same symmetric matrix with `per_row` off-diagonal zeros a row on average stored as well (symmetric
    pattern, columns in no order)."""
    import scipy.sparse as sp
    n = ia.size - 1
    rng = np.random.default_rng(seed)
    k = n * per_row // 2
    i = rng.integers(0, n, k)
    j = (i + rng.integers(1, min(n, 200), k)) % n
    M = sp.csr_matrix((va, ja, ia), shape=(n, n)).tocoo()
    have = set(zip(M.row.tolist(), M.col.tolist()))
    new = sorted({p for a, b in zip(i.tolist(), j.tolist()) for p in ((a, b), (b, a)) if p not in have and a != b})
    r = np.concatenate([M.row, np.array([p[0] for p in new], np.int64)])
    c = np.concatenate([M.col, np.array([p[1] for p in new], np.int64)])
    v = np.concatenate([M.data, np.zeros(len(new))])
    order = np.lexsort((rng.random(r.size), r))
    r, c, v = r[order], c[order], v[order]
    ia2 = np.zeros(n + 1, np.int32)
    ia2[1:] = np.cumsum(np.bincount(r, minlength=n))
    return ia2, c.astype(np.int32), v


# rows per slice and entries per slice: a last slice of one row (m = 41: 1,600 rows = 25 slices; 45: 1,936 = 30
# slices and 16 rows), slices of up to 1,024 entries (staged in LDS) and of more (30 zeros a row)
@pytest.mark.parametrize("m,per_row", [(41, 3), (45, 8), (45, 30)])
@pytest.mark.parametrize("smoother", [capi.SMOOTHER_L1DIAG, capi.SMOOTHER_GS])
def test_solve_with_stored_zeros(lib, orc, libc, m, per_row, smoother):
    """The solve's matrix copies leave stored off-diagonal zeros out: the same solution as without them in the
    matrix, and the oracle's (which multiplies by them) within the PCG bars."""
    ia, ja, va = _with_stored_zeros(*problems.poisson2d_p1(m), per_row, seed=m)
    b = problems.uniform_rhs(ia.size - 1, seed=5)
    A = capi.HostCSR(ia, ja, va)
    res = _solve_both(lib, orc, libc, A, b, tol=1e-10, maxit=400, aggregation=capi.HEM, smoother=smoother,
                      coarse_dof=100, theta=0.04)
    (ig, xg), (io, xo) = res["gpu"], res["oracle"]
    # Gauss-Seidel sweeps in another row order than the oracle: its iterations may differ by a quarter
    assert ig > 0 and abs(ig - io) <= (1 if smoother == capi.SMOOTHER_L1DIAG else max(2, io // 4))
    # two iterates below 1e-10 of a system of condition below 2e3 (2-D Laplacian, h = 1/45)
    tol = 1e-10 if smoother == capi.SMOOTHER_L1DIAG else 2e-7
    assert np.linalg.norm(xg - xo) / np.linalg.norm(xo) < tol


def _dirichlet_rows(m):
    """2-D Laplacian with every 7th unknown turned into an identity row (rows outside every aggregate)."""
    import scipy.sparse as sp
    ia, ja, va = problems.poisson2d_p1(m)
    n = ia.size - 1
    M = sp.csr_matrix((va, ja, ia), shape=(n, n))
    keep = np.arange(n) % 7 != 3
    D = sp.diags(keep.astype(float))
    M = (D @ M @ D + sp.diags(1.0 - keep)).tocsr()
    M.eliminate_zeros()
    M.sort_indices()
    return M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data


def _star(ia, ja, va, entries):
    """The matrix with `entries` weak couplings of row 0, spread over all rows, added."""
    import scipy.sparse as sp
    n = ia.size - 1
    j = np.linspace(n // 3, n - 1, entries).astype(np.int64)
    S = sp.coo_matrix((np.full(entries, -1e-3), (np.zeros(entries, np.int64), j)), shape=(n, n)).tocsr()
    S = S + S.T
    M = (sp.csr_matrix((va, ja, ia), shape=(n, n)) + S - sp.diags(np.asarray(S.sum(axis=1)).ravel())).tocsr()
    M.sort_indices()
    return M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data


def _long_row(m, entries):
    """2-D Laplacian with `entries` weak couplings of row 0 added (symmetric, diagonally dominant)."""
    import scipy.sparse as sp
    ia, ja, va = problems.poisson2d_p1(m)
    n = ia.size - 1
    M = sp.csr_matrix((va, ja, ia), shape=(n, n)).tolil()
    for k in range(1, entries + 1):
        j = (k * 13) % (n - 1) + 1
        M[0, j] -= 0.01
        M[j, 0] -= 0.01
        M[0, 0] += 0.01
        M[j, j] += 0.01
    M = M.tocsr()
    M.sort_indices()
    return M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data


def _two_diagonals(m):
    """2-D Laplacian whose rows store their diagonal as two entries, 3 and 1."""
    ia, ja, va = problems.poisson2d_p1(m)
    n = ia.size - 1
    row = np.repeat(np.arange(n), np.diff(ia))
    va = va.copy()
    va[ja == row] = 3.0
    r, c, v = np.concatenate([row, np.arange(n)]), np.concatenate([ja, np.arange(n)]), np.concatenate([va, np.ones(n)])
    order = np.argsort(r, kind="stable")
    ia2 = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    return ia2, c[order].astype(np.int32), v[order]


FUSED = {
    "p2d_hec": (lambda: problems.poisson2d_p1(80), capi.HEC),         # aggregates of uneven size, last workgroup part full
    "p2d_vmb": (lambda: problems.poisson2d_p1(61), capi.VMB),         # larger aggregates
    "kuhn_hem": (lambda: problems.poisson3d_kuhn(22), capi.HEM),      # pairs, zeros left out
    "aniso_hec": (lambda: problems.aniso3d_kuhn(24, 0.7, 0.05), capi.HEC),   # rows of over 16 entries below
    "large_hem": (lambda: problems.aniso3d_kuhn(46, 0.7, 0.05), capi.HEM),   # 91,125 rows: widths by slice
    "row45": (lambda: _star(*problems.aniso3d_kuhn(46, 0.7, 0.05), 45), capi.HEM),   # places, one wide slice a level
    "dirichlet": (lambda: _dirichlet_rows(50), capi.HEC),             # rows in no aggregate: the list-walking kernels
    "row64": (lambda: _long_row(40, 59), capi.HEC),                   # the longest row that the merge takes
    "two_diagonals": (lambda: _two_diagonals(40), capi.HEC),          # Jacobi: the list-walking kernels
    "row200": (lambda: _long_row(40, 195), capi.HEC),                 # longer: the list-walking kernels
}


@pytest.mark.parametrize("case", list(FUSED))
@pytest.mark.parametrize("smoother", [capi.SMOOTHER_L1DIAG, capi.SMOOTHER_JACOBI])
def test_fused_cycle_kernels_vs_oracle(lib, orc, libc, case, smoother):
    """One preconditioner application (both fused kernels on every level that takes them) against the oracle's cycle:
    FP64 within 1e-12 relative (two summation orders of at most 200 terms over at most 10 levels, whose coarsest
    solve amplifies by its condition number, below 1e3); the FP32 and BF16 cycles within their bounds of the FP64
    one (2e-5: 10 levels of 2^-24 roundings; 5e-2: 2^-9 in the values)."""
    import oracle
    make, agg = FUSED[case]
    ia, ja, va = make()
    n = ia.size - 1
    A = capi.HostCSR(ia, ja, va)
    kw = dict(aggregation=agg, smoother=smoother, coarse_dof=60, theta=0.04)
    opts = capi.hz_options()
    lib.hz_get_options(C.byref(opts))
    old = opts.vcycle_precision, opts.jacobi_weight
    opts.jacobi_weight = w = 2.0 / 3.0 if smoother == capi.SMOOTHER_JACOBI else 1.0
    orc.orc_set_jacobi_weight.argtypes = [C.c_double]
    r = problems.uniform_rhs(n, seed=9)
    z = {}
    try:
        orc.orc_set_jacobi_weight(w)
        _, amgo = oracle.params(**kw)
        libc.srand(1)
        h = orc.orc_precond_create(A.ptr(), C.byref(amgo))
        z["oracle"] = np.zeros(n)
        orc.orc_precond_apply(h, capi.dptr(r), capi.dptr(z["oracle"]))
        orc.orc_precond_free(h)
        for precision in (0, 1, 2):
            opts.vcycle_precision = precision
            lib.hz_set_options(C.byref(opts))
            _, amg = capi.solver_params(lib, **kw)
            libc.srand(1)
            pc = lib.create_precond_amg(A.ptr(), C.byref(amg))
            assert pc
            z[precision] = np.zeros(n)
            lib.apply_precond(capi.dptr(r), capi.dptr(z[precision]), pc)
            lib.hz_precond_free(pc)
    finally:
        orc.orc_set_jacobi_weight(1.0)
        opts.vcycle_precision, opts.jacobi_weight = old
        lib.hz_set_options(C.byref(opts))

    def off(a, b):
        return np.linalg.norm(z[a] - z[b]) / np.linalg.norm(z[b])
    assert off(0, "oracle") < 1e-12
    assert off(1, 0) < 2e-5
    assert off(2, 0) < 5e-2


def test_fused_layout_memory_with_a_long_row(lib, libc):
    """A row of 60 entries in a level of 287,496 rows of 15 costs the fused layout its own slice's padding: the solve's
    pool grows by no more than one of its chunks (with the longest row's room in every slice, A and A P took 24 bytes
    times 45 more entries a row there and as many again on the levels below, 600 MB)."""
    base = problems.aniso3d_kuhn(67, 0.7, 0.05)
    held = []
    for ia, ja, va in (base, _star(*base, 45)):
        A = capi.HostCSR(ia, ja, va)
        n = ia.size - 1
        lib.hz_release_device_memory()
        b, x = capi.HostVec(problems.uniform_rhs(n, seed=4)), capi.HostVec(np.zeros(n))
        it, amg = capi.solver_params(lib, tol=1e-6, maxit=200, aggregation=capi.HEM, smoother=capi.SMOOTHER_L1DIAG,
                                     coarse_dof=1000, theta=0.04)
        libc.srand(1)
        r = lib.linear_solver_dcsr_krylov_amg(A.ptr(), b.ptr(), x.ptr(), C.byref(it), C.byref(amg))
        assert r > 0
        held.append(lib.hz_device_pool_bytes())
    lib.hz_release_device_memory()
    print(f"[fused] pool {held[0] >> 20} MB, with the long row {held[1] >> 20} MB", flush=True)
    assert held[1] - held[0] <= 256 << 20


# thread counts of the one-row-a-thread CG are 64, 256, 512 and 1,024; 1,025 rows run the general form; 20
# off-diagonal entries a row read past the 16 held in registers
@pytest.mark.parametrize("n", [1, 5, 63, 64, 65, 255, 256, 257, 512, 513, 1024, 1025])
@pytest.mark.parametrize("per_row", [4, 20])
def test_coarse_cg_sizes_vs_oracle(lib, orc, n, per_row):
    """The coarsest level's CG against the oracle's: iterations within one; solutions of systems of condition below
    10 at relative residuals of 1e-8 differ by less than 2e-7; and on a nonsymmetric matrix of the same size CG
    fails and GMRES takes over, as the oracle's does."""
    import scipy.sparse as sp
    rng = np.random.default_rng(n + per_row)
    k = min(per_row // 2, max(0, n - 1))
    i = np.repeat(np.arange(n), k)
    j = rng.integers(0, n, i.size)
    off = sp.csr_matrix((rng.uniform(-1.0, 0.0, i.size), (i, j)), shape=(n, n))
    off = off + off.T
    off.setdiag(0.0)
    off.eliminate_zeros()
    A = (off + sp.diags(1.0 + 1.5 * np.abs(off).sum(axis=1).A1)).tocsr()
    A.sort_indices()
    b = problems.uniform_rhs(n, seed=2)
    Ah = capi.HostCSR(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(np.float64))
    x, xcg, xo = np.zeros(n), np.zeros(n), np.zeros(n)
    st_cg = capi.INT()
    st = lib.hz_coarse_itsolver(Ah.ptr(), capi.dptr(b), capi.dptr(x), 1e-8, C.byref(st_cg), capi.dptr(xcg))
    so = orc.orc_coarse_itsolver(Ah.ptr(), capi.dptr(b), capi.dptr(xo), 1e-8)
    assert st == st_cg.value > 0 and abs(st - so) <= 1
    assert np.array_equal(x, xcg)
    assert np.linalg.norm(x - xo) <= 2e-7 * np.linalg.norm(xo)


@pytest.mark.parametrize("m", [7, 16, 20, 32])
def test_coarse_gmres_after_small_cg_vs_oracle(lib, orc, m):
    from test_gpu_semantics import _coarse_gpu, _convdiff
    A = _convdiff(m, 6.0, 4.0)
    n = A.shape[0]
    b = problems.uniform_rhs(n, seed=3)
    st, st_cg, x, xcg, Ah = _coarse_gpu(lib, A, b)
    xo = xcg.copy()
    so = orc.orc_pvgmres(Ah.ptr(), capi.dptr(b), capi.dptr(xo), 1e-8, 20 * n, 30)
    assert st_cg < 0 < st and abs(st - so) <= 2
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


def _gs_matrix(rows, per_row, symmetric, long_row=0):
    """Diagonally dominant matrix with about per_row off-diagonal entries a row within 300 of the diagonal, and row
    rows / 2 coupled to `long_row` others spread over all rows."""
    import scipy.sparse as sp
    rng = np.random.default_rng(rows + per_row)
    i = np.repeat(np.arange(rows), per_row // 2 if symmetric else per_row)
    j = (i + rng.integers(1, max(2, min(rows, 300)), i.size)) % rows
    off = sp.csr_matrix((rng.uniform(-1.0, 1.0, i.size), (i, j)), shape=(rows, rows))
    if long_row:
        j = np.linspace(0, rows - 1, long_row).astype(np.int64)
        off = off + sp.csr_matrix((rng.uniform(-1.0, 1.0, long_row), (np.full(long_row, rows // 2), j)),
                                  shape=(rows, rows))
    if symmetric:
        off = off + off.T
    off.setdiag(0.0)
    off.eliminate_zeros()
    A = (off + sp.diags(1.0 + np.asarray(np.abs(off).sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    return capi.HostCSR(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(np.float64)), rng


def _gs_bitexact(lib, orc, M, rows, rng, smoother):
    b, x0 = rng.standard_normal(rows), rng.standard_normal(rows)
    for post in (0, 1):
        order, cptr = np.zeros(rows, np.int32), np.zeros(rows + 2, np.int32)
        nc = capi.INT()
        xg = x0.copy()
        assert lib.hz_gs_smooth(M.ptr(), capi.dptr(b), capi.dptr(xg), smoother, post, 2, 0.8, capi.dptr(order, capi.INT),
                                capi.dptr(cptr, capi.INT), C.byref(nc)) == 0
        xo = x0.copy()
        orc.orc_gs_smooth_ordered(M.ptr(), capi.dptr(b), capi.dptr(xo), smoother, post, 2, 0.8,
                                  capi.dptr(order, capi.INT), capi.dptr(cptr, capi.INT), nc.value)
        assert np.array_equal(np.sort(order), np.arange(rows))
        assert np.array_equal(xg, xo)


# positions (64 per slice, colours padded): one workgroup up to 18,432, colour launches above; rows of up to 8, up to
# 16 and over 16 off-diagonal entries; a nonsymmetric pattern; more than 65,536 rows: widths by slice
@pytest.mark.parametrize("rows,per_row,symmetric", [(1, 0, True), (70, 6, True), (3000, 6, True), (3000, 14, True),
                                                    (3000, 30, True), (3000, 8, False), (21000, 6, True),
                                                    (21000, 20, False), (70001, 6, True)])
@pytest.mark.parametrize("smoother", [capi.SMOOTHER_GS, capi.SMOOTHER_SGS, capi.SMOOTHER_SGSOR])
def test_gauss_seidel_forms_bitexact(lib, orc, rows, per_row, symmetric, smoother):
    """Smoothing calls (two sweeps, before and after the coarse correction) in the library's colour order, bit for bit
    as the oracle sweeps the rows in that order, on every form that the level's size and rows choose."""
    M, rng = _gs_matrix(rows, per_row, symmetric)
    _gs_bitexact(lib, orc, M, rows, rng, smoother)


# one workgroup, colour launches, and more than 65,536 rows; the long row's slices alone are that wide
@pytest.mark.parametrize("rows,long_row", [(3000, 2000), (15000, 9000), (21000, 9000), (70001, 30000)])
@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("smoother", [capi.SMOOTHER_GS, capi.SMOOTHER_SGSOR])
def test_gauss_seidel_long_row(lib, orc, rows, long_row, symmetric, smoother):
    """One row far longer than the others: the same bits as the oracle, and memory for the slices' own widths (at the
    longest row's everywhere the entries alone would take 12 rows long_row bytes, up to 25 GB)."""
    M, rng = _gs_matrix(rows, 6, symmetric, long_row)
    lib.hz_release_device_memory()
    _gs_bitexact(lib, orc, M, rows, rng, smoother)
    assert lib.hz_device_pool_bytes() <= 512 << 20   # two of the pool's chunks


# tiles of 64 rows over 256 workgroups: fewer tiles than workgroups, as many, one more, and several a workgroup with a
# last tile of one row
@pytest.mark.parametrize("B", [65, 16384, 16385, 40001])
def test_mlp_gradient_tiles_vs_fp64(lib, B):
    """Loss and gradient against the same network in FP64: sums of B terms in FP32 over at most 256 partials are within
    2e-5 of the gradient's norm (64-row tiles: 2^-24 times a few hundred roundings)."""
    from scipy.special import erf
    rng = np.random.default_rng(B)
    th = np.zeros(capi.MLP_PARAMS, np.float32)
    lib.hz_mlp_init(capi.fptr(th), 3)
    X = rng.standard_normal((B, capi.MLP_INPUTS)).astype(np.float32)
    T = rng.standard_normal((B, capi.MLP_OUTPUTS)).astype(np.float32)
    grad, loss = np.zeros(capi.MLP_PARAMS, np.float32), np.zeros(1, np.float32)
    assert lib.hz_mlp_loss_grad(capi.fptr(th), capi.fptr(X), capi.fptr(T), B, capi.fptr(grad), capi.fptr(loss)) == 0
    t = th.astype(np.float64)
    o = np.cumsum([0, 16 * 64, 64, 64 * 64, 64, 64 * 16, 16])
    W1, b1, W2, b2, W3, b3 = (t[o[k]:o[k + 1]] for k in range(6))
    W1, W2, W3 = W1.reshape(16, 64), W2.reshape(64, 64), W3.reshape(64, 16)
    x = np.pad(X.astype(np.float64), ((0, 0), (0, 4)))

    def cdf(z):
        return 0.5 * (1.0 + erf(z / np.sqrt(2.0)))

    def dgelu(z):
        return cdf(z) + z * np.exp(-0.5 * z * z) / np.sqrt(2.0 * np.pi)
    z1 = x @ W1 + b1
    h1 = z1 * cdf(z1)
    z2 = h1 @ W2 + b2
    h2 = z2 * cdf(z2)
    d = (h2 @ W3 + b3)[:, :2] - T
    dy = np.zeros((B, 16))
    dy[:, :2] = d / B
    dz2 = (dy @ W3.T) * dgelu(z2)
    dz1 = (dz2 @ W2.T) * dgelu(z1)
    ref = np.concatenate([(x.T @ dz1).ravel(), dz1.sum(0), (h1.T @ dz2).ravel(), dz2.sum(0), (h2.T @ dy).ravel(),
                          dy.sum(0)])
    assert np.linalg.norm(grad - ref) < 2e-5 * np.linalg.norm(ref)
    assert abs(loss[0] - (d ** 2).mean()) < 2e-6 * (d ** 2).mean()


# sweeps before and after (a zero start without sweeps, the last sweep writing z or not), and largest coarsest blocks:
# below 64 rows, above 512; systems of 31^2 + 1 chunk ends: 961 rows (below a chunk of 1,024), 1,024 (one), 1,089 (one
# and a rest); 25 rows are solved at level 0
@pytest.mark.parametrize("pre,post,coarse", [(1, 1, 30), (2, 2, 600), (0, 1, 100), (1, 0, 100), (0, 0, 30)])
def test_batch_cycle_forms_vs_single_system(lib, libc, pre, post, coarse):
    """Every pair as the single-system solver with the same FP32 cycle.  Three iterations on every form of the cycle,
    also those whose iteration does not converge: the iterates differ by what the cycles' applications do, each at most
    2e-5 (the FP32 cycle's bound against FP64) and each step from the one before, 1e-4 in all.  Solves to 1e-8 with
    smoothing on both sides: the iteration at which it is passed moves by at most one; both solutions are within 1e-8
    times the condition number (below 1e4 here) of the true one, 1e-4 of each other."""
    systems = [problems.aniso2d_p1(m, 0.4 + 0.1 * m, 0.3) for m in (32, 6, 33, 34, 48)]
    B = [problems.batch_rhs(s[0].size - 1, k, nrhs=3) for k, s in enumerate(systems)]

    def params(maxit):
        it, amg = capi.solver_params(lib, tol=1e-8, maxit=maxit, aggregation=capi.HEM, smoother=capi.SMOOTHER_JACOBI,
                                     coarse_dof=coarse, theta=0.04)
        amg.presmooth_iter, amg.postsmooth_iter = pre, post
        return it, amg

    old = _set_precision(lib, 1)
    try:
        for maxit in (3, 60) if pre and post else (3,):
            X = [np.zeros_like(b) for b in B]
            r, iters = capi.batch_solve(lib, systems, B, X, *params(maxit))
            for k, (ia, ja, va) in enumerate(systems):
                A = capi.HostCSR(ia, ja, va)
                direct = ia.size - 1 <= coarse   # solved by the coarsest inverse alone: one step, or two
                for q in range(3):
                    its, amgs = params(maxit)
                    x, b = capi.HostVec(np.zeros(ia.size - 1)), capi.HostVec(B[k][q])
                    libc.srand(1)
                    rs = lib.linear_solver_dcsr_krylov_amg(A.ptr(), b.ptr(), x.ptr(), C.byref(its), C.byref(amgs))
                    off = np.linalg.norm(X[k][q] - x.arr) / np.linalg.norm(x.arr)
                    print(f"[batch] {pre},{post},{coarse} {maxit} system {k} rhs {q}: {iters[k, q]} single {rs}, {off:.1e}",
                          flush=True)
                    if direct:
                        assert rs > 0 and 0 < iters[k, q] <= rs + 1
                    elif maxit == 3 or k == 4:   # system 4's anisotropy needs more than 60
                        assert rs == iters[k, q] == -48
                    else:
                        assert rs > 0 and abs(int(iters[k, q]) - rs) <= 1
                    assert off <= 1e-4 or (k == 4 and maxit == 60)
    finally:
        _set_precision(lib, old)


def _banded(n, offsets, classes, diags):
    """Symmetric diagonally dominant matrix with entries at +-offsets[k], value -(1 + class) of `classes` classes by
    (i + j) and `diags` diagonal values: 2 len(offsets) classes + diags different (offset, value) pairs."""
    import scipy.sparse as sp
    parts, val = [], []
    for o in offsets:
        i = np.arange(n - o)
        v = -(1.0 + ((2 * i + o) // 2 % classes) / classes)
        parts += [(i, i + o, v), (i + o, i, v)]
    i = np.arange(n)
    parts.append((i, i, 4.0 * len(offsets) + 1.0 + (i % diags)))
    A = sp.coo_matrix((np.concatenate([p[2] for p in parts]),
                       (np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts]))), shape=(n, n))
    A = A.tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(np.float64)


# pairs: 255 have codes, 256 do not; words of a row: 1, 2 (8 entries at once), 3 (16), 5 (a second round of 16: 19
# entries); rows: 65,536 (full slices), 65,601 (a last slice of one row) and 65,576 (three wavefronts past a last slice
# of 40 rows, whose entries above the diagonal would lead past the vectors)
@pytest.mark.parametrize("n,offsets,classes,diags,coded", [
    (65601, [1], 127, 1, True), (65601, [1], 127, 2, False), (65536, [1, 50, 51], 1, 1, True),
    (65576, [1, 30, 31], 1, 1, True),
    (65601, [1, 50, 51, 700], 2, 3, True), (65601, [1, 2, 3, 50, 51, 52, 900, 901, 902], 3, 1, True)])
# (the FP32 cycle has no Gauss-Seidel)
@pytest.mark.parametrize("smoother,precision", [("jacobi", 0), ("jacobi", 1), ("l1", 0), ("l1", 1), ("cheb", 0),
                                                ("cheb", 1), ("sgs", 0)])
def test_entry_codes_bitexact(lib, libc, monkeypatch, n, offsets, classes, diags, coded, smoother, precision):
    """The kernels over entry codes add the same products in the same order as those over columns and values: the same
    iterations and solution bits with the codes off (HZ_COL16=0).  Where the matrix has them an iteration's product alone
    streams 11 bytes an entry fewer and no row pointers; 16-bit column offsets alone save 2 in each of at most 3 kernels."""
    A = capi.HostCSR(*_banded(n, offsets, classes, diags))
    b = problems.uniform_rhs(n, seed=5)
    kw = dict(tol=1e-8, maxit=30, aggregation=capi.HEM, coarse_dof=500,
              smoother=dict(jacobi=capi.SMOOTHER_JACOBI, l1=capi.SMOOTHER_L1DIAG, cheb=capi.SMOOTHER_CHEBY,
                            sgs=capi.SMOOTHER_SGS)[smoother])
    out = {}
    old = _set_precision(lib, precision)
    try:
        for flag in ("0", "1"):
            monkeypatch.setenv("HZ_COL16", flag)
            x = capi.HostVec(np.zeros(n))
            it, amg = capi.solver_params(lib, **kw)
            libc.srand(1)
            r = lib.linear_solver_dcsr_krylov_amg(A.ptr(), capi.HostVec(b).ptr(), x.ptr(), C.byref(it), C.byref(amg))
            info = capi.hz_solve_info()
            lib.hz_get_last_info(C.byref(info))
            assert r > 0
            out[flag] = (r, x.arr.copy(), info.solve_alg_bytes)
    finally:
        _set_precision(lib, old)
    assert out["0"][0] == out["1"][0]
    assert np.array_equal(out["0"][1], out["1"][1])
    saved = (out["0"][2] - out["1"][2]) / (A.ja.size * out["1"][0])
    assert (saved > 10.5) == coded


# outputs of the generator: below and at a step of 64, a whole chunk of 4,096 and one more; rows: the most the shuffle in
# LDS takes, and one more
@pytest.mark.parametrize("n", [3, 65, 66, 4097, 4098, 19456, 19457])
def test_hec_turn_order_sizes_vs_oracle(lib, orc, libc, n):
    """The aggregates of a chain depend on every position of the turn order: the same as the oracle's, whose order is
    the loop over rand(), and rand() goes on from the same place."""
    A = capi.HostCSR(*_banded(n, [1], 97, 1))
    (lg, _, rg), (lo, _, ro) = _hierarchies(lib, orc, libc, A, capi.HEC, 0.0, coarse_dof=2)
    assert rg == ro and len(lg) == len(lo)
    for g, o in zip(lg, lo):
        if "agg" in o:
            assert np.array_equal(g["agg"], o["agg"])


_ABOVE_LIMIT = """
import ctypes as C, sys
import numpy as np
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from hazmath_amd import capi, problems
from test_gpu_kernel_forms import _banded
from test_gpu_parity import _set_precision
lib = capi.load_library()
o = capi.hz_options()
lib.hz_get_options(C.byref(o))
o.return_on_fatal = 1
lib.hz_set_options(C.byref(o))
n = int(sys.argv[2])
A = capi.HostCSR(*_banded(n, [1], 1, 1))
b = problems.uniform_rhs(n, seed=3)
out = {}
for precision in (0, 1):
    _set_precision(lib, precision)
    x = capi.HostVec(np.zeros(n))
    it, amg = capi.solver_params(lib, tol=1e-8, maxit=60, aggregation=capi.HEM, smoother=capi.SMOOTHER_L1DIAG,
                                 coarse_dof=1000)
    r = lib.linear_solver_dcsr_krylov_amg(A.ptr(), capi.HostVec(b).ptr(), x.ptr(), C.byref(it), C.byref(amg))
    out["r%d" % precision], out["x%d" % precision] = r, x.arr
np.savez(sys.argv[3], **out)
"""


def test_fused_levels_above_their_default_limit(lib, tmp_path):
    """HZ_FUSE_DOWN_MAX puts a chain's first level of 2,100,000 rows in pairs on the fused kernels: C = 120 coarse rows a
    workgroup are 8,750 workgroups, a partial each, more than the n / 256 + 1 = 8,204 of the kernels over slices.  Two
    solutions below 1e-8 of a system of condition 7 / 3 (diagonal 5, off-diagonal entries -1)."""
    import os
    import subprocess
    import sys
    from pathlib import Path
    n = 2_100_000
    assert n // 240 > max(8192, n // 256 + 1)
    root = str(Path(__file__).resolve().parents[1])
    out = {}
    for limit in ("300000", "4000000"):
        f = tmp_path / f"x{limit}.npz"
        r = subprocess.run([sys.executable, "-c", _ABOVE_LIMIT, root, str(n), str(f)], timeout=110, capture_output=True,
                           text=True, env=dict(os.environ, HZ_FUSE_DOWN_MAX=limit))
        assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
        out[limit] = dict(np.load(f))
    for precision in (0, 1):
        a, c = out["300000"], out["4000000"]
        assert a[f"r{precision}"] > 0 and abs(int(a[f"r{precision}"]) - int(c[f"r{precision}"])) <= 1
        xa, xc = a[f"x{precision}"], c[f"x{precision}"]
        assert np.linalg.norm(xa - xc) <= 5e-8 * np.linalg.norm(xa)
