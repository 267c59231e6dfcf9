"""The work that users of this library have it do, as cases that can be timed.

Every case goes through a public entry point of the C ABI (hazmath_amd.capi):

* solve    hz_krylov_amg_device: AMG setup and PCG on arrays already in HBM
* host     linear_solver_dcsr_krylov_amg: the same call on host arrays, upload
           and download included
* learned  hz_krylov_amg_learned: smoothed aggregation with the parameter
           network, host arrays
* batch    hz_batch_krylov_amg_device: many 2-D systems x 8 right-hand sides
* precond  hz_precond_amg_apply_device: one cycle of a preconditioner that the
           program set up once (it runs its own Krylov method around it)
* mlp      hz_mlp_loss_grad: forward and backward pass of the parameter network

The systems are the P1 finite-element ones of hazmath_amd.problems (Poisson,
piecewise-constant coefficients with jumps, rotated anisotropy; the 15-point
Kuhn pattern in 3-D with the structural zeros an assembled matrix holds),
assembled here with torch so that making them is quick.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from hazmath_amd import capi, learned, problems

AGG = {"hem": capi.HEM, "hec": capi.HEC, "vmb": capi.VMB}
SMOOTHER = {"jacobi": capi.SMOOTHER_JACOBI, "l1": capi.SMOOTHER_L1DIAG, "gs": capi.SMOOTHER_GS,
            "sgs": capi.SMOOTHER_SGS, "ssor": capi.SMOOTHER_SSOR, "cheb": capi.SMOOTHER_CHEBY}
BUDGET = 400          # iterations the learned method may take before the plain one is used


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest whole solve: a 2-D system of 16,129 rows from host arrays, HEC pairs and
        # damped Jacobi, as a small application calls the drop-in once a time step
        dict(name="host_2d_hec_jacobi", kind="host", problem="poisson2d", m=128, agg="hec", smoother="jacobi",
             sweeps=1, cycle="v", coarse_dof=100, tol=1e-8),
        # what a program gets that only calls the two param_*_init functions: W-cycle, Gauss-Seidel,
        # HEC, CG on the coarsest level
        dict(name="host_2d_defaults", kind="host", problem="poisson2d", m=101, agg="defaults", smoother="gs",
             sweeps=1, cycle="w", coarse_dof=200, tol=1e-6),
        # the headline: 3-D Kuhn Poisson with 128^3 cells (2,048,383 rows, 30,340,171 stored entries)
        dict(name="poisson3d_128", kind="solve", problem="poisson3d", m=128, agg="hem", smoother="l1", sweeps=1,
             precision=0, coarse_dof=1000, tol=1e-10),
        # an ordinary size that is a multiple of nothing, entries without zeros, long iteration counts
        dict(name="aniso3d_77", kind="solve", problem="aniso3d", m=77, agg="hem", smoother="l1", sweeps=1,
             precision=0, coarse_dof=1000, tol=1e-10, theta=2.529, eps=1e-2),
        # jumping coefficients (8^3 blocks over six decades) with the FP32 cycle under the FP64 PCG
        dict(name="coef3d_128_fp32", kind="solve", problem="coef3d", m=128, agg="hem", smoother="l1", sweeps=1,
             precision=1, coarse_dof=1000, tol=1e-10),
        # a symmetric Gauss-Seidel smoother, the usual choice on CPUs
        dict(name="poisson3d_64_sgs", kind="solve", problem="poisson3d", m=64, agg="hem", smoother="sgs", sweeps=1,
             precision=0, coarse_dof=1000, tol=1e-10),
        # smoothed aggregation with Chebyshev smoothing and constant parameters, FP64
        dict(name="sa_aniso3d_64", kind="solve", problem="aniso3d", m=64, agg="vmb", smoother="cheb", sweeps=2,
             precision=0, coarse_dof=1000, tol=1e-10, theta=0.8, eps=1e-2, sa=True),
        # the learned method on the strongly anisotropic 128^3 problem, from host arrays
        dict(name="learned_aniso3d_128", kind="learned", m=128, theta=2.529, eps=1e-3, sweeps=4, coarse_sweeps=2,
             precision=1, coarse_dof=1000, tol=1e-10),
        # many small systems at once (a parameter study): 48 anisotropic 2-D systems x 8 right-hand sides
        dict(name="batch_48", kind="batch", count=48, side_lo=33, side_hi=257, spec_seed=4, eps_lo=-3.0,
             coarse_dof=200, tol=1e-10),
        # one cycle of a kept preconditioner on a small 2-D system: latency and launches alone
        dict(name="precond_2d_96", kind="precond", problem="poisson2d", m=96, agg="hec", smoother="l1", sweeps=1,
             precision=0, coarse_dof=200),
        # ... and on a 3-D system of ordinary size
        dict(name="precond_3d_80", kind="precond", problem="coef3d", m=80, agg="hem", smoother="l1", sweeps=1,
             precision=0, coarse_dof=1000),
        # one gradient of the parameter network over its whole training set
        dict(name="mlp_grad_84400", kind="mlp", rows=84400),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "solve", "solve", "solve", "gs", "sa", "learned", "batch", "precond", "precond", "mlp",
                       "defaults"])
    theta = round(rng.uniform(0.0, math.pi), 4)
    eps = round(10.0 ** rng.uniform(-3.0, 0.0), 6)
    if kind == "host":
        return dict(kind="host", problem=rng.choice(["poisson2d", "aniso2d"]), m=_log_int(rng, 33, 257),
                    agg=rng.choice(["hec", "hem", "vmb"]), smoother=rng.choice(["jacobi", "l1"]),
                    sweeps=rng.choice([1, 2]), cycle="v", coarse_dof=100, tol=rng.choice([1e-8, 1e-10]), theta=theta,
                    eps=max(eps, 0.05))
    if kind == "defaults":
        return dict(kind="host", problem="poisson2d", m=_log_int(rng, 24, 140), agg="defaults", smoother="gs",
                    sweeps=1, cycle="w", coarse_dof=200, tol=1e-6)
    if kind == "solve":
        return dict(kind="solve", problem=rng.choice(["poisson3d", "coef3d", "aniso3d"]), m=_log_int(rng, 17, 128),
                    agg=rng.choice(["hem", "hem", "hec"]), smoother=rng.choice(["l1", "l1", "jacobi"]),
                    sweeps=rng.choice([1, 1, 2]), precision=rng.choice([0, 0, 1]),
                    coarse_dof=rng.choice([200, 500, 1000]), tol=1e-10, theta=theta, eps=eps)
    if kind == "gs":
        return dict(kind="solve", problem=rng.choice(["poisson3d", "coef3d"]), m=_log_int(rng, 17, 80), agg="hem",
                    smoother=rng.choice(["gs", "sgs", "ssor"]), sweeps=1, precision=0, coarse_dof=1000, tol=1e-10)
    if kind == "sa":
        return dict(kind="solve", problem="aniso3d", m=_log_int(rng, 17, 80), agg="vmb", smoother="cheb",
                    sweeps=rng.choice([2, 3, 4]), precision=rng.choice([0, 1]), coarse_dof=1000, tol=1e-10,
                    theta=theta, eps=min(eps, 0.1), sa=True)
    if kind == "learned":
        return dict(kind="learned", m=_log_int(rng, 24, 110), theta=theta, eps=min(eps, 0.1),
                    sweeps=rng.choice([2, 4]), coarse_sweeps=2, precision=rng.choice([0, 1]), coarse_dof=1000,
                    tol=1e-10)
    if kind == "batch":
        return dict(kind="batch", count=_log_int(rng, 4, 48), side_lo=33, side_hi=rng.choice([129, 257]),
                    spec_seed=rng.randrange(1000), eps_lo=-3.0, coarse_dof=200, tol=1e-10)
    if kind == "precond":
        two_d = rng.random() < 0.5
        return dict(kind="precond", problem="poisson2d" if two_d else rng.choice(["poisson3d", "coef3d", "aniso3d"]),
                    m=_log_int(rng, 33, 257) if two_d else _log_int(rng, 17, 96), agg=rng.choice(["hem", "hec"]),
                    smoother=rng.choice(["l1", "jacobi"]), sweeps=rng.choice([1, 2]), precision=rng.choice([0, 1]),
                    coarse_dof=rng.choice([200, 1000]), theta=theta, eps=eps)
    return dict(kind="mlp", rows=_log_int(rng, 100, 84400))


# ---------------------------------------------------------------------------
# systems
# ---------------------------------------------------------------------------
def _stencil(shape, offsets, values):
    """CSR (int32, int32, float64 on the GPU) of a stencil on the grid `shape` (z, y, x; x fastest), entries
    that leave the grid dropped, columns ascending.  values[k]: a number, or a value per grid point."""
    nz, ny, nx = shape
    n = nz * ny * nx
    dev = torch.device("cuda")
    lin = [(dz * ny + dy) * nx + dx for dz, dy, dx in offsets]
    order = sorted(range(len(offsets)), key=lambda k: lin[k])
    i = torch.arange(n, device=dev)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    col = torch.empty((n, len(offsets)), dtype=torch.int32, device=dev)
    val = torch.empty((n, len(offsets)), dtype=torch.float64, device=dev)
    ok = torch.empty((n, len(offsets)), dtype=torch.bool, device=dev)
    for c, k in enumerate(order):
        dz, dy, dx = offsets[k]
        ok[:, c] = ((x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz))
        col[:, c] = (i + lin[k]).to(torch.int32)
        val[:, c] = values[k]
    ia = torch.zeros(n + 1, dtype=torch.int32, device=dev)
    ia[1:] = torch.cumsum(ok.sum(1), 0).to(torch.int32)
    return ia, col[ok].contiguous(), val[ok].contiguous()


_OFFSETS3 = [(0, 0, 0)] + [tuple(s * a for a in ax) for ax in ((0, 0, 1), (0, 1, 0), (1, 0, 0)) for s in (1, -1)] + \
            [tuple(s * a for a in d) for d in problems.KUHN_DIAGONALS for s in (1, -1)]
_OFFSETS2 = [(0, 0, 0), (0, 0, 1), (0, 0, -1), (0, 1, 0), (0, -1, 0), (0, 1, 1), (0, -1, -1)]


def _cell_values(cell, offsets, weight, dim):
    """Stencil values assembled from the cell matrix `cell`, each cell weighted: weight(cz, cy, cx) is a number or
    an array over the grid points for the cell in which the point is the corner (cz, cy, cx)."""
    out = []
    for dz, dy, dx in offsets:
        v = 0.0
        for c in range(2 ** dim):
            cx, cy, cz = c & 1, (c >> 1) & 1, (c >> 2) & 1
            ex, ey, ez = cx + dx, cy + dy, cz + dz
            if min(ex, ey, ez) < 0 or max(ex, ey, ez) > 1 or (dim == 2 and ez):
                continue
            k = float(cell[c, ex + 2 * ey + 4 * ez])
            if k != 0.0:
                v = v + k * weight(cz, cy, cx)
        out.append(v)
    return out


def _system(case, seed):
    kind, m = case["problem"], case["m"]
    k = m - 1
    if kind == "poisson2d":
        return _stencil((1, k, k), _OFFSETS2[:5], [4.0, -1.0, -1.0, -1.0, -1.0])
    if kind == "aniso2d":
        cell = problems._p1_cell_matrix(2, problems.anisotropic_tensor(2, case["theta"], case["eps"]))
        return _stencil((1, k, k), _OFFSETS2, _cell_values(cell, _OFFSETS2, lambda *_: 1.0, 2))
    if kind == "aniso3d":
        cell = problems._p1_cell_matrix(3, problems.anisotropic_tensor(3, case["theta"], case["eps"]))
        return _stencil((k, k, k), _OFFSETS3, _cell_values(cell, _OFFSETS3, lambda *_: 1.0 / m, 3))
    if kind == "poisson3d":
        return _stencil((k, k, k), _OFFSETS3, [6.0 / m] + [-1.0 / m] * 6 + [0.0] * 8)
    # coef3d: the coefficients come with the inputs
    kappa = torch.from_numpy(problems.block_coefficients(8, seed)).cuda()
    cb = (torch.arange(m, device="cuda") * 8) // m
    kc = kappa[cb][:, cb][:, :, cb]
    vals = _cell_values(problems.KUHN_CUBE_K6, _OFFSETS3,
                        lambda cz, cy, cx: (1.0 / (6 * m)) * kc[1 - cz:m - cz, 1 - cy:m - cy, 1 - cx:m - cx].reshape(-1),
                        3)
    return _stencil((k, k, k), _OFFSETS3, vals)


def _rhs(n, seed, cols=None):
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)
    shape = (n,) if cols is None else (n, cols)
    return 2.0 * torch.rand(shape, dtype=torch.float64, device="cuda", generator=g) - 1.0


def _batch_system(case):
    """The systems stacked into one block-diagonal CSR, and their row offsets."""
    specs = problems.batch_anisotropic_2d(case["count"], case["spec_seed"], (case["side_lo"], case["side_hi"]))
    off, nnz, ias, jas, vas = [0], 0, [], [], []
    for d in specs:
        eps = d["eps"] ** (-case["eps_lo"] / 4.0)      # 10^U[eps_lo, 0]
        ia, ja, va = _system(dict(problem="aniso2d", m=d["side"] - 1, theta=d["theta"], eps=eps), 0)
        ias.append(ia[:-1] + nnz)
        jas.append(ja + off[-1])
        vas.append(va)
        nnz += int(ja.numel())
        off.append(off[-1] + ia.numel() - 1)
    ias.append(torch.tensor([nnz], dtype=torch.int32, device="cuda"))
    return torch.cat(ias), torch.cat(jas), torch.cat(vas), off


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
_LIBC = C.CDLL(None)


def _set_options(lib, case):
    """The options that AMG_param does not hold (process-wide, so each call states them)."""
    o = capi.hz_options()
    lib.hz_get_options(C.byref(o))
    o.jacobi_weight = 2.0 / 3.0 if case.get("smoother") == "jacobi" else 1.0
    o.vcycle_precision = case.get("precision", 0)
    o.cheb_coarse_steps = case.get("coarse_sweeps", 0)
    o.return_on_fatal = 1
    lib.hz_set_options(C.byref(o))


def _params(lib, case):
    if case.get("agg") == "defaults":
        it, amg = capi.default_itsolver_param(lib), capi.default_amg_param(lib)
        it.linear_itsolver_type = capi.SOLVER_CG
        it.linear_precond_type = capi.PREC_AMG
        it.linear_tol = case["tol"]
        return it, amg
    it, amg = capi.solver_params(lib, tol=case.get("tol", 1e-10), maxit=2000, aggregation=AGG[case.get("agg", "hem")],
                                 smoother=SMOOTHER[case.get("smoother", "l1")], coarse_dof=case["coarse_dof"],
                                 coarse_solver=capi.SOLVER_UMFPACK, max_levels=20, theta=0.04)
    amg.presmooth_iter = amg.postsmooth_iter = case.get("sweeps", 1)
    if case.get("sa"):
        amg.AMG_type = capi.SA_AMG
    return it, amg


class _Precond:
    """A preconditioner object and its release."""

    def __init__(self, lib, A, amg):
        self.lib, self.pc = lib, lib.create_precond_amg(A.ptr(), C.byref(amg))
        if not self.pc:
            raise RuntimeError("create_precond_amg failed")
        self.data = self.pc.contents.data

    def __del__(self):
        if self.pc:
            self.lib.hz_precond_free(self.pc)
            self.pc = None


def prepare(case, seed):
    lib = capi.load_library()
    if lib.hz_device_count() < 1:
        raise RuntimeError("no HIP device")
    kind = case["kind"]
    st = dict(case=case, lib=lib, seed=seed)
    if kind == "mlp":
        rng = np.random.default_rng(seed)
        st["theta"] = learned.load_model()
        st["x"] = rng.random((case["rows"], capi.MLP_INPUTS), dtype=np.float32)
        st["t"] = (0.3 + rng.random((case["rows"], capi.MLP_OUTPUTS), dtype=np.float32)).astype(np.float32)
        st["grad"] = np.zeros(capi.MLP_PARAMS, np.float32)
        st["loss"] = np.zeros(1, np.float32)
        return st
    if kind == "batch":
        ia, ja, va, off = _batch_system(case)
        st.update(ia=ia, ja=ja, va=va, off=(capi.INT * len(off))(*off), b=_rhs(off[-1], seed, capi.BATCH_RHS),
                  iters=np.zeros(case["count"] * capi.BATCH_RHS, np.int32))
        st["x"] = torch.zeros_like(st["b"])
    else:
        sysc = dict(case, problem="aniso3d") if kind == "learned" else case
        ia, ja, va = _system(sysc, seed)
        b = _rhs(ia.numel() - 1, seed)
        if kind == "solve":
            st.update(ia=ia, ja=ja, va=va, b=b, x=torch.zeros_like(b))
        else:
            st["A"] = capi.HostCSR(ia.cpu().numpy(), ja.cpu().numpy(), va.cpu().numpy())
            if kind == "precond":
                _set_options(lib, case)
                _LIBC.srand(1 + seed)
                st["pc"] = _Precond(lib, st["A"], _params(lib, case)[1])
                st.update(r=b, z=torch.empty_like(b))
            else:
                st["b"] = capi.HostVec(b.cpu().numpy())
                st["x"] = capi.HostVec(np.zeros(b.numel()))
                if kind == "learned":
                    st["theta"] = learned.load_model()
    torch.cuda.synchronize()
    return st


def run(st):
    case, lib, kind = st["case"], st["lib"], st["case"]["kind"]
    if kind == "mlp":
        r = lib.hz_mlp_loss_grad(capi.fptr(st["theta"]), capi.fptr(st["x"]), capi.fptr(st["t"]), case["rows"],
                                 capi.fptr(st["grad"]), capi.fptr(st["loss"]))
        if r != 0:
            raise RuntimeError(f"hz_mlp_loss_grad returned {r}")
        return [st["grad"], st["loss"]]
    if kind == "precond":
        lib.hz_precond_amg_apply_device(st["r"].data_ptr(), st["z"].data_ptr(), st["pc"].data)
        return st["z"]
    _set_options(lib, case)
    _LIBC.srand(1 + st["seed"])       # HEC draws its turn order from the C library's rand()
    it, amg = _params(lib, case)
    if kind in ("solve", "batch"):
        # the library works on its own stream: a caller waits for the initial guess it has queued
        x = st["x"].zero_()
        torch.cuda.current_stream().synchronize()
        if kind == "solve":
            r = lib.hz_krylov_amg_device(x.numel(), st["ja"].numel(), st["ia"].data_ptr(), st["ja"].data_ptr(),
                                         st["va"].data_ptr(), st["b"].data_ptr(), x.data_ptr(), C.byref(it),
                                         C.byref(amg))
        else:
            r = lib.hz_batch_krylov_amg_device(case["count"], st["off"], st["ja"].numel(), st["ia"].data_ptr(),
                                               st["ja"].data_ptr(), st["va"].data_ptr(), st["b"].data_ptr(),
                                               x.data_ptr(), C.byref(it), C.byref(amg),
                                               capi.dptr(st["iters"], capi.INT))
            r = min(int(r), int(st["iters"].min()))
        out = x
    else:
        st["x"].arr[:] = 0.0
        if kind == "host":
            r = lib.linear_solver_dcsr_krylov_amg(st["A"].ptr(), st["b"].ptr(), st["x"].ptr(), C.byref(it),
                                                  C.byref(amg))
        else:
            r = lib.hz_krylov_amg_learned(st["A"].ptr(), st["b"].ptr(), st["x"].ptr(), C.byref(it), C.byref(amg),
                                          capi.fptr(st["theta"]), BUDGET, case["sweeps"])
        out = st["x"].arr
    if r < 0:
        raise RuntimeError(f"{kind} returned {r}")
    return out


# ---------------------------------------------------------------------------
# work, tolerance, exact results
# ---------------------------------------------------------------------------
def _rows_nnz(case):
    kind = case["kind"]
    if kind == "batch":
        specs = problems.batch_anisotropic_2d(case["count"], case["spec_seed"], (case["side_lo"], case["side_hi"]))
        ks = [d["side"] - 2 for d in specs]
        return sum(k * k for k in ks), sum(k * k + 4 * k * (k - 1) + 2 * (k - 1) ** 2 for k in ks)
    k = case["m"] - 1
    if case.get("problem") == "poisson2d":
        return k * k, k * k + 4 * k * (k - 1)
    if case.get("problem") == "aniso2d":
        return k * k, k * k + 4 * k * (k - 1) + 2 * (k - 1) ** 2
    return k ** 3, k ** 3 + 6 * k * k * (k - 1) + 6 * k * (k - 1) ** 2 + 2 * (k - 1) ** 3


def work(case):
    """The inputs read once, the outputs written once, and one product with the matrix (one forward and backward
    pass of the network)."""
    if case["kind"] == "mlp":
        B = case["rows"]
        mac = 12 * 64 + 64 * 64 + 64 * 2
        return {"bytes": 4 * (B * 14 + 2 * capi.MLP_PARAMS + 1), "flops": 2 * B * (3 * mac - 12 * 64)}
    n, nnz = _rows_nnz(case)
    cols = capi.BATCH_RHS if case["kind"] == "batch" else 1
    vectors = 2 if case["kind"] == "precond" else 3      # b (r), x in, x out (z)
    return {"bytes": 12 * nnz + 4 * (n + 1) + 8 * vectors * n * cols, "flops": 2 * nnz * cols}


def tolerance(case):
    """A solve stops at the first iterate whose residual is below tol, and the order of the sums moves that by an
    iteration at most: two solutions differ by what each is off by (measured against exact(): up to 5 tol on the listed
    and drawn systems)."""
    if case["kind"] == "mlp":
        return {"rel": 1e-5}
    if case["kind"] == "precond":
        return {"rel": 2e-5} if case.get("precision") else {"rel": 1e-12}
    return {"rel": 40.0 * case["tol"]}


def _cg(ia, ja, va, b, groups=None, tol=1e-14, maxit=6000):
    """Conjugate gradients in FP64 with the diagonal as preconditioner, columns of b solved together; groups: the
    row's system, each (system, column) with its own step lengths.  Runs on to the level of rounding."""
    n = b.shape[0]
    dev = b.device
    cnt = (ia[1:] - ia[:-1]).long()
    K = int(cnt.max())
    row = torch.repeat_interleave(torch.arange(n, device=dev), cnt)
    pos = torch.arange(ja.numel(), device=dev) - ia[:-1].long()[row]
    col = torch.zeros((n, K), dtype=torch.int32, device=dev)
    val = torch.zeros((n, K), dtype=torch.float64, device=dev)
    col[row, pos] = ja
    val[row, pos] = va
    dinv = 1.0 / (val * (col == torch.arange(n, device=dev)[:, None])).sum(1)
    if b.dim() > 1:
        dinv = dinv[:, None]
    ns = 1 if groups is None else int(groups.max()) + 1
    shape = (ns,) + tuple(b.shape[1:])

    def mv(p):
        y = torch.zeros_like(p)
        for k in range(K):
            v = val[:, k] if p.dim() == 1 else val[:, k, None]
            y += v * p[col[:, k]]
        return y

    if groups is not None:
        # sums per system: chunks of 1024 of its rows, then over its chunks (row n is a row of zeros)
        sizes = torch.bincount(groups, minlength=ns).tolist()
        idx, owner, o = [], [], 0
        for g, size in enumerate(sizes):
            c = -(-size // 1024)
            j = torch.arange(c * 1024, device=dev)
            idx.append(torch.where(j < size, j + o, n).reshape(c, 1024))
            owner += [g] * c
            o += size
        idx, owner = torch.cat(idx), torch.tensor(owner, device=dev)

    def dot(p, q):
        if groups is None:
            return (p * q).sum(0, keepdim=True)
        pq = torch.cat([p * q, torch.zeros_like(p[:1])])
        return torch.zeros(shape, dtype=torch.float64, device=dev).index_add_(0, owner, pq[idx].sum(1))

    def spread(s):
        return s if groups is None else s[groups]

    x = torch.zeros_like(b)
    r = b.clone()
    z = dinv * r
    p = z.clone()
    rz = dot(r, z)
    stop = (tol ** 2) * dot(b, b)
    for k in range(maxit):
        t = mv(p)
        a = rz / dot(p, t).clamp_min(1e-300)
        x += spread(a) * p
        r -= spread(a) * t
        z = dinv * r
        new = dot(r, z)
        p = z + spread(new / rz.clamp_min(1e-300)) * p
        rz = new
        if k % 50 == 49 and bool((dot(r, r) <= stop).all()):
            break
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        st = prepare(case, seed)
        th = torch.from_numpy(st["theta"]).double().cuda()
        sizes = [(16, 64), (64, 64), (64, 16)]
        parts, o = [], 0
        for i, j in sizes:
            parts += [th[o:o + i * j].reshape(i, j).clone().requires_grad_(),
                      th[o + i * j:o + i * j + j].clone().requires_grad_()]
            o += i * j + j
        x = torch.nn.functional.pad(torch.from_numpy(st["x"]).double().cuda(), (0, 4))
        h = torch.nn.functional.gelu(x @ parts[0] + parts[1])
        h = torch.nn.functional.gelu(h @ parts[2] + parts[3])
        y = (h @ parts[4] + parts[5])[:, :2]
        loss = ((y - torch.from_numpy(st["t"]).double().cuda()) ** 2).mean()
        grads = torch.autograd.grad(loss, parts)
        return [torch.cat([g.reshape(-1) for g in grads]).cpu().numpy(), loss.detach().reshape(1).cpu().numpy()]
    if kind == "precond":
        return None                  # one cycle is defined by the hierarchy, which plain torch does not have
    if kind == "batch":
        ia, ja, va, off = _batch_system(case)
        sizes = torch.tensor([off[i + 1] - off[i] for i in range(case["count"])], device="cuda")
        groups = torch.repeat_interleave(torch.arange(case["count"], device="cuda"), sizes)
        return _cg(ia, ja, va, _rhs(off[-1], seed, capi.BATCH_RHS), groups)
    sysc = dict(case, problem="aniso3d") if kind == "learned" else case
    ia, ja, va = _system(sysc, seed)
    x = _cg(ia, ja, va, _rhs(ia.numel() - 1, seed))
    return x if kind == "solve" else x.cpu().numpy()
