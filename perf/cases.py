"""Timing cases: the work a frequency-domain modelling or inversion program has this library do.

Grids run from 61 x 41 to 1601 x 401 cells with the PML, batches from one right-hand side to
8 frequencies x 200 shots, in FP64 and in FP32 with FP64 refinement, forward (M) and adjoint
(M, M^H, M^T).  The kinds of case:

* solve: the panel solves alone, on factors a program keeps;
* dropin: the UMFPACK entry points as an unmodified host code calls them, host arrays in and out;
* forward: fdfd.forward_shots, with factor storage of its own or in a kept Workspace;
* gradient: fdfd.grad_obj, one FWI gradient (forward and adjoint panels, residuals, shot sums);
* step: model to wavefields for a batch of frequencies through the batched entry points.

The matrices of solve and dropin are built here in double, so `exact` can solve the same systems
in 64 bits by block elimination; the other kinds' matrices are defined by the single-precision
rounding of the assembled coefficients and have no plain 64-bit value.
"""
import ctypes
import math

import numpy as np
import torch

import germaine_amd as G
from germaine_amd import fdfd, models

PRECISION = {"fp64": G.FP64, "fp32": G.FP32}
PHYSICS = {"ac": G.AC, "sh": G.SH, "te": G.TE}
TOL = 1e-10


def listed():
    return [
        # one shot on the smallest grid in use: launches and latency alone
        dict(name="solve_61x41_1shot", kind="solve", nx=61, ny=41, nfreq=1, nrhs=1, prec="fp64", sys=0, refine=False),
        # one shot on the large grid: every factor entry is read for one vector
        dict(name="solve_1601x401_1shot", kind="solve", nx=1601, ny=401, nfreq=1, nrhs=1, prec="fp64", sys=0,
             refine=False),
        # the two-inclusion example's grid (250 x 125 and a 10-cell PML): a program linked against the
        # UMFPACK names factors one frequency and solves shot after shot with default refinement
        dict(name="dropin_270x145_8shots", kind="dropin", nx=270, ny=145, nrhs=8, sys=0),
        # a marine line's forward panels on kept FP64 factors, all frequencies in one call
        dict(name="solve_801x187_4f_100shots", kind="solve", nx=801, ny=187, nfreq=4, nrhs=100, prec="fp64", sys=0,
             refine=False),
        # the adjoint panels of an inversion on kept FP32 factors, refined to the FP64 residual
        dict(name="adjoint_801x201_4f_80shots_fp32", kind="solve", nx=801, ny=201, nfreq=4, nrhs=80, prec="fp32",
             sys=2, refine=True),
        # the two-inclusion example's 264 shots of one frequency, storage made for the call
        dict(name="forward_270x145_264shots", kind="forward", phys="ac", nx=270, ny=145, nfreq=1, nrhs=264,
             nrec=264, prec="fp64", ws=False),
        # the 201 x 101 example in a loop that keeps its storage: small launches, all phases
        dict(name="forward_201x101_10shots", kind="forward", phys="ac", nx=201, ny=101, nfreq=1, nrhs=10, nrec=100,
             prec="fp64", ws=True),
        # shear waves, an odd-sized grid and a ragged panel, FP32 with refinement
        dict(name="forward_sh_503x333_3f_37shots_fp32", kind="forward", phys="sh", nx=503, ny=333, nfreq=3, nrhs=37,
             nrec=121, prec="fp32", ws=True),
        # one acoustic FWI gradient on the inversion workload
        dict(name="gradient_ac_801x201_4f_80shots", kind="gradient", phys="ac", nx=801, ny=201, nfreq=4, nrhs=80,
             nrec=320, ws=True),
        # one radar gradient (adjoint with M^T, two materials), odd sizes
        dict(name="gradient_te_403x207_2f_31shots", kind="gradient", phys="te", nx=403, ny=207, nfreq=2, nrhs=31,
             nrec=125, ws=True),
        # model to wavefields for 8 frequencies x 200 shots, the benchmark's step
        dict(name="step_1601x401_8f_200shots_fp32", kind="step", phys="ac", nx=1601, ny=401, nfreq=8, nrhs=200,
             prec="fp32"),
        # the same with FP64 factors and no refinement, half the frequencies
        dict(name="step_1601x401_4f_200shots_fp64", kind="step", phys="ac", nx=1601, ny=401, nfreq=4, nrhs=200,
             prec="fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "dropin", "forward", "gradient", "step"])
    most = 642001 * 800                       # unknowns x right-hand sides of the FP64 step
    while True:
        nx, ny = _log_int(rng, 61, 1601), _log_int(rng, 41, 401)
        nfreq, nrhs = rng.randint(1, 8), _log_int(rng, 1, 200)
        if kind == "dropin":
            nfreq, nrhs = 1, rng.randint(1, 12)
            if nx * ny > 170000:
                continue
        if nx * ny * nfreq * nrhs <= most and nx * ny * nfreq <= 642001 * 4:
            break
    prec = rng.choice(["fp64", "fp64", "fp32"])
    c = dict(kind=kind, nx=nx, ny=ny)
    if kind == "solve":
        c.update(nfreq=nfreq, nrhs=nrhs, prec=prec, sys=rng.choice([0, 0, 1, 2]), refine=prec == "fp32")
    elif kind == "dropin":
        c.update(nrhs=nrhs, sys=rng.choice([0, 0, 2]))
    elif kind == "forward":
        c.update(phys=rng.choice(["ac", "ac", "sh", "te"]), nfreq=nfreq, nrhs=nrhs, nrec=_log_int(rng, 10, 400),
                 prec=prec, ws=rng.choice([True, True, False]))
    elif kind == "gradient":
        c.update(phys=rng.choice(["ac", "ac", "te"]), nfreq=min(nfreq, 4), nrhs=nrhs, nrec=_log_int(rng, 10, 400),
                 ws=True)
    elif kind == "step":
        c.update(phys="ac", nfreq=nfreq, nrhs=nrhs, prec=prec)
    return c


# ---- models and matrices ---------------------------------------------------------

def _seed(case, seed, salt=0):
    return [int(seed), case["nx"], case["ny"], salt]


def _npml(case):
    return 10 if min(case["nx"], case["ny"]) < 150 else 20


def _model(case, seed, smooth=False):
    """(m1, m2) float32 [ny, nx]: layers with faults, and for radar layers with ellipses."""
    npml = _npml(case)
    nxi, nyi = case["nx"] - 2 * npml, case["ny"] - 2 * npml
    rng_seed = int(np.random.default_rng(_seed(case, seed)).integers(1 << 31))
    if case.get("phys") == "te":
        a, b = models.te_interior(nxi, nyi, rng_seed)
    else:
        layers = max(2, min(12, nyi // 8))
        a, b = models.layered_fault_interior(nxi, nyi, rng_seed, n_layers=layers)
        if case.get("phys") == "sh":
            a = (a / np.float32(1.8)).astype(np.float32)
    if smooth:
        a = models.gaussian_smooth(a, 4.0)
        b = models.gaussian_smooth(b, 4.0)
    return models.extend_pml(a, npml), models.extend_pml(b, npml)


def _spacing(case):
    return 0.04 if case["phys"] == "te" else 12.5


def _freqs(case):
    nf = case["nfreq"]
    return [1e8 * (k + 1) / (2 if nf > 4 else 1) for k in range(nf)] if case["phys"] == "te" else \
        [2.0 * (k + 1) for k in range(nf)]


def _row(case, count, row=2):
    return models.acquisition_row(case["nx"], _npml(case), _spacing(case), row, count)


def _stencil(nx, ny, freq, rng):
    """The nine diagonals of a 9-point Helmholtz operator with an absorbing frame:
    {(dj, di): [ny, nx] complex128}, row (j, i), column (j + dj, i + di)."""
    jj, ii = np.mgrid[0:ny, 0:nx]
    a, b = rng.uniform(0.0, 2 * np.pi, 2)
    v = 2000.0 + 3500.0 * jj / ny + 400.0 * np.sin(2 * np.pi * (ii / 97.0 + a)) * np.cos(2 * np.pi * jj / 61.0 + b)
    v += rng.uniform(-50.0, 50.0, (ny, nx))
    k2 = (2.0 * np.pi * freq * 12.5 / v) ** 2

    def stretch(m):
        x = np.arange(2 * m + 1) / 2.0 - 0.5                     # whole and half points
        d = np.maximum(0.0, np.maximum(10 - x, x - (m - 1 - 10)) / 10.0)
        s = 1.0 - 3.0j * d * d
        return s[1::2], s[0::2]

    sx, sxh = stretch(nx)
    sy, syh = stretch(ny)
    e, w = sy[:, None] / sxh[None, 1:], sy[:, None] / sxh[None, :-1]
    s, n = sx[None, :] / syh[1:, None], sx[None, :] / syh[:-1, None]
    c = 0.55
    D = {(0, 1): c * e, (0, -1): c * w, (1, 0): c * s, (-1, 0): c * n}
    for dj, y in ((1, s), (-1, n)):
        for di, x in ((1, e), (-1, w)):
            D[dj, di] = 0.25 * (1.0 - c) * (x + y)
    D[0, 0] = -sum(D.values())
    for off in D:
        weight = 0.62 if off == (0, 0) else 0.0938 if 0 in off else 0.0012
        rolled = k2[np.clip(jj + off[0], 0, ny - 1), np.clip(ii + off[1], 0, nx - 1)]
        D[off] = D[off] + weight * rolled * sy[:, None] * sx[None, :]
    return D


def _csc(D, nx, ny):
    """Values in canonical CSC order of the 9-point pattern."""
    vals = np.zeros((ny, nx, 9), np.complex128)
    have = np.zeros((ny, nx, 9), bool)
    for k in range(9):
        a, b = k // 3 - 1, k % 3 - 1                              # row of the entry relative to its column
        j = slice(max(0, -a), ny - max(0, a))
        i = slice(max(0, -b), nx - max(0, b))
        jr = slice(max(0, a), ny + min(0, a))
        ir = slice(max(0, b), nx + min(0, b))
        vals[j, i, k] = D[-a, -b][jr, ir]
        have[j, i, k] = True
    return vals[have]


def _systems(case, seed):
    rng = np.random.default_rng(_seed(case, seed))
    return [_stencil(case["nx"], case["ny"], 4.0 + 1.5 * f, rng) for f in range(case.get("nfreq", 1))]


def _sources(case, seed):
    """[nfreq, nrhs, n] complex128 on the GPU: point sources for forward systems, weighted
    receivers along a row for adjoint ones."""
    rng = np.random.default_rng(_seed(case, seed, 1))
    nx, ny, nf, nr = case["nx"], case["ny"], case.get("nfreq", 1), case["nrhs"]
    B = np.zeros((nf, nr, nx if case["sys"] else 1), np.complex128)
    B[:] = rng.standard_normal(B.shape) + 1j * rng.standard_normal(B.shape)
    at = rng.integers(0, nx, (nf, nr))
    return B, at, min(11, ny // 4) * nx


def _panel(case, seed, device):
    B, at, row = _sources(case, seed)
    nf, nr, width = B.shape
    P = torch.zeros((nf, nr, case["nx"] * case["ny"]), dtype=torch.complex128, device=device)
    B = torch.as_tensor(B, device=device)
    if width > 1:
        P[:, :, row:row + width] = B
    else:
        P.scatter_(2, torch.as_tensor(at, device=device)[:, :, None] + row, B)
    return P


# ---- prepare ---------------------------------------------------------------------

def _prepare_solve(case, seed):
    plan = fdfd.Plan(case["nx"], case["ny"])
    vals = torch.as_tensor(np.stack([_csc(D, case["nx"], case["ny"]) for D in _systems(case, seed)]), device="cuda")
    F = plan.factor(vals, PRECISION[case["prec"]])
    B = _panel(case, seed, "cuda")
    return dict(F=F, B=B, X=torch.empty_like(B), freqs=list(range(case["nfreq"])))


class _Symbolic:
    """The analysis object a host program keeps for one grid."""

    def __init__(self, n, Ap, Ai):
        self.h = ctypes.c_void_p()
        G.check(G.lib().umfpack_zi_symbolic(n, n, Ap.ctypes.data, Ai.ctypes.data, None, None, ctypes.byref(self.h),
                                            None, None), "umfpack_zi_symbolic")

    def __del__(self):
        G.lib().umfpack_zi_free_symbolic(ctypes.byref(self.h))


def _prepare_dropin(case, seed):
    Ap, Ai = fdfd.Plan(case["nx"], case["ny"]).pattern()
    vals = _csc(_systems(case, seed)[0], case["nx"], case["ny"])
    B = _panel(case, seed, "cpu")[0].numpy()
    return dict(Ap=Ap, Ai=Ai, Ax=vals.real.copy(), Az=vals.imag.copy(), Bx=B.real.copy(), Bz=B.imag.copy(),
                Xx=np.empty(B.shape), Xz=np.empty(B.shape), S=_Symbolic(case["nx"] * case["ny"], Ap, Ai),
                sys=case["sys"])


def _prepare_path(case, seed):
    plan = fdfd.Plan(case["nx"], case["ny"])
    phys, freqs = PHYSICS[case["phys"]], _freqs(case)
    prec = PRECISION[case.get("prec", "fp64")]
    m1, m2 = (torch.as_tensor(m, device="cuda") for m in _model(case, seed, smooth=case["kind"] == "gradient"))
    st = dict(plan=plan, phys=phys, dh=_spacing(case), freqs=freqs, m1=m1, m2=m2, npml=_npml(case), prec=prec,
              src=_row(case, case["nrhs"]))
    if "nrec" in case:
        st["rec"] = _row(case, case["nrec"], row=3)
    if case["kind"] == "step":
        n, nf, ns = plan.n, len(freqs), case["nrhs"]
        st["vals"] = torch.empty((nf, plan.nnz), dtype=torch.complex128, device="cuda")
        plan.assemble(phys, st["dh"], freqs, m1, m2, npml=st["npml"], out=st["vals"])
        st["F"] = plan.factor(st["vals"], prec)
        st["k"] = torch.as_tensor(np.asarray(st["src"], np.int32), device="cuda")
        st["B"] = torch.empty((nf, ns, n), dtype=torch.complex128, device="cuda")
        st["X"] = torch.empty((nf, ns, n), dtype=torch.complex128, device="cuda")
        return st
    if case["kind"] == "gradient":
        t1, t2 = (torch.as_tensor(m, device="cuda") for m in _model(case, seed))
        st["pobs"] = fdfd.forward_shots(plan, phys, st["dh"], freqs, t1, t2, st["src"], st["rec"], npml=st["npml"],
                                        tol=None)["data"]
    st["ws"] = fdfd.Workspace(plan, len(freqs), prec) if case["ws"] else None
    return st


def prepare(case, seed):
    if case["kind"] == "solve":
        return dict(_prepare_solve(case, seed), case=case)
    if case["kind"] == "dropin":
        return dict(_prepare_dropin(case, seed), case=case)
    return dict(_prepare_path(case, seed), case=case)


# ---- run -------------------------------------------------------------------------

def _run_solve(st):
    c, F, B, X = st["case"], st["F"], st["B"], st["X"]
    if c["nfreq"] == 1:
        if c["refine"]:
            return F.solve_refine(0, B[0], sys=c["sys"], tol=TOL, out=X[0])[0]
        return F.solve(0, B[0], sys=c["sys"], out=X[0])
    if c["refine"]:
        return F.solve_refine_batch(st["freqs"], B, sys=c["sys"], tol=TOL, out=X)[0]
    return F.solve_batch(st["freqs"], B, sys=c["sys"], out=X)


def _run_dropin(st):
    L, num = G.lib(), ctypes.c_void_p()
    A = [st[k].ctypes.data for k in ("Ap", "Ai", "Ax", "Az")]
    G.check(L.umfpack_zi_numeric(*A, st["S"].h, ctypes.byref(num), None, None), "umfpack_zi_numeric")
    for s in range(len(st["Bx"])):
        G.check(L.umfpack_zi_solve(st["sys"], *A, st["Xx"][s].ctypes.data, st["Xz"][s].ctypes.data,
                                   st["Bx"][s].ctypes.data, st["Bz"][s].ctypes.data, num, None, None),
                "umfpack_zi_solve")
    L.umfpack_zi_free_numeric(ctypes.byref(num))
    return st["Xx"], st["Xz"]


def _run_step(st):
    plan, F, B, X = st["plan"], st["F"], st["B"], st["X"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    vals = plan.assemble(st["phys"], st["dh"], st["freqs"], st["m1"], st["m2"], npml=st["npml"], out=st["vals"])
    F.refactor_graph(vals)
    for f, fr in enumerate(st["freqs"]):
        amp = fdfd.source_amp(st["phys"], fr, 0.0, st["dh"])
        G.check(G.lib().gfdfd_spike_panel(plan.n, B.shape[1], ctypes.c_void_p(st["k"].data_ptr()), amp.real, amp.imag,
                                          ctypes.c_void_p(B[f].data_ptr()), stream), "gfdfd_spike_panel")
    sel = list(range(len(st["freqs"])))
    if st["prec"] == G.FP32:
        return F.solve_refine_batch(sel, B, tol=TOL, max_iter=20, out=X)[0]
    return F.solve_batch(sel, B, out=X)


def run(st):
    kind = st["case"]["kind"]
    if kind == "solve":
        return _run_solve(st)
    if kind == "dropin":
        return _run_dropin(st)
    if kind == "step":
        return _run_step(st)
    path = (st["plan"], st["phys"], st["dh"], st["freqs"], st["m1"], st["m2"], st["src"], st["rec"])
    if kind == "forward":
        return fdfd.forward_shots(*path, npml=st["npml"], precision=st["prec"], ws=st["ws"])["data"]
    return fdfd.grad_obj(*path, st["pobs"], npml=st["npml"], ws=st["ws"])


# ---- work and exact values -------------------------------------------------------

def work(case):
    n = case["nx"] * case["ny"]
    info = fdfd.Plan(case["nx"], case["ny"]).info
    nf, nr = case.get("nfreq", 1), case["nrhs"]
    es = 8 if case.get("prec") == "fp32" else 16
    lu, panel = es * info.nnz_lu * nf, 16.0 * n * nr * nf
    solve = 8.0 * info.nnz_lu * nr * nf
    if case["kind"] == "solve":                  # factors and right-hand sides in, solutions out
        return {"bytes": lu + 2 * panel, "flops": solve}
    values, factor = 16.0 * info.nnz * nf, info.factor_flops * nf
    if case["kind"] == "dropin":
        return {"bytes": values + 2 * lu + 2 * panel, "flops": factor + solve}
    model = 8.0 * n
    if case["kind"] == "step":                   # model in, solutions out
        return {"bytes": model + 2 * lu + panel, "flops": factor + solve}
    if case["kind"] == "forward":                # model in, receiver samples out
        return {"bytes": model + 2 * lu + 8.0 * nr * case["nrec"] * nf, "flops": factor + solve}
    # two sweeps of the factors, both panels read once by the shot sums
    return {"bytes": model + 3 * lu + 2 * panel, "flops": factor + 2 * solve}


def _block_solve(D, sys, B):
    """x of op(M) x = B [nrhs, ny, nx] by block elimination along the longer side, in 64 bits."""
    if sys:
        ny, nx = D[0, 0].shape
        T = {}
        for (dj, di) in D:
            A = np.zeros((ny, nx), np.complex128)
            j, i = slice(max(0, -dj), ny - max(0, dj)), slice(max(0, -di), nx - max(0, di))
            A[j, i] = D[-dj, -di][max(0, dj):ny + min(0, dj), max(0, di):nx + min(0, di)]
            T[dj, di] = A.conj() if sys == 1 else A
        D = T
    swap = D[0, 0].shape[1] > D[0, 0].shape[0]
    E = {((d[1], d[0]) if swap else d): (A.T if swap else A) for d, A in D.items()}
    B = B.transpose(2, 1, 0) if swap else B.transpose(1, 2, 0)       # [block, point, rhs]
    nb, w, _ = B.shape
    rows = np.arange(w)

    def band(t, dt):
        A = np.zeros((w, w), np.complex128)
        A[rows, rows] = E[dt, 0][t]
        A[rows[1:], rows[:-1]] = E[dt, -1][t, 1:]
        A[rows[:-1], rows[1:]] = E[dt, 1][t, :-1]
        return A

    def times(t, dt, X):                                              # band(t, dt) @ X
        Y = E[dt, 0][t][:, None] * X
        Y[1:] += E[dt, -1][t, 1:, None] * X[:-1]
        Y[:-1] += E[dt, 1][t, :-1, None] * X[1:]
        return Y

    H, Z = [], []
    for t in range(nb):
        S, y = band(t, 0), B[t].astype(np.complex128)
        if t:
            S -= times(t, -1, H[-1])
            y -= times(t, -1, Z[-1])
        R = np.linalg.solve(S, np.concatenate([band(t, 1), y], axis=1))
        H.append(np.ascontiguousarray(R[:, :w]))
        Z.append(np.ascontiguousarray(R[:, w:]))
    X = np.empty((nb, w, B.shape[2]), np.complex128)
    X[-1] = Z[-1]
    for t in range(nb - 2, -1, -1):
        X[t] = Z[t] - H[t] @ X[t + 1]
    return X.transpose(2, 1, 0) if swap else X.transpose(2, 0, 1)


def exact(case, seed):
    if case["kind"] not in ("solve", "dropin"):
        return None
    nx, ny, nf = case["nx"], case["ny"], case.get("nfreq", 1)
    long, short = max(nx, ny), min(nx, ny)
    if nf * long * short ** 2 * (short + 2.0 * case["nrhs"]) > 1.1e11:
        return None
    B = _panel(case, seed, "cpu").numpy().reshape(nf, case["nrhs"], ny, nx)
    X = np.stack([_block_solve(D, case["sys"], B[f]) for f, D in enumerate(_systems(case, seed))])
    X = X.reshape(nf, case["nrhs"], nx * ny)
    if case["kind"] == "dropin":
        return X[0].real.copy(), X[0].imag.copy()
    return X if nf > 1 else X[0]
