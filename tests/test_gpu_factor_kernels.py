"""The factorisation's kernels at the sizes where their code changes: orders
around one and two rows per lane, panels shorter than a block, pivoting that
moves rows, against the banded oracle."""
import numpy as np
import pytest

import germaine_amd as G
from germaine_amd import fdfd
from oracle import oracle as O
from tests._grids import smooth_model
from tests.test_gpu_parity import dev, oracle_system, random_grid_csc, rel, say

pytestmark = pytest.mark.gpu


def solve_and_check(pl, nx, ny, mats, precision, tol64, sys=0):
    F = pl.factor(dev(np.stack([c[2] + 1j * c[3] for c in mats])), precision)
    assert np.all(F.singular() == 0)
    rng = np.random.default_rng(nx * ny)
    nf = len(mats)
    B = rng.standard_normal((nf, 5, nx * ny)) + 1j * rng.standard_normal((nf, 5, nx * ny))
    if precision == G.FP64:
        X = F.solve_batch(list(range(nf)), dev(B), sys=sys).cpu().numpy()
    else:
        X = F.solve_refine_batch(list(range(nf)), dev(B), sys=sys, tol=1e-12, max_iter=30)[0].cpu().numpy()
    for z, c in enumerate(mats):
        Xr, _ = O.band_solve(*c, B[z].T, sys=sys, perm=O.grid_transpose_perm(nx, ny))
        assert rel(X[z], Xr.T) <= (tol64 if precision == G.FP64 else 1e-8), z


# small fronts of one and of two rows per lane (small_max up to 64, and above), leaves from 2 x 2 on
@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
@pytest.mark.parametrize("leaf_area,small_max", [(4, 13), (9, 30), (32, 64), (32, 66), (50, 90)])
def test_small_fronts_match_oracle(leaf_area, small_max, precision):
    nx, ny = 53, 47
    say("small fronts", leaf_area, small_max, precision)
    pl = fdfd.Plan(nx, ny, leaf_area=leaf_area, small_max=small_max)
    m = pl.fronts()["m"]
    assert m[m <= small_max].max() > 0.7 * small_max
    m1, m2 = smooth_model(nx, ny, seed=3)
    helm = [oracle_system(G.AC, nx, ny, 6, 10.0, f, m1, m2)[1] for f in (4.0, 9.0)]
    fdfd.factor_tuning(0, 0, fdfd.NO_DEEP)
    try:
        solve_and_check(pl, nx, ny, helm, precision, 1e-10)
        # random values: rows move in every panel
        solve_and_check(pl, nx, ny, [random_grid_csc(nx, ny, s) for s in (7, 8)], precision, 1e-8)
    finally:
        fdfd.factor_tuning()


# panels in registers at every workgroup width (separators of up to 45, 109, 230, 300 and 530 rows: one to
# eight waves in FP64 and, past 512 rows, the global-memory panel; sixteen waves in FP32), last panels of
# fewer than 32 columns, one panel and two per step
@pytest.mark.parametrize("deep", [0, fdfd.NO_DEEP])
@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
@pytest.mark.parametrize("nx,ny", [(61, 45), (131, 109)])
def test_register_panels_match_oracle(nx, ny, precision, deep):
    say("register panels", nx, ny, precision, deep)
    pl = fdfd.Plan(nx, ny, small_max=24)
    m1, m2 = smooth_model(nx, ny, seed=9)
    fdfd.factor_tuning(0, 0, deep)
    try:
        solve_and_check(pl, nx, ny, [oracle_system(G.AC, nx, ny, 8, 10.0, 6.0, m1, m2)[1], random_grid_csc(nx, ny, 5)],
                        precision, 1e-8, sys=2)
    finally:
        fdfd.factor_tuning()


@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
@pytest.mark.parametrize("nx,ny", [(300, 230), (341, 307), (561, 531)])
def test_wide_register_panels_residual(nx, ny, precision):
    """Larger separators: the residual of the solution (FP64, from the values), on random
    matrices, whose pivoting moves rows between the waves' slots."""
    say("wide register panels", nx, ny, precision)
    pl = fdfd.Plan(nx, ny)
    c = random_grid_csc(nx, ny, 3)
    vals = dev((c[2] + 1j * c[3])[None, :])
    rng = np.random.default_rng(1)
    B = dev(rng.standard_normal((5, nx * ny)) + 1j * rng.standard_normal((5, nx * ny)))
    fdfd.factor_tuning(0, 0, fdfd.NO_DEEP)
    try:
        F = pl.factor(vals, precision)
    finally:
        fdfd.factor_tuning()
    assert F.singular()[0] == 0
    X, it, rr = F.solve_refine(0, B, tol=1e-12, max_iter=30)
    R = pl.residual(vals[0], B, X).cpu().numpy()
    say("  iterations", it, "relres", rr)
    assert rr <= 1e-12
    assert np.max(np.linalg.norm(R, axis=1) / np.linalg.norm(B.cpu().numpy(), axis=1)) <= 1e-11


# panel sweeps of the multi-block levels at each tile width (16 and 32 right-hand sides per workgroup, by how
# many tiles a launch has): one column past a tile, several frequencies, single last blocks
@pytest.mark.parametrize("sys", [0, 1, 2])
@pytest.mark.parametrize("nf,nrhs,precision", [(1, 17, G.FP64), (3, 33, G.FP64), (8, 129, G.FP64), (3, 65, G.FP32)])
def test_block_tiles_match_oracle(nf, nrhs, precision, sys):
    nx, ny = 131, 109
    say("block tiles", nf, nrhs, precision, sys)
    pl = fdfd.Plan(nx, ny)
    m1, m2 = smooth_model(nx, ny, seed=2)
    mats = [oracle_system(G.AC, nx, ny, 8, 10.0, 3.0 + f, m1, m2)[1] for f in range(nf)]
    F = pl.factor(dev(np.stack([c[2] + 1j * c[3] for c in mats])), precision)
    rng = np.random.default_rng(nrhs)
    B = rng.standard_normal((nf, nrhs, nx * ny)) + 1j * rng.standard_normal((nf, nrhs, nx * ny))
    if precision == G.FP64:
        X = F.solve_batch(list(range(nf)), dev(B), sys=sys).cpu().numpy()
    else:
        X = F.solve_refine_batch(list(range(nf)), dev(B), sys=sys, tol=1e-12, max_iter=30)[0].cpu().numpy()
    cols = [0, nrhs // 2, nrhs - 1]
    for z, c in enumerate(mats):
        Xr, _ = O.band_solve(*c, B[z][cols].T, sys=sys, perm=O.grid_transpose_perm(nx, ny))
        assert rel(X[z][cols], Xr.T) <= (1e-10 if precision == G.FP64 else 1e-8), z


# forward launches large enough that the update of the rows below runs apart from the block pairs' solve; 257
# right-hand sides leave one column in the last tile
@pytest.mark.parametrize("sys", [0, 1, 2])
@pytest.mark.parametrize("nf,nrhs,precision", [(9, 257, G.FP64), (18, 257, G.FP32)])
def test_split_forward_matches_oracle(nf, nrhs, precision, sys):
    fr = fdfd.Plan(131, 109).fronts()
    tiles = [-(-int(fr["m"][s].max()) // 64) * int(s.sum()) * -(-nrhs // 64) * nf
             for s in (fr["level"] == l for l in np.unique(fr["level"])) if fr["p"][s].max() > 32]
    assert max(tiles) > (512 if precision == G.FP64 else 1024)
    test_block_tiles_match_oracle(nf, nrhs, precision, sys)


# a threshold between the blocked levels' orders: two-panel and one-panel levels in one factorisation
@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
def test_mixed_schedule_matches_oracle(precision):
    nx, ny, deep = 97, 81, 110
    say("mixed schedule", precision)
    pl = fdfd.Plan(nx, ny, small_max=16)
    fr = pl.fronts()
    top = [fr["m"][fr["level"] == l].max() for l in np.unique(fr["level"]) if fr["p"][fr["level"] == l].max() > 32]
    assert min(top) < deep <= max(top)
    m1, m2 = smooth_model(nx, ny, seed=6)
    fdfd.factor_tuning(0, 0, deep)
    solve_and_check(pl, nx, ny, [oracle_system(G.AC, nx, ny, 8, 10.0, 6.0, m1, m2)[1], random_grid_csc(nx, ny, 2)],
                    precision, 1e-8, sys=2)


def test_default_schedule_after_other_calls():
    """factor_tuning() returns to the schedule the library starts with: FP64 levels and FP32 levels of few
    tiles one panel per step, FP32 levels of at least 1536 tiles with fronts of order >= 384 two.  On 300 x 300
    a level of order 450 has 221 depth-64 tiles per frequency and the next one 183 at order 451, so eight
    frequencies lie between the two."""
    nx, ny = 300, 300
    say("default schedule")
    pl = fdfd.Plan(nx, ny)
    fr = pl.fronts()
    tiles = []
    for l in np.unique(fr["level"]):
        s = fr["level"] == l
        if fr["m"][s].max() >= 384:
            tiles.append(int((((fr["m"][s] - np.minimum(64, fr["p"][s]) + 63) // 64) ** 2).sum()))
    assert min(tiles) * 8 < 1536 < max(tiles) * 8
    m1, m2 = smooth_model(nx, ny, seed=1)
    vals = pl.assemble(G.AC, 10.0, [2.0 + 0.7 * k for k in range(8)], dev(m1), dev(m2), npml=10)
    rng = np.random.default_rng(3)
    B = dev(rng.standard_normal((5, pl.n)) + 1j * rng.standard_normal((5, pl.n)))

    def solution(v, precision, *tuning):
        fdfd.factor_tuning(0, 1, 0)
        fdfd.factor_tuning(*tuning)
        F = pl.factor(v, precision)
        rr = F.solve_refine(0, B, tol=1e-12, max_iter=30)[2]
        assert rr <= 1e-12
        return F.solve(0, B).cpu().numpy()

    none = (0, 0, fdfd.NO_DEEP)
    assert np.array_equal(solution(vals[:1], G.FP64), solution(vals[:1], G.FP64, *none))
    assert np.array_equal(solution(vals[:1], G.FP32), solution(vals[:1], G.FP32, *none))
    some = solution(vals, G.FP32)
    assert not np.array_equal(some, solution(vals, G.FP32, *none))
    assert not np.array_equal(some, solution(vals, G.FP32, 0, 0, 384))


def small_terms_system(nx, per_ulp, precision):
    """(values, c) of a 64 x 2 grid's matrix [[T, a I], [-b I, I]], T the tridiagonal
    (-1, 2, -1) with a first entry of 1, whose factors are all +-1: the Schur
    complement is I + c K, K[i, j] = nx - max(i, j), and every entry of it the sum of
    that many equal terms c = a b of per_ulp units in the last place of 1."""
    ulp = 2.0 ** (-52 if precision == G.FP64 else -23)
    a, b = ulp, per_ulp
    pl = fdfd.Plan(nx, 2, leaf_area=2 * nx, small_max=8)
    cp, ri = pl.pattern()
    col = np.repeat(np.arange(pl.n), np.diff(cp))
    top_r, top_c = ri < nx, col < nx
    v = np.zeros(pl.nnz, np.complex128)
    v[top_r & top_c & (ri == col)] = 2.0
    v[(ri == 0) & (col == 0)] = 1.0
    v[top_r & top_c & (abs(ri - col) == 1)] = -1.0
    v[top_r & ~top_c & (col - ri == nx)] = a
    v[~top_r & top_c & (ri - col == nx)] = -b
    v[~top_r & ~top_c & (ri == col)] = 1.0
    return pl, v, a * b



def small_terms_error(pl, v, c, precision):
    """Largest error, in units of the last place of 1, of solutions with right-hand
    sides in the second grid row, where the Schur complement I + c K stands."""
    F = pl.factor(dev(v[None]), precision)
    assert F.singular()[0] == 0
    nx = pl.n // 2
    rows = [0, 1, 2, 5, 9]
    B = np.zeros((5, 2 * nx), np.complex128)
    B[np.arange(5), nx + np.array(rows)] = 1.0
    X = F.solve(0, dev(B)).cpu().numpy()
    # (I + c K)^-1 e to second order in c K, whose norm is below 3e-5
    K = c * (nx - np.maximum(*np.mgrid[0:nx, 0:nx])).astype(np.longdouble)
    E = B[:, nx:].real.T.astype(np.longdouble)
    ref = E - K @ E + K @ (K @ E)
    err = float(np.abs(X[:, nx:] - ref.T).max() * 2.0 ** (52 if precision == G.FP64 else 23))
    say("  error in units of the last place of 1:", err)
    return err


# the trailing update's terms are summed before they meet the entry they update: 64 terms of 0.12 units in the
# last place each are lost when they are added to it one by one (or four by four), 7.7 units in all.  Summed
# first, the entry is rounded once or twice and its inverse once: 3 units at most.  One panel and two per step.
@pytest.mark.parametrize("deep", [0, fdfd.NO_DEEP])
@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
def test_trailing_update_keeps_small_terms(precision, deep):
    say("trailing update, small terms", precision, deep)
    fdfd.factor_tuning(0, 0, deep)
    assert small_terms_error(*small_terms_system(64, 0.12, precision), precision) <= 3.0


# the same inside a panel, whose columns are eliminated eight at a time: 16 terms of 0.3 units, lost one by one
# (4.8 units); summed over the eight columns the entry is rounded twice and its inverse once
@pytest.mark.parametrize("precision", [G.FP64, G.FP32])
def test_panel_keeps_small_terms(precision):
    say("panel, small terms", precision)
    assert small_terms_error(*small_terms_system(16, 0.3, precision), precision) <= 2.0


# the forward update of the rows below, where it runs apart from the block pairs' solve: 64 terms of 0.12 units in
# the last place of the entry, lost one by one (7.7 units); summed first the entry is rounded once
@pytest.mark.parametrize("precision,nrhs", [(G.FP64, 257 * 64 - 3), (G.FP32, 513 * 64 - 3)])
def test_split_forward_keeps_small_terms(precision, nrhs):
    nx, bits = 64, 52 if precision == G.FP64 else 23
    say("split forward, small terms", precision)
    assert -(-2 * nx // 64) * -(-nrhs // 64) > (512 if precision == G.FP64 else 1024)
    # [[T, 0], [-I / 4, I]]: L21 is -1/4 on and above the diagonal, y of the first rows 0.48 units throughout
    pl, v, _ = small_terms_system(nx, 0.25, precision)
    v[v == 2.0 ** -bits] = 0.0
    F = pl.factor(dev(v[None]), precision)
    t = float(np.float32(0.48)) * 2.0 ** -bits
    B = np.zeros((1, 2 * nx), np.complex128)
    B[0, 0], B[0, nx:] = t, 1.0
    X = F.solve(0, dev(B).expand(nrhs, -1).contiguous()).cpu().numpy()
    ref = 1.0 + 0.25 * np.longdouble(t) * (nx - np.arange(nx))
    err = float(np.abs(X[:, nx:] - ref).max() * 2.0 ** bits)
    say("  error in units of the last place of 1:", err)
    assert err <= 1.0


# more right-hand-side tiles than a launch's grid holds in z: 2 x 32769 of 32 columns
@pytest.mark.parametrize("sys", [0, 2])
def test_more_tiles_than_one_launch(sys):
    torch = pytest.importorskip("torch")
    nx, ny, nrhs = 13, 6, 32 * 32768 + 17
    say("tiles beyond one launch", sys)
    pl = fdfd.Plan(nx, ny, leaf_area=36)
    assert pl.info.max_pivots > 32
    mats = [random_grid_csc(nx, ny, s) for s in (3, 4)]
    F = pl.factor(dev(np.stack([c[2] + 1j * c[3] for c in mats])), G.FP64)
    rng = np.random.default_rng(0)
    B = rng.standard_normal((2, 7, nx * ny)) + 1j * rng.standard_normal((2, 7, nx * ny))
    pick = torch.arange(nrhs, device="cuda") % 7
    X = F.solve_batch([0, 1], dev(B)[:, pick].contiguous(), sys=sys)
    for z, c in enumerate(mats):
        Xr, _ = O.band_solve(*c, B[z].T, sys=sys, perm=O.grid_transpose_perm(nx, ny))
        ref = dev(np.ascontiguousarray(Xr.T))
        assert float((X[z] - ref[pick]).abs().max()) <= 1e-10 * float(ref.abs().max())
