"""Frequencies solved together by the workflows: the grouping rule, and the workflows' results
against the same calls one frequency at a time."""
import numpy as np
import pytest

import germaine_amd as G
from germaine_amd import fdfd, models
from tests._grids import smooth_model, te_model


@pytest.mark.parametrize("nfreq,nrhs,n", [(1, 1, 2501), (8, 200, 642001), (8, 104, 642001), (70, 3, 2501), (5, 0, 10)])
def test_groups_cover_every_frequency_once_within_the_limits(nfreq, nrhs, n):
    groups = fdfd._groups(nfreq, nrhs, n)
    assert [f for g in groups for f in g] == list(range(nfreq))
    for g in groups:
        assert 1 <= len(g) <= 64
        assert len(g) == 1 or len(g) * nrhs * n <= fdfd._GROUP_ENTRIES


@pytest.mark.gpu
@pytest.mark.parametrize("phys,precision,nshots", [(G.AC, G.FP64, 7), (G.AC, G.FP32, 7), (G.TE, G.FP64, 3)])
def test_grouped_frequencies_equal_one_at_a_time(phys, precision, nshots, monkeypatch):
    torch = pytest.importorskip("torch")
    nx, ny, npml = 61, 47, 8
    if phys == G.TE:
        (m1, m2), dh, freqs = te_model(nx, ny, seed=4), 0.04, [1.0e8, 2.0e8, 3.0e8]
    else:
        (m1, m2), dh, freqs = smooth_model(nx, ny, seed=4), 10.0, [4.0, 7.0, 9.0]
    m1, m2 = (torch.as_tensor(m, device="cuda") for m in (m1, m2))
    src = models.acquisition_row(nx, npml, dh, 2, nshots)
    rec = models.acquisition_row(nx, npml, dh, 6, 11)
    pl = fdfd.Plan(nx, ny)
    rng = np.random.default_rng(2)
    pobs = [torch.as_tensor((rng.standard_normal((nshots, 11)) + 1j * rng.standard_normal((nshots, 11)))
                            .astype(np.complex64), device="cuda") for _ in freqs]
    args = (pl, phys, dh, freqs, m1, m2, src, rec)
    kw = dict(npml=npml, precision=precision, tol=1e-12, max_iter=30)

    def results():
        fwd = fdfd.forward_shots(*args, keep_fields=True, **kw)
        l2, grad = fdfd.grad_obj(*args, pobs, **kw)
        out = [x.cpu().numpy() for x in fwd["fields"] + fwd["data"]]
        out += [g.cpu().numpy() for g in (grad if isinstance(grad, tuple) else (grad,))]
        hess = fdfd.hessian_gn(*args, **kw)
        out += [h.cpu().numpy() for h in (hess if isinstance(hess, tuple) else (hess,))]
        return out + [np.array([l2, fdfd.objective(*args, pobs, **kw)])]

    together = results()
    monkeypatch.setattr(fdfd, "_GROUP_ENTRIES", 1)
    assert [len(g) for g in fdfd._groups(3, nshots, pl.n)] == [1, 1, 1]
    # FP32 factors stop at a 1e-12 residual along different corrections; receiver samples round to float
    for a, b in zip(together, results()):
        assert np.linalg.norm(a - b) <= (2e-7 if a.dtype == np.complex64 else 1e-7) * np.linalg.norm(b)


@pytest.mark.gpu
def test_kept_fields_own_their_storage():
    """A field kept, dropped or saved by itself is one frequency's panel, not its group's."""
    torch = pytest.importorskip("torch")
    nx, ny, npml = 41, 37, 6
    m1, m2 = (torch.as_tensor(m, device="cuda") for m in smooth_model(nx, ny, seed=4))
    pl = fdfd.Plan(nx, ny)
    src = models.acquisition_row(nx, npml, 10.0, 2, 5)
    fields = fdfd.forward_shots(pl, G.AC, 10.0, [4.0, 7.0, 9.0], m1, m2, src, npml=npml, keep_fields=True)["fields"]
    assert [tuple(x.shape) for x in fields] == [(5, pl.n)] * 3
    assert all(x.untyped_storage().nbytes() == 5 * pl.n * 16 for x in fields)


@pytest.mark.gpu
def test_frequencies_of_any_sized_iterable():
    """Frequencies need a length and an order, not an index: a dict's keys, as a list of them."""
    torch = pytest.importorskip("torch")
    nx, ny, npml = 41, 37, 6
    m1, m2 = (torch.as_tensor(m, device="cuda") for m in smooth_model(nx, ny, seed=4))
    src, rec = models.acquisition_row(nx, npml, 10.0, 2, 5), models.acquisition_row(nx, npml, 10.0, 5, 7)
    args = (fdfd.Plan(nx, ny), G.AC, 10.0)
    pobs = [torch.ones((5, 7), dtype=torch.complex64, device="cuda")] * 2

    def results(freqs):
        fwd = fdfd.forward_shots(*args, freqs, m1, m2, src, rec, npml=npml)["data"]
        return fwd + [fdfd.hessian_shin(*args, freqs, m1, m2, src, npml=npml),
                      fdfd.hessian_gn(*args, freqs, m1, m2, src, rec, npml=npml),
                      fdfd.grad_obj(*args, freqs, m1, m2, src, rec, pobs, npml=npml)[1]]

    for a, b in zip(results([4.0, 7.0]), results({4.0: "a", 7.0: "b"}.keys())):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["library", "torch"])
def test_group_beyond_memory_goes_one_at_a_time(kind, monkeypatch):
    """A group whose second panel solve runs out of memory gives what its frequencies give one by one; other
    errors, and one frequency's own, are the caller's."""
    torch = pytest.importorskip("torch")
    nx, ny, npml = 41, 37, 6
    m1, m2 = (torch.as_tensor(m, device="cuda") for m in smooth_model(nx, ny, seed=4))
    src, rec = models.acquisition_row(nx, npml, 10.0, 2, 5), models.acquisition_row(nx, npml, 10.0, 5, 7)
    args = (fdfd.Plan(nx, ny), G.AC, 10.0, [4.0, 7.0, 9.0], m1, m2, src, rec)
    pobs = [torch.ones((5, 7), dtype=torch.complex64, device="cuda")] * 3

    def results():
        fwd = fdfd.forward_shots(*args, npml=npml)
        l2, grad = fdfd.grad_obj(*args, pobs, npml=npml)
        return fwd["data"] + [fdfd.hessian_gn(*args, npml=npml), grad], [l2, fdfd.objective(*args, pobs, npml=npml)]

    monkeypatch.setattr(fdfd, "_GROUP_ENTRIES", 1)
    ref = results()
    monkeypatch.undo()
    solve, calls = fdfd.Factors.solve_refine_batch, []

    def limited(self, freqs, *a, **kw):
        calls.append(len(freqs))
        if len(freqs) > 1 and len(calls) % 2 == 0:
            raise (G.GfdfdError("hipMalloc of 1 bytes: out of memory") if kind == "library" else
                   torch.OutOfMemoryError("HIP out of memory."))
        return solve(self, freqs, *a, **kw)

    monkeypatch.setattr(fdfd.Factors, "solve_refine_batch", limited)
    got = results()
    assert max(calls) == 3 and 1 in calls
    assert got[1] == ref[1] and all(torch.equal(a, b) for a, b in zip(got[0], ref[0]))

    def failing(self, freqs, *a, **kw):
        raise G.GfdfdError("out of memory" if len(freqs) == 1 else "singular")

    monkeypatch.setattr(fdfd.Factors, "solve_refine_batch", failing)
    with pytest.raises(G.GfdfdError, match="singular"):
        fdfd.forward_shots(*args, npml=npml)
    monkeypatch.setattr(fdfd, "_GROUP_ENTRIES", 1)
    with pytest.raises(G.GfdfdError, match="out of memory"):
        fdfd.forward_shots(*args, npml=npml)


def test_groups_are_even():
    n = fdfd._GROUP_ENTRIES // 3
    assert [len(g) for g in fdfd._groups(4, 1, n)] == [2, 2]
    assert [len(g) for g in fdfd._groups(7, 1, n)] == [3, 3, 1]
    assert fdfd._groups(0, 1, n) == []
