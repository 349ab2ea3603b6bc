"""force_eig_r at the edges of its kernel: one band and one atom, 1 .. 32 projectors (sweeps of 9),
FD orders 1 .. 4 and every number of periodic directions, against the oracle.

Bar: both sum the same products in different orders; the largest sums run over natinf list points
times 2 nf differences, then projector pairs and bands, so eps times that count times the size of
the terms (bounded by the largest force of the run with all signs made positive) is generous at
1e-11 of the largest component."""
import numpy as np
import pytest

from rspacedist_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kk():
    from rspacedist_amd import kukan
    kukan.init(0)
    return kukan


@pytest.mark.parametrize("nprj", [1, 9, 10, 18, 32])
@pytest.mark.parametrize("nf,nperi,bands,atoms", [(4, 3, 5, 3), (1, 0, 1, 1), (2, 1, 3, 2), (3, 2, 66, 2)])
def test_force_eig_edges(kk, orc, nprj, nf, nperi, bands, atoms):
    s = synth.make_system(12, 0.4, atoms, bands, seed=nprj + nf)
    rng = np.random.default_rng(nprj * 10 + nf)
    sym = lambda a: a + a.transpose(1, 0, *range(2, a.ndim))  # noqa: E731
    kw = synth.abi_args(s, nf=nf, nperi=nperi, nprjmx=nprj, nprj=np.array([nprj], dtype=np.int32),
                        vnlocp=np.asfortranarray(rng.standard_normal((s.num_list, nprj, atoms))),
                        dij=np.asfortranarray(sym(rng.standard_normal((nprj, nprj, 1, atoms)))),
                        sss=np.asfortranarray(sym(rng.standard_normal((nprj, nprj, 1)))))
    arr = dict(svecre=synth.random_bands(s), sval=rng.standard_normal(bands), fnele=rng.random(bands))
    out = []
    for call in (kk.call, orc.call):
        f = [np.zeros(atoms) for _ in range(3)]
        call("force_eig_r", **kw, **arr, fatx=f[0], faty=f[1], fatz=f[2])
        out.append(np.stack(f))
    np.testing.assert_allclose(out[0], out[1], rtol=0, atol=1e-11 * np.abs(out[1]).max())


@pytest.mark.parametrize("nprj", [1, 9, 16, 18, 32])
@pytest.mark.parametrize("bands,n", [(7, 12), (8, 12), (17, 11), (40, 14)])
def test_gather_edges(kk, nprj, bands, n):
    """<p|psi> of a band block (orthogonalization_r's rspsep at nflag = 1, one pass over all
    bands) and the adjoint's four-table pass against numpy: fewer bands than the matrix-core
    kernel takes, ragged band and projector counts, lists that end inside a 16-point step.  Each
    value is a sum of natinf products: off by at most natinf 2^-53 times their absolute sum."""
    s = synth.make_system(n, 0.4, 3, bands, seed=nprj + bands)
    rng = np.random.default_rng(nprj)
    tabs = [np.asfortranarray(rng.standard_normal((s.num_list, nprj, s.natom))) for _ in range(4)]
    dij = rng.standard_normal((nprj, nprj, 1, s.natom))
    dij = np.asfortranarray(dij + dij.transpose(1, 0, 2, 3))
    f = rng.random(bands)
    kw = synth.abi_args(s, nprjmx=nprj, nprj=np.array([nprj], dtype=np.int32), vnlocp=tabs[0], dij=dij)
    psi = synth.random_bands(s)
    dedv, dedr = np.zeros(s.npts), np.zeros((s.natom, 3), order="F")
    kk.call("energy_adjoint_r", **kw, dvnlocp=np.asfortranarray(np.stack(tabs[1:], axis=-1)), svecre=psi, fnele=f,
            dedv=dedv, dedr=dedr)
    want, bound = np.zeros((s.natom, 3)), np.zeros((s.natom, 3))
    for a in range(s.natom):
        m = s.natinf[a]
        w = psi[s.lstvec2[:m, a] - 1]
        r = [t[:m, :, a].T @ w for t in tabs]
        ra = [np.abs(t[:m, :, a]).T @ np.abs(w) for t in tabs]
        for d in range(3):
            want[a, d] = 2 * np.einsum("l,il,ij,jl->", f, r[1 + d], dij[:, :, 0, a], r[0], optimize=True)
            bound[a, d] = 2 * np.einsum("l,il,ij,jl->", f, ra[1 + d], np.abs(dij[:, :, 0, a]), ra[0], optimize=True)
    eps = (2 * s.num_list + nprj * nprj + bands) * 2.0 ** -53
    assert np.all(np.abs(dedr - want) <= eps * bound)
    np.testing.assert_allclose(dedv, s.dv * (f * psi * psi).sum(axis=1), rtol=bands * 2.0 ** -52)
    # the one-table pass: <p|psi> of the orthonormal bands it returns
    rp = np.zeros((nprj, s.natom, bands), order="F")
    kk.call("orthogonalization_r", **dict(kw, sss=np.zeros((nprj, nprj, 1), order="F")), nflag=1, svecre=psi,
            ssvre=psi, rspsep=rp)
    kappa = 50.0  # of the triangular factor applied to psi and to <p|psi> alike
    for a in range(s.natom):
        m = s.natinf[a]
        w = psi[s.lstvec2[:m, a] - 1]
        err = np.abs(rp[:, a] - tabs[0][:m, :, a].T @ w)
        assert np.all(err <= kappa * (s.num_list + s.npts) * 2.0 ** -53 * (np.abs(tabs[0][:m, :, a]).T @ np.abs(w)))


@pytest.mark.parametrize("bands", [7, 8, 40])
def test_species_with_different_projector_counts(kk, orc, bands):
    """Atoms of three species with 0, 9 and 4 projectors on one table: the atom without projectors
    contributes nothing and leaves its neighbours' <p|psi> alone, through the orthonormalisation,
    the adjoint's four-table pass, the band energy, the forces and both band solvers.  Bounds of
    the sums as in test_gather_edges and above; the two band solvers against the oracle after one
    iteration, to the rounding of test_gpu_seqcg's iterates (1e-8 of the largest entry)."""
    nprj, natom = np.array([0, 9, 4], dtype=np.int32), 5
    s = synth.make_system(12, 0.4, natom, bands, seed=bands)
    assert s.natinf.min() > 16
    rng = np.random.default_rng(bands)
    spe = np.array([1, 2, 3, 1, 2], dtype=np.int32)
    count = nprj[spe - 1]
    tabs = [rng.standard_normal((s.num_list, 9, natom)) for _ in range(4)]
    dij = rng.standard_normal((9, 9, 1, natom))
    dij = dij + dij.transpose(1, 0, 2, 3)
    for a, c in enumerate(count):  # zeros past a species' count
        dij[c:, :, :, a] = dij[:, c:, :, a] = 0.0
        for t in tabs:
            t[:, c:, a] = 0.0
    tabs, dij = [np.asfortranarray(0.01 * t) for t in tabs], np.asfortranarray(0.1 * dij)
    kw = synth.abi_args(s, num_spe=3, nprj=nprj, indspe=spe, ntyppp=np.full(3, synth.KEY_PP_PAW, dtype=np.int32),
                        sss=np.zeros((9, 9, 3), order="F"), vnlocp=tabs[0], dij=dij)
    f, e = rng.random(bands), rng.standard_normal(bands)
    psi0 = synth.smooth_bands(synth.random_bands(s), s.n, s.h, width=0.6 * s.h)
    out = []
    for call in (kk.call, orc.call):
        psi, rp = psi0.copy(order="F"), np.zeros((9, natom, bands), order="F")
        call("orthogonalization_r", **kw, nflag=1, svecre=psi, ssvre=psi.copy(order="F"), rspsep=rp)
        fa = [np.zeros(natom) for _ in range(3)]
        call("force_eig_r", **kw, svecre=psi, sval=e, fnele=f, fatx=fa[0], faty=fa[1], fatz=fa[2])
        st = dict(svecre=psi.copy(order="F"), ssvre=psi.copy(order="F"), hsvre=np.zeros_like(psi, order="F"),
                  rspsep=rp.copy(order="F"), sval=np.zeros(bands), residual_states=np.zeros(bands))
        call("kscg_r", **dict(kw, nsdmax=1, epssd=1e-14), **st)
        out.append(dict(st, psi=psi, rp=rp, force=np.stack(fa)))
    for k in ("psi", "force"):
        np.testing.assert_allclose(out[0][k], out[1][k], rtol=0, atol=1e-11 * np.abs(out[1][k]).max(), err_msg=k)
    for k in ("svecre", "hsvre", "rspsep", "sval"):
        np.testing.assert_allclose(out[0][k], out[1][k], rtol=0, atol=1e-8 * np.abs(out[1][k]).max(), err_msg=k)
    psi, rp = out[0]["psi"], out[0]["rp"]
    eb, dedv, dedr = np.zeros(bands), np.zeros(s.npts), np.zeros((natom, 3), order="F")
    kk.call("band_energy_r", **kw, svecre=psi, eband=eb)
    kk.call("energy_adjoint_r", **kw, dvnlocp=np.asfortranarray(np.stack(tabs[1:], axis=-1)), svecre=psi, fnele=f,
            dedv=dedv, dedr=dedr)
    want, bound = np.zeros((natom, 3)), np.zeros((natom, 3))
    for a, c in enumerate(count):
        m = s.natinf[a]
        w, D = psi[s.lstvec2[:m, a] - 1], dij[:c, :c, 0, a]
        r = [t[:m, :c, a].T @ w for t in tabs]
        ra = [np.abs(t[:m, :c, a]).T @ np.abs(w) for t in tabs]
        assert np.all(np.abs(rp[:c, a] - r[0]) <= 50.0 * (s.num_list + s.npts) * 2.0 ** -53 * ra[0])
        assert not rp[c:, a].any()
        for d in range(3):
            want[a, d] = 2 * np.einsum("l,il,ij,jl->", f, r[1 + d], D, r[0], optimize=True)
            bound[a, d] = 2 * np.einsum("l,il,ij,jl->", f, ra[1 + d], np.abs(D), ra[0], optimize=True)
    assert np.all(np.abs(dedr - want) <= (2 * s.num_list + 81 + bands) * 2.0 ** -53 * bound)
    # one iteration's eigenvalue estimate is <psi|H|psi> of the orthonormal bands it starts from
    np.testing.assert_allclose(eb[0], out[0]["sval"][0], rtol=0, atol=1e-11 * np.abs(eb).max())
