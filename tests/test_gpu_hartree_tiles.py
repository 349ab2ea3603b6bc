"""The Hartree CG's tiled iteration on grids whose edges do not fill its tiles (32 x 8 or 16 x 16
columns; 2, 4 or 8 planes), every stencil width and number of periodic directions, against the
solution by the eigenvectors of each axis' operator.

Bar: the solve stops at sqrt(mean r^2) <= eps, so |V - V*| <= eps sqrt(n) / lambda_min with
lambda_min the operator's smallest nonzero eigenvalue."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kk():
    from rspacedist_amd import kukan
    kukan.init(0)
    kukan.set_param("hartree_persistent", 0)
    return kukan


def _axis(n, h, nf, periodic):
    a = -0.5 * H.fd_weights(nf) / h ** 2
    t = np.zeros((n, n))
    for i in range(n):
        t[i, i] += a[0]
        for m in range(1, nf + 1):
            for j in (i - m, i + m):
                if periodic or 0 <= j < n:
                    t[i, j % n] += a[m]
    return np.linalg.eigh(t)


@pytest.mark.parametrize("dims", [(8, 8, 8), (33, 9, 13), (16, 17, 6), (47, 31, 34), (64, 40, 100), (70, 66, 68),
                                  (258, 10, 9)])
@pytest.mark.parametrize("nperi,nfh", [(3, 4), (0, 6), (1, 5), (2, 4)])
def test_tiles(kk, dims, nperi, nfh):
    h, eps = 0.3, 1e-9
    if min(dims) < nfh:
        pytest.skip("edge below the stencil radius")
    rng = np.random.default_rng(sum(dims) + nperi)
    rho = np.asfortranarray(rng.random(dims))
    v = np.asfortranarray(0.1 * rng.standard_normal(dims))  # a warm start far from the solution
    z = np.zeros(1)
    kk.call("scf_hartree", nd=1, ncpx_d=dims[0], ncpy_d=dims[1], ncpz_d=dims[2], nfh=nfh, ndisp=6, nperi=nperi,
            ncgres=801, ncgmin=1, ncgmax=3000, xmax=dims[0] * h / 2, ymax=dims[1] * h / 2, zmax=dims[2] * h / 2,
            epsvh=eps, rho_aug_dense=rho, boundx=z, boundy=z, boundz=z, vh_dense=v)
    b = 2 * np.pi * rho
    if nperi == 3:
        b, v = b - b.mean(), v - v.mean()
    lam, q = zip(*(_axis(n, h, nfh, nperi > ax) for ax, n in enumerate(dims)))
    c = np.einsum("xyz,xa,yb,zc->abc", b, *q, optimize=True)
    d = lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :]
    live = d > 1e-8
    ref = np.einsum("abc,xa,yb,zc->xyz", np.where(live, c / np.where(live, d, 1.0), 0.0), *q, optimize=True)
    assert np.linalg.norm(v - ref) <= 1.01 * eps * np.sqrt(rho.size) / d[live].min()
    assert kk.get_param("hartree_iterations") < 3000


# 1064 and 1300 tiles of 32 x 8 / 16 x 16 columns by four planes (four from 1024 tiles on), 8320 and
# 8280 (eight past 8192), every edge ending inside a tile
@pytest.mark.parametrize("dims,nperi,nfh", [((124, 56, 149), 3, 4), ((124, 55, 150), 0, 6), ((70, 66, 205), 1, 5),
                                            ((250, 121, 257), 3, 6), ((251, 122, 259), 1, 4), ((248, 119, 273), 2, 5)])
def test_taller_tiles(kk, dims, nperi, nfh):
    test_tiles(kk, dims, nperi, nfh)


def test_lock_step(kk):
    """Cells of different edges advanced together, their rule changed from step to step (an
    iteration count inside, at and past a block of 16): each against its own solve from the same
    density and start.  CG iterates of a few tens of iterations agree to the rounding of their
    recurrences, ~1e-15 of the potential an iteration."""
    from rspacedist_amd import batch, synth
    b = batch.Batch()
    cells = []
    for n, h, m in ((8, 0.4, 2), (33, 0.3, 3), (17, 0.35, 1), (50, 0.3, 4)):
        s = synth.make_system(n, h, 2, m, seed=n)
        q, _ = np.linalg.qr(synth.smooth_bands(synth.random_bands(s), n, h))
        b.add(s, np.asfortranarray(q / np.sqrt(s.dv)))
        cells.append([s, np.zeros(s.npts)])
    z = np.zeros(1)
    for batched, ncgmax in ((True, 1), (True, 16), (False, 17), (True, 33), (False, 1), (True, 15)):
        b.step(batched=batched, ncgmax=ncgmax, epsvh=1e-30)
        for i, (s, start) in enumerate(cells):
            psi, _, vh, its = b.get(i)
            ref = start.copy()
            kk.call("scf_hartree", nd=1, ncpx_d=s.n, ncpy_d=s.n, ncpz_d=s.n, nfh=4, ndisp=6, nperi=3, ncgres=801,
                    ncgmin=1, ncgmax=ncgmax, xmax=s.xmax, ymax=s.xmax, zmax=s.xmax, epsvh=1e-30,
                    rho_aug_dense=(psi ** 2).sum(axis=1), boundx=z, boundy=z, boundz=z, vh_dense=ref)
            assert its == ncgmax
            np.testing.assert_allclose(vh, ref, rtol=0, atol=1e-11 * np.abs(ref).max())
            cells[i][1] = vh.copy()
    b.close()


@pytest.mark.parametrize("sizes", [(66, 70, 62), (150, 149, 131)])
def test_lock_step_taller_tiles(kk, sizes):
    """Cells together large enough for tiles of four and of eight planes (1131 tiles of 16 x 16
    columns by four planes, 10025 of 32 x 8), none of whose edges ends with a tile; bar as above."""
    from rspacedist_amd import batch, synth
    b = batch.Batch()
    cells = []
    for n in sizes:
        s = synth.make_system(n, 0.3, 1, 1, seed=n)
        psi = np.asfortranarray(synth.random_bands(s))
        b.add(s, psi / np.linalg.norm(psi) / np.sqrt(s.dv))
        cells.append([s, np.zeros(s.npts)])
    z = np.zeros(1)
    for batched, ncgmax in ((True, 5), (False, 18)):
        b.step(batched=batched, ncgmax=ncgmax, epsvh=1e-30)
        for i, (s, start) in enumerate(cells):
            psi, _, vh, its = b.get(i)
            ref = start.copy()
            kk.call("scf_hartree", nd=1, ncpx_d=s.n, ncpy_d=s.n, ncpz_d=s.n, nfh=4, ndisp=6, nperi=3, ncgres=801,
                    ncgmin=1, ncgmax=ncgmax, xmax=s.xmax, ymax=s.xmax, zmax=s.xmax, epsvh=1e-30,
                    rho_aug_dense=(psi ** 2).sum(axis=1), boundx=z, boundy=z, boundz=z, vh_dense=ref)
            assert its == ncgmax
            np.testing.assert_allclose(vh, ref, rtol=0, atol=1e-11 * np.abs(ref).max())
            cells[i][1] = vh.copy()
    b.close()
