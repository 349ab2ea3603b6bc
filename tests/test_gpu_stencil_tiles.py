"""The block CG's H passes with enough bands for 1024-thread stencil tiles, on grids whose rows and
planes do not fill them, in the plain, symmetric and general combination forms (a symmetric or
unsymmetric dij).

H psi of the returned bands, which the passes build up by linearity, is H applied to them in
numpy: only rounding differs, ~1e-15 of |H| |psi| per update, 1e-12 of the largest entry.  The
scalars (the passes' partial sums) are those of the same update with the direction stored and its H
formed by the plain pass: two iterations and the closing orthonormalisation of random bands carry
~1e-15 on by at most ~1e4, 1e-10 of the largest entry."""
import numpy as np
import pytest

from rspacedist_amd import synth
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kk():
    from rspacedist_amd import kukan
    kukan.init(0)
    kukan.set_param("precision", 0)
    kukan.set_param("kscg_mode", 1)
    yield kukan
    kukan.set_param("kscg_mode", 0)
    kukan.set_param("bcg_comb", 1)


def h_apply(s, dims, nperi, kw, psi):
    u = psi.T.reshape((-1,) + dims[::-1])  # band, z, y, x
    w = -0.5 * H.fd_weights(s.nf) / s.h ** 2
    out = 3 * w[0] * u + kw["veff"][:, 0].reshape(dims[::-1]) * u
    for ax in range(3):
        for m in range(1, s.nf + 1):
            for k in (m, -m):
                v = np.roll(u, k, axis=3 - ax)
                if nperi <= ax:  # isolated: nothing beyond the edge
                    v = np.moveaxis(v, 3 - ax, 0)
                    v[slice(0, k) if k > 0 else slice(k, None)] = 0.0
                    v = np.moveaxis(v, 0, 3 - ax)
                out += w[m] * v
    out = np.ascontiguousarray(out.reshape(len(u), -1).T)
    for a in range(s.natom):
        c = s.natinf[a]
        p, rows = s.vnlocp[:c, :, a], s.lstvec2[:c, a] - 1
        out[rows] += p @ (kw["dij"][:, :, 0, a].T @ (p.T @ psi[rows])) / s.dv
    return out


@pytest.mark.parametrize("dims,nf,nperi,m", [((24, 20, 17), 4, 3, 1030), ((8, 70, 10), 4, 1, 1029),
                                             ((33, 65, 8), 3, 2, 400), ((100, 21, 8), 2, 0, 400),
                                             ((256, 8, 9), 4, 3, 600)])
@pytest.mark.parametrize("sym", [True, False])
def test_block_step(kk, dims, nf, nperi, m, sym):
    n = int(np.prod(dims))
    s = synth.make_system(12, 0.45, 3, m, seed=sum(dims), nf=nf)
    rng = np.random.default_rng(7)
    q, _ = np.linalg.qr(rng.standard_normal((n, m)))
    dij = s.dij.copy(order="F")
    if not sym:
        dij[0, 1] += 0.01
    kw = dict(neigmx=m, nperi=nperi, nsdmax=2, epssd=1e-14, ncpx=dims[0], ncpy=dims[1], ncpz=dims[2], dij=dij,
              veff=np.asfortranarray(0.3 * rng.standard_normal((n, 1))))
    out = []
    for comb in (1, 0):
        kk.set_param("bcg_comb", comb)
        psi = np.asfortranarray(q / np.sqrt(s.dv))
        a = dict(svecre=psi, ssvre=psi.copy(order="F"), hsvre=np.zeros_like(psi, order="F"),
                 rspsep=np.zeros((9, s.natom, m), order="F"), sval=np.zeros(m), residual_states=np.zeros(m))
        kk.call("orthogonalization_r", **synth.abi_args(s, **kw), nflag=1,
                **{k: a[k] for k in ("svecre", "ssvre", "rspsep")})
        kk.call("kscg_r", **synth.abi_args(s, **kw), **a)
        out.append(a)
    ref = h_apply(s, dims, nperi, kw, out[0]["svecre"])
    np.testing.assert_allclose(out[0]["hsvre"], ref, rtol=0, atol=1e-12 * np.abs(ref).max())
    for k in ("svecre", "sval", "hsvre", "rspsep"):
        np.testing.assert_allclose(out[0][k], out[1][k], rtol=0, atol=1e-10 * np.abs(out[1][k]).max(), err_msg=k)


def block_step(kk, s, dims, nperi, m, precision=0, nsdmax=1, tiled=1, seed=3):
    """(starting bands, results) of one block-CG call."""
    n = int(np.prod(dims))
    rng = np.random.default_rng(seed)
    kw = dict(neigmx=m, nperi=nperi, nsdmax=nsdmax, epssd=1e-14, ncpx=dims[0], ncpy=dims[1], ncpz=dims[2], dij=s.dij,
              veff=np.asfortranarray(0.3 * rng.standard_normal((n, 1))))
    q, _ = np.linalg.qr(rng.standard_normal((n, m)))
    psi = np.asfortranarray(q / np.sqrt(s.dv))
    a = dict(svecre=psi, ssvre=psi.copy(order="F"), hsvre=np.zeros_like(psi, order="F"),
             rspsep=np.zeros((9, s.natom, m), order="F"), sval=np.zeros(m), residual_states=np.zeros(m))
    kk.set_param("stencil_lds", tiled)
    kk.set_param("precision", precision)
    try:
        kk.call("orthogonalization_r", **synth.abi_args(s, **kw), nflag=1,
                **{k: a[k] for k in ("svecre", "ssvre", "rspsep")})
        start = a["svecre"].copy()
        kk.call("kscg_r", **synth.abi_args(s, **kw), **a)
    finally:
        kk.set_param("stencil_lds", 1)
        kk.set_param("precision", 0)
    return kw, start, a


def shifted(u, ax, k, periodic):
    """u (band, z, y, x) at +k along axis ax (0: x), zero beyond an isolated edge."""
    v = np.roll(u, -k, axis=3 - ax)
    if not periodic:
        v = np.moveaxis(v, 3 - ax, 0)
        v[slice(-k, None) if k > 0 else slice(0, -k)] = 0.0
        v = np.moveaxis(v, 0, 3 - ax)
    return v


@pytest.mark.parametrize("dims,nf,nperi", [((6, 22, 21), 4, 1), ((12, 7, 30), 3, 3), ((300, 9, 8), 4, 2),
                                           ((24, 20, 17), 4, 3)])
def test_block_step_outside_the_tiles(kk, dims, nf, nperi):
    """A block-CG iteration on grids that the stencil tiles do not take (an axis below 8 points, x
    above 256): its eigenvalue estimates <psi|H psi> and residuals <r|K r> of the bands it starts
    from, against numpy.  Bar: sums of 2500 to 20000 terms of the size of |H| |psi|^2, 1e-11."""
    m = 7
    s = synth.make_system(12, 0.45, 3, m, seed=sum(dims), nf=nf)
    kw, psi, a = block_step(kk, s, dims, nperi, m)
    h = h_apply(s, dims, nperi, kw, psi)
    eps = s.dv * (psi * h).sum(axis=0)
    r = (eps * psi - h).T.reshape((-1,) + dims[::-1])
    k = 0.5 * r
    for ax in range(3):
        for d in (1, -1):
            k = k + shifted(r, ax, d, nperi > ax) / 12.0
    res = s.dv * (r * k).sum(axis=(1, 2, 3))
    np.testing.assert_allclose(a["sval"], eps, rtol=0, atol=1e-11 * np.abs(eps).max())
    np.testing.assert_allclose(a["residual_states"], res, rtol=0, atol=1e-11 * np.abs(res).max())


def test_block_step_tiled_or_not(kk):
    """The same two iterations with and without the tiles (param stencil_lds), and on a long grid
    outside them with split-precision products: the first to rounding (bar as above), the second to
    the split's 2^-22 carried through two iterations."""
    m = 9
    s = synth.make_system(12, 0.45, 3, m, seed=5)
    x, y = (block_step(kk, s, (24, 20, 17), 3, m, nsdmax=2, tiled=t)[2] for t in (1, 0))
    for k in ("svecre", "sval", "residual_states", "rspsep"):
        np.testing.assert_allclose(y[k], x[k], rtol=0, atol=1e-10 * np.abs(x[k]).max(), err_msg=k)
    x, y = (block_step(kk, s, (300, 15, 16), 3, m, precision=p, nsdmax=2)[2] for p in (0, 1))
    for k in ("svecre", "sval", "residual_states"):
        np.testing.assert_allclose(y[k], x[k], rtol=0, atol=1e-5 * np.abs(x[k]).max(), err_msg=k)
