"""The FP64 matrix-core products at the edges of their tiles, against numpy in extended precision.

Bound: a sum of K products in any order is off by at most K 2^-53 (1 + O(K 2^-53)) times the sum
of their absolute values (numpy's longdouble reference adds nothing at this level)."""
import numpy as np
import pytest

from rspacedist_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kk():
    from rspacedist_amd import kukan
    kukan.init(0)
    kukan.set_param("precision", 0)
    return kukan


# one column .. past a tile of 64 and 128 on either side; inner lengths below, at and past a
# 16-deep step, and odd ones (columns that are not 16-byte aligned)
@pytest.mark.parametrize("m1,m2,k", [(1, 1, 1), (3, 5, 15), (16, 16, 16), (64, 64, 17), (65, 63, 257), (128, 128, 4096),
                                     (129, 127, 4098), (130, 130, 4097), (200, 131, 1000), (300, 70, 2049),
                                     (70, 300, 333), (260, 260, 515)])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_tn_product(kk, m1, m2, k, beta):
    rng = np.random.default_rng(m1 * 1000 + m2 + k)
    A, B = (np.asfortranarray(rng.standard_normal((k, m))) for m in (m1, m2))
    C0 = np.asfortranarray(rng.standard_normal((m1, m2)))
    C = C0.copy(order="F") if beta else np.full_like(C0, np.nan)  # beta = 0 must not read C
    kk.subspace_gemm(1, m1, m2, k, 0.7, A, k, B, k, beta, C, m1)
    ref = 0.7 * (A.astype(np.longdouble).T @ B.astype(np.longdouble)) + beta * C0
    bound = (k + 4) * 2.0 ** -53 * (0.7 * (np.abs(A).T @ np.abs(B)) + np.abs(beta * C0))
    assert np.all(np.abs(C - ref) <= bound)


# at most 32 columns (32 x 32 tiles), and either side of the shortest K of the 128 x 128 tiles
@pytest.mark.parametrize("m1,m2,k", [(2, 32, 1), (32, 32, 4099), (17, 31, 100), (1, 32, 300), (32, 33, 258),
                                     (200, 131, 1022), (200, 131, 1024)])
def test_tn_product_narrow(kk, m1, m2, k):
    test_tn_product(kk, m1, m2, k, -0.5)


@pytest.mark.parametrize("m,ld", [(32, 16_700_000), (64, 8_380_000), (64, 8_388_610)])
def test_tn_product_long_columns(kk, m, ld):
    """Columns so far apart that the last one of a tile lies almost 2^32 bytes from the first (the
    direct kernels' offsets), and one length past that for 64 columns; bound as above."""
    k = 70
    rng = np.random.default_rng(m)
    dev, host = [], []
    for _ in range(2):
        x = rng.standard_normal((m, k))
        d = kk.DeviceArray((ld, m))
        for j in range(m):
            kk._ck(kk.lib().kukan_memcpy(d.device_ptr + 8 * ld * j, x[j].ctypes.data, 8 * k, 1), "kukan_memcpy")
        kk.synchronize()
        dev.append(d)
        host.append(x)
    C = np.full((m, m), np.nan, order="F")
    kk.subspace_gemm(1, m, m, k, 0.7, dev[0], ld, dev[1], ld, 0.0, C, m)
    ref = 0.7 * (host[0].astype(np.longdouble) @ host[1].astype(np.longdouble).T)
    assert np.all(np.abs(C - ref) <= (k + 4) * 2.0 ** -53 * 0.7 * (np.abs(host[0]) @ np.abs(host[1]).T))


@pytest.mark.parametrize("n,m", [(12, 5), (11, 70), (12, 129), (16, 300)])
def test_orthogonalisation_triangles(kk, n, m):
    """orthogonalization_r forms a Gram triangle and applies the triangular inverse in place, over
    one to three column tiles and for even and odd band lengths: Q^T Q dV = 1, and Q spans the
    input with the positive-diagonal factor of the Householder QR.  Random bands have a Gram
    condition number kappa of order 10, and both factorisations are off by a few n eps kappa."""
    s = synth.make_system(n, 0.4, 2, m, seed=n + m)
    psi0 = synth.random_bands(s)
    psi = psi0.copy(order="F")
    kk.call("orthogonalization_r", **synth.abi_args(s), nflag=1, svecre=psi, ssvre=psi,
            rspsep=np.zeros((9, s.natom, m), order="F"))
    kappa = np.linalg.cond(psi0) ** 2
    np.testing.assert_allclose(psi.T @ psi * s.dv, np.eye(m), rtol=0, atol=s.npts * 2.0 ** -53 * kappa)
    q, r = np.linalg.qr(psi0 * np.sqrt(s.dv))
    q *= np.sign(np.diag(r))
    np.testing.assert_allclose(psi * np.sqrt(s.dv), q, rtol=0, atol=s.npts * 2.0 ** -53 * kappa)


@pytest.mark.parametrize("dims,m", [((32, 32, 32), 32), ((32, 32, 32), 33), ((31, 32, 33), 40), ((32, 33, 34), 129),
                                    ((46, 27, 31), 260)])
def test_orthogonalisation_long_bands(kk, dims, m):
    """As above for bands long and many enough (32768 points, more than 32) that the inverse factor
    is applied by the matrix-core product instead of dtrsm: both sides of the line, one to three
    column tiles, points that end inside a tile."""
    s = synth.make_system(12, 0.4, 2, m, seed=m)
    n = int(np.prod(dims))
    psi0 = np.asfortranarray(np.random.default_rng(m).standard_normal((n, m)))
    psi = psi0.copy(order="F")
    kk.call("orthogonalization_r", **synth.abi_args(s, ncpx=dims[0], ncpy=dims[1], ncpz=dims[2]), nflag=1, svecre=psi,
            ssvre=psi, rspsep=np.zeros((9, s.natom, m), order="F"))
    bound = n * 2.0 ** -53 * np.linalg.cond(psi0) ** 2
    np.testing.assert_allclose(psi.T @ psi * s.dv, np.eye(m), rtol=0, atol=bound)
    q, r = np.linalg.qr(psi0 * np.sqrt(s.dv))
    np.testing.assert_allclose(psi * np.sqrt(s.dv), q * np.sign(np.diag(r)), rtol=0, atol=bound)


@pytest.mark.parametrize("m", [66, 130, 257])
def test_block_cg_projection_triangle(kk, m):
    """One block-CG step in FP64 with the triangular projection product and with every product
    on rocBLAS (params gemm_f64 1 / 0): the same step to rounding."""
    s = synth.make_system(14, 0.35, 2, m, seed=m)
    psi = synth.smooth_bands(synth.random_bands(s), s.n, s.h, width=0.6 * s.h)
    out = []
    for own in (1, 0):
        kk.set_param("gemm_f64", own)
        kk.set_param("kscg_mode", 1)
        st = dict(svecre=psi.copy(order="F"), rspsep=np.zeros((9, s.natom, m), order="F"), sval=np.zeros(m),
                  residual_states=np.zeros(m), hsvre=np.zeros_like(psi, order="F"))
        st["ssvre"] = st["svecre"]
        kk.call("orthogonalization_r", **synth.abi_args(s), nflag=1, **{k: st[k] for k in ("svecre", "ssvre", "rspsep")})
        kk.call("scf_diag", **synth.abi_args(s, nsdmax=2, epssd=1e-14), **st)
        out.append(st)
        kk.set_param("gemm_f64", 1)
        kk.set_param("kscg_mode", 0)
    np.testing.assert_allclose(out[0]["sval"], out[1]["sval"], rtol=0, atol=1e-10 * np.abs(out[1]["sval"]).max())
    rho = [(o["svecre"] ** 2).sum(axis=1) for o in out]
    np.testing.assert_allclose(rho[0], rho[1], rtol=0, atol=1e-9 * rho[1].max())


def test_timed_flops(kk):
    """The work booked beside a product's time: 2 m1 m2 k of a full one, half of it (with the
    diagonal) where one triangle is asked for."""
    m, n = 200, 16
    s = synth.make_system(n, 0.4, 2, m, seed=1)
    psi = synth.random_bands(s)
    st = dict(svecre=psi, ssvre=psi, rspsep=np.zeros((9, s.natom, m), order="F"))

    def booked(f):
        kk.timing_reset()
        kk.set_param("timing", 1)
        f()
        kk.synchronize()
        kk.set_param("timing", 0)
        return kk.timing()["gemm_f64"][2]
    C = np.zeros((m, m), order="F")
    assert booked(lambda: kk.subspace_gemm(1, m, m, s.npts, 1.0, psi, s.npts, psi, s.npts, 0.0, C, m)) == 2 * m * m * s.npts
    gram = booked(lambda: kk.call("orthogonalization_r", **synth.abi_args(s), nflag=1, **st))
    assert gram == m * (m + 1) * s.npts
    # one block-CG step: the Gram triangles before and after, the projection's two
    kw = dict(synth.abi_args(s, nsdmax=1, epssd=1e-14), hsvre=np.zeros_like(psi, order="F"), sval=np.zeros(m),
              residual_states=np.zeros(m))
    kk.set_param("kscg_mode", 1)
    total = booked(lambda: kk.call("kscg_r", **kw, **st))
    kk.set_param("kscg_mode", 0)
    assert total == 4 * gram
