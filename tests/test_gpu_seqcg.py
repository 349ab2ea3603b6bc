"""The band-sequential CG (kscg_r, kscg_c) on grids whose edges do not fill its tiles, every number
of periodic directions, the stencil's widths, its options (northo, nkscg, nprecon_cg), bands that
stop early, and band counts on both sides of the one (128) where the projections are folded by a
launch of their own, against the oracle.

Bar: both sides follow the same iterates; an iteration carries the rounding of its vectors (~1e-16
of their size, sums of 1728 terms ~1e-15) on through the division by the norm of a direction
that the projection has shortened, at most ~1e3 per iteration here: 1e-8 of the largest entry
leaves that for two of them."""
import numpy as np
import pytest

from rspacedist_amd import synth
from tests import helpers as H
from tests.test_gpu_bloch import init_c
from tests.test_oracle_bloch import K

pytestmark = pytest.mark.gpu

CASES = [  # 1728 points each
    dict(dims=(9, 16, 12), nperi=2, nf=8),
    dict(dims=(27, 8, 8), nperi=1, nf=5),
    dict(dims=(8, 6, 36), nperi=3, nf=6, q=2.0),
    dict(dims=(18, 32, 3), nperi=0, nf=1, nkscg=0),
    dict(dims=(12, 12, 12), northo=2, q=2.0),
    dict(dims=(12, 12, 12), northo=2),
    dict(dims=(12, 12, 12), nprecon_cg=0, q=2.0, nf=2),
    dict(dims=(36, 4, 12), nf=3, nsdmax=1, m=1),
    dict(dims=(12, 12, 12), nsdmax=19, epssd=0.3, q=2.0),
    dict(dims=(12, 12, 12), nsdmax=2, m=128),
    dict(dims=(12, 12, 12), nsdmax=2, m=131, q=2.0),
]


@pytest.fixture(scope="module")
def kk():
    from rspacedist_amd import kukan
    kukan.init(0)
    kukan.set_param("kscg_mode", 0)
    return kukan


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_iterates(kk, orc, case, cplx):
    c = dict(nperi=3, northo=1, nkscg=1, nprecon_cg=1, nsdmax=3, nf=4, q=0.0, m=7, epssd=1e-14)
    c.update(CASES[case])
    s = synth.make_system(12, 0.45, 3, c["m"], seed=50 + case, nf=c["nf"], q_scale=c["q"])
    kw = {k: c[k] for k in ("nperi", "northo", "nkscg", "nprecon_cg", "nsdmax", "epssd")}
    kw.update(zip(("ncpx", "ncpy", "ncpz"), c["dims"]))
    if cplx:
        st, name, args = init_c(orc, s), "kscg_c", synth.bloch_args(s, K, **kw)
        vec = ("sveccm", "ssvcm", "hsvcm", "cspsep")
    else:
        st, name, args = H.init_state(s, orc), "kscg_r", synth.abi_args(s, **kw)
        vec = ("svecre", "ssvre", "hsvre", "rspsep")
    out = []
    for f in (kk.call, orc.call):
        a = {k: v.copy(order="F") for k, v in st.items()}
        a["_ret"] = f(name, **args, **a)
        out.append(a)
    g, o = out
    for k in vec + ("sval",):
        np.testing.assert_allclose(g[k], o[k], rtol=0, atol=1e-8 * np.abs(o[k]).max(), err_msg=k)
    np.testing.assert_allclose(g["residual_states"], o["residual_states"], rtol=1e-6, atol=1e-14)
    assert g["_ret"]["ksitmax"] == o["_ret"]["ksitmax"]
    assert g["_ret"]["ksconv"] == o["_ret"]["ksconv"]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("dims,nf", [((17, 17, 260), 4), ((17, 18, 1030), 3), ((18, 17, 1029), 8)])
def test_long_grids(kk, orc, dims, nf, cplx):
    """More tiles than the H kernel's 512 work-groups (520 tiles of two planes), and enough for
    tiles of four planes (past 2048 of two; a last one of two planes or one), with partial tiles
    along every axis and vectors longer than one sweep of the elementwise kernels.  Bar as above,
    for sums over 75000 to 315000 terms."""
    m, n = 3, int(np.prod(dims))
    s = synth.make_system(12, 0.45, 3, m, seed=sum(dims), nf=nf, q_scale=1.0)
    rng = np.random.default_rng(nf)
    kw = dict(zip(("ncpx", "ncpy", "ncpz"), dims), nperi=3, nsdmax=2, epssd=1e-14,
              veff=np.asfortranarray(0.3 * rng.standard_normal((n, 1))))
    psi = rng.standard_normal((n, m))
    z = lambda *d: np.zeros(d, dtype=np.complex128 if cplx else np.float64, order="F")  # noqa: E731
    if cplx:
        psi = psi + 1j * rng.standard_normal((n, m))
        name, gs, args = "kscg_c", "orthogonalization_c", synth.bloch_args(s, K, **kw)
        st = dict(sveccm=np.asfortranarray(psi), ssvcm=z(n, m), cspsep=z(9, s.natom, m))
        vec = ("sveccm", "ssvcm", "hsvcm", "cspsep")
    else:
        name, gs, args = "kscg_r", "orthogonalization_r", synth.abi_args(s, **kw)
        st = dict(svecre=np.asfortranarray(psi), ssvre=z(n, m), rspsep=z(9, s.natom, m))
        vec = ("svecre", "ssvre", "hsvre", "rspsep")
    orc.call(gs, **args, nflag=1, **st)
    st.update({vec[2]: z(n, m), "sval": np.zeros(m), "residual_states": np.zeros(m)})
    out = []
    for f in (kk.call, orc.call):
        a = {k: v.copy(order="F") for k, v in st.items()}
        f(name, **args, **a)
        out.append(a)
    g, o = out
    for k in vec + ("sval",):
        np.testing.assert_allclose(g[k], o[k], rtol=0, atol=1e-8 * np.abs(o[k]).max(), err_msg=k)
    np.testing.assert_allclose(g["residual_states"], o["residual_states"], rtol=1e-6, atol=1e-14)
