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
