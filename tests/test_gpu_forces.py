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
