"""The Gram-Schmidt step of the Davidson at the edges of its register splits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# npw below and above 4 and 9 elements a thread of 1,024
@pytest.mark.parametrize("cell, nr", [(8.0, 24), (19.5, 54), (19.8, 54), (25.7, 72), (25.9, 72)])
def test_gram_schmidt(gpu, cell, nr):
    from west_amd import wfreq
    from west_amd.groundstate import GroundState, from_real
    from west_amd.gsphere import make_gamma_basis
    b = make_gamma_basis(np.eye(3) * cell, 16.0, nr=(nr, nr, nr))
    n = b.npw
    rng = np.random.default_rng(3)
    x = rng.normal(size=(2 * n - 1, 2)) / (1.0 + np.concatenate([b.g2kin, b.g2kin[1:]]))[:, None]
    evc = from_real(np.linalg.qr(x)[0].T.copy(), n, n, 2)
    gs = GroundState(basis=b, npwx=n, vrs=rng.random(b.nnr), vkb=np.zeros((0, n), complex), dvan=np.zeros(0), evc=evc,
                     et=np.zeros(2), nbndval=2, occ=np.ones(2), weight=2.0, alpha_pv=1.0)
    sqvc = np.zeros(gs.npwx)
    sqvc[1:] = np.sqrt(8.0 * np.pi / gs.basis.g2kin[1:])
    gpu.set_ground_state(gs, sqvc=sqvc)
    _, _, v, _ = gpu.davidson_diago(5, n_pdep_maxiter=3, trev_pdep=1e-1, trev_pdep_rel=1e-1, tr2_dfpt=1e-6)
    # an orthonormal basis of at most 20 rows combined with orthonormal coefficients, 10,000-term sums
    assert np.abs(wfreq.glbrak_gamma(v, v) - np.eye(5)).max() <= 1e-11
