"""The FP64 products at the edges of their tiles and K splits: <a|b> (bra) and
the projector update of the operator (ket) against NumPy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(gpu, nv, nr, cell, ecut, alpha_pv):
    from west_amd.groundstate import GroundState, from_real
    from west_amd.gsphere import make_gamma_basis
    b = make_gamma_basis(np.eye(3) * cell, ecut, nr=(nr, nr, nr))
    n = b.npw
    rng = np.random.default_rng(nv + n)
    evc = from_real(np.linalg.qr(rng.normal(size=(2 * n - 1, nv)))[0].T.copy(), n, n, 2)
    gs = GroundState(basis=b, npwx=n, vrs=np.zeros(b.nnr), vkb=np.zeros((0, n), complex), dvan=np.zeros(0),
                     evc=evc, et=np.zeros(nv), nbndval=nv, occ=np.ones(nv), weight=2.0, alpha_pv=alpha_pv)
    gpu.set_ground_state(gs)
    return gs, rng


def _vecs(rng, m, n):
    x = rng.normal(size=(m, n)) + 1j * rng.normal(size=(m, n))
    x[:, 0] = x[:, 0].real
    return x


# spheres of one K chunk and of up to 34; rows and columns
# around 32, 64, 128 and 256
@pytest.mark.parametrize("nr, cell, ecut", [(12, 8.0, 2.0), (32, 12.0, 12.0), (60, 20.0, 16.0)])
@pytest.mark.parametrize("na, nb", [(33, 1), (33, 31), (32, 257), (31, 300), (48, 32), (64, 33), (65, 64), (127, 65),
                                    (128, 127), (129, 129), (300, 257), (1, 513)])
def test_bra(gpu, nr, cell, ecut, na, nb):
    from west_amd import wfreq
    gs, rng = _system(gpu, 2, nr, cell, ecut, 1.0)
    a, b = _vecs(rng, na, gs.npwx), _vecs(rng, nb, gs.npwx)

    def real(x):
        return np.concatenate([x.real, x.imag], axis=1)

    ref = 2.0 * (real(a) @ real(b).T) - np.outer(a[:, 0].real, b[:, 0].real)
    size = 2.0 * (np.abs(real(a)) @ np.abs(real(b)).T)
    # sums of up to 8,710 terms, both sides: sqrt(8,710) roundings of 1.1e-16, times ten, twice
    assert np.all(np.abs(wfreq.glbrak_gamma(a, b) - ref) <= 2e-13 * size)


@pytest.mark.parametrize("nv, m", [(33, 1), (33, 31), (16, 300), (40, 64), (47, 65), (48, 129), (49, 128), (127, 63),
                                   (129, 257)])
def test_ket(gpu, nv, m):
    gs, rng = _system(gpu, nv, 32, 12.0, 12.0, 0.75)
    x = _vecs(rng, m, gs.npwx)
    got = gpu.apply_sternheimerop_to_m_wfcs(nv, x, np.zeros(m), gs.alpha_pv)
    ps = 2.0 * (gs.evc.real @ x.real.T + gs.evc.imag @ x.imag.T) - np.outer(gs.evc[:, 0].real, x[:, 0].real)
    ref = gs.basis.g2kin * x + gs.alpha_pv * (ps.T @ gs.evc)
    # kinetic terms up to 12 and a sum over up to 129 bands
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
