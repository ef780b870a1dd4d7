"""The Lanczos step kernel at the sphere sizes where its split changes (4, 9,
18 and 36 elements a thread of 512, and r in memory), one to four chains,
against a NumPy restatement of the recurrence on the library's own operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gdot(a, b):
    return 2.0 * np.sum(a.real * b.real + a.imag * b.imag, axis=1) - a[:, 0].real * b[:, 0].real


# npw just below and above 512 x 4, 9, 18 and 36: cubic cells at 16 Ry
@pytest.mark.parametrize("cell, nr, nrhs, nls", [(14.2, 45, 1, 7), (14.5, 45, 3, 1), (18.7, 54, 2, 6),
                                                 (19.3, 54, 4, 2), (23.7, 72, 2, 5), (24.2, 72, 3, 3),
                                                 (30.1, 90, 1, 4), (30.9, 90, 2, 5)])
def test_recurrence(gpu, cell, nr, nrhs, nls):
    from west_amd import wfreq
    from west_amd.groundstate import GroundState, from_real
    from west_amd.gsphere import make_gamma_basis
    b = make_gamma_basis(np.eye(3) * cell, 16.0, nr=(nr, nr, nr))
    n = b.npw
    rng = np.random.default_rng(nr + nrhs)
    x = rng.normal(size=(2 * n - 1, 2)) / (1.0 + np.concatenate([b.g2kin, b.g2kin[1:]]))[:, None]
    evc = from_real(np.linalg.qr(x)[0].T.copy(), n, n, 2)
    gs = GroundState(basis=b, npwx=n, vrs=rng.normal(size=b.nnr), vkb=np.zeros((0, n), complex), dvan=np.zeros(0),
                     evc=evc, et=np.zeros(2), nbndval=2, occ=np.ones(2), weight=2.0, alpha_pv=1.0)
    gpu.set_ground_state(gs)
    rhs = (rng.normal(size=(nrhs, n)) + 1j * rng.normal(size=(nrhs, n))) / (1.0 + b.g2kin)
    rhs[:, 0] = rhs[:, 0].real

    def pc(f):
        ps = 2.0 * (evc.real @ f.real.T + evc.imag @ f.imag.T) - np.outer(evc[:, 0].real, f[:, 0].real)
        return f - (ps.T @ evc.real + 1j * (ps.T @ evc.imag))

    rhs = pc(rhs)
    a, bt, q, bn = wfreq.solve_deflated_lanczos_w_full_ortho(2, rhs, nls)
    r, beta, qs = rhs, np.sqrt(_gdot(rhs, rhs)), []
    np.testing.assert_allclose(bn, beta, rtol=1e-13)
    for il in range(nls):
        qs.append(r / beta[:, None])
        r = pc(gpu.apply_sternheimerop_to_m_wfcs(2, qs[il], np.zeros(nrhs), 0.0))
        if il:
            r = r - qs[il - 1] * beta[:, None]
        al = _gdot(qs[il], r)
        r = r - qs[il] * al[:, None]
        for ia in range(il - 1):
            r = r - qs[ia] * _gdot(qs[ia], r)[:, None]
        beta = np.sqrt(_gdot(r, r))
        # sums of up to 20,000 terms in another order, a few steps of growth
        assert np.abs(a[:, il] - al).max() <= 1e-11 * np.abs(a).max()
        if il + 1 < nls:
            assert np.abs(bt[:, il] - beta).max() <= 1e-11 * beta.max()
        assert np.abs(q[il] - qs[il]).max() <= 1e-10 * np.abs(qs[il]).max()
