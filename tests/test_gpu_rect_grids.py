"""Orthorhombic grids on the device: the plane kernels of n1 != n2 (two radices
per length), of n1 = n2 with another n3, and the run-time-radix kernels behind
them, through the operator and the response without a solve (its forward and
inverse transforms, the real-space potentials and the density), against the
FP64 oracle."""
import numpy as np
import pytest

from oracle.dfpt import dfpt as dfpt_ref
from oracle.hamiltonian import apply_sternheimerop
from west_amd.groundstate import GroundState, from_real
from west_amd.gsphere import make_gamma_basis

pytestmark = pytest.mark.gpu

ECUT = 16.0


def _ground_state(nr, nbnd, nkb, seed):
    """Orthonormal random states on a sphere that fills a quarter of each
    grid length (its widest), a random potential and projectors: neither the
    operator nor the unsolved response needs eigenstates."""
    at = np.diag([2.0 * np.pi * (n // 4 + 0.3) / np.sqrt(ECUT) for n in nr])
    b = make_gamma_basis(at, ECUT, nr=nr)
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.normal(size=(2 * b.npw - 1, nbnd + nkb)))
    rows = from_real(q.T.copy(), b.npw, b.npw + 3, 2)
    return GroundState(basis=b, npwx=b.npw + 3, vrs=rng.normal(size=b.nnr), vkb=rows[nbnd:], dvan=rng.normal(size=nkb),
                       evc=rows[:nbnd], et=rng.normal(size=nbnd), nbndval=nbnd, occ=np.ones(nbnd), weight=2.0,
                       alpha_pv=1.3)


# two radices a length with even and odd lengths and chunks, a plane that
# leaves one workgroup a CU, a length of 75 (run-time radices), n1 = n2 != n3
@pytest.mark.parametrize("nr, nbnd, nkb, m", [
    ((15, 16, 18), 1, 0, 1),
    ((40, 18, 25), 3, 2, 5),
    ((27, 54, 20), 4, 3, 4),
    ((100, 72, 18), 2, 1, 3),
    ((81, 25, 27), 3, 0, 2),
    ((75, 20, 18), 2, 1, 3),
    ((36, 36, 20), 3, 2, 3),
    ((45, 45, 96), 2, 0, 3),
])
def test_operator_and_response(nr, nbnd, nkb, m):
    from west_amd import wstat
    gs = _ground_state(nr, nbnd, nkb, seed=sum(nr))
    n = gs.basis.npw
    wstat.init(0)
    wstat.set_ground_state(gs)
    rng = np.random.default_rng(5)
    psi = np.zeros((m, gs.npwx), complex)
    psi[:, :n] = rng.normal(size=(m, n)) + 1j * rng.normal(size=(m, n))
    psi[:, 0] = psi[:, 0].real
    e = rng.normal(size=m)
    out = wstat.apply_sternheimerop_to_m_wfcs(nbnd, psi, e, gs.alpha_pv)
    ref = apply_sternheimerop(gs, psi, e, gs.alpha_pv)
    # FP64 transforms and sums of a few thousand terms: 1e-12 of the largest value
    assert np.abs(out - ref)[:, :n].max() <= 1e-12 * np.abs(ref).max()
    dv = psi / (1.0 + np.pad(gs.basis.g2kin, (0, gs.npwx - n)))
    got = wstat.dfpt(m, dv, -1.0)
    want = dfpt_ref(gs, dv, -1.0)
    assert np.abs(got - want)[:, :n].max() <= 1e-12 * np.abs(want).max()


# n1 = n2 with another n3: every plane kernel that such a grid can take, the last
# workgroup short of planes (n3 no multiple of 2, 3 or 4); the quad-lane kernels
# at 60, 72 and 100, the LDS-pass kernel above 64, the density in two halves at 100
# and 108 (its scratch by planes)
@pytest.mark.parametrize("nr", [(54, 54, 25), (60, 60, 20), (60, 60, 25), (72, 72, 25), (80, 80, 18), (100, 100, 27),
                                (108, 108, 20)])
def test_square_planes(nr, monkeypatch):
    from west_amd import wstat
    gs = _ground_state(nr, 2, 1, seed=sum(nr))
    n = gs.basis.npw
    wstat.init(0)
    rng = np.random.default_rng(6)
    psi = np.zeros((3, gs.npwx), complex)
    psi[:, :n] = rng.normal(size=(3, n)) + 1j * rng.normal(size=(3, n))
    psi[:, 0] = psi[:, 0].real
    e = rng.normal(size=3)
    ref = apply_sternheimerop(gs, psi, e, gs.alpha_pv)
    for variant in range(1, 10):   # LDS passes, register lines, quad lanes; beyond the last the last again
        monkeypatch.setenv("WH_PLANE_OCC", str(variant))
        wstat.set_ground_state(gs)
        out = wstat.apply_sternheimerop_to_m_wfcs(2, psi, e, gs.alpha_pv)
        assert np.abs(out - ref)[:, :n].max() <= 1e-12 * np.abs(ref).max(), variant
    dv = psi / (1.0 + np.pad(gs.basis.g2kin, (0, gs.npwx - n)))
    got = wstat.dfpt(3, dv, -1.0)
    want = dfpt_ref(gs, dv, -1.0)
    assert np.abs(got - want)[:, :n].max() <= 1e-12 * np.abs(want).max()
