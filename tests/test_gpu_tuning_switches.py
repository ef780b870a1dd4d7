"""The switches that force a transform path: that the path is the one that
runs, and that its results are the others' up to rounding."""
import numpy as np
import pytest

from west_amd.groundstate import GroundState, from_real
from west_amd.gsphere import make_gamma_basis
from west_amd.kpoint import make_h2_crystal, make_k_ground_state

pytestmark = pytest.mark.gpu


def _gamma(gpu, nr, seed=4):
    """Random states and potential on a sphere that fills a quarter of each grid length."""
    ecut = 16.0
    b = make_gamma_basis(np.diag([2.0 * np.pi * (n // 4 + 0.3) / np.sqrt(ecut) for n in nr]), ecut, nr=nr)
    rng = np.random.default_rng(seed)
    rows = from_real(np.linalg.qr(rng.normal(size=(2 * b.npw - 1, 3)))[0].T.copy(), b.npw, b.npw, 2)
    gpu.set_ground_state(GroundState(basis=b, npwx=b.npw, vrs=rng.normal(size=b.nnr), vkb=rows[:0], dvan=np.zeros(0),
                                     evc=rows, et=np.zeros(3), nbndval=3, occ=np.ones(3), weight=2.0, alpha_pv=1.0))
    return b


# two radices for the first two lengths, no compiled third
@pytest.mark.parametrize("nr", [(40, 18, 25), (27, 45, 25)])
def test_runtime_size_kernels_on_orthorhombic_grids(gpu, nr, monkeypatch):
    out = []
    for generic in ("0", "1"):
        monkeypatch.setenv("WH_FFT_GENERIC", generic)
        b = _gamma(gpu, nr)
        rng = np.random.default_rng(2)
        x = rng.normal(size=(3, b.npw)) + 1j * rng.normal(size=(3, b.npw))
        x[:, 0] = x[:, 0].real
        out.append([gpu.apply_sternheimerop_to_m_wfcs(3, x, np.zeros(3), 0.5), gpu.dfpt(3, x / (1.0 + b.g2kin), -1.0)])
    for a, c in zip(*out):
        assert np.abs(a - c).max() <= 1e-12 * np.abs(a).max()
        # other radices: thousands of sums do not all round alike
        assert not np.array_equal(a, c)


@pytest.fixture(scope="module")
def kgs_30():
    # 30 x 25 x 27: beyond the LDS, with stick kernels
    at = np.diag((9.0, 7.8, 8.4)) + np.array([[0, 0.1, 0.2], [0, 0, 0.1], [0, 0, 0]])
    return make_k_ground_state(make_h2_crystal(25.0, cell=at), (2, 1, 1), nbnd=4)


def _at_q(gpu, kgs, m=3, tr2=1e-18):
    """chi0 at the second q point and the profile's counts of the kernels behind it."""
    qb = kgs.qpts[1].basis
    rng = np.random.default_rng(3)
    dv = np.zeros((m, kgs.npwqx), complex)
    dv[:, :qb.npw] = (rng.normal(size=(m, qb.npw)) + 1j * rng.normal(size=(m, qb.npw))) / (1.0 + qb.g2kin)
    gpu.profile(True)
    try:
        out = gpu.dfpt(m, dv, tr2, iq=2)
        return out, {k: gpu.profile_query(k)[1] for k in ("kzinv", "plane_vloc", "cg_iter_lds", "kvloc_lds", "kgrid_lds")}
    finally:
        gpu.profile(False)


def test_runtime_size_kernels_at_q(gpu, kgs_30, monkeypatch):
    out = []
    for generic in ("0", "1"):
        monkeypatch.setenv("WH_FFT_GENERIC", generic)
        gpu.set_k_ground_state(kgs_30)
        r, n = _at_q(gpu, kgs_30)
        assert (n["kzinv"] > 0) == (generic == "0")
        out.append(r)
    # solves to tr2 = 1e-18
    assert np.abs(out[0] - out[1]).max() <= 1e-9 * np.abs(out[0]).max()


def test_plane_variant_at_q(gpu, monkeypatch):
    # 30 x 30 x 18: compiled plane kernels
    at = np.diag((9.0, 9.0, 5.3)) + np.array([[0, 0.1, 0.2], [0, 0, 0.1], [0, 0, 0]])
    kgs = make_k_ground_state(make_h2_crystal(25.0, cell=at), (1, 1, 2), nbnd=4)
    out = []
    for v in ("1", "9"):   # LDS passes, the last of the register-line kernels
        monkeypatch.setenv("WH_PLANE_OCC", v)
        gpu.set_k_ground_state(kgs)
        out.append(_at_q(gpu, kgs)[0])
    assert np.abs(out[0] - out[1]).max() <= 1e-9 * np.abs(out[0]).max()
    assert not np.array_equal(out[0], out[1])


def test_full_grid_switch_leaves_lds_grids(gpu, kgs_30, monkeypatch):
    """WH_KSTICKS=0 is about grids beyond the LDS: on one that fits, the fused CG
    iteration and the solve over all k points stay, bit for bit."""
    at = np.diag((7.2, 5.9, 5.3)) + np.array([[0, 0.1, 0.2], [0, 0, 0.1], [0, 0, 0]])   # 24 x 20 x 18
    kgs = make_k_ground_state(make_h2_crystal(25.0, cell=at), (2, 1, 1), nbnd=4)
    out = []
    for v in ("1", "0"):
        monkeypatch.setenv("WH_KSTICKS", v)
        gpu.set_k_ground_state(kgs)
        r, n = _at_q(gpu, kgs)
        assert n["cg_iter_lds"] > 0 and n["kgrid_lds"] > 0 and n["kzinv"] == 0
        out.append(r)
    assert np.array_equal(out[0], out[1])
    # beyond the LDS it does keep the full grid
    gpu.set_k_ground_state(kgs_30)
    assert _at_q(gpu, kgs_30)[1]["kzinv"] == 0
