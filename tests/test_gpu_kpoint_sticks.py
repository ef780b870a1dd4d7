"""The q-point path on grids beyond the LDS (stick transforms or the fused
iteration, one CG over the columns of every k point) against the oracle: the operator and the CG at each
k point, chi0(q) with all k points in one solve and one after another, and a
grid whose planes take the two-radix kernels or the compiled ones."""
import numpy as np
import pytest

from west_amd.kpoint import make_h2_crystal, make_k_ground_state

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def _smooth(n, npwx, m, g2, seed):
    rng = np.random.default_rng(seed)
    a = np.zeros((m, npwx), complex)
    a[:, :n] = (rng.normal(size=(m, n)) + 1j * rng.normal(size=(m, n))) / (1.0 + g2[None, :n])
    return a


# (30, 25, 27): n1 != n2; (27, 20, 20): an odd length; (25, 25, 30) n1 = n2 not
# compiled; (30, 30, 18): n1 = n2 compiled; (24, 24, 20): the fused CG
# iteration, whose rows fit the LDS where the whole grid does not
CASES = {"n30x25x27": ((9.0, 7.8, 8.4), (2, 1, 1)), "n27x20x20": ((8.4, 5.9, 5.9), (3, 1, 1)),
         "n24x24x20": ((7.2, 7.2, 5.9), (2, 1, 1)),
         "n25x25x30": ((7.8, 7.8, 9.0), (1, 2, 1)), "n30x30x18": ((9.0, 9.0, 5.3), (1, 1, 2))}


@pytest.fixture(scope="module", params=list(CASES), ids=list(CASES))
def ksys(gpu, request):
    cell, nk = CASES[request.param]
    print(f"case {request.param}: ground state", flush=True)
    at = np.diag(cell) + np.array([[0, 0.1, 0.2], [0, 0, 0.1], [0, 0, 0]])
    kgs = make_k_ground_state(make_h2_crystal(25.0, cell=at), nk, nbnd=4)
    assert "n" + "x".join(str(n) for n in kgs.nr) == request.param
    h = gpu.system_create()
    gpu.system_select(h)
    gpu.set_k_ground_state(kgs)
    yield kgs
    gpu.system_select(0)
    gpu.system_destroy(h)


# tolerances as in test_gpu_kpoint.py: FP64 operator 1e-12, converged solves 1e-9
def test_operator_at_k(gpu, ksys):
    from oracle import kpoint as K
    for ik in range(ksys.nks):
        v = K.KView(ksys, ik)
        for m in (1, 5):
            psi = _smooth(v.basis.npw, ksys.npwx, m, v.basis.g2kin, 10 + ik)
            e = np.linspace(-0.6, 0.1, m)
            gpu.set_current_k(ik + 1)
            out = gpu.apply_sternheimerop_to_m_wfcs(ksys.nbndval, psi, e, ksys.alpha_pv)
            assert _rel(out, K.apply_sternheimerop_k(v, psi, e, ksys.alpha_pv)) < 1e-12


def test_linsolve_at_k(gpu, ksys):
    from oracle import kpoint as K
    from oracle.linsolve import linsolve_sternheimer_m_wfcts
    v = K.KView(ksys, ksys.nks - 1)
    m, nb = 3, ksys.nbndval
    b = _smooth(v.basis.npw, ksys.npwx, m, v.basis.g2kin, 3)
    e = np.full(m, float(v.et[:nb].min()) - 0.3)
    ep = K.set_eprec_k(v, v.evc[:1]).repeat(m)
    x0 = K.precondition_k(v, b, ep)
    xr, br = x0.copy(), b.copy()
    linsolve_sternheimer_m_wfcts(v, nb, br, xr, e, ep, 1e-22, 250, None)
    gpu.set_current_k(ksys.nks)
    x = x0.copy()
    assert gpu.linsolve_sternheimer_m_wfcts(nb, m, b.copy(), x, e, ep, 1e-22) == 0
    assert _rel(x, xr) < 1e-9


@pytest.mark.parametrize("kbatch", ["1", "0"])
def test_dfpt_at_q(gpu, ksys, kbatch, monkeypatch):
    from oracle import kpoint as K
    monkeypatch.setenv("WH_KBATCH", kbatch)
    for iq in range(len(ksys.qpts)):
        qb = ksys.qpts[iq].basis
        dv = _smooth(qb.npw, ksys.npwqx, 3, qb.g2kin, 40 + iq)
        for tr2, tol in ((-1.0, 1e-12), (1e-22, 1e-9)):
            out, ierr = gpu.dfpt(3, dv, tr2, iq=iq + 1, return_ierr=True)
            assert not ierr.any()
            assert _rel(out, K.dfpt_q(ksys, iq, dv, tr2)) < tol


def test_iteration_limit_counts_unconverged(gpu, ksys):
    """n_dfpt_maxiter = 2 leaves every column unconverged: nks nbndval a perturbation."""
    try:
        gpu.set_k_ground_state(ksys, n_dfpt_maxiter=2)
        qb = ksys.qpts[0].basis
        dv = _smooth(qb.npw, ksys.npwqx, 2, qb.g2kin, 7)
        with pytest.warns(UserWarning):
            _, ierr = gpu.dfpt(2, dv, 1e-22, iq=1, return_ierr=True)
        assert list(ierr) == [ksys.nks * ksys.nbndval] * 2
    finally:
        gpu.set_k_ground_state(ksys)


# the last: |i| = n1 / 2, a point whose row has no mirror row
@pytest.mark.parametrize("nr, a1, imax", [((12, 10, 9), 6.4, 5), ((20, 16, 15), 11.5, 9), ((15, 12, 16), 8.9, 7),
                                          ((12, 10, 9), 7.2, 6)])
def test_wide_sphere_on_lds_grid(gpu, nr, a1, imax, monkeypatch):
    """Spheres wider than a quarter of the grid (a density cutoff below four times
    the wave functions') keep the fused iteration."""
    import dataclasses
    from oracle import kpoint as K
    from west_amd import kpoint
    from west_amd.gsphere import grid_index, make_gamma_basis
    at = np.diag((a1, 5.9, 5.3))
    s = make_h2_crystal(25.0, cell=at)
    wide, plain = s.basis, kpoint.make_k_basis

    def on_small_grid(_, xk):   # spheres from the full grid, indexed on this one
        b = plain(wide, xk)
        return dataclasses.replace(b, nr=nr, nl=(grid_index(b.mill, nr) + 1).astype(np.int32))

    monkeypatch.setattr(kpoint, "make_k_basis", on_small_grid)
    s = dataclasses.replace(s, basis=make_gamma_basis(at, 25.0, nr=nr))
    kgs = make_k_ground_state(s, (2, 1, 1), nbnd=4, vrs=-np.random.default_rng(6).random(nr[0] * nr[1] * nr[2]))
    assert max(int(np.abs(k.basis.mill[:, 0]).max()) for k in kgs.kpts) == imax > nr[0] // 4
    assert all(len(np.unique(k.basis.nl)) == k.basis.npw for k in kgs.kpts)
    qb = kgs.qpts[1].basis
    dv = _smooth(qb.npw, kgs.npwqx, 3, qb.g2kin, 8)
    h = gpu.system_create()
    gpu.system_select(h)
    try:
        gpu.set_k_ground_state(kgs)
        gpu.profile(True)
        out, ierr = gpu.dfpt(3, dv, 1e-22, iq=2, return_ierr=True)
        assert gpu.profile_query("cg_iter_lds")[1] > 0
        gpu.profile(False)
    finally:
        gpu.system_select(0)
        gpu.system_destroy(h)
    assert not ierr.any()
    # converged solves, as above
    assert _rel(out, K.dfpt_q(kgs, 1, dv, 1e-22)) < 1e-9


def test_workspace_stays_within_the_grid_budget(gpu):
    """The solve over every k point and its sticks share one budget of 2 GiB: 8 k
    points of 16 states on 36^3 points, 40 perturbations (1.8 GiB of vectors and
    grids; the sticks of their 5,120 columns would be 1.25 GiB more)."""
    import torch
    from west_amd.gsphere import make_gamma_basis
    from west_amd.kpoint import KGroundState, KPoint, make_k_basis, make_qpoint, mp_grid
    nb, m = 16, 40
    gb = make_gamma_basis(np.eye(3) * 10.26, 25.0, nr=(36, 36, 36))
    kc, kx = mp_grid(gb, (2, 2, 2))
    bases = [make_k_basis(gb, k) for k in kx]
    npwx = max(b.npw for b in bases)
    rng = np.random.default_rng(2)
    kpts = []
    for b in bases:
        evc = np.zeros((nb, npwx), complex)
        evc[:, :b.npw] = np.linalg.qr(rng.normal(size=(b.npw, nb)) + 1j * rng.normal(size=(b.npw, nb)))[0].T
        kpts.append(KPoint(basis=b, npwx=npwx, evc=evc, et=np.zeros(nb), vkb=np.zeros((0, npwx), complex), weight=0.25))
    kgs = KGroundState(gbasis=gb, nk=(2, 2, 2), kcryst=kc, kpts=kpts, vrs=rng.random(36 ** 3), dvan=np.zeros(0),
                       nbndval=nb, alpha_pv=1.0, qpts=[make_qpoint(gb, kc, kc[1])])
    dv = _smooth(kgs.qpts[0].basis.npw, kgs.npwqx, m, kgs.qpts[0].basis.g2kin, 1)
    h = gpu.system_create()
    gpu.system_select(h)
    try:
        gpu.set_k_ground_state(kgs, n_dfpt_maxiter=2)
        free = torch.cuda.mem_get_info()[0]
        gpu.profile(True)
        with pytest.warns(UserWarning):   # (two iterations)
            gpu.dfpt(m, dv, 1e-22, iq=1)
        assert gpu.profile_query("kzinv")[1] > 0
        gpu.profile(False)
        used = free - torch.cuda.mem_get_info()[0]
    finally:
        gpu.system_select(0)
        gpu.system_destroy(h)
    # and the products' partial sums, the in- and outputs, the sphere's tables
    assert used <= (2 << 30) + (256 << 20)


def test_linsolve_waits_for_device_inputs(gpu, ksys):
    """Device arrays that null-stream work queued before the call still writes."""
    import torch
    v = ksys.kpts[0].basis
    m, nb = 3, ksys.nbndval
    b = torch.from_numpy(_smooth(v.npw, ksys.npwx, m, v.g2kin, 3)).cuda()
    e, ep = np.full(m, -1.5), np.full(m, 1.5)
    big = torch.ones(1 << 28, device="cuda")
    gpu.set_current_k(1)
    out = []
    for late in (False, False, True):   # (the first call sizes the workspaces)
        x, bb = torch.zeros_like(b), torch.zeros_like(b)
        torch.cuda.synchronize()
        if late:
            for _ in range(20):   # some 10 ms
                big.mul_(1.0)
        bb.copy_(b)
        if not late:
            torch.cuda.synchronize()
        assert gpu.linsolve_sternheimer_m_wfcts(nb, m, bb, x, e, ep, 1e-20) == 0
        out.append(x)
    assert torch.equal(out[1], out[2])
