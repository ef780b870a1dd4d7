"""The CG iteration for few projector rows (operator by band, then one kernel)
against the general iteration, at the edges of its register and row splits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _state(cell, nr, nv, nproj, pad, seed):
    from west_amd.groundstate import GroundState, from_real
    from west_amd.gsphere import make_gamma_basis
    b = make_gamma_basis(np.eye(3) * cell, 16.0, nr=(nr, nr, nr))
    n = b.npw
    rng = np.random.default_rng(seed)
    # (33 rows whatever the pad, so that both sides get the same ones)
    x = rng.normal(size=(2 * n - 1, nv + 33)) / (1.0 + np.concatenate([b.g2kin, b.g2kin[1:]]))[:, None]
    rows = from_real(np.linalg.qr(x)[0].T.copy(), n, n, 2)[:nv + nproj + pad]
    dvan = np.concatenate([0.1 + rng.random(33)[:nproj], np.zeros(pad)])
    return GroundState(basis=b, npwx=n, vrs=np.random.default_rng(1).random(b.nnr), vkb=rows[nv:], dvan=dvan, evc=rows[:nv], et=np.zeros(nv),
                       nbndval=nv, occ=np.ones(nv), weight=2.0, alpha_pv=1.0)


# npw 258 to 9,200 (4 or 9 elements a thread of 1,024), 1 to 32 rows in groups of 1 to
# 7, up to 256 columns; 33 rows (those added have coefficient zero) take the
# general products
@pytest.mark.parametrize("cell, nr, nv, nproj, m, kin", [
    (8.0, 24, 1, 0, 1, False), (8.0, 24, 2, 1, 256, False), (14.2, 45, 2, 0, 3, False), (14.2, 45, 4, 3, 5, False),
    (14.2, 45, 4, 5, 5, False), (14.2, 45, 16, 16, 7, False), (19.5, 54, 5, 0, 2, False), (19.5, 54, 4, 0, 1, True),
    (19.8, 54, 1, 0, 2, False), (19.8, 54, 2, 0, 1, False), (19.8, 54, 6, 0, 3, False), (25.7, 72, 4, 1, 2, False),
    (25.7, 72, 20, 11, 2, True)])
def test_linsolve(gpu, cell, nr, nv, nproj, m, kin):
    if kin:   # the bands are the only rows
        nproj = 0
    tr2 = 1e-20
    out = []
    for pad in (0, 33 - nproj):
        gs = _state(cell, nr, nv, nproj, pad, 7)
        # (kinetic only: bands beyond nv, with no column of their own, cannot be added; the dense solution instead)
        gpu.set_ground_state(gs, l_kinetic_only=kin)
        rng = np.random.default_rng(m)
        b = (rng.normal(size=(m, gs.npwx)) + 1j * rng.normal(size=(m, gs.npwx))) / (1.0 + gs.basis.g2kin)
        b[:, 0] = b[:, 0].real
        x = np.zeros_like(b)
        e = -0.5 - rng.random(m)
        assert gpu.linsolve_sternheimer_m_wfcts(nv, m, b.copy(), x, e, np.full(m, 1.5), tr2) == 0
        out.append(x)
        if kin:
            # (g2 - e) x + sum_v |v><v|x> = b, by the small system of <v|x>
            d = 1.0 / (gs.basis.g2kin[None] - e[:, None])

            def dot(u, w):
                return 2.0 * (u.real @ w.real.T + u.imag @ w.imag.T) - np.outer(u[:, 0].real, w[:, 0].real)

            ref = np.zeros_like(b)
            for i in range(m):
                w = gs.evc * d[i]
                c = np.linalg.solve(np.eye(nv) + dot(gs.evc, w), dot(gs.evc, (d[i] * b[i])[None])[:, 0])
                ref[i] = d[i] * b[i] - c @ w
            out.append(ref)
            break
    # <M^-1 r|r> < 1e-20 in each solve, M <= 16/1.5 and the operator above 0.5:
    # each is within sqrt(1e-20 11) / 0.5 = 7e-10 of the solution (two-norm)
    err = np.sqrt(2.0 * np.sum(np.abs(out[0] - out[1]) ** 2, axis=1))
    assert err.max() <= 1.4e-9


@pytest.mark.parametrize("cell, nr, nv, m", [(8.0, 24, 1, 256), (14.2, 45, 2, 3), (14.2, 45, 5, 2), (14.2, 45, 7, 1),
                                             (14.2, 45, 31, 2), (19.5, 54, 6, 1), (19.8, 54, 1, 2), (19.8, 54, 2, 2),
                                             (19.8, 54, 9, 1), (25.7, 72, 32, 2), (25.7, 72, 4, 1)])
def test_projector(gpu, cell, nr, nv, m):
    """The operator's projector part for few columns against NumPy."""
    gs = _state(cell, nr, nv, 0, 0, 5)
    gs.vrs = np.zeros_like(gs.vrs)
    gpu.set_ground_state(gs)
    rng = np.random.default_rng(m)
    x = rng.normal(size=(m, gs.npwx)) + 1j * rng.normal(size=(m, gs.npwx))
    x[:, 0] = x[:, 0].real
    got = gpu.apply_sternheimerop_to_m_wfcs(nv, x, np.zeros(m), 0.75)
    ps = 2.0 * (gs.evc.real @ x.real.T + gs.evc.imag @ x.imag.T) - np.outer(gs.evc[:, 0].real, x[:, 0].real)
    ref = gs.basis.g2kin * x + 0.75 * (ps.T @ gs.evc)
    # kinetic terms up to 16 and sums of 18,000 terms
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()


# npw 4,193 and 9,163 (9 elements a thread): threes, twos and fours of rows, one
# group and several, and the columns (129 up) that take the kernel with many
# rows; 4 elements: rows in twos
@pytest.mark.parametrize("cell, nr, nv, m", [(19.8, 54, 6, 1), (19.8, 54, 5, 3), (25.7, 72, 3, 2), (19.8, 54, 9, 129),
                                             (25.7, 72, 32, 256), (25.7, 72, 30, 130), (19.8, 54, 10, 131),
                                             (14.2, 45, 10, 2), (14.2, 45, 13, 3)])
def test_projector_row_groups(gpu, cell, nr, nv, m):
    gpu.profile(True)
    try:
        test_projector(gpu, cell, nr, nv, m)
        assert gpu.profile_query("project")[1] == 1
    finally:
        gpu.profile(False)


# either side of the rule that picks the CG's kernel: npw 1,536 (always), 4,193 (5
# elements a thread: 8 columns beyond ten rows), 9,163 (9: 30 columns, 48 beyond 20 rows)
@pytest.mark.parametrize("cell, nr, nv, m, kernel", [
    (14.2, 45, 32, 1, True), (19.8, 54, 10, 1, True), (19.8, 54, 11, 7, False), (19.8, 54, 11, 8, True),
    (25.7, 72, 10, 2, True), (25.7, 72, 20, 29, False), (25.7, 72, 20, 30, True), (25.7, 72, 21, 47, False),
    (25.7, 72, 21, 48, True), (25.7, 72, 32, 3, False)])
def test_solve_on_either_side_of_the_rule(gpu, cell, nr, nv, m, kernel):
    from oracle.hamiltonian import apply_sternheimerop
    gs = _state(cell, nr, nv, 0, 0, 3)
    gpu.set_ground_state(gs)
    rng = np.random.default_rng(m)
    b = (rng.normal(size=(m, gs.npwx)) + 1j * rng.normal(size=(m, gs.npwx))) / (1.0 + gs.basis.g2kin)
    b[:, 0] = b[:, 0].real
    x = np.zeros_like(b)
    e = -0.5 - rng.random(m)
    gpu.profile(True)
    try:
        assert gpu.linsolve_sternheimer_m_wfcts(nv, m, b.copy(), x, e, np.full(m, 1.5), 1e-20) == 0
        assert (gpu.profile_query("cg_project")[1] > 0) == kernel
    finally:
        gpu.profile(False)
    # the first and the last column's residual r by the oracle's operator: <M^-1 r|r>
    # < 1e-20 at the end, M <= 16/1.5, and roundings of sums of order ten
    for i in {0, m - 1}:
        r = apply_sternheimerop(gs, x[i:i + 1], e[i:i + 1], gs.alpha_pv) - b[i:i + 1]
        assert 2.0 * np.sum(np.abs(r) ** 2) - np.abs(r[0, 0]) ** 2 <= 11e-20 + (1e-12) ** 2
