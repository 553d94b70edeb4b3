"""HEOM propagation in the commutator form against classical RK4 on the sparse
generator: every block size the compile-time kernels serve, one and two
Matsubara terms, hierarchies whose last level has no upward edges, one and
several samples (small and large tiles, the XCD map), real and complex
Hamiltonians, both pictures, FP64 and MIXED."""
import numpy as np
import pytest
import torch

from qspectra_amd import CM_FS, CM_K, DebyeBath, ElectronicHamiltonian, HEOMModel
from qspectra_amd.simulate.utils import propagate_heom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('sites,K,levels,members,imag', [
    (2, 1, 2, 1, False), (2, 2, 4, 11, False), (3, 1, 5, 1, True), (3, 2, 3, 9, False),
    (4, 1, 3, 3, False), (5, 1, 3, 8, True), (6, 2, 2, 1, False), (7, 1, 3, 1, False),
    (7, 2, 2, 17, True), (8, 1, 3, 2, False)])
def test_commutator_form_matches_rk4(gpu, sites, K, levels, members, imag):
    rs = np.random.RandomState(sites * 10 + K)
    hams = []
    for _ in range(members):
        J = np.triu(rs.normal(0, 60, (sites, sites)) + imag * 1j * rs.normal(0, 60, (sites, sites)),
                    1)
        H = J + J.conj().T + np.diag(rs.uniform(12200, 12700, sites))
        hams.append(ElectronicHamiltonian(H, bath=DebyeBath(CM_K * 300, 35., 106.),
                                          dipoles=np.ones((sites, 3))))
    models = [HEOMModel(h, rw_freq=12450., hilbert_subspace='ge', unit_convert=CM_FS,
                        level_cutoff=levels, K=K) for h in hams]
    batch = models[0]
    if members > 1:
        batch = batch.with_hamiltonians([h.in_rotating_frame(12450.) for h in hams])
    dt, t = 0.5, np.array([0.0, 1.5, 4.0])
    for heisenberg in (False, True):
        eom = batch.equation_of_motion('ee', heisenberg)
        y0 = rs.normal(size=(members, eom.size)) + 1j * rs.normal(size=(members, eom.size))
        want = []
        for m, y in zip(models, y0):
            L = m.HEOM_tensor('ee', heisenberg) * CM_FS
            out = [y]
            for g in range(8):
                k1 = L @ y
                k2 = L @ (y + dt / 2 * k1)
                k3 = L @ (y + dt / 2 * k2)
                y = y + dt / 6 * (k1 + 2 * k2 + 2 * k3 + L @ (y + dt * k3))
                if g + 1 in (3, 8):
                    out.append(y)
            want.append(out)
        want = np.array(want)
        yd = torch.as_tensor(y0).to(eom.Hop.device)
        # FP64: 32 sums of fewer than 60 products; MIXED: 8 steps of terms rounded
        # to 24 bits, which add up to at most 1.1 times the state (the fastest
        # damping, 0.74 a step): 8 x 1.1 x 2^-24 = 5e-7
        for precision, tol in (('fp64', 1e-12), ('mixed', 5e-7)):
            whole = propagate_heom(eom, yd, t, dt=dt, precision=precision, full_states=True)
            assert np.abs(whole.cpu().numpy() - want).max() <= tol * np.abs(want).max()
            ado0 = propagate_heom(eom, yd, t, dt=dt, precision=precision).cpu().numpy()
            assert np.abs(ado0 - want[:, :, :eom.M]).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize('sites,K,levels,members', [
    (2, 1, 4, 3), (5, 1, 4, 60), (7, 2, 3, 30), (8, 1, 3, 70), (8, 2, 3, 9)])
def test_batches_match_their_members(gpu, sites, K, levels, members):
    """Real and complex Hamiltonians in one batch, at batch sizes whose launches
    give a thread one, two and three elements, against batches of one: the
    same sums in the same order, so the same bits."""
    rs = np.random.RandomState(sites + members)
    bath = DebyeBath(CM_K * 300, 35., 106.)
    hams = []
    for imag in (0, 1, 0):
        J = np.triu(rs.normal(0, 60, (sites, sites)) + imag * 1j * rs.normal(0, 60, (sites, sites)),
                    1)
        hams.append(ElectronicHamiltonian(J + J.conj().T + np.diag(rs.uniform(12200, 12700, sites)),
                                          bath=bath, dipoles=np.ones((sites, 3)))
                    .in_rotating_frame(12450.))
    model = HEOMModel(hams[0], rw_freq=12450., hilbert_subspace='ge', unit_convert=CM_FS,
                      level_cutoff=levels, K=K)
    pick = rs.randint(0, 3, members)
    pick[:3] = 0, 1, 2
    batch = model.with_hamiltonians([hams[i] for i in pick]).equation_of_motion('ee')
    y0 = rs.normal(size=(3, batch.size)) + 1j * rs.normal(size=(3, batch.size))
    y0 = torch.as_tensor(y0).to(batch.Hop.device)
    t = np.array([0.0, 2.0])
    for precision in ('fp64', 'mixed'):
        got = propagate_heom(batch, y0[pick], t, dt=0.5, precision=precision, full_states=True)
        for i in range(3):
            one = model.with_hamiltonians([hams[i]]).equation_of_motion('ee')
            want = propagate_heom(one, y0[i:i + 1], t, dt=0.5, precision=precision,
                                  full_states=True)
            for b in np.flatnonzero(pick == i):
                assert torch.equal(got[b], want[0]), (precision, i, b)
