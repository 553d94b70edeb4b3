"""The column form of the ZOFE propagation (diagonal couplings, at most eight
states) against the element-wise kernel, which every other case runs: odd and
even state counts, one and two columns per thread, few and many right-hand
sides, every form of the rho equation, full states and projections, fields."""
import copy

import numpy as np
import pytest
import torch

from qspectra_amd import CM_FS, ElectronicHamiltonian, PseudomodeBath, ZOFEModel, _native

pytestmark = pytest.mark.gpu


def _eom(sites, modes, subspace, members=1, **forms):
    rs = np.random.RandomState(sites * 100 + modes)
    H = rs.normal(0, 60, (members, sites, sites))
    H = H + H.transpose(0, 2, 1) + np.eye(sites) * 300
    one = np.ones((modes, sites))
    bath = PseudomodeBath(modes, rs.uniform(-300, 900, (modes, 1)) * one + 0j,
                          rs.uniform(40, 300, (modes, 1)) * one + 0j,
                          rs.uniform(0.01, 0.2, (modes, 1)) * one + 0j)
    hams = [ElectronicHamiltonian(12000 * np.eye(sites) + h, bath=bath,
                                  dipoles=rs.normal(size=(sites, 3))) for h in H]
    m = ZOFEModel(hams[0], rw_freq=12000., hilbert_subspace=subspace, unit_convert=CM_FS, **forms)
    if members > 1:
        m = m.with_hamiltonians([h.in_rotating_frame(12000.) for h in hams])
    return m.equation_of_motion('ee')


@pytest.mark.parametrize('sites,modes,subspace,members,R', [
    (1, 1, 'e', 1, 1), (2, 1, 'e', 1, 3), (2, 16, 'ge', 2, 1), (3, 5, 'e', 1, 2),
    (3, 3, 'gef', 2, 2), (4, 16, 'e', 3, 1), (4, 17, 'e', 1, 1), (5, 12, 'ge', 1, 2),
    (6, 16, 'e', 2, 1), (7, 5, 'e', 1, 1), (7, 16, 'e', 1, 2), (7, 16, 'ge', 1, 1),
    (8, 10, 'e', 1, 1)])
def test_columns_match_elements(gpu, sites, modes, subspace, members, R):
    rs = np.random.RandomState(5)
    for ham_hermit in (False, True):
        for rho_hermit in (False, True):
            eom = _eom(sites, modes, subspace, members, ham_hermit=ham_hermit,
                       rho_hermit=rho_hermit)
            assert eom.flags & 4
            general = copy.copy(eom)
            general.flags = eom.flags & 3
            dev = eom.H.device
            y0 = rs.normal(size=(members, R, eom.size)) + 1j * rs.normal(
                size=(members, R, eom.size))
            y0 = torch.as_tensor(y0).to(dev)
            nsub = torch.tensor([0, 2, 0, 3], dtype=torch.int32, device=dev)
            h = torch.tensor([0.0, 0.4, 0.0, 0.25], dtype=torch.float64, device=dev)
            proj = torch.as_tensor(rs.normal(size=(1, 2, eom.N ** 2)) + 0j).to(dev)
            V = torch.as_tensor(rs.normal(size=(1, 2, eom.N, eom.N)) + 0j).to(dev)
            F = torch.as_tensor(rs.normal(size=(1, 5, 3, 2)) * 0.01 + 0.01j).to(dev)
            for kw in (dict(), dict(proj=proj), dict(V=V, F=F)):
                a, sa = _native.zofe_propagate(eom, y0, nsub, h, **kw)
                b, sb = _native.zofe_propagate(general, y0, nsub, h, **kw)
                assert int(sa.item()) == int(sb.item()) == 0
                # 20 stages, each a sum of fewer than 100 products in another
                # order: well under 1e4 ulp of the largest entry
                assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_columns_report_missing_field_samples_and_non_finite_states(gpu):
    eom = _eom(3, 4, 'e')
    dev = eom.H.device
    y0 = torch.ones((1, 1, eom.size), dtype=torch.complex128, device=dev)
    nsub = torch.tensor([3], dtype=torch.int32, device=dev)
    h = torch.tensor([0.1], dtype=torch.float64, device=dev)
    V = torch.ones((1, 1, 3, 3), dtype=torch.complex128, device=dev)
    F = torch.ones((1, 2, 3, 1), dtype=torch.complex128, device=dev)
    assert int(_native.zofe_propagate(eom, y0, nsub, h, V=V, F=F)[1].item()) == 2
    y0[0, 0, 1] = float('nan')
    assert int(_native.zofe_propagate(eom, y0, nsub, h)[1].item()) == 1


def test_first_stage_does_not_depend_on_what_the_lds_held(gpu):
    """One step of many members right after models with other site lists have
    used the same LDS: the first stage's sums over sites are those of the
    element-wise kernel."""
    rs = np.random.RandomState(6)
    eoms = [_eom(*args) for args in ((7, 16, 'e', 700), (3, 3, 'gef', 700), (7, 5, 'ge', 700))]
    dev = eoms[0].H.device
    nsub = torch.tensor([1], dtype=torch.int32, device=dev)
    h = torch.tensor([0.4], dtype=torch.float64, device=dev)
    for _ in range(2):
        for eom in eoms:
            general = copy.copy(eom)
            general.flags = eom.flags & 3
            y0 = rs.normal(size=(700, 1, eom.size)) + 1j * rs.normal(size=(700, 1, eom.size))
            y0 = torch.as_tensor(y0).to(dev)
            a, sa = _native.zofe_propagate(eom, y0, nsub, h)
            b, sb = _native.zofe_propagate(general, y0, nsub, h)
            assert int(sa.item()) == int(sb.item()) == 0
            # four stages, sums of fewer than 100 products in another order
            assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


@pytest.mark.parametrize('sites,modes,subspace', [(5, 2, 'ge'), (6, 1, 'ge')])
def test_crowded_batches_of_few_modes(gpu, sites, modes, subspace):
    """Many right-hand sides of six and seven states with few modes take the
    element-wise kernel (bit by bit), fewer the column form (to rounding)."""
    eom = _eom(sites, modes, subspace)
    general = copy.copy(eom)
    general.flags = eom.flags & 3
    dev = eom.H.device
    rs = np.random.RandomState(7)
    nsub = torch.tensor([2], dtype=torch.int32, device=dev)
    h = torch.tensor([0.4], dtype=torch.float64, device=dev)
    for members in (300, 800):
        y0 = rs.normal(size=(members, 1, eom.size)) + 1j * rs.normal(size=(members, 1, eom.size))
        y0 = torch.as_tensor(y0).to(dev)
        a, sa = _native.zofe_propagate(eom, y0, nsub, h)
        b, sb = _native.zofe_propagate(general, y0, nsub, h)
        assert int(sa.item()) == int(sb.item()) == 0
        assert torch.equal(a, b) if members == 800 else \
            float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
