"""Parity of the HEOM kernels (qsx_heom_apply / qsx_heom_propagate) with the
reference's sparse hierarchy generator (golden CSR matrices) and its
tight-tolerance zvode trajectory.

FP64: the right-hand side to 1e-13 relative; RK4 trajectories against the
oracle's RK4 on the same CSR and schedule to 1e-11; against zvode at the RK4
truncation error of the step used.  MIXED (complex64 stage vectors): 1e-5.
"""
import numpy as np
import pytest
import torch

import qspectra_amd as qa
from qspectra_amd import _native
from oracle import propagate as P
from tests.conftest import golden, golden_csr, rel_err

pytestmark = pytest.mark.gpu


def _model(name='redfield_dimer', T=qa.CM_K * 300, rw=12800.0, **kw):
    g = golden(name)
    ham = qa.ElectronicHamiltonian(g['in_H1'], bath=qa.DebyeBath(T, 35, 106),
                                   dipoles=g['in_dipoles'], energy_spread_extra=float(g['extra']),
                                   disorder=100 / qa.GAUSSIAN_SD_FWHM)
    kw.setdefault('level_cutoff', 3)
    kw.setdefault('K', 1)
    return qa.HEOMModel(ham, rw_freq=rw, hilbert_subspace='ge', unit_convert=qa.CM_FS, **kw)


@pytest.mark.parametrize('name,kw', [('dimer', dict(level_cutoff=3, K=1)),
                                     ('dimer_mod', dict(level_cutoff=3, K=1, modified_HEOM=True)),
                                     ('dimer_nolt', dict(level_cutoff=3, K=2,
                                                         low_temp_corr=False))])
def test_heom_rhs_matches_reference(gpu, name, kw):
    gh = golden('heom')
    m = _model(**kw)
    rs = np.random.RandomState(0)
    for s in ('ee', 'gg,ge,eg,ee', 'eg'):
        L = golden_csr(gh, '%s_%s' % (name, s.replace(',', '_')))
        y = rs.randn(L.shape[0]) + 1j * rs.randn(L.shape[0])
        for heis in (False, True):
            eom = m.equation_of_motion(s, heisenberg_picture=heis)
            ref = (L.T if heis else L) @ y
            assert rel_err(eom(0, y), ref) < 1e-13, (name, s, heis)


def test_heom_propagation_matches_oracle_rk4(gpu):
    gh = golden('heom')
    m = _model()
    for s, key in (('ee', 'dimer_ee'), ('gg,ge,eg,ee', 'dimer_gg_ge_eg_ee')):
        L = golden_csr(gh, key)
        eom = m.equation_of_motion(s)
        y0 = np.zeros(L.shape[0], complex)
        y0[:eom.M] = np.random.RandomState(1).randn(eom.M)
        t = np.arange(0, 60.0, 2.0)
        ref = P.integrate_rk4(L, y0, t, dt=0.5)
        got = qa.integrate(eom, y0, t, dt=0.5)
        assert got.shape == ref.shape
        assert rel_err(got, ref) < 1e-11, s
        gm = qa.integrate(eom, y0, t, dt=0.5, precision='mixed')
        assert rel_err(gm, ref) < 1e-5, s


def test_heom_dynamics_matches_reference_zvode(gpu):
    gh = golden('heom')
    m = _model()
    rho0 = np.zeros((2, 2))
    rho0[0, 0] = 1
    t, rho = qa.simulate_dynamics(m, rho0, times=gh['dyn_t'], dt=float(gh['dyn_time_step']) / 8)
    ref = gh['dyn_y'][:, :4].reshape(-1, 2, 2, order='F')
    assert rel_err(rho, ref) < 1e-6
    # the default step (calibrated by probe runs to rtol = 1e-6 over the span)
    t, rho = qa.simulate_dynamics(m, rho0, times=gh['dyn_t'])
    assert rel_err(rho, ref) < 1e-5
    # 7-site hierarchy (level_cutoff 3): RK4 against the oracle on the golden CSR
    g7 = golden('redfield_7site')
    m7 = _model('redfield_7site', rw=float(gh['agg7_rw_freq']))
    L7 = golden_csr(gh, 'agg7_ee')
    rho0 = np.zeros((7, 7))
    rho0[0, 0] = 1
    t = np.arange(0, 40.0, 0.5)
    _, rho = qa.simulate_dynamics(m7, rho0, times=t, dt=0.5)
    y0 = np.zeros(L7.shape[0], complex)
    y0[0] = 1
    ref = P.integrate_rk4(L7, y0, t, dt=0.5)[:, :49].reshape(-1, 7, 7, order='F')
    assert rel_err(rho, ref) < 1e-11


def test_heom_ensemble_batch_one_launch(gpu):
    """8 disorder samples in one launch (XCD-mapped tiles) vs one at a time."""
    m = _model('redfield_7site', rw=float(golden('heom')['agg7_rw_freq']))
    rho0 = np.zeros((7, 7))
    rho0[2, 2] = 1
    t = np.arange(0, 20.0, 0.5)
    hams = [m.hamiltonian.sample(n) for n in range(8)]
    mb = m.with_hamiltonians(hams)
    eom = mb.equation_of_motion('ee')
    assert eom.batch == 8
    y0 = np.zeros((8, eom.size), complex)
    y0[:, :49] = rho0.reshape(-1, order='F')
    got = qa.integrate(eom, y0, t, dt=0.5)
    for n in range(8):
        single = _model('redfield_7site', rw=float(golden('heom')['agg7_rw_freq']))
        single.hamiltonian = hams[n]
        e1 = single.equation_of_motion('ee')
        ref = qa.integrate(e1, y0[n], t, dt=0.5)
        assert rel_err(got[n], ref) < 1e-13, n
    _, avg = qa.simulate_dynamics(m, rho0, times=t, ensemble_size=8, dt=0.5)
    assert rel_err(avg, got[:, :, :49].mean(axis=0).reshape(-1, 7, 7, order='F')) < 1e-12


@pytest.mark.parametrize('per_pass', ['3', '8', '0'])
def test_heom_sample_passes_match_one_pass(gpu, monkeypatch, per_pass):
    """Samples propagated in passes of a few (each pass runs all its steps
    before the next starts) equal the single pass over all samples, FP64 and
    MIXED, with an uneven last pass."""
    m = _model('redfield_7site', rw=float(golden('heom')['agg7_rw_freq']), level_cutoff=2)
    rho0 = np.zeros((7, 7))
    rho0[1, 1] = 1
    t = np.arange(0, 10.0, 0.5)
    mb = m.with_hamiltonians([m.hamiltonian.sample(n) for n in range(11)])
    eom = mb.equation_of_motion('ee')
    y0 = np.zeros((11, eom.size), complex)
    y0[:, :49] = rho0.reshape(-1, order='F')
    for prec in ('fp64', 'mixed'):
        monkeypatch.setenv('QSX_HEOM_SAMPLES_PER_PASS', '0')
        ref = qa.integrate(eom, y0, t, dt=0.5, precision=prec)
        monkeypatch.setenv('QSX_HEOM_SAMPLES_PER_PASS', per_pass)
        got = qa.integrate(eom, y0, t, dt=0.5, precision=prec)
        assert np.array_equal(got, ref), (prec, per_pass)


def _spectra_models(**kw):
    from oracle import system as S, liouville as Lv
    g = golden('redfield_dimer')
    hp = qa.ElectronicHamiltonian(g['in_H1'], bath=qa.DebyeBath(qa.CM_K * 77, 35, 106),
                                  dipoles=g['in_dipoles'], energy_spread_extra=float(g['extra']))
    ho = S.ElectronicHamiltonian(g['in_H1'], bath=S.DebyeBath(S.CM_K * 77, 35, 106),
                                 dipoles=g['in_dipoles'], energy_spread_extra=float(g['extra']))
    return (qa.HEOMModel(hp, hilbert_subspace='gef', unit_convert=qa.CM_FS, **kw),
            Lv.HEOMOracleModel(ho, hilbert_subspace='gef', unit_convert=S.CM_FS, **kw))


@pytest.mark.parametrize('name,kw', [('lt', dict(level_cutoff=3, K=1)),
                                     ('nolt', dict(level_cutoff=3, K=1, low_temp_corr=False))])
def test_heom_third_order_matches_oracle_and_reference(gpu, name, kw, monkeypatch):
    """HEOM third-order responses (the hierarchy through t1 and t2, per-ADO
    dipoles, Heisenberg t3): the dense-generator path and the stage-kernel
    path against the oracle's RK4 on the same schedule (FP64 1e-10) and the
    reference's tight zvode (tests/golden/heom_spectra.npz, 1e-7 at 1/8 of
    the model step); mixed 1e-6."""
    from qspectra_amd.simulate import response
    g = golden('heom_spectra')
    mp, mo = _spectra_models(**kw)
    dt = float(g['time_step']) / 8
    for geom in ('-++', '++-'):
        key = '%s_R3_%s' % (name, geom.replace('-', 'm').replace('+', 'p'))
        (t1, t2, t3), R = qa.third_order_response(mp, 8.5, population_times=[0., 3., 7.],
                                                  geometry=geom, dt=dt)
        _, Ro = P.third_order_response(mo, 8.5, population_times=[0., 3., 7.], geometry=geom,
                                       dt=dt)
        np.testing.assert_allclose(t1, g['t1'])
        assert rel_err(R, Ro) < 1e-10, key
        assert rel_err(R, g[key]) < 1e-7, key
        _, Rm = qa.third_order_response(mp, 8.5, population_times=[0., 3., 7.], geometry=geom,
                                        dt=dt, precision='mixed')
        assert rel_err(Rm, Ro) < 1e-6, key
        monkeypatch.setattr(response, 'HEOM_DENSE_MAX', 0)       # stage-kernel path
        _, Rk = qa.third_order_response(mp, 8.5, population_times=[0., 3., 7.], geometry=geom,
                                        dt=dt)
        monkeypatch.undo()
        assert rel_err(Rk, Ro) < 1e-10, key
    f, X = qa.absorption_spectra(mp, 150.5, dt=dt)
    np.testing.assert_allclose(f, g[name + '_abs_f'])
    assert rel_err(X, g[name + '_abs_X']) < 1e-7
    # default steps: the dense-generator path (rate-bound step) and the stage
    # kernel (calibrated step) against the tight zvode outputs
    key = '%s_R3_mpp' % name
    _, Rd = qa.third_order_response(mp, 8.5, population_times=[0., 3., 7.])
    assert rel_err(Rd, g[key]) < 1e-5
    monkeypatch.setattr(response, 'HEOM_DENSE_MAX', 0)
    _, Rk = qa.third_order_response(mp, 8.5, population_times=[0., 3., 7.])
    monkeypatch.undo()
    assert rel_err(Rk, g[key]) < 1e-5
    (f1, t2, f3), X2 = qa.two_dimensional_spectra(mp, 8.5, population_times=[0., 3.], dt=dt)
    assert X2.shape == (len(f1), 2, len(f3)) and np.isfinite(X2).all()


def test_heom_rectangular_commutator_blocks(gpu, monkeypatch):
    """Single Liouville blocks XY with X != Y through the commutator form
    -i unit (H_X rho - rho H_Y): forced on the dimer's 'eg' block against
    the reference's CSR generator, and the 7-site 'fe' block (M = 147, above
    the dense-block limit) against the oracle's sparse generator, in both
    pictures (RHS 1e-13)."""
    from qspectra_amd.dynamics import heom as heom_mod
    from oracle import system as S
    from oracle import liouville as Lv
    gh = golden('heom')
    rs = np.random.RandomState(4)
    monkeypatch.setattr(heom_mod, 'DENSE_BLOCK_MAX', 0)
    m = _model()
    L = golden_csr(gh, 'dimer_eg')
    y = rs.randn(L.shape[0]) + 1j * rs.randn(L.shape[0])
    for heis in (False, True):
        eom = m.equation_of_motion('eg', heisenberg_picture=heis)
        assert eom.n_comm == 2
        assert rel_err(eom(0, y), (L.T if heis else L) @ y) < 1e-13, heis
    monkeypatch.undo()
    g7 = golden('redfield_7site')
    hp = qa.ElectronicHamiltonian(g7['in_H1'], bath=qa.DebyeBath(qa.CM_K * 300, 35, 106),
                                  dipoles=g7['in_dipoles'])
    ho = S.ElectronicHamiltonian(g7['in_H1'], bath=S.DebyeBath(S.CM_K * 300, 35, 106),
                                 dipoles=g7['in_dipoles']).in_rotating_frame(12400.0)
    mp = qa.HEOMModel(hp, rw_freq=12400.0, hilbert_subspace='gef', unit_convert=qa.CM_FS,
                      level_cutoff=2, K=1)
    for heis in (False, True):
        Lo = Lv.heom_evolve_matrix(ho, 'gef', 'fe', S.CM_FS, K=1, level_cutoff=2,
                                   heisenberg_picture=heis)
        eom = mp.equation_of_motion('fe', heisenberg_picture=heis)
        assert eom.M == 147 and eom.n_comm == 21
        y = rs.randn(Lo.shape[0]) + 1j * rs.randn(Lo.shape[0])
        assert rel_err(eom(0, y), Lo @ y) < 1e-13, heis


def test_heom_7site_esa_third_order_matches_oracle(gpu):
    """ESA pathways of a 7-site HEOM model (Heisenberg t3 in the 147-element
    'fe' block on the stage kernel) against the oracle's RK4 on the same
    schedule (FP64 1e-10)."""
    from oracle import system as S
    from oracle import liouville as Lv
    g7 = golden('redfield_7site')
    extra = float(g7['extra'])
    hp = qa.ElectronicHamiltonian(g7['in_H1'], bath=qa.DebyeBath(qa.CM_K * 300, 35, 106),
                                  dipoles=g7['in_dipoles'], energy_spread_extra=extra)
    ho = S.ElectronicHamiltonian(g7['in_H1'], bath=S.DebyeBath(S.CM_K * 300, 35, 106),
                                 dipoles=g7['in_dipoles'], energy_spread_extra=extra)
    mp = qa.HEOMModel(hp, hilbert_subspace='gef', unit_convert=qa.CM_FS, level_cutoff=2, K=1)
    mo = Lv.HEOMOracleModel(ho, hilbert_subspace='gef', unit_convert=S.CM_FS, level_cutoff=2,
                            K=1)
    dt = mp.time_step / 4
    kw = dict(population_times=[0., 3.], geometry='-++', include_signal='ESA')
    (t1, t2, t3), R = qa.third_order_response(mp, 5.5, dt=dt, **kw)
    _, Ro = P.third_order_response(mo, 5.5, dt=dt, **kw)
    assert R.shape == (len(t1), 2, len(t3)) and len(t1) >= 2
    assert rel_err(R, Ro) < 1e-10


def test_heom_fields_match_oracle_and_reference(gpu):
    """simulate_pump / simulate_with_fields of a HEOM model (the dipole
    commutators on every ADO, eom.py:79-103 with heom.py:22-58): FP64 against
    the oracle's time-dependent RK4 on the same schedule (1e-10), MIXED 1e-6,
    and the default step against the reference's tight zvode hierarchy
    states (tests/golden/heom_fields.npz, 1e-5)."""
    from oracle import system as S, liouville as Lv
    g = golden('heom_fields')
    gd = golden('redfield_dimer')
    hp = qa.ElectronicHamiltonian(gd['in_H1'], bath=qa.DebyeBath(qa.CM_K * 77, 35, 106),
                                  dipoles=gd['in_dipoles'], energy_spread_extra=float(gd['extra']))
    ho = S.ElectronicHamiltonian(gd['in_H1'], bath=S.DebyeBath(S.CM_K * 77, 35, 106),
                                 dipoles=gd['in_dipoles'], energy_spread_extra=float(gd['extra']))
    mp = qa.HEOMModel(hp, hilbert_subspace='gef', unit_convert=qa.CM_FS, level_cutoff=3, K=1)
    mo = Lv.HEOMOracleModel(ho, hilbert_subspace='gef', unit_convert=S.CM_FS, level_cutoff=3, K=1)
    assert abs(mp.time_step - float(g['time_step'])) < 1e-12
    pp = qa.GaussianPulse(12750., 20., t_peak=0., scale=0.02, freq_convert=qa.CM_FS)
    po = S.GaussianPulse(12750., 20., t_peak=0., scale=0.02, freq_convert=S.CM_FS)
    dt = mp.time_step / 4
    t, y = qa.simulate_pump(mp, pp, 'x', time_extra=30., dt=dt)
    to, yo = P.simulate_pump(mo, po, 'x', time_extra=30., dt=dt)
    np.testing.assert_allclose(t, to)
    assert np.asarray(y).shape == yo.shape
    assert rel_err(np.asarray(y), yo) < 1e-10
    _, ym = qa.simulate_pump(mp, pp, 'x', time_extra=30., dt=dt, precision='mixed')
    assert rel_err(np.asarray(ym), yo) < 1e-6
    t, y = qa.simulate_pump(mp, pp, 'x', time_extra=30.)          # default step
    np.testing.assert_allclose(t, g['pump_t'])
    assert rel_err(np.asarray(y), g['pump_y']) < 1e-5
    p1 = qa.GaussianPulse(12700., 15., t_peak=-10., scale=0.015, freq_convert=qa.CM_FS)
    p2 = qa.GaussianPulse(12900., 25., t_peak=5., scale=0.01 * np.exp(0.6j),
                          freq_convert=qa.CM_FS, t_limits_multiple=2.5)
    t, y = qa.simulate_with_fields(mp, [p1, p2], '-+', 'xy', times=[0., 4., 10.])
    np.testing.assert_allclose(t, g['two_t'])
    assert rel_err(np.asarray(y), g['two_y']) < 1e-5
    # one Liouville block: the field term vanishes, the hierarchy evolves freely
    t, y = qa.simulate_pump(mp, pp, 'x', time_extra=10., liouville_subspace='gg', dt=dt)
    to, yo = P.simulate_pump(mo, po, 'x', time_extra=10., liouville_subspace='gg', dt=dt)
    assert rel_err(np.asarray(y), yo) < 1e-10


def test_ensemble_of_a_model_that_has_been_used(gpu):
    """The ensemble average does not depend on whether the model has
    propagated its own Hamiltonian before."""
    rho0 = np.zeros((2, 2))
    rho0[1, 1] = 1
    t = np.arange(0, 20.0, 1.0)
    out = []
    for used in (False, True):
        ham = qa.ElectronicHamiltonian(np.array([[12000., 50.], [50., 12100.]]),
                                       bath=qa.DebyeBath(53.5, 35., 106.), dipoles=np.eye(2, 3),
                                       disorder=100., random_seed=0)
        m = qa.HEOMModel(ham, rw_freq=12000., hilbert_subspace='ge', unit_convert=qa.CM_FS,
                         level_cutoff=3, K=1)
        if used:
            qa.simulate_dynamics(m, rho0, times=t, dt=0.5)
        out.append(qa.simulate_dynamics(m, rho0, times=t, ensemble_size=3, dt=0.5)[1])
    assert np.array_equal(*out)


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_heom_propagation_under_capture(gpu, precision):
    """A captured propagation replays the eager one bit by bit, with eager
    work between the replays (the launch shape comes from a host query)."""
    m = _model('redfield_7site', rw=float(golden('heom')['agg7_rw_freq']))
    eom = m.with_hamiltonians([m.hamiltonian.sample(n) for n in range(3)]).equation_of_motion('ee')
    rs = np.random.RandomState(0)
    y0 = torch.as_tensor(rs.normal(size=(3, eom.size)) + 1j * rs.normal(size=(3, eom.size))).cuda()
    mode = _native.QSX_FP64 if precision == 'fp64' else _native.QSX_MIXED

    def go():
        return _native.heom_propagate(eom, y0, [2, 3], [0.5, 0.25], mode)[0]
    want = go()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = go()
    for scale in (1.0, -2.0, 0.5):
        y0.mul_(scale)
        want = go()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
