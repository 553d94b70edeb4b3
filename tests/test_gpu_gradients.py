"""Reverse mode on the GPU: the adjoint propagation kernel against torch's
autograd of the same recursion (CPU, complex128), the RK4-propagator VJP,
and gradients of ensemble absorption spectra with respect to site energies,
couplings and the reorganization energy against central finite differences
of the GPU forward pass and of the oracle."""
import numpy as np
import pytest
import torch

import qspectra_amd as qa
from qspectra_amd import _native
from qspectra_amd import gradients as G
from qspectra_amd import workloads as W
from oracle import system as S
from oracle import liouville as Lv
from oracle import propagate as P
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

BATH = (S.CM_K * 77, 35.0, 106.0)


def _cplx(rng, *shape):
    return rng.normal(size=shape) + 1j * rng.normal(size=shape)


def _cpu_loop(A, y0, nsub):
    """states [B, R, nsave, M] of y <- A y by plain torch (CPU autograd)."""
    outs, y = [], y0
    for n in nsub:
        for _ in range(int(n)):
            y = torch.einsum('bij,brj->bri', A, y)
        outs.append(y)
    return torch.stack(outs, dim=2)


@pytest.mark.parametrize('M,B,R,shared', [(5, 3, 2, False), (7, 4, 1, True), (13, 2, 3, False),
                                          (24, 2, 1, False), (49, 1, 2, False),
                                          (100, 1, 2, False), (147, 2, 1, True)])
def test_adjoint_kernel_matches_autograd(gpu, M, B, R, shared):
    rng = np.random.RandomState(M)
    A = _cplx(rng, 1 if shared else B, M, M)
    A = A / np.abs(np.linalg.eigvals(A)).max(axis=-1)[:, None, None] * 0.98
    y0 = _cplx(rng, B, R, M)
    nsub = np.array([0, 3, 1, 0, 5, 2, 7, 1])
    w = _cplx(rng, B, R, len(nsub), M)
    At = torch.tensor(A, requires_grad=True)
    yt = torch.tensor(y0, requires_grad=True)
    ref = _cpu_loop(At.expand(B, M, M) if shared else At, yt, nsub)
    (ref * torch.as_tensor(w)).real.sum().backward()
    for ckpt in (1, 3, 4, 64):
        Ad = torch.tensor(A, device='cuda', requires_grad=True)
        yd = torch.tensor(y0, device='cuda', requires_grad=True)
        out = G.propagate(Ad, yd, nsub, ckpt=ckpt)
        assert rel_err(out.detach().cpu().numpy(), ref.detach().numpy()) < 1e-12
        (out * torch.as_tensor(w, device='cuda')).real.sum().backward()
        assert rel_err(Ad.grad.cpu().numpy(), At.grad.numpy()) < 1e-11, ckpt
        assert rel_err(yd.grad.cpu().numpy(), yt.grad.numpy()) < 1e-11, ckpt


def test_adjoint_rejects_oversized_block_and_short_workspace(gpu):
    A = torch.zeros((1, 161, 161), dtype=torch.complex128, device='cuda')
    y0 = torch.zeros((1, 1, 161), dtype=torch.complex128, device='cuda')
    n = torch.ones(2, dtype=torch.int32, device='cuda')
    g = torch.zeros((1, 1, 2, 161), dtype=torch.complex128, device='cuda')
    with pytest.raises(_native.NativeError):
        _native.propagate_adjoint(A, y0, n, 2, g)
    # checkpoints that do not fit the workspace set status 2 (no access beyond
    # it), in the register-resident and in the large-block kernel
    for M in (4, 100):
        A = torch.eye(M, dtype=torch.complex128, device='cuda')[None]
        y0 = torch.ones((1, 1, M), dtype=torch.complex128, device='cuda')
        n = torch.tensor([0, 40, 40], dtype=torch.int32, device='cuda')
        g = torch.ones((1, 1, 3, M), dtype=torch.complex128, device='cuda')
        _, _, st = _native.propagate_adjoint(A, y0, n, 8, g, ckpt=4)   # sized for 8 steps
        assert int(st.item()) == 2, M


def test_rk4_propagator_vjp(gpu):
    rng = np.random.RandomState(3)
    L = _cplx(rng, 3, 9, 9) * 0.1
    h = 0.7
    Gw = _cplx(rng, 3, 9, 9)
    Lt = torch.tensor(L, requires_grad=True)
    X = h * Lt
    I = torch.eye(9, dtype=torch.complex128)
    Pt = I + X + X @ X / 2 + X @ X @ X / 6 + X @ X @ X @ X / 24
    (Pt * torch.as_tensor(Gw)).real.sum().backward()
    Ld = torch.tensor(L, device='cuda', requires_grad=True)
    Pd = G.rk4_propagator(Ld, h)
    assert rel_err(Pd.detach().cpu().numpy(), Pt.detach().numpy()) < 1e-13
    (Pd * torch.as_tensor(Gw, device='cuda')).real.sum().backward()
    assert rel_err(Ld.grad.cpu().numpy(), Lt.grad.numpy()) < 1e-12


def _aggregate7():
    from qspectra_amd import workloads as W
    H, d, _ = W.aggregate7_hamiltonian()
    return H, d


def _theta(H):
    iu = np.triu_indices(len(H), 1)
    mk = lambda a: torch.tensor(np.array(a, dtype=float), device='cuda', requires_grad=True)
    return mk(np.diag(H)), mk(H[iu]), mk(BATH[1])


def _spec(d, size, steps, **kw):
    return G.RedfieldAbsorption(d, BATH[2], BATH[0], 12450.0, steps * 1.0, 1.0,
                                disorder=100 / S.GAUSSIAN_SD_FWHM if size else None,
                                ensemble_size=size, random_seed=0, **kw)


def test_absorption_forward_matches_product_path_and_oracle(gpu):
    H, d = _aggregate7()
    spec = _spec(d, 6, 384)
    E, J, lam = _theta(H)
    f, Sg = spec(E, J, lam)
    ham = qa.ElectronicHamiltonian(H, bath=qa.DebyeBath(*BATH), dipoles=d,
                                   disorder=100 / S.GAUSSIAN_SD_FWHM)
    members = list(ham.sample_ensemble(6))
    from qspectra_amd.batched import absorption_batch
    fb, Xb = absorption_batch(members, 384.0, rw_freq=12450.0, dt=1.0,
                              model_kwargs=dict(secular=False))
    assert np.allclose(f, fb) and rel_err(Sg.detach().cpu().numpy(), Xb.mean(0)) < 1e-12

    class _FixedStep(Lv.LiouvilleModel):
        time_step = 1.0
    ref = 0
    for h in members:
        om = _FixedStep(S.ElectronicHamiltonian(h.H_1exc, bath=S.DebyeBath(*BATH), dipoles=d),
                        rw_freq=12450.0, hilbert_subspace='ge', unit_convert=S.CM_FS,
                        secular=False)
        ref = ref + P.absorption_spectra(om, 384.0, dt=1.0)[1] / len(members)
    assert rel_err(Sg.detach().cpu().numpy(), ref) < 1e-10


def _loss_fn(spec, target):
    def loss(E, J, lam):
        return ((spec(E, J, lam)[1] - target) ** 2).sum()
    return loss


def test_absorption_gradient_matches_finite_differences(gpu):
    """All 29 parameters (7 E, 21 J, lam) of an 8-member ensemble, 1024 RK4
    steps with checkpoints every 64; central differences with h = 1e-3 cm^-1
    of the FP64 forward pass."""
    H, d = _aggregate7()
    spec = _spec(d, 8, 1024, ckpt=64)
    rng = np.random.RandomState(3)
    Ht = H.copy()
    Ht[np.diag_indices(7)] += rng.uniform(-50, 50, 7)
    iu = np.triu_indices(7, 1)
    dJ = rng.uniform(-10, 10, len(iu[0]))
    Ht[iu] += dJ
    Ht[iu[1], iu[0]] += dJ
    Et, Jt, lt = _theta(Ht)
    with torch.no_grad():
        target = spec(Et, Jt, lt + rng.uniform(-5, 5))[1]
    loss = _loss_fn(spec, target)
    E, J, lam = _theta(H)
    loss(E, J, lam).backward()
    grad = torch.cat([E.grad, J.grad, lam.grad[None]]).cpu().numpy()
    theta0 = [E.detach(), J.detach(), lam.detach()]
    fd = []
    h = 1e-3
    with torch.no_grad():
        for which, t in enumerate(theta0):
            for i in range(t.numel()):
                val = []
                for sgn in (1, -1):
                    th = [x.clone() for x in theta0]
                    th[which].reshape(-1)[i] += sgn * h
                    val.append(float(loss(*th)))
                fd.append((val[0] - val[1]) / (2 * h))
    fd = np.array(fd)
    err = np.abs(grad - fd).max() / np.abs(fd).max()
    assert err < 1e-5, err


def test_absorption_gradient_matches_oracle_differences(gpu):
    """Site-energy and lam gradients against central differences of the
    oracle's absorption spectra (the reference algorithm, RK4 at the same
    step), 3 members, 256 steps."""
    H, d = _aggregate7()
    spec = _spec(d, 3, 256)
    shifts = spec.shifts

    class _FixedStep(Lv.LiouvilleModel):
        time_step = 1.0

    def oracle_spectrum(Hc, lam):
        out = 0
        for n in range(3):
            om = _FixedStep(S.ElectronicHamiltonian(Hc + np.diag(shifts[n]),
                                                    bath=S.DebyeBath(BATH[0], lam, BATH[2]),
                                                    dipoles=d),
                            rw_freq=12450.0, hilbert_subspace='ge', unit_convert=S.CM_FS,
                            secular=False)
            out = out + P.absorption_spectra(om, 256.0, dt=1.0)[1] / 3
        return out

    target = oracle_spectrum(H + np.diag(np.linspace(-20, 20, 7)), BATH[1] + 3.0)
    E, J, lam = _theta(H)
    ((spec(E, J, lam)[1] - torch.as_tensor(target, device='cuda')) ** 2).sum().backward()
    h = 1e-3
    for i in (0, 3, 6):
        dH = np.zeros((7, 7))
        dH[i, i] = h
        lp = ((oracle_spectrum(H + dH, BATH[1]) - target) ** 2).sum()
        lm = ((oracle_spectrum(H - dH, BATH[1]) - target) ** 2).sum()
        fd = (lp - lm) / (2 * h)
        assert abs(float(E.grad[i]) - fd) <= 1e-5 * abs(fd), i
    lp = ((oracle_spectrum(H, BATH[1] + h) - target) ** 2).sum()
    lm = ((oracle_spectrum(H, BATH[1] - h) - target) ** 2).sum()
    fd = (lp - lm) / (2 * h)
    assert abs(float(lam.grad) - fd) <= 1e-5 * abs(fd)


def _sym_h(n, B, seed):
    rng = np.random.RandomState(seed)
    H = rng.normal(0.0, 60.0, (B, n, n))
    H = (H + H.transpose(0, 2, 1)) / 2
    for b in range(B):
        H[b][np.diag_indices(n)] = rng.uniform(12200, 12700, n)
    return H


def _flags(secular=False, real=False, heis=False, eigen=False):
    return ((_native.QSX_SECULAR if secular else 0) | (_native.QSX_REAL_CORR if real else 0)
            | (_native.QSX_HEISENBERG if heis else 0) | (_native.QSX_EIGEN_BASIS if eigen else 0))


@pytest.mark.parametrize('X,Y', [(1, 0), (0, 1), (1, 1), (0, 0)])
@pytest.mark.parametrize('secular,real,heis', [(False, False, False), (True, False, True),
                                               (False, True, True), (True, True, False)])
def test_redfield_vjp_matches_torch_autograd(gpu, X, Y, secular, real, heis):
    """qsx_redfield_block_vjp against torch's autograd through the torch
    restatement of the block (eigh, C(w), tensor, basis change) on the CPU:
    the symmetric part of dl/dH1 and dl/dlam, 1e-9 relative."""
    from tests import torch_redfield as TR
    n, B = 5, 3
    H = _sym_h(n, B, 7 + X + 2 * Y)
    rw = np.array([12450.0, 12380.0, 12510.0])
    rng = np.random.RandomState(11)
    flags = _flags(secular, real, heis)
    Hd = torch.as_tensor(H).cuda()
    rwd = torch.as_tensor(rw).cuda()
    L = _native.redfield_block(Hd, rwd, BATH[0], BATH[1], BATH[2], X, Y, flags, S.CM_FS)
    gL = torch.as_tensor(_cplx(rng, *L.shape)).cuda()
    gH, glam = _native.redfield_block_vjp(Hd, rwd, BATH[0], BATH[1], BATH[2], X, Y, flags,
                                          S.CM_FS, gL)
    gH, glam = gH.cpu().numpy(), glam.cpu().numpy()
    for b in range(B):
        Ht = torch.tensor(H[b:b + 1], requires_grad=True)
        lam = torch.tensor(BATH[1], dtype=torch.float64, requires_grad=True)
        Lt = TR.redfield_block(Ht, lam, BATH[2], BATH[0], rw[b], 'ge'[X], 'ge'[Y], secular,
                               real, S.CM_FS)
        if heis:
            Lt = Lt.transpose(-1, -2)
        assert rel_err(L[b].cpu().numpy(), Lt[0].detach().numpy()) < 1e-12
        loss = (torch.conj(gL[b:b + 1].cpu()) * Lt).real.sum()
        loss.backward()
        # the g block does not depend on H1 (and 'gg' on nothing)
        ref = Ht.grad[0].numpy() if Ht.grad is not None else np.zeros((n, n))
        ref = (ref + ref.T) / 2
        ref_lam = float(lam.grad) if lam.grad is not None else 0.0
        scale = max(np.abs(ref).max(), 1e-300)
        if X or Y:
            assert np.abs(gH[b] - ref).max() / scale < 1e-9, (b, np.abs(gH[b] - ref).max(), scale)
        else:
            assert np.abs(gH[b]).max() == 0.0
        assert abs(glam[b] - ref_lam) <= 1e-9 * abs(ref_lam), b


@pytest.mark.parametrize('X,Y,secular,heis,eigen', [
    (2, 1, False, True, False), (2, 1, True, False, False), (1, 2, False, False, True),
    (2, 2, False, False, False), (2, 2, True, True, False), (1, 1, False, False, True),
    (2, 0, False, True, False), (1, 0, False, False, True)])
def test_redfield_vjp_matches_finite_differences(gpu, X, Y, secular, heis, eigen):
    """Blocks with the two-exciton space, the secular mask and the eigen
    basis: dl/dH1 along symmetric directions and dl/dlam against central
    differences (h = 1e-3 cm^-1, 1e-4 for lam) of the GPU forward pass."""
    n, B = 4, 2
    H = _sym_h(n, B, 3 + X + 3 * Y)
    rwd = torch.as_tensor(np.array([12450.0, 12400.0])).cuda()
    flags = _flags(secular, False, heis, eigen)
    rng = np.random.RandomState(5)

    def block(Hn, lam=BATH[1]):
        return _native.redfield_block(torch.as_tensor(Hn).cuda(), rwd, BATH[0], lam, BATH[2],
                                      X, Y, flags, S.CM_FS)
    L0 = block(H)
    gL = torch.as_tensor(_cplx(rng, *L0.shape)).cuda()
    gH, glam = _native.redfield_block_vjp(torch.as_tensor(H).cuda(), rwd, BATH[0], BATH[1],
                                          BATH[2], X, Y, flags, S.CM_FS, gL)
    gH, glam = gH.cpu().numpy(), glam.cpu().numpy()

    def loss(Hn, lam=BATH[1]):
        return (torch.conj(gL) * block(Hn, lam)).real.sum(dim=(1, 2)).cpu().numpy()
    h = 1e-3
    for (p, q) in [(0, 0), (1, 2), (0, 3), (3, 3), (2, 1)]:
        D = np.zeros((n, n))
        D[p, q] = D[q, p] = 1.0
        fd = (loss(H + h * D) - loss(H - h * D)) / (2 * h)
        an = (gH * D).sum(axis=(1, 2))
        scale = np.abs(gH).max(axis=(1, 2))
        assert np.all(np.abs(fd - an) <= 1e-6 * scale), (p, q, fd, an)
    fdl = (loss(H, BATH[1] + 1e-4) - loss(H, BATH[1] - 1e-4)) / 2e-4
    assert np.all(np.abs(fdl - glam) <= 1e-6 * np.abs(fdl)), (fdl, glam)


@pytest.mark.parametrize('n', [1, 2, 12, 13, 17, 33])
def test_records_across_widths(gpu, n):
    """Block records over the lanes per Matsubara sum (16 down to 1, pairs
    in several trips) and both work-group widths (the line lies at 12
    states): block eg and its cotangents against the torch restatement, with
    the bounds of the comparison above."""
    from tests import torch_redfield as TR
    H = _sym_h(n, 2, n)
    rw = np.array([12450.0, 12380.0])
    rng = np.random.RandomState(n)
    Hd, rwd = torch.as_tensor(H).cuda(), torch.as_tensor(rw).cuda()
    L = _native.redfield_block(Hd, rwd, *BATH, 1, 0, 0, S.CM_FS)
    gL = torch.as_tensor(_cplx(rng, *L.shape)).cuda()
    gH, glam = _native.redfield_block_vjp(Hd, rwd, *BATH, 1, 0, 0, S.CM_FS, gL)
    for b in range(2):
        Ht = torch.tensor(H[b:b + 1], requires_grad=True)
        lam = torch.tensor(BATH[1], dtype=torch.float64, requires_grad=True)
        Lt = TR.redfield_block(Ht, lam, BATH[2], BATH[0], rw[b], 'e', 'g', False, False, S.CM_FS)
        assert rel_err(L[b].cpu().numpy(), Lt[0].detach().numpy()) < 1e-12
        (torch.conj(gL[b:b + 1].cpu()) * Lt).real.sum().backward()
        ref = (Ht.grad[0] + Ht.grad[0].T).numpy() / 2
        assert np.abs(gH[b].cpu().numpy() - ref).max() < 1e-9 * np.abs(ref).max()
        assert abs(float(glam[b]) - float(lam.grad)) < 1e-9 * abs(float(lam.grad))


def test_signal_vector_keeps_its_gradient(gpu):
    """A signal vector that is differentiated is contracted with the states:
    its gradient equals that of the explicit contraction."""
    H, d, _ = W.aggregate7_hamiltonian()
    spec = G.RedfieldAbsorption(d, 106.0, BATH[0], 12450.0, 200.0, 1.0)
    E = torch.tensor(np.diag(H).copy(), device='cuda')
    J = torch.tensor(H[np.triu_indices(7, 1)], device='cuda')
    plain = spec.signal(E, J, 35.0)
    spec.v = spec.v.clone().requires_grad_(True)
    x = spec.signal(E, J, 35.0)
    assert rel_err(x.detach().cpu().numpy(), plain.cpu().numpy()) < 1e-12
    (x.abs() ** 2).sum().backward()
    P = G.rk4_propagator(spec.liouvillian(spec.hamiltonians(E, J), 35.0), spec.dt)
    y = G.propagate(P, spec.y0, spec.nsub)[0, 0]
    want = 2 * (y.conj() * x.detach()[:, None]).sum(dim=0)
    assert rel_err(spec.v.grad.cpu().numpy(), want.cpu().numpy()) < 1e-12
