"""qsx_propagate_pieces and its reverse mode (blocks of at most 16 states,
parallel in time) against the step-by-step recursion: states, signals and
gradients over the smallest and largest blocks, shared and per-member
operators, several right-hand sides, one to several pieces with a partial last
one, saves before the first step, repeated and unevenly spaced saves."""
import numpy as np
import pytest
import torch

from qspectra_amd import _native
from qspectra_amd import gradients as G

pytestmark = pytest.mark.gpu


def _problem(M, B, R, shared, seed):
    rs = np.random.RandomState(seed)
    A = rs.normal(size=(1 if shared else B, M, M)) + 1j * rs.normal(size=(1 if shared else B, M, M))
    A = A / np.abs(np.linalg.eigvals(A)).max(axis=1)[:, None, None] * 0.999
    y0 = rs.normal(size=(B, R, M)) + 1j * rs.normal(size=(B, R, M))
    v = rs.normal(size=M) + 1j * rs.normal(size=M)
    return [torch.as_tensor(x).to('cuda') for x in (A, y0, v)]


def _reference(A, y0, nsub, gout):
    """States, dLoss/dA and dLoss/dy0 of the step-by-step recursion (numpy)."""
    A, y0 = A.cpu().numpy(), y0.cpu().numpy()
    B, R, M = y0.shape
    A = np.broadcast_to(A, (B, M, M))
    ys, out, at = [y0], [], []
    for n in nsub:
        for _ in range(n):
            ys.append(np.einsum('bij,brj->bri', A, ys[-1]))
        out.append(ys[-1])
        at.append(len(ys) - 1)
    lam = np.zeros_like(y0)
    gA = np.zeros((B, R, M, M), dtype=complex)
    p = len(ys) - 1
    for s in reversed(range(len(nsub))):
        while p > at[s]:
            gA += lam[..., :, None] * ys[p - 1].conj()[..., None, :]
            lam = np.einsum('bji,brj->bri', A.conj(), lam)
            p -= 1
        lam = lam + gout[:, :, s]
    while p > 0:
        gA += lam[..., :, None] * ys[p - 1].conj()[..., None, :]
        lam = np.einsum('bji,brj->bri', A.conj(), lam)
        p -= 1
    return np.stack(out, axis=2), gA, lam


def _rel(a, b):
    a = a.detach().cpu().numpy()
    return np.abs(a - b).max() / np.abs(b).max()


SCHEDULES = {
    'ones': [0] + [1] * 200, 'one piece': [8], 'two': [9], 'exact': [0] + [1] * 64,
    'uneven': [0, 0, 3, 0, 70, 1, 1, 0, 0, 40], 'late': [130, 0, 0],
    'no end': [5, 60, 0, 2] + [7] * 30}


@pytest.mark.parametrize('schedule', sorted(SCHEDULES))
@pytest.mark.parametrize('M,B,R,shared', [(1, 3, 1, False), (2, 1, 5, True), (7, 6, 1, False),
                                          (15, 2, 2, True), (16, 3, 3, False)])
def test_pieces_match_steps(gpu, M, B, R, shared, schedule):
    nsub = SCHEDULES[schedule]
    A, y0, v = _problem(M, B, R, shared, M + len(nsub))
    sched = _native.PieceSchedule(nsub, y0.device)
    rs = np.random.RandomState(3)
    ns = len(nsub)
    for signal in ((False, True) if M < 16 else (False,)):
        g = rs.normal(size=(B, R, ns) + (() if signal else (M,))) + 0.5j
        vn = v.cpu().numpy()
        states, gA, gy = _reference(A, y0, nsub, g[..., None] * vn.conj() if signal else g)
        out, Q, Y, status = _native.propagate_pieces(A, y0, sched, v if signal else None)
        # at most 270 products of 16 terms each: 270 x 16 ulp with the block's
        # norm amplification, far below 1e-11
        assert _rel(out, states @ vn if signal else states) <= 1e-11
        assert int(status.item()) == 0
        dA, dy, status = _native.propagate_pieces_adjoint(
            A, y0, sched, Q, Y, torch.as_tensor(g).to(y0.device), v if signal else None)
        assert _rel(dA, gA) <= 1e-11 and _rel(dy, gy) <= 1e-11
        assert int(status.item()) == 0


def test_propagate_uses_pieces_and_keeps_its_gradients(gpu):
    """gradients.propagate: the same states and gradients on both routes."""
    A, y0, _ = _problem(7, 4, 2, True, 9)
    nsub = np.array([0] + [1] * 150)
    got = []
    for limit in (G.PIECE_BYTES, 0):
        before, G.PIECE_BYTES = G.PIECE_BYTES, limit
        try:
            a, y = A.clone().requires_grad_(True), y0.clone().requires_grad_(True)
            states = G.propagate(a, y, nsub)
            (states.abs() ** 2).sum().backward()
        finally:
            G.PIECE_BYTES = before
        got.append((states, a.grad, y.grad))
    for p, q in zip(*got):
        assert _rel(p, q.detach().cpu().numpy()) <= 1e-11


def test_pieces_report_non_finite_states(gpu):
    A, y0, _ = _problem(3, 2, 1, False, 4)
    y0[1, 0, 2] = float('inf')
    sched = _native.PieceSchedule([0] + [1] * 80, y0.device)
    assert int(_native.propagate_pieces(A, y0, sched)[3].item()) == 1
    with pytest.raises(ValueError):
        _native.propagate_pieces(A[:, :2], y0, sched)


@pytest.mark.parametrize('M', [5, 20])
def test_lazily_conjugated_operands_and_cotangents(gpu, M):
    """gradients.propagate on both routes (16 states at most: pieces) with a
    loss whose cotangent arrives as a pending conjugation, and operands that
    are conjugate views, against the recursion in numpy."""
    A, y0, _ = _problem(M, 2, 2, False, M)
    nsub = [0] + [1] * 100
    w = torch.as_tensor(np.random.RandomState(2).normal(size=(2, 2, 101, M)) + 0.5j).to(y0.device)
    a, y = A.clone().requires_grad_(True), y0.clone().requires_grad_(True)
    states = G.propagate(a, y, nsub)
    (w * states.conj()).sum().real.backward()
    # d Re sum(w conj(s)) with respect to s: w
    want, gA, gy = _reference(A, y0, nsub, w.cpu().numpy())
    assert _rel(states, want) <= 1e-11
    assert _rel(a.grad, gA.sum(axis=1)) <= 1e-11 and _rel(y.grad, gy) <= 1e-11
    conj = G.propagate(A.conj(), y0.conj(), nsub)
    assert _rel(conj, want.conj()) <= 1e-11


@pytest.mark.parametrize('n', [40, 2500])
def test_transforms_of_lazily_conjugated_rows(gpu, n):
    """Forward, real-part and adjoint transforms of x.conj() equal those of
    the conjugated copy."""
    x = torch.as_tensor(np.random.RandomState(n).normal(size=(700, n)) + 0.3j).to('cuda')
    N, lo = 2 * n - 1, n - 1
    c = x.conj().resolve_conj()
    for f in (lambda v: _native.fourier_transform(v, N, lo, -1, 0.5),
              lambda v: _native.fourier_transform_real(v, N, lo, -1, 0.5)):
        assert torch.equal(f(x.conj()), f(c))
    g = _native.fourier_transform(x, N, lo, -1, 0.5)
    assert torch.equal(_native.fourier_transform_adjoint(g.conj(), n, lo, -1, 0.5),
                       _native.fourier_transform_adjoint(g.conj().resolve_conj(), n, lo, -1, 0.5))


def test_powers_that_overflow_where_no_state_does(gpu):
    """A mode that grows by 1e6 a step and is not in the states: its 64th power
    overflows, the states and gradients of the recursion are finite; with it
    in the states both routes report it."""
    A = torch.diag(torch.tensor([1e6, 0.9], dtype=torch.complex128)).to('cuda')[None]
    y0 = torch.tensor([[[0, 1 + 1j]]], dtype=torch.complex128, device='cuda')
    nsub = [0] + [1] * 300
    a, y = A.clone().requires_grad_(True), y0.clone().requires_grad_(True)
    states = G.propagate(a, y, nsub)
    (states[..., 1].abs() ** 2).sum().backward()
    g = np.zeros((1, 1, 301, 2), dtype=complex)
    g[0, 0, :, 1] = 2 * (1 + 1j) * 0.9 ** np.arange(301)
    want, gA, gy = _reference(A, y0, nsub, g)
    assert _rel(states, want) <= 1e-11
    assert _rel(a.grad, gA.sum(axis=1)) <= 1e-11 and _rel(y.grad, gy) <= 1e-11
    with pytest.raises(FloatingPointError):
        G.propagate(A, torch.ones_like(y0), nsub)
