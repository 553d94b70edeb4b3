"""qsx_fourier_transform (the reference's zero-padded symmetric FFT,
qspectra/simulate/utils.py:128-219, on the GPU: a direct sum for rows
shorter than 2048 samples or points, the chirp-z form with FFTs in LDS for
longer ones) against the oracle's numpy FFT pipeline: grids starting at,
before and after t = 0 (the zero padding on either side), both signs,
batched rows along any axis, and the adjoint against the conjugate-transposed
transform matrix, through autograd, and (long rows) against numpy's inverse
FFT run through the transposed pipeline.  Tolerance 1e-13 relative
(max-norm)."""
import numpy as np
import pytest
import torch

import qspectra_amd as qa
from qspectra_amd import _native
from qspectra_amd.simulate.utils import fourier_transform_device
from oracle import propagate as P
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,t0,dt', [(2, 0.0, 1.0), (7, 0.0, 0.7), (64, -20.0, 0.5),
                                     (300, 11.0, 0.25), (1989, 0.0, 5.0297804513411934),
                                     (4096, -4096 * 0.5, 0.5), (5000, 7.0, 2.0)])
def test_matches_numpy_fft_pipeline(gpu, n, t0, dt):
    rs = np.random.RandomState(n)
    _check_against_oracle(rs, n, t0, dt)


def _check_against_oracle(rs, n, t0, dt):
    t = t0 + dt * np.arange(n)
    x = rs.randn(3, n) + 1j * rs.randn(3, n)
    for sign in (1, -1):
        for conv in ('angular', 'linear'):
            fo, Xo = P.fourier_transform(t, x, axis=-1, rw_freq=123.0, unit_convert=0.3,
                                         sign=sign, convention=conv)
            f, X = qa.fourier_transform(t, x, axis=-1, rw_freq=123.0, unit_convert=0.3,
                                        sign=sign, convention=conv)
            assert np.array_equal(f, fo)
            assert rel_err(X, Xo) < 1e-13, (n, sign)


def test_axes_and_adjoint(gpu):
    rs = np.random.RandomState(1)
    t1 = 0.5 * np.arange(40)
    t3 = 0.5 * np.arange(33)
    R = rs.randn(40, 5, 33) + 1j * rs.randn(40, 5, 33)
    f1, A = P.fourier_transform(t1, R, axis=0, sign=-1)
    f3, B = P.fourier_transform(t3, A, axis=2)
    _, Ag = qa.fourier_transform(t1, R, axis=0, sign=-1)
    _, Bg = qa.fourier_transform(t3, Ag, axis=2)
    assert rel_err(Ag, A) < 1e-13 and rel_err(Bg, B) < 1e-13
    # adjoint: <F x, g> = <x, F^H g>, and the autograd backward is F^H g
    t = -3.0 + 0.25 * np.arange(21)
    x = torch.as_tensor(rs.randn(21) + 1j * rs.randn(21)).cuda().requires_grad_(True)
    _, X = fourier_transform_device(t, x, -1, 0.0, 1.0, sign=1)
    g = torch.as_tensor(rs.randn(X.shape[-1]) + 1j * rs.randn(X.shape[-1])).cuda()
    (gx,) = torch.autograd.grad((X * g.conj()).sum().real, x)
    F = np.stack([P.fourier_transform(t, e, sign=1)[1] for e in np.eye(21)], axis=1)
    assert rel_err(gx.cpu().numpy(), F.conj().T @ g.cpu().numpy()) < 1e-13
    ga = _native.fourier_transform_adjoint(g[None], 21, 0, 1, 0.25)[0].cpu().numpy()
    assert rel_err(ga, F.conj().T @ g.cpu().numpy()) < 1e-13


def _adjoint_numpy(t, g, sign):
    """The oracle's pipeline transposed: flip (sign +1), ifftshift (the
    transpose of fftshift), N * ifft (the conjugate transpose of fft),
    fftshift (the transpose of ifftshift), the sample positions of the
    zero-padded grid, times dt."""
    t_sym, _ = P.symmetrize(t, np.zeros(t.size))
    lo = int(np.searchsorted(t_sym, t[0]))
    N = g.shape[-1]
    h = g[..., ::-1] if sign == 1 else g
    y = np.fft.fftshift(N * np.fft.ifft(np.fft.ifftshift(h, axes=-1), axis=-1), axes=-1)
    return (t[1] - t[0]) * y[..., lo:lo + t.size], lo


@pytest.mark.parametrize('n,t0,dt,rows', [(4096, 0.0, 1.0, 37), (2048, -3.0, 0.5, 5),
                                          (6000, 11.0, 0.25, 3)])
def test_long_rows_forward_and_adjoint(gpu, n, t0, dt, rows):
    """Rows of 2048 samples and more (the chirp-z path: one piece and two
    output chunks for 4096 samples from t = 0, two pieces and three chunks
    for 6000) against the numpy FFT pipeline, with a scale; the adjoint
    against the transposed numpy pipeline."""
    rs = np.random.RandomState(n + rows)
    t = t0 + dt * np.arange(n)
    x = rs.randn(rows, n) + 1j * rs.randn(rows, n)
    for sign in (1, -1):
        fo, Xo = P.fourier_transform(t, x, axis=-1, sign=sign)
        f, X = fourier_transform_device(t, torch.as_tensor(x).cuda(), -1, sign=sign,
                                        scale=-2.5)
        assert np.array_equal(f, fo)
        assert rel_err(X.cpu().numpy(), -2.5 * Xo) < 1e-13, (n, sign)
        g = rs.randn(rows, Xo.shape[-1]) + 1j * rs.randn(rows, Xo.shape[-1])
        xa_ref, lo = _adjoint_numpy(t, g, sign)
        xa = _native.fourier_transform_adjoint(torch.as_tensor(g).cuda(), n, lo, sign, dt)
        assert rel_err(xa.cpu().numpy(), xa_ref) < 1e-13, (n, sign)


@pytest.mark.parametrize('rows,n,lo,N', [(1, 1, 0, 1), (2, 2, 1, 4), (3, 17, 0, 33), (5, 16, 15, 31),
                                         (5, 600, 599, 1199), (700, 300, 0, 600),
                                         (2100, 70, 69, 139), (1, 513, 100, 1024),
                                         (9, 40, 300, 1000), (3, 40, 700, 1000),
                                         (2100, 100, 1400, 1500), (700, 257, 0, 514),
                                         (2, 64, 63, 127), (4200, 65, 64, 129)])
def test_direct_sum_row_groups(gpu, rows, n, lo, N):
    """The direct sum over one, two and four rows per thread, odd and even
    grids, sample counts that are no multiple of the twiddle block or tile,
    placed anywhere on the grid (also all before or all after its zero), pair
    counts at the edges of a wavefront and a work-group: against the sum in numpy, forward (both
    signs) and adjoint.  n products of unit twiddles accurate to a few ulp:
    1e-12 of the row's scale."""
    rs = np.random.RandomState(n)
    x = rs.normal(size=(rows, n)) + 1j * rs.normal(size=(rows, n))
    c = N // 2
    for sign in (-1, 1):
        s = np.arange(N) - c if sign == -1 else N - 1 - c - np.arange(N)
        F = 0.5 * np.exp(-2j * np.pi * ((s[:, None] * (lo + np.arange(n) - c)) % N) / N)
        got = _native.fourier_transform(torch.as_tensor(x).to('cuda'), N, lo, sign, 0.5)
        want = x @ F.T
        assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
        g = torch.as_tensor(want).to('cuda')
        back = _native.fourier_transform_adjoint(g, n, lo, sign, 0.5)
        want = want @ F.conj()
        assert np.abs(back.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.parametrize('rows,n,sign', [(2, 2048, -1), (3, 2049, 1), (4, 3000, -1),
                                         (5, 4096, 1), (2, 4095, -1)])
def test_paired_real_parts(gpu, rows, n, sign):
    """Real parts of two rows per transform against the complex transform:
    one and two chunks, odd batches, rows of very different magnitude, a zero
    and a non-finite row beside a finite one.  The rounding of log2(8192) = 13
    passes each way, some tens of ulp: 1e-13 of the row's own scale."""
    rs = np.random.RandomState(n)
    N, lo = 2 * n - 1, n - 1
    x = rs.normal(size=(rows, n)) + 1j * rs.normal(size=(rows, n))
    x[1] *= 1e-12
    if rows > 2:
        x[2] = 0
    if rows > 4:
        x[2, 7] = np.nan
    xd = torch.as_tensor(x).to('cuda')
    want = _native.fourier_transform(xd, N, lo, sign, 0.5).real.cpu().numpy()
    got = _native.fourier_transform_real(xd, N, lo, sign, 0.5, pairs=True).cpu().numpy()
    assert got.dtype == np.float64 and got.shape == (rows, N)
    for b in range(rows):
        if np.isnan(x[b]).any():
            assert np.isnan(got[b]).all()
        else:
            assert np.abs(got[b] - want[b]).max() <= 1e-13 * np.abs(want[b]).max()


def test_direct_sum_on_a_grid_beyond_2_30_points(gpu):
    """Twiddle indices of a grid whose residues' sums pass 2^31: 48 samples
    (three exact twiddles each) onto 2^30 + 5 points, a few of the outputs
    against the sum in numpy with exponents reduced in Python integers."""
    N, n, lo = (1 << 30) + 5, 48, 12345
    if torch.cuda.get_device_properties(0).total_memory < 48 << 30:
        pytest.skip('needs 35 GB of device memory')
    rs = np.random.RandomState(0)
    x = rs.normal(size=n) + 1j * rs.normal(size=n)
    out = _native.fourier_transform(torch.as_tensor(x).to('cuda'), N, lo, -1, 0.5)
    c = N // 2
    at = np.concatenate([[0, 1, 2, N - 1, c - 1, c, c + 1], rs.randint(0, N, 200)])
    got = out[torch.as_tensor(at).to('cuda')].cpu().numpy()
    del out
    torch.cuda.empty_cache()
    want = [0.5 * sum(x[j] * np.exp(-2j * np.pi * (((int(r) - c) * (lo + j - c)) % N) / N)
                      for j in range(n)) for r in at]
    assert np.abs(got - want).max() <= 1e-12 * np.abs(x).sum()


@pytest.mark.parametrize('a,b', [(1e306, 1e200), (1e-300, 1e-200), (1e-310, 1.0), (1e160, 1e10),
                                 (1e140, 1e290), (1e-140, 1e-290)])
def test_paired_rows_at_the_ends_of_the_exponent_range(gpu, a, b):
    """A row beside one that overflows or is almost denormal: its real part is
    that of the row alone (1e-13 of its own scale, as above)."""
    rs = np.random.RandomState(3)
    n = 2100
    N, lo = 2 * n - 1, n - 1
    x = rs.normal(size=(2, n)) + 1j * rs.normal(size=(2, n))
    xd = torch.as_tensor(x * [[a], [b]]).to('cuda')
    got = _native.fourier_transform_real(xd, N, lo, -1, 0.5, pairs=True).cpu().numpy()
    with np.errstate(over='ignore', invalid='ignore'):
        want = _native.fourier_transform(torch.as_tensor(x).to('cuda'), N, lo, -1,
                                         0.5).real.cpu().numpy() * [[a], [b]]
    for g, w in zip(got, want):
        if 1e-290 < np.abs(w).max() < 1e305:
            assert np.isfinite(g).all()
            assert np.abs(g - w).max() <= 1e-13 * np.abs(w).max()
