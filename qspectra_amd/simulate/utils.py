"""Time integration on the GPU and Fourier-transform utilities
(qspectra/simulate/utils.py API).

``integrate`` replaces scipy's zvode loop (utils.py:16-109) with the fused
fixed-step RK4 kernel qsx_rk4_dense: every right-hand side (rows of a 2-D
y0) and every ensemble member is propagated in one launch, and a linear
save_func (the operators' commutator / expectation value / bra) is applied
inside the kernel at each output time.

Extra keyword arguments (all optional):
  dt         maximum RK4 step (default: chosen from rtol, see step_size)
  precision  'fp64' (default) or 'mixed' (complex64 products with the FP64
             diagonal, FP64 state and update)
  rtol       target relative accuracy for the default step (1e-6, zvode's
             default); atol, nsteps and other zvode options are accepted and
             ignored.
  schedule   'auto' (default), 'rk4' or 'propagator' (see propagate)
"""
import numpy as np
import torch

from .. import _native
from ..engine import rk4_schedule, schedule_tensors
from ..lti import split_diagonal
from ..schedules import Stage, stepper_operator, _mode
from ..dynamics.liouville_space import DeviceEOM, LinearMap
from ..dynamics.heom import DeviceHEOM
from ..dynamics.zofe import DeviceZOFE

ZVODE_OPTIONS = ('rtol', 'atol', 'nsteps', 'method', 'with_jacobian', 'lband', 'uband',
                 'order', 'first_step', 'min_step', 'max_step')


class IntegratorError(Exception):
    pass


def step_size(L, span, rtol=1e-6):
    """RK4 step with estimated global error <= rtol over ``span``.

    With rho >= the spectral radius of L (its max absolute row sum), the
    local error of one step of length h is about (rho h)^5 / 120, so
    (rho h)^4 rho span / 120 <= rtol bounds the accumulated error."""
    rho = float(torch.max(torch.sum(torch.abs(L), dim=-1)).item())
    if rho == 0 or span <= 0:
        return float('inf')
    return (120.0 * rtol / (rho * span)) ** 0.25 / rho


def _prepare_precision(L, proj, precision):
    if precision in ('fp64', 'double', None):
        return L, None, proj, _native.QSX_FP64
    if precision != 'mixed':
        raise ValueError("precision must be 'fp64' or 'mixed'")
    Lm, diag = split_diagonal(L)
    pm = None if proj is None else proj.to(torch.complex64).contiguous()
    return Lm, diag, pm, _native.QSX_MIXED


def project_states(states, proj):
    """out[b, r, s, :] = proj[b] @ states[b, r, s, :] as one batched complex128
    GEMM (in every precision: dipole maps are a small share of the work)."""
    B, R, ns, M = states.shape
    K = proj.shape[-2]
    projT = proj.transpose(-1, -2).to(torch.complex128).contiguous()
    out = _native.zgemm(states.reshape(B, R * ns, M).contiguous(), projT)
    return out.reshape(B, R, ns, K)


def propagate(eom, y0, t, t0=None, proj=None, dt=None, precision='fp64', rtol=1e-6,
              want_final=False, schedule='auto'):
    """Device-level driver: y0 [B, R, M] complex128 tensor, proj [B|1, K, M]
    tensor or None.  Returns out [B, R, len(t), K] (and the final state).

    schedule: 'rk4' (four Liouvillian products per step), 'propagator' (one
    product per step with the RK4 propagator; needs a uniform step),
    'blocked' (propagator powers / time chunks, see schedules.Stage) or
    'auto' (blocked whenever every step has the same length)."""
    t = np.asarray(t, dtype=float).reshape(-1)
    if t0 is None:
        t0 = float(t[0])
    if dt is None:
        dt = step_size(eom.L, float(t[-1]) - float(t0), rtol)
        spacing = np.diff(np.concatenate([[t0], t]))
        spacing = spacing[spacing > 0]
        if spacing.size:
            dt = min(dt, float(spacing.min()))
        if not np.isfinite(dt):
            dt = None
    n_host, h_host = rk4_schedule(t, t0, dt)
    nsub, h = schedule_tensors(t, t0, dt, eom.L.device)
    steps = int(n_host.sum())
    M = eom.L.shape[-1]
    if M > _native.MAX_REGISTER_BLOCK:
        L, diag, pj, mode = _prepare_precision(eom.L, proj, precision)
        out, yfin, status = _native.rk4_dense(L, y0, nsub, h, pj, mode, diag, want_final,
                                              steps=steps)
    else:
        if schedule not in ('auto', 'rk4', 'propagator', 'blocked'):
            raise ValueError("schedule must be 'auto', 'rk4', 'propagator' or 'blocked'")
        stage = Stage(eom, t, t0, dt, precision, schedule, y0.shape[1])
        statuses = []
        states = stage.run(y0, statuses)
        yfin = states[:, :, -1].contiguous() if want_final else None
        status = sum(statuses) if statuses else torch.zeros(1, dtype=torch.int32,
                                                            device=y0.device)
        if not statuses and not bool(torch.isfinite(torch.view_as_real(states[:, :, -1])).all()):
            status = torch.ones(1, dtype=torch.int32, device=y0.device)
        out = states if proj is None else project_states(states, proj)
    if int(status.item()) != 0:
        raise IntegratorError('integration failed: non-finite state between t=%g and t=%g'
                              % (t0, t[-1]))
    return (out, yfin) if want_final else out


def heom_rate(eom, iters=40):
    """Spectral-radius estimate of a hierarchy generator (times 1.5): power
    iteration with qsx_heom_apply from a fixed pseudo-random start, the
    largest growth factor over the samples; cached on the equation of
    motion."""
    cached = getattr(eom, '_rate_estimate', None)
    if cached is not None:
        return cached
    gen = torch.Generator().manual_seed(12345)
    B, S = eom.batch, eom.size
    v = torch.complex(torch.randn(B, S, generator=gen, dtype=torch.float64),
                      torch.randn(B, S, generator=gen, dtype=torch.float64)).to(eom.Hop.device)
    growth = torch.zeros(B, dtype=torch.float64, device=v.device)
    for _ in range(iters):
        v = v / v.abs().amax(dim=1, keepdim=True).clamp_min(1e-300)
        w = _native.heom_apply(eom, v)
        growth = w.abs().amax(dim=1)
        v = w
    rate = 1.5 * float(growth.max().item())
    eom._rate_estimate = rate
    return rate


def heom_step(eom, y0, span, rtol=1e-6, t0=0.0):
    """Default RK4 step of a hierarchy over ``span``: calibrate_step between
    the stable step 2 / rate and the rate-bound step (rate from heom_rate),
    probing from the initial hierarchy states y0 [B, n_ado * M]."""
    rate = heom_rate(eom)
    if rate == 0 or span <= 0:
        return None
    h_safe = (120.0 * rtol / (rate * span)) ** 0.25 / rate

    def probe(H, n):
        ends = []
        for hp, steps in ((H, n), (H / 2, 2 * n)):
            _, yf, status = _native.heom_propagate(eom, y0, [steps], [hp], _native.QSX_FP64,
                                                   want_final=True)
            if int(status.item()) != 0:
                return None
            ends.append(yf)
        return ends
    return calibrate_step(probe, h_safe, 2.0 / rate, span, rtol)


def propagate_heom(eom, y0, t, t0=None, dt=None, precision='fp64', full_states=False,
                   rtol=1e-6):
    """Hierarchy propagation: y0 [B, n_ado * M] complex128 tensor.  Returns
    ADO 0 at every output time, [B, len(t), M], or with full_states the
    whole hierarchy, [B, len(t), n_ado * M] (one launch per output time).
    Without ``dt`` the step is calibrated to ``rtol`` (heom_step)."""
    t = np.asarray(t, dtype=float).reshape(-1)
    if t0 is None:
        t0 = float(t[0])
    if dt is None:
        dt = heom_step(eom, y0, float(t[-1]) - float(t0), rtol, float(t0))
        gaps = np.diff(np.concatenate([[t0], t]))
        gaps = gaps[gaps > 0]
        if gaps.size:
            dt = float(gaps.min()) if dt is None else min(dt, float(gaps.min()))
    n, h = rk4_schedule(t, t0, dt)
    mode = _mode(precision)
    if not full_states:
        out, _, status = _native.heom_propagate(eom, y0, n, h, mode)
        if int(status.item()) != 0:
            raise IntegratorError('integration failed: non-finite state')
        return out
    states = []
    y = y0
    for ni, hi in zip(n, h):
        _, y, status = _native.heom_propagate(eom, y, [ni], [hi], mode, want_final=True)
        if int(status.item()) != 0:
            raise IntegratorError('integration failed: non-finite state')
        states.append(y)
    return torch.stack(states, dim=1)


def _zofe_rate(eom, field_rate=0.0):
    """Rate bound of the ZOFE equation: unit * (2 max row sum |H| + max |w|
    + 2 S sum_p max_s |Gamma / w|) (+ the fields' rate)."""
    H = eom.H.abs().sum(dim=-1).max().item()
    w = eom.w.abs()
    rate = abs(eom.unit_convert) * (2 * H + float(w.max().item())
                                    + 2 * eom.S * float((eom.Gamma.abs() / w).max(dim=-1)
                                                        .values.sum().item()))
    return rate + field_rate


def calibrate_step(probe, h_safe, h_max, span, rtol, window=0.0):
    """The largest RK4 step, from h_max down and never below h_safe, whose
    error estimate is below rtol / 4.  probe(H, n) returns the end states
    of n steps of H and of 2 n steps of H / 2 from the initial states (None
    when a run is not finite); their difference (x 16/15, Richardson) is the
    error of the H run, extrapolated linearly from the probe's n H to the
    span.  The probe covers max(span / 20, window) (16 to 256 steps)."""
    if h_safe is None or span <= 0:
        return h_safe
    H = min(h_max, span)
    for _ in range(12):
        if H <= h_safe:
            return h_safe
        n = int(min(256, max(16, np.ceil(max(span / 20.0, window) / H))))
        ends = probe(H, n)
        est = float('inf')
        if ends is not None:
            scale = float(ends[1].abs().max().item())
            diff = float((ends[0] - ends[1]).abs().max().item())
            est = (16.0 / 15.0) * diff / max(scale, 1e-300) * max(span / (n * H), 1.0)
        if np.isfinite(est) and est <= 0.25 * rtol:
            return H
        shrink = 0.5
        if np.isfinite(est) and est > 0:
            shrink = min(0.5, 0.9 * (0.25 * rtol / est) ** 0.25)
        H *= shrink
    return h_safe


def zofe_step(eom, span, rtol=1e-6, field_rate=0.0, y0=None, fields=None, t0=0.0,
              window=0.0):
    """RK4 step for the ZOFE equation with estimated global error <= rtol
    over ``span``.  The rate bound (as step_size for a Liouvillian) gives a
    step that is safe for any state, and far too small for the strongly
    damped pseudomodes: with the initial states y0 [B, R, size] the step is
    calibrated instead (calibrate_step, from the stable step 2 / rate).
    ``fields(t_out, t0, dt)`` -> (V, F) gives the field terms of a probe
    schedule (None: undriven); ``window`` the time the probe must cover (the
    pulses)."""
    rate = _zofe_rate(eom, field_rate)
    if rate == 0 or span <= 0:
        return None
    h_safe = (120.0 * rtol / (rate * span)) ** 0.25 / rate
    if y0 is None:
        return h_safe

    def probe(H, n):
        ends = []
        for hp in (H, H / 2):
            tp = np.array([t0 + n * H])
            nsub, hh = schedule_tensors(tp, t0, hp, y0.device)
            V, F = fields(tp, t0, hp) if fields is not None else (None, None)
            out, status = _native.zofe_propagate(eom, y0, nsub, hh, V=V, F=F)
            if int(status.item()) != 0:
                return None
            ends.append(out[:, :, -1])
        return ends
    return calibrate_step(probe, h_safe, 2.0 / rate, span, rtol, window)


def propagate_zofe(eom, y0, t, t0=None, dt=None, proj=None, V=None, F=None, rtol=1e-6,
                   field_rate=0.0):
    """ZOFE propagation: y0 [B, R, size] complex128 device tensor (the
    reference's state layout); proj [B|1, K, N*N] rows on vec(rho) or None
    (full states); field terms V / F as _native.zofe_propagate.  Returns
    out [B, R, len(t), K or size]."""
    t = np.asarray(t, dtype=float).reshape(-1)
    if t0 is None:
        t0 = float(t[0])
    if dt is None:
        if V is None:
            dt = zofe_step(eom, float(t[-1]) - float(t0), rtol, field_rate, y0=y0, t0=t0)
        else:
            dt = zofe_step(eom, float(t[-1]) - float(t0), rtol, field_rate)
        gaps = np.diff(np.concatenate([[t0], t]))
        gaps = gaps[gaps > 0]
        if gaps.size:
            dt = gaps.min() if dt is None else min(dt, float(gaps.min()))
    nsub, h = schedule_tensors(t, t0, dt, y0.device)
    out, status = _native.zofe_propagate(eom, y0, nsub, h, proj=proj, V=V, F=F)
    if int(status.item()) != 0:
        raise IntegratorError('integration failed: non-finite state between t=%g and t=%g'
                              % (t0, t[-1]))
    return out


def zofe_projection(eom, save_func):
    """The rows of a LinearMap save function on a ZOFE state, restricted to
    vec(rho), as [1, K, N*N] (None when the map also reads the auxiliary
    operators), and whether it returns a scalar."""
    mat = np.asarray(save_func.matrix)
    scalar = mat.ndim == 1
    mat = np.atleast_2d(mat)
    n2 = eom.N * eom.N
    if np.any(mat[:, n2:] != 0):
        return None, scalar
    return _native.to_device(mat[None, :, :n2].copy()), scalar


def integrate(f, y0, t, t0=None, method_name='zvode', f_params=None, save_func=None, **kwargs):
    """Solves dy/dt = f(t, y) from y(t0) = y0 and returns save_func(y(t_i))
    for every t_i: shape [..., len(t), *save_shape] for y0 of shape [..., M]
    (leading axes are independent right-hand sides, propagated together).

    ``f`` must be an equation of motion produced by a qspectra_amd model
    (the GPU needs the operator, not a Python callback)."""
    if isinstance(f, DeviceHEOM):
        return _integrate_heom(f, y0, t, t0, save_func, kwargs)
    if isinstance(f, DeviceZOFE):
        return _integrate_zofe(f, y0, t, t0, save_func, kwargs)
    if not isinstance(f, DeviceEOM):
        raise TypeError('integrate needs an equation of motion from a qspectra_amd model '
                        '(DynamicalModel.equation_of_motion); arbitrary Python callables '
                        'have no GPU form')
    if f_params:
        raise TypeError('f_params are not supported by the Liouvillian equations of motion')
    dt = kwargs.pop('dt', None)
    precision = kwargs.pop('precision', 'fp64')
    rtol = kwargs.pop('rtol', 1e-6)
    schedule = kwargs.pop('schedule', 'auto')
    unknown = set(kwargs) - set(ZVODE_OPTIONS)
    if unknown:
        raise TypeError('unexpected integrate options: %s' % sorted(unknown))
    y0 = np.asarray(y0)
    M = f.size
    if y0.shape[-1] != M:
        raise ValueError('y0 has %d components, the subspace has %d' % (y0.shape[-1], M))
    lead = y0.shape[:-1]
    B = f.batch
    if B > 1:
        if not lead or lead[0] != B:
            raise ValueError('a batched equation of motion needs y0 with leading axis %d' % B)
        y = y0.reshape(B, -1, M)
    else:
        y = y0.reshape(1, -1, M)
    dev = f.L.device
    proj, scalar, host_save = None, False, None
    if isinstance(save_func, LinearMap):
        mat = save_func.matrix
        scalar = mat.ndim == 1
        proj = _native.to_device(np.atleast_2d(mat)[None], dev=dev)
    elif save_func is not None:
        host_save = save_func
    out = propagate(f, _native.to_device(y, dev=dev), t, t0, proj, dt, precision, rtol,
                    schedule=schedule)
    out = out.cpu().numpy()                      # [B, R, nt, K]
    nt = out.shape[2]
    if scalar:
        out = out[..., 0]
    result = out.reshape(lead + (nt,) + out.shape[3:])
    if host_save is not None:
        saved = [host_save(v) for v in result.reshape(-1, M)]
        saved = np.asarray(saved)
        result = saved.reshape(lead + (nt,) + saved.shape[1:])
    return result


def _integrate_zofe(f, y0, t, t0, save_func, kwargs):
    dt = kwargs.pop('dt', None)
    rtol = kwargs.pop('rtol', 1e-6)
    kwargs.pop('precision', None)
    kwargs.pop('schedule', None)
    unknown = set(kwargs) - set(ZVODE_OPTIONS)
    if unknown:
        raise TypeError('unexpected integrate options: %s' % sorted(unknown))
    y0 = np.asarray(y0)
    if y0.shape[-1] != f.size:
        raise ValueError('y0 has %d components, the ZOFE state %d' % (y0.shape[-1], f.size))
    lead = y0.shape[:-1]
    B = f.batch
    y = y0.reshape(B, -1, f.size) if B > 1 else y0.reshape(1, -1, f.size)
    proj, scalar, host_save = None, False, None
    if isinstance(save_func, LinearMap):
        proj, scalar = zofe_projection(f, save_func)
        if proj is None:
            host_save = save_func
    elif save_func is not None:
        host_save = save_func
    out = propagate_zofe(f, _native.to_device(y), t, t0, dt, proj=proj, rtol=rtol)
    out = out.cpu().numpy()                                     # [B, R, nt, K or size]
    nt = out.shape[2]
    if scalar and proj is not None:
        out = out[..., 0]
    result = out.reshape(lead + (nt,) + out.shape[3:])
    if host_save is not None:
        saved = np.asarray([host_save(v) for v in result.reshape(-1, f.size)])
        result = saved.reshape(lead + (nt,) + saved.shape[1:])
    return result


def _integrate_heom(f, y0, t, t0, save_func, kwargs):
    dt = kwargs.pop('dt', None)
    precision = kwargs.pop('precision', 'fp64')
    rtol = kwargs.pop('rtol', 1e-6)
    kwargs.pop('schedule', None)
    unknown = set(kwargs) - set(ZVODE_OPTIONS)
    if unknown:
        raise TypeError('unexpected integrate options: %s' % sorted(unknown))
    y0 = np.asarray(y0)
    lead = y0.shape[:-1]
    B = f.batch
    y = y0.reshape(B, f.size) if B > 1 else y0.reshape(-1, f.size)
    if y.shape[0] != B:
        raise ValueError('hierarchy states must have a leading axis of %d samples' % B)
    out = propagate_heom(f, _native.to_device(y), t, t0, dt, precision, full_states=True,
                         rtol=rtol)
    out = out.cpu().numpy().reshape(lead + (len(np.atleast_1d(t)), f.size))
    if save_func is not None:
        flat = out.reshape(-1, f.size)
        saved = np.asarray([save_func(v) for v in flat])
        out = saved.reshape(lead + (len(np.atleast_1d(t)),) + saved.shape[1:])
    return out


# ------------------------------------------------------------ Fourier tools
def slice_along_axis(start=None, stop=None, step=None, axis=0, ndim=1):
    return tuple(slice(start, stop, step) if (n == axis or n == ndim + axis) else slice(None)
                 for n in range(ndim))


def is_constant(x, atol=1e-7, positive=None):
    x = np.asarray(x)
    return (np.max(np.abs(x - x[0])) < atol
            and (np.all((x > 0) == positive) if positive is not None else True))


def _symmetrize(t, x, axis=-1):
    """Zero-pads x along ``axis`` to a grid symmetric about t = 0."""
    if not is_constant(np.diff(t), positive=True):
        raise ValueError('sample times must differ by a positive constant')
    t = np.asarray(t)
    x = np.asarray(x)
    dt = t[1] - t[0]
    T = max(t[-1], -t[0])
    n_after = int((T - t[-1]) / dt) + 1
    n_before = int((T + t[0]) / dt) + 1
    t_sym = np.concatenate([t[0] - dt * np.arange(1, n_before)[::-1], t,
                            t[-1] + dt * np.arange(1, n_after)])
    shape = list(x.shape)
    shape[axis] = t_sym.size
    x_sym = np.zeros(shape, dtype=x.dtype)
    lo, hi = (int(np.searchsorted(t_sym, ti)) for ti in (t[0], t[-1]))
    x_sym[slice_along_axis(lo, hi + 1, axis=axis, ndim=x.ndim)] = x
    return t_sym, x_sym


class _SymmetricFourier(torch.autograd.Function):
    """The transform of the last axis onto the zero-padded symmetric grid
    (qsx_fourier_transform); backward: its conjugate transpose."""

    @staticmethod
    def forward(ctx, x, N, lo, sign, dt):
        ctx.meta = (x.shape[-1], lo, sign, dt)
        return _native.fourier_transform(x, N, lo, sign, dt)

    @staticmethod
    def backward(ctx, g):
        n, lo, sign, dt = ctx.meta
        return _native.fourier_transform_adjoint(g, n, lo, sign, dt), None, None, None, None


def fourier_transform_device(t, x, axis=-1, rw_freq=0, unit_convert=1, sign=1,
                             convention='angular', scale=1.0, real=False):
    """fourier_transform on a complex128 device tensor x (result stays on the
    device; differentiable): the zero-padded symmetric grid, ifftshift, DFT,
    fftshift of utils.py:128-219, evaluated by qsx_fourier_transform (a
    direct sum for short rows, the chirp-z form with FFTs in LDS for long
    ones), the result times ``scale``.  With ``real`` its real part only (not
    differentiable)."""
    t = np.asarray(t, dtype=float)
    if t.ndim != 1:
        raise ValueError('t must be one dimensional')
    ax = axis % x.dim()
    if t.size != x.shape[ax]:
        raise ValueError('t must have the same length as the shape of x along the given axis')
    if sign not in (-1, 1):
        raise ValueError('sign must be +1 or -1')
    if convention == 'angular':
        unit_convert = unit_convert / (2 * np.pi)
    elif convention != 'linear':
        raise ValueError("convention must be 'angular' or 'linear'")
    t_sym, _ = _symmetrize(t, np.zeros(t.size), 0)
    lo = int(np.searchsorted(t_sym, t[0]))
    N = t_sym.size
    dt = t_sym[1] - t_sym[0]
    xm = x.to(torch.complex128).movedim(ax, -1)
    factor = float(dt) * float(scale)
    if real:
        X = _native.fourier_transform_real(xm.detach(), N, lo, sign, factor).movedim(-1, ax)
    else:
        X = _SymmetricFourier.apply(xm, N, lo, sign, factor).movedim(-1, ax)
    f = np.fft.fftshift(np.fft.fftfreq(N, dt * unit_convert))
    if sign == 1:
        f = -f[::-1]
    return f + rw_freq, X


def fourier_transform(t, x, axis=-1, rw_freq=0, unit_convert=1, sign=1, convention='angular'):
    """X(w) = int exp(i sign (w - rw) t) x(t) dt on the symmetric, zero-padded
    grid (qspectra/simulate/utils.py:154-219); the FFT runs on the GPU."""
    t = np.asarray(t)
    if t.ndim != 1:
        raise ValueError('t must be one dimensional')
    x = np.asarray(x)
    if t.size != x.shape[axis]:
        raise ValueError('t must have the same length as the shape of x along the given axis')
    if not is_constant(np.diff(t), positive=True):
        raise ValueError('sample times must differ by a positive constant')
    f, X = fourier_transform_device(t, _native.to_device(x), axis, rw_freq, unit_convert, sign,
                                    convention)
    return f, X.cpu().numpy()


def bound_signal(ticks, signal, bounds, axis=0):
    if signal.shape[axis] != len(ticks):
        raise ValueError('ticks must have same shape as signal along given axis')
    i0, i1 = sorted(int(np.argmin(np.abs(ticks - b))) for b in bounds)
    return ticks[i0:i1 + 1], signal[slice_along_axis(i0, i1 + 1, axis=axis,
                                                     ndim=signal.ndim)]
