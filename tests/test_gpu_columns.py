"""Two steps of a flow of a few Fourier modes, up to 1024^3, against the same steps on the modes
themselves: the nonlinear term by convolution, wrapped as the grid wraps it, then the update of
every mode (turb.f90:634-691).  One mode reaches every point of a column and every mode of the
result, so each plan of the register transforms (forward, update and inverse, in all tile
widths) is held to values from outside at its own size, and everything else has to be zero."""
import ctypes

import numpy as np
import pytest

DT, RNU = 1e-3, 1e-4


def _modes(N, seed):
    """Wave vectors (kx > 0, and one with kx = 0) inside the sphere, some on its edge, and their
    solenoidal amplitudes."""
    rng = np.random.default_rng(seed)
    nek = int(N / 2 - 1.5)
    k = [(nek, 0, 0), (0, 3, nek - 2), (2, nek - 1, -3), (1, 1, -1)]
    while len(k) < 10:
        c = rng.integers(-nek, nek + 1, 3)
        if c[0] > 0 and np.sqrt((c ** 2).sum()) < nek:
            k.append(tuple(c))
    k = np.array(k)
    a = rng.standard_normal((len(k), 3)) + 1j * rng.standard_normal((len(k), 3))
    a -= k * ((k * a).sum(1) / (k * k).sum(1))[:, None]
    return k, a


def _whole(k, a):
    """The modes of the real field: k and -k (one of each pair is given where kx = 0)."""
    return np.concatenate([k, -k]), np.concatenate([a, a.conj()])


def _half(N, k, a):
    """Sums over equal wave vectors of the N^3 grid, kx in [0, N/2), inside the sphere; of a pair
    with kx = 0 both."""
    k = (k + N // 2 - 1) % N - N // 2 + 1
    keep = (np.floor(np.sqrt((k * k).sum(1)) + 0.5) <= int(N / 2 - 1.5)) & (k[:, 0] >= 0) & (k[:, 0] < N // 2)
    k, at = np.unique(k[keep], axis=0, return_inverse=True)
    out = np.zeros((len(k), 3), dtype=complex)
    np.add.at(out, at.reshape(-1), a[keep])
    return k, out


def _nonlinear(N, k, a):
    """u x w of the whole set of modes, half the modes of the result."""
    w = 1j * np.cross(k, a)
    n = np.cross(a[:, None, :], w[None, :, :]).reshape(-1, 3)
    return _half(N, (k[:, None, :] + k[None, :, :]).reshape(-1, 3), n)


def _step(N, ku, u, ko, o):
    """(modes of u, of the stored nonlinear term) after a step without forcing, half sets."""
    pos = ku[:, 0] > 0
    first = pos | ((ku[:, 0] == 0) & ((ku[:, 1] > 0) | ((ku[:, 1] == 0) & (ku[:, 2] > 0))))
    kn, n = _nonlinear(N, *_whole(ku[first], u[first]))
    k = np.concatenate([ku, kn, ko])
    ac = 0.5 * DT * RNU * (ku * ku).sum(1)
    v = np.concatenate([(1 - ac)[:, None] * u, 1.5 * DT * n, -0.5 * DT * o])
    k, v = _half(N, k, v)
    live = (k * k).sum(1) > 0
    k, v = k[live], v[live]
    k2 = (k * k).sum(1)
    v -= k * ((k * v).sum(1) / k2)[:, None]
    return (k, v / (1 + 0.5 * DT * RNU * k2)[:, None]), (kn, n)


def _two_steps(N, seed):
    k, a = _modes(N, seed)
    zero = k[:, 0] == 0
    start = (np.concatenate([k, -k[zero]]), np.concatenate([a, a[zero].conj()]))
    u1, o1 = _step(N, *start, np.zeros((0, 3), dtype=int), np.zeros((0, 3)))
    return start, u1, *_step(N, *u1, *o1)


def _fill(N, k, a):
    """The reference's arrays (kz, kx re/im, ky) of a half set."""
    out = []
    for c in range(3):
        f = np.zeros((N + 2, N + 2, N), order="F")
        f[k[:, 2] % N, 2 * k[:, 0], k[:, 1] % N] = a[:, c].real
        f[k[:, 2] % N, 2 * k[:, 0] + 1, k[:, 1] % N] = a[:, c].imag
        out.append(f)
    return out


def _largest_difference(N, f, k, a):
    """max |f - (the component a of the modes k)|; f is overwritten."""
    f[k[:, 2] % N, 2 * k[:, 0], k[:, 1] % N] -= a.real
    f[k[:, 2] % N, 2 * k[:, 0] + 1, k[:, 1] % N] -= a.imag
    return max(f.max(), -f.min())


def _velocity(N, k, a, at):
    """The velocity at nodes at (z, y, x)."""
    zero = k[:, 0] == 0
    ph = np.exp(2j * np.pi / N * ((at[:, None, ::-1] * k[None]).sum(2) % N))
    return (ph * np.where(zero, 1.0, 2.0)) @ a


def test_the_steps_of_the_modes_are_the_oracles(ddns, oracle_mod):
    N = 32
    start, u1, u2, o2 = _two_steps(N, 5)
    with oracle_mod.Oracle(ddns.default_params(N=N, dt=DT, rnu=RNU, forcing=0)) as o:
        zero = _fill(N, start[0][:0], start[1][:0])
        o.set_flow(_fill(N, *start), zero)
        o.flow_only(True)
        o.step(2)
        got = o.get_flow()
        vel = o.physical_velocity()
    for f, (k, a) in zip(got, (u2, o2)):
        for c in range(3):
            assert _largest_difference(N, f[c].copy(order="F"), k, a[:, c]) < 1e-13 * np.abs(a).max()
    at = np.random.default_rng(1).integers(0, N, (500, 3))
    want = _velocity(N, *u1, at)
    for c in range(3):
        assert np.abs(vel[c][at[:, 0], at[:, 1], at[:, 2]] - want[:, c].real).max() < 1e-13 * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("N,precision,wide", [(32, 0, 0), (64, 1, 0), (128, 0, 0), (128, 1, 1), (256, 0, 0), (256, 0, 1),
                                              (256, 1, 0), (256, 1, 1), (512, 0, 0), (512, 0, 1), (512, 1, 0), (512, 1, 1),
                                              (1024, 0, 0), (1024, 1, 0)])
def test_two_steps_of_a_few_modes(ddns, monkeypatch, N, precision, wide):
    """wide: twice the default width of the y and z tiles, each where it fits."""
    p = ddns.default_params(N=N, precision=precision, dt=DT, rnu=RNU, forcing=0)
    monkeypatch.setenv("DDNS_TUNE", "0")
    if wide:
        with ddns.Solver(p) as s:
            t = s.tuning()
        monkeypatch.setenv("DDNS_KY_TC", str(2 * t["ky_tc_default"]))
        monkeypatch.setenv("DDNS_KZ_NT", str(2 * t["kz_nt_default"]))
    start, u1, u2, o2 = _two_steps(N, N + precision)
    at = np.random.default_rng(1).integers(0, N, (2000, 3))
    want = _velocity(N, *u1, at)
    tol = 2e-6 if precision else 1e-13
    f = np.zeros((N + 2, N + 2, N), order="F")
    g = np.zeros((N, N, N))
    pointer = lambda a, c, n: [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) if q == c else None for q in range(n)]
    with ddns.Solver(p) as s:
        assert (s.tuning()["ky_tc"] != s.tuning()["ky_tc_default"]) == bool(wide)
        s.set_flow(_fill(N, *start))
        s.step(2)
        for c in range(6):
            k, a = u2 if c < 3 else o2
            assert s.lib.ddns_get_flow(s.h, *pointer(f, c, 6)) == 0
            err = _largest_difference(N, f, k, a[:, c % 3]) / np.abs(a).max()
            print(f"N={N} precision={precision} wide={wide}: {'uo'[c // 3]}{c % 3} {err:.1e}", flush=True)
            assert err < tol
        for c in range(3):
            assert s.lib.ddns_get_physical_velocity(s.h, *pointer(g, c, 3)) == 0
            assert np.abs(g[at[:, 0], at[:, 1], at[:, 2]] - want[:, c].real).max() < tol * np.abs(want).max()
