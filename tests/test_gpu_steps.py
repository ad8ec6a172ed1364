"""Steps queued several to a call, the stochastic forcing beside the x stage, states with modes
beyond the dealiasing sphere, and the transforms at the sizes whose columns sit in registers."""
import numpy as np
import pytest

from helpers import random_spectral, rel_l2

pytestmark = pytest.mark.gpu


def _flow(s):
    return [a for q in s.get_flow() for a in q]


@pytest.mark.parametrize("forcing", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 17])
def test_steps_of_one_call_are_single_steps(ddns, n, forcing):
    p = ddns.default_params(N=32, precision=1, forcing=forcing, dt=1e-3, rnu=0.02)
    out = []
    for calls in ([n], [1] * n):
        with ddns.Solver(p) as s:
            s.init_flow(ddns.SPEC_K4_GAUSS, 11, 4.0, 1.0)
            for k in calls:
                s.step(k)
            out.append(_flow(s))
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("N,precision", [(32, 0), (64, 0), (64, 1), (128, 1), (256, 1)])
def test_forcing_beside_the_x_stage(ddns, N, precision):
    """Without droplets a work-group of the x stage does the stochastic forcing, with them a kernel
    of its own: the flow, which does not see the droplets, is the same, bit for bit."""
    out = []
    for droplets in (0, 1):
        p = ddns.default_params(N=N, precision=precision, forcing=2, dt=5e-4, rnu=0.01, npart=10 * droplets,
                                radius=[20.0])
        with ddns.Solver(p) as s:
            s.init_flow(ddns.SPEC_K4_GAUSS, 11, 4.0, 1.0)
            if droplets:
                s.init_droplets(seed=5)
            s.step(3)
            s.step(2)
            out.append(_flow(s))
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def test_modes_beyond_the_sphere(ddns, oracle_mod):
    """A state with energy beyond the dealiasing sphere, the corners included (in FP64: the shells
    that the forcing rescales hold little of it, and FP32 rounding alone gives 2e-5)."""
    N = 32
    kw = dict(N=N, forcing=1, dt=1e-3, rnu=0.02)
    v = random_spectral(N, seed=17, kmax=15, amp=1.0)
    with ddns.Solver(ddns.default_params(precision=0, **kw)) as s, oracle_mod.Oracle(ddns.default_params(**kw)) as o:
        for x in (s, o):
            x.set_flow(v, v)
        o.flow_only(True)
        for n in (1, 2):
            s.step(n)
            o.step(n)
            a, b = s.get_flow(), o.get_flow()
            for q in range(2):
                assert rel_l2(a[q], b[q]) < 1e-11


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [128, 256])
def test_transforms(ddns, N, precision):
    rng = np.random.default_rng(N)
    phys = np.zeros((N + 2, N + 2, N), order="F")
    phys[:N, :N] = rng.standard_normal((N, N, N))
    with ddns.Solver(ddns.default_params(N=N, precision=precision)) as s:
        g = s.fft_r2c(phys)
        back = s.fft_c2r(g)
    # physical (x, y, z), spectral (kz, kx re/im, ky)
    c = np.fft.rfftn(phys[:N, :N], axes=(1, 2, 0)) / N ** 3
    c[N // 2] = 0.0                                          # the GPU does not store kx = N/2
    got = (g[:N, 0:N:2] + 1j * g[:N, 1:N:2]).transpose(1, 2, 0)
    tol = 1e-13 if precision == 0 else 2e-6
    assert np.abs(got - c[:N // 2]).max() <= tol * np.abs(c).max()
    want = np.fft.irfftn(c, s=(N, N, N), axes=(1, 2, 0)) * N ** 3
    assert np.abs(back[:N, :N] - want).max() <= tol * np.abs(want).max()
