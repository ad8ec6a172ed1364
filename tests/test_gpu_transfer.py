"""State transfers: the layouts are formed on the device, in pieces where an array is larger
than the staging buffer."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [32, 64, 512])
def test_flow_round_trip(ddns, N, precision):
    """What is set comes back, rounded to the handle's type, with the padding zero; 512^3 takes
    several pieces."""
    if N == 512 and precision == 0:
        pytest.skip("one large case is enough")
    rng = np.random.default_rng(N + precision)
    v = [np.asfortranarray(rng.standard_normal((N, N + 2, N + 2)).T) for _ in range(1 if N == 512 else 3)]
    with ddns.Solver(ddns.default_params(N=N, precision=precision)) as s:
        s.set_flow((v * 3)[:3])
        got = s.get_flow()[0]
    for a, b in zip(v, got):
        want = np.zeros_like(a)
        want[:N, :N] = a[:N, :N] if precision == 0 else a[:N, :N].astype(np.float32)
        assert np.array_equal(b, want)


def test_physical_velocity_in_pieces(ddns):
    N = 256
    with ddns.Solver(ddns.default_params(N=N, precision=0, dt=1e-4)) as s:
        s.init_flow(ddns.SPEC_K4_GAUSS, 3, 4.0, 1.0)
        v = s.get_flow()[0]
        s.step(1)
        u = s.physical_velocity()
    for a, b in zip(v, u):
        c = (a[:N, 0:N:2] + 1j * a[:N, 1:N:2]).transpose(0, 2, 1)                     # kz, ky, kx
        c = np.concatenate([c, np.zeros((N, N, 1))], axis=2)
        want = np.fft.irfftn(c, s=(N, N, N), axes=(0, 1, 2)) * N ** 3
        assert np.abs(b - want).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("n", [1, 255, 1000])
def test_droplet_round_trip(ddns, n):
    rng = np.random.default_rng(n)
    p = ddns.default_params(N=32, precision=0, npart=1000, nset=1, radius=[20.0])
    yp = np.asfortranarray(rng.random((8, n)))
    a = dict(fvp=np.asfortranarray(rng.random((3, 3, n))), fdp=np.asfortranarray(rng.random((3, 4, n))),
             pertvel=np.asfortranarray(rng.random((3, n))))
    with ddns.Solver(p) as s:
        s.set_droplets(yp, **a)
        d = s.get_droplets()
        assert np.array_equal(d["yp"], yp) and all(np.array_equal(d[k], a[k]) for k in a)
        s.set_droplets(yp[:, :n // 2])
        d = s.get_droplets()
        assert np.array_equal(d["yp"], yp[:, :n // 2]) and not any(d[k].any() for k in a)


@pytest.mark.parametrize("n", [3, 6800, 27000, 40000])
def test_some_of_the_droplet_arrays(ddns, n):
    """Each array alone, pairs of them and all give the same values: outputs of up to 2 MB go to the
    caller through one copy, larger ones array by array."""
    rng = np.random.default_rng(n)
    p = ddns.default_params(N=32, precision=0, npart=n, nset=1, radius=[5.0], dt=1e-6)
    size = dict(yp=8, fvp=9, fdp=12, pertvel=3, vp=3, dmove=3)
    with ddns.Solver(p) as s:
        s.init_flow(ddns.SPEC_K4_GAUSS, 3, 4.0, 0.1)
        s.init_droplets(seed=5)
        s.step(2)
        d = s.get_droplets()
        s.set_droplets(d["yp"], d["fvp"], d["fdp"], np.asfortranarray(rng.random((3, n))))
        every = {k: np.ravel(a, order="F") for k, a in s.get_droplets().items()}
        assert all(every[k].size == size[k] * n and every[k].any() for k in size)
        for chosen in ([k] for k in size):
            chosen = chosen + list(size)[::3]
            out = {k: np.full(size[k] * n, np.nan) for k in chosen}
            ptr = [out[k].ctypes.data_as(ctypes.POINTER(ctypes.c_double)) if k in out else None for k in size]
            assert s.lib.ddns_get_droplets(s.h, None, *ptr) == 0
            assert all(np.array_equal(out[k], every[k]) for k in out)
