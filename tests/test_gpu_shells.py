"""The shell sums of the diagnostics (E, D and, with the nonlinear term, T) against the field
they are taken of, on grids where the work-groups of their kernel hold 16 and 8 wavefronts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [32, 64, 128, 256])
def test_shell_sums_against_the_field(ddns, N, precision):
    p = ddns.default_params(N=N, precision=precision, dt=0.0005, rnu=0.01)
    with ddns.Solver(p) as s:
        s.init_flow(ddns.SPEC_KOLMOGOROV, 5)
        s.step(1)
        e, d, t = s.spectra()
        ek = s.spectrum()
        m = s.monitors()
        v, _ = s.get_flow()
    k = np.where(np.arange(N) <= N // 2, np.arange(N), np.arange(N) - N).astype(float)
    kx = np.arange(N // 2).astype(float)
    k2 = k[:, None, None] ** 2 + kx[None, :, None] ** 2 + k[None, None, :] ** 2      # kz, kx, ky
    shell = np.floor(np.sqrt(k2) + 0.5).astype(int)
    e2 = sum(a[:N, 0:N:2] ** 2 + a[:N, 1:N:2] ** 2 for a in v)
    e2[:, 0] *= 0.5
    nek = len(e)
    want_e = np.bincount(shell.ravel(), weights=e2.ravel(), minlength=nek + 1)[1:nek + 1]
    want_d = np.bincount(shell.ravel(), weights=(2 * p.rnu * k2 * e2).ravel(), minlength=nek + 1)[1:nek + 1]
    # sums of up to N^3 / 2 doubles of one sign in another order: N^3 eps at the very worst
    assert np.allclose(e, want_e, rtol=1e-12, atol=0) and np.allclose(d, want_d, rtol=1e-12, atol=0)
    assert np.allclose(ek, want_e, rtol=1e-12, atol=0)
    assert abs(m.qq - want_e.sum()) <= 1e-12 * m.qq and abs(m.dissp - want_d.sum()) <= 1e-12 * m.dissp
    # the nonlinear term conserves energy: T sums to zero to the precision of its transforms
    assert abs(t.sum()) <= (1e-11 if precision == 0 else 1e-4) * np.abs(t).sum()


def test_shell_sums_eight_wavefronts(ddns):
    """512^3: the tables of three sums leave a work-group 8 wavefronts."""
    with ddns.Solver(ddns.default_params(N=512, precision=1, dt=0.0005, rnu=0.01)) as s:
        s.init_flow(ddns.SPEC_KOLMOGOROV, 5)
        e, d, t = s.spectra()
        m = s.monitors()
        assert np.allclose(e, s.spectrum(), rtol=1e-12, atol=0)
        assert abs(m.dissp - d.sum()) <= 1e-12 * m.dissp
        assert abs(t.sum()) <= 1e-4 * np.abs(t).sum()
