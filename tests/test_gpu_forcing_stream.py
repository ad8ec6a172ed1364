"""The random stream of the stochastic forcing from states at the edge of ranff: a seed that the
generator's modulus divides, and tables that hold a zero, which make it seed itself again
between two draws of one step (accesories.f90:49-58)."""
import numpy as np
import pytest

from helpers import rel_l2

pytestmark = pytest.mark.gpu

IM = 2147483647


@pytest.mark.parametrize("iseedf,iyf,zeros", [
    (-232300, 0, None),                 # an ordinary seed
    (-1, 0, None),
    (-IM, 0, None),                     # seeds itself to zeros, then to 1 at the second draw
    (IM, 5, ()),
    (12345, 0, ()),                     # seeds itself with 1
    (12345, 777777777, ()),
    (12345, 777777777, (0, 11, 31)),    # hands out zeros, and seeds itself after each
    (12345, 777777777, range(32)),
])
def test_draws_as_the_reference(ddns, oracle_mod, iseedf, iyf, zeros):
    N = 32
    iv = np.zeros(32, dtype=np.int32)
    if zeros is not None:
        iv[:] = np.random.default_rng(3).integers(1, IM, 32)
        iv[list(zeros)] = 0
    p = ddns.default_params(N=N, precision=0, forcing=2, dt=1e-3, rnu=0.02)
    with ddns.Solver(p) as s, oracle_mod.Oracle(p) as o:
        rest = [np.zeros((N + 2, N + 2, N), order="F") for _ in range(3)]
        o.flow_only(True)
        for x in (s, o):
            x.set_flow(rest, rest)
            x.set_forcing_state(np.zeros(450), iseedf, iyf, iv)
        for _ in range(2):
            s.step(1)
            o.step(1)
            (b, *a), (c, *d) = s.get_forcing_state(), o.get_forcing_state()
            assert a[:2] == d[:2] and np.array_equal(a[2], d[2])
            assert np.abs(b - c).max() <= 1e-13 * np.abs(c).max()
        assert rel_l2(s.get_flow()[0], o.get_flow()[0]) < 1e-11
