"""Neighbour walks: rows of cells as runs of the sorted droplets, across the periodic faces, on the
coarsest grids, on a shared grid and on two, with one or four lanes a row."""
import numpy as np
import pytest

from helpers import random_droplets

pytestmark = pytest.mark.gpu


def _params(ddns, n, trunc, radius, **over):
    return ddns.default_params(N=32, precision=0, npart=n, radius=radius, forcing=0, dt=1e-3, rnu=0.02, gravity=980.0,
                               hdi_included=1, hdi_trunc=trunc, nonoverlap=1, new_particle=1, gmres_tol=1e-12,
                               gmres_maxiter=50, **over)


def _apart(n, rad, box, seed):
    """n droplets in box = (low, high) per axis that do not overlap: random places, the later of
    two close ones dropped."""
    from scipy.spatial import cKDTree
    yp = random_droplets(2 * n + 50, seed, rad)
    low, high = np.array(box, dtype=float).T
    yp[:3] = (low + (high - low) * yp[:3].T / (2 * np.pi)).T
    pairs = cKDTree(np.mod(yp[:3].T, 2 * np.pi), boxsize=2 * np.pi).query_pairs(2.2 * np.max(rad), output_type="ndarray")
    keep = np.ones(yp.shape[1], bool)
    keep[pairs.max(axis=1) if len(pairs) else []] = False
    yp = yp[:, keep][:, :n]
    assert yp.shape[1] == n
    yp[7] = np.arange(1, n + 1)
    return np.asfortranarray(yp)


# reach of the HI lists in box lengths / 2 pi: three cells an axis, five, many; the fullest
# of them has more than four droplets a cell, so the collision search gets its own grid
@pytest.mark.parametrize("n,reach,span", [(60, 2.0, 1.0), (700, 1.2, 1.0), (400, 0.5, 0.4), (3000, 0.35, 0.35), (3000, 0.35, 1.0)])
def test_two_steps_match_oracle(ddns, oracle_mod, n, reach, span):
    p = _params(ddns, n, 10.0, [25.0, 40.0])
    with oracle_mod.Oracle(p) as o:
        rad = o.scaling()["radius"][:2]
    p.hdi_trunc = reach / rad[1]
    yp = _apart(n, rad, [(-0.5 * span, 2 * np.pi * span - 0.5 * span)] * 3 if span < 1 else [(0, 2 * np.pi)] * 3, n)
    yp[:3] = np.mod(yp[:3], 2 * np.pi)
    with oracle_mod.Oracle(p) as o, ddns.Solver(p) as s:
        for x in (o, s):
            x.set_droplets(yp)
            x.step(2)
        a, b = s.get_droplets(), o.get_droplets()
        ca, cb = s.collision_counts(), o.collision_counts()
        assert (ca.ncoll, list(ca.icc), list(ca.nir)) == (cb.ncoll, list(cb.icc), list(cb.nir))
        assert np.allclose(a["yp"], b["yp"], rtol=1e-9, atol=1e-9)
        assert np.abs(a["pertvel"] - b["pertvel"]).max() <= 1e-9 * np.abs(b["pertvel"]).max()


def test_one_lane_a_row_as_four(ddns, oracle_mod):
    """131 072 droplets share four lanes a row; one more, beyond the reach of all others, has every
    row walked by a single lane.  The others' solution is the same to the solver's tolerance."""
    n = 131072
    p = _params(ddns, n + 1, 10.0, [8.0])
    p.capacity = n + 1
    with oracle_mod.Oracle(_params(ddns, 10, 10.0, [8.0])) as o:
        rad = o.scaling()["radius"][:1]
    p.hdi_trunc = 0.12 / rad[0]
    yp = _apart(n + 1, rad, [(0, 2 * np.pi), (0, 2 * np.pi), (0, 6.0)], 5)
    yp[:3, n] = (1.0, 1.0, 6.14)                     # 0.14 from both ends of the others
    got = []
    for m in (n, n + 1):
        with ddns.Solver(p) as s:
            s.set_droplets(np.asfortranarray(yp[:, :m]))
            s.step(1)
            got.append(s.get_droplets()["pertvel"][:, :n])
    assert np.abs(got[0]).max() > 0
    assert np.abs(got[0] - got[1]).max() <= 1e-9 * np.abs(got[0]).max()
