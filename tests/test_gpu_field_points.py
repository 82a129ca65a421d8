"""The scattered field over its launch shapes (one point, a tile's edges, chunks
of 8, 16 and 64 sources, enough points for a single chunk), media and distances
(arguments beyond the short reduction of sine and cosine), against the oracle.

Tolerance: a sum of about 10^4 terms in FP64, 1e-12; at a distance of a
kilometre k R is 1e10 and its rounding alone 1e-6.
"""
import numpy as np
import pytest

from oracle import oracle as O
from specklesim_amd import SieTriMlfmm, meshes

pytestmark = pytest.mark.gpu
LAM = 633e-9


@pytest.mark.parametrize("npts,dist,eps1,tol", [
    (1, 3 * LAM, 1.0, 1e-12), (63, 2 * LAM, 1.0, 1e-12), (64, 2 * LAM, 1.3 - 0.05j, 1e-12),
    (65, 1e3 * LAM, 1.0, 1e-11), (900, 2 * LAM, 1.3 - 0.05j, 1e-12), (7, 1e3, 1.0, 1e-5),
    (7, 1e3, 1.3 - 1e-10j, 1e-5), (131073, 2 * LAM, 1.0, 1e-12),
])
def test_scattered_field(npts, dist, eps1, tol):
    pp, tt = meshes.rough_surface(9, 7, 0.9, 0.7, 0.1, 0.5, 3, LAM)
    g = SieTriMlfmm(LAM, 2.25, eps_r1=eps1, formulation="ICTF", normal_convention=2)
    g.precalculation_tri(pp, tt)
    rng = np.random.default_rng(2)
    x = rng.standard_normal(2 * g.N) + 1j * rng.standard_normal(2 * g.N)
    d = rng.standard_normal((npts, 3))
    pts = d / np.linalg.norm(d, axis=1)[:, None] * dist
    E, H = g.scattered_field(pts, x)
    some = np.unique(np.r_[0, npts - 1, rng.integers(0, npts, 40)])
    o = O.Oracle(pp, tt, LAM, 2.25, eps_r1=eps1, formulation="ICTF", normal_convention=2)
    Eo, Ho = o.scattered_field(pts[some], x)
    assert np.linalg.norm(E[some] - Eo) < tol * np.linalg.norm(Eo)
    assert np.linalg.norm(H[some] - Ho) < tol * np.linalg.norm(Ho)
