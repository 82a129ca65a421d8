"""The near fill by (test edge, source triangle) against the general
evaluation of single blocks (spk_near_blocks), where it can go wrong: row
tiles with remainders, several column chunks per box, a closed surface, lossy
media, each formulation it takes and, beside them, the calls that stay on the
general fill (an edge of three triangles, the seven-point rule, MCTF2, CNF).

Tolerance: coordinates of a few wavelengths are rounded to 1e-16 of
themselves, up to 1e-13 of a distance between neighbouring points, and the
kernel's 1/R^3 terms triple that; the Taylor term's remainder is 1e-15.  1e-11
of the row's largest entry holds both with room.
"""
import numpy as np
import pytest

from specklesim_amd import SieTriMlfmm, meshes

pytestmark = pytest.mark.gpu
LAM = 633e-9


def _fin(pp, tt):
    """A third triangle on an interior edge."""
    a, b = tt[0][0], tt[0][2]
    top = 0.5 * (pp[a - 1] + pp[b - 1]) + np.array([0, 0, 0.1 * LAM])
    return np.vstack([pp, top]), np.vstack([tt, [[a, b, len(pp) + 1]]]).astype(np.int32)


def _mesh(kind):
    if kind == "sphere":
        return meshes.icosphere(2, 0.5 * LAM)
    if kind == "wide":  # 1157 columns in one box's rows: two chunks
        return meshes.rough_surface(21, 19, 2.1, 1.9, 0.1, 0.5, 6, LAM)
    pp, tt = meshes.rough_surface(15, 14, 1.5, 1.4, 0.1, 0.5, 6, LAM)
    return _fin(pp, tt) if kind == "fin" else (pp, tt)


@pytest.mark.parametrize("form,kind,s_opt,eps,ng", [
    ("ICTF", "patch", 250, 2.25, 3),
    ("ICTF", "patch", 20, 2.25, 3),
    ("ICTF", "patch", 4000, 2.25 - 0.3j, 3),
    ("PMCHWT", "sphere", 60, 2.25, 3),
    ("PMCHWT", "patch", 4000, 2.25 - 0.3j, 3),
    ("MCTF", "patch", 100, 4.0, 3),
    ("PMCHWT-S", "sphere", 4000, 2.25 - 0.3j, 3),
    ("PMCHWT-S", "patch", 50, 2.25, 3),
    ("ICTF", "wide", 4000, 2.25, 3),
    ("PMCHWT-S", "wide", 4000, 2.25 - 0.3j, 3),
    ("ICTF", "fin", 100, 2.25, 3),
    ("ICTF", "patch", 250, 2.25, 7),
    ("MCTF2", "patch", 250, 2.25, 3),
    ("CNF", "sphere", 250, 2.25, 3),
])
def test_near_blocks_equal_single_blocks(form, kind, s_opt, eps, ng):
    pp, tt = _mesh(kind)
    g = SieTriMlfmm(LAM, eps, formulation=form, ng=ng, tree_s_opt=s_opt).precalculation_tri(pp, tt)
    ia, ja, v = g.near_csr()
    assert kind != "wide" or np.diff(ia).max() > 1024
    rows = np.repeat(np.arange(g.N), np.diff(ia))
    pick = np.random.default_rng(1).permutation(len(ja))[:6000]
    # every column of the first and the last row too
    pick = np.unique(np.concatenate([pick, np.arange(ia[1]), np.arange(ia[-2], ia[-1])]))
    ref = g.impedance_edges(rows[pick], ja[pick]).reshape(-1, 4)
    got = v.reshape(-1, 4)[pick]
    assert np.isfinite(got).all()
    scale = np.zeros((g.N, 4))
    np.maximum.at(scale, rows, np.abs(v.reshape(-1, 4)))
    err = np.abs(got - ref) / np.maximum(scale[rows[pick]], 1e-300)
    assert err.max() < 1e-11, (err.max(), np.unravel_index(err.argmax(), err.shape))
