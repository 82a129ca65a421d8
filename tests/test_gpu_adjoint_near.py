"""The near-block share of the adjoint gradient by triangle pairs, for every
formulation that takes it, media with losses and a closed surface, against
dense algebra: on a surface of one octree level every pair is near, so Z and its
central difference come from single blocks of the moved meshes
(spk_near_blocks), the currents and the adjoint vector from dense solves.  The
seven-point rule and MCTF2 stay on the per-entry kernel.

Tolerance: the solves of the library stop at 1e-10, on systems of condition up
to 1e4; 1e-5 of the largest share.
"""
import numpy as np
import pytest

from specklesim_amd import SieTriMlfmm, meshes, plane_wave

pytestmark = pytest.mark.gpu
LAM = 633e-9
DZ = 1e-6 * LAM


def _dense(pp, tt, kw):
    g = SieTriMlfmm(LAM, **kw).precalculation_tri(pp, tt)
    N = g.N
    i, j = np.divmod(np.arange(N * N), N)
    b = g.impedance_edges(i, j).reshape(N, N, 2, 2)
    return g, b.transpose(2, 0, 3, 1).reshape(2 * N, 2 * N)


@pytest.mark.parametrize("form,eps,kind,ng", [
    ("ICTF", 2.25, "patch", 3), ("ICTF", 2.25 - 0.4j, "sphere", 3), ("PMCHWT", 2.25, "sphere", 3),
    ("MCTF", 2.25, "patch", 3), ("PMCHWT-S", 2.25 - 0.4j, "patch", 3), ("ICTF", 2.25, "patch", 7),
    ("MCTF2", 2.25, "patch", 3),
])
def test_near_share(form, eps, kind, ng):
    if kind == "patch":
        pp, tt = meshes.rough_surface(7, 6, 0.7, 0.6, 0.1, 0.5, 3, LAM)
    else:
        pp, tt = meshes.icosphere(1, 0.3 * LAM)
    kw = dict(eps_r2=eps, formulation=form, normal_convention=2, ng=ng)
    g, Z = _dense(pp, tt, kw)
    k, e = plane_wave(0.3, 0.0, 2, "TM")
    d = np.random.default_rng(1).standard_normal((6, 3))
    pts = 50 * LAM * d / np.linalg.norm(d, axis=1)[:, None]
    w = np.ones(6)
    nodes = np.array([0, 9, 17, 30])
    _, _, info, terms = g.adjoint_height_gradient(k, e, pts, w, nodes, dz=DZ, tolerance=1e-10,
                                                  return_terms=True)
    I = np.linalg.solve(Z, g.get_vector_b_tri(k, e))
    E, _ = g.scattered_field(pts, I)
    F = np.stack([g.scattered_field(pts, u)[0].ravel()
                  for u in np.eye(2 * g.N, dtype=complex)], axis=1)
    nu = np.linalg.solve(Z.T, F.T @ np.conj(E.ravel()))
    ref = []
    for n in nodes:
        dZ = 0
        for s in (1, -1):
            q = pp.copy()
            q[n, 2] += s * DZ
            dZ = dZ + s * _dense(q, tt, kw)[1]
        ref.append(-2 * (nu @ dZ @ I).real / (2 * DZ))
    ref = np.array(ref)
    assert np.abs(terms[:, 2] - ref).max() < 1e-5 * np.abs(ref).max(), (terms[:, 2], ref, info)
