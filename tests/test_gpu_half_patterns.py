"""Pattern rows that keep half of the sample directions (media of real
wavenumber) and whole rows (media with losses), in every kernel that reads
them: patterns, products of one and several vectors in both precisions and the
transposed product, for odd and even truncation numbers (an even K leaves an
odd half, padded), against the oracle's operator on all samples.

Tolerances: the products are held to 1e-9, the bound of the translation sums'
cancellation on these leaf boxes (0.58 wavelengths, K <= 19: 4e-11 measured);
complex64 has 2^29 times FP64's rounding, held to 1e-2 as a whole.  The far part
alone (the complex64 product less its near part, each half of the vector by
itself) is held to four times what is measured: 3.2e-6 for K <= 13, where the
translation sums hardly cancel and complex64's own rounding and the near part's
are what is left, 5.4e-3 for K = 19, where they cancel 1e5 times their result.
An edge left out of a box changes it by some 1e-2.
"""
import numpy as np
import pytest

from oracle import oracle as O
from specklesim_amd import SieTriMlfmm, meshes

pytestmark = pytest.mark.gpu
LAM = 633e-9


@pytest.fixture(scope="module")
def mesh():
    return meshes.rough_surface(24, 24, 2.4, 2.4, 0.1, 0.5, 9, LAM)


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _far_err(g, X, far, y, batched):
    """the worst half of the worst vector"""
    f = y.astype(np.complex128) - g.near_product_lowp(X, "c64", batched=batched)
    return max(_rel(f[r, h], far[r, h]) for r in range(len(X))
               for h in (slice(0, g.N), slice(g.N, None)))


@pytest.mark.parametrize("K,eps1,eps2", [
    (19, 1.0, 2.25), (12, 1.0, 2.25), (13, 1.0, 2.25 - 0.2j), (12, 1.2 - 0.1j, 2.25),
    (8, 1.2 - 0.1j, 2.25 - 0.2j), (3, 1.0, 2.25),
])
def test_products_on_half_and_whole_rows(mesh, K, eps1, eps2):
    _check(*mesh, K, eps1, eps2)


@pytest.mark.parametrize("K,eps1,eps2", [(12, 1.0, 2.25), (9, 1.0, 2.25 - 0.2j),
                                         (8, 1.2 - 0.1j, 2.25 - 0.2j)])
def test_boxes_of_more_edges_than_a_stage(K, eps1, eps2):
    """147 to 176 edges a box: two stages of the single-vector aggregation's x
    and two tiles of the matrix-core disaggregation."""
    _check(*meshes.rough_surface(30, 30, 3.0, 3.0, 0.1, 0.5, 9, LAM), K, eps1, eps2)


def _check(pp, tt, K, eps1, eps2):
    kw = dict(eps_r1=eps1, formulation="ICTF", normal_convention=2)
    o = O.Oracle(pp, tt, LAM, eps2, K=K, **kw)
    o.tree()
    o.near_csr(fill=True)
    o.mlfmm_setup()
    g = SieTriMlfmm(LAM, eps2, truncation_number=K, precision="mixed", **kw).precalculation_tri(pp, tt)
    pat = g.patterns(0, 40)
    for m in (0, 7, 39):
        ref = o.pattern(m)
        assert np.abs(pat[m] - ref).max() < 1e-12 * np.abs(ref).max()
    rng = np.random.default_rng(3)
    X = rng.standard_normal((16, 2 * g.N)) + 1j * rng.standard_normal((16, 2 * g.N))
    Y = np.stack([o.matvec(x) for x in X])
    assert _rel(g.calculate_vector_b_tri(X[0]), Y[0]) < 1e-9
    assert _rel(g.calculate_vector_b_tri_c64(X[0]), Y[0]) < 1e-2
    for R in (1, 2, 3, 7, 9, 16):
        assert _rel(g.calculate_vector_b_tri_batch(X[:R]), Y[:R]) < 1e-9, R
        assert _rel(g.calculate_vector_b_tri_batch(X[:R], c64=True), Y[:R]) < 1e-2, R
    F = X.astype(np.complex64)
    near, far = (np.stack(v) for v in zip(*[g.matvec_parts(x) for x in F]))
    assert _rel(near + far, Y) < 1e-6  # F is X to 24 bits
    tol = 1.3e-5 if K <= 13 else 2.2e-2
    assert _far_err(g, F[:1], far, g.calculate_vector_b_tri_c64(F[0])[None], False) < tol
    for R in (1, 2, 3, 7, 9, 16):
        assert _far_err(g, F[:R], far, g.calculate_vector_b_tri_batch(F[:R], c64=True), True) < tol, R
    # u.(Z^T v) = v.(Z u)
    g.set_transposed(True)
    far_t = g.matvec_parts(F[0])[1][None]
    assert _far_err(g, F[:1], far_t, g.calculate_vector_b_tri_c64(F[0])[None], False) < tol
    t = X[1] @ g.calculate_vector_b_tri(X[2])
    assert abs(t - X[2] @ Y[1]) < 1e-9 * np.linalg.norm(X[2]) * np.linalg.norm(Y[1])
