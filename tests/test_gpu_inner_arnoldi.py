"""The inner Arnoldi steps of the near-field preconditioned solves against
flexible GMRES written out in numpy with the same operator and near blocks:
inner lengths at the edges of the update's column groups, one vector and a
batch (whose row chunks differ), on FP64 handles with the exact blocks and on
mixed ones, whose columns are complex64 and whose product is the fp8 or bf16 one
(in numpy too, one call of it per inner step).  The inner solve is the same
mathematics in another order, so the outer iteration counts may differ by one
where an estimate meets the tolerance; a wrong coefficient or scale in a
column costs many.  Zero inner residuals (a right-hand side of zeros) end at
once.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from specklesim_amd import DeviceBuffer, SieTriMlfmm, meshes, plane_wave

pytestmark = pytest.mark.gpu
LAM = 633e-9
TOL = 1e-6


def _gmres(mul, prec, b, steps, tol=0.0):
    """min |b - A sum z_j| over z_j = prec(v_j): the solution and the steps."""
    beta = np.linalg.norm(b)
    V, Z = [b / beta], []
    H = np.zeros((steps + 1, steps), complex)
    e = np.zeros(steps + 1)
    e[0] = beta
    for j in range(steps):
        Z.append(prec(V[j]))
        w = mul(Z[j])
        for _ in range(2):
            for i in range(j + 1):
                c = np.vdot(V[i], w)
                H[i, j] += c
                w = w - c * V[i]
        H[j + 1, j] = np.linalg.norm(w)
        y = np.linalg.lstsq(H[:j + 2, :j + 1], e[:j + 2], rcond=None)[0]
        if np.linalg.norm(e[:j + 2] - H[:j + 2, :j + 1] @ y) <= tol * beta:
            break
        V.append(w / H[j + 1, j])
    return np.column_stack(Z) @ y, j + 1


@pytest.fixture(scope="module")
def case():
    pp, tt = meshes.rough_surface(16, 16, 2.0, 2.0, 0.1, 0.5, 6, LAM)
    s = SieTriMlfmm(LAM, 2.25, formulation="ICTF", normal_convention=2).precalculation_tri(pp, tt)
    ia, ja, v = s.near_csr()
    v = v.reshape(-1, 4)
    A = sp.bmat([[sp.csr_matrix((v[:, 2 * i + j], ja, ia), shape=(s.N, s.N)) for j in range(2)]
                 for i in range(2)], format="csr")
    B = [s.get_vector_b_tri(*plane_wave(0.1 * r, 0.0, 2, "TM")) for r in range(5)]
    return s, A, B


@pytest.mark.parametrize("kin,tol", [(1, 0.1), (2, 0.03), (8, 1e-3), (9, 1e-3), (33, 1e-6), (64, 1e-6)])
def test_outer_iterations_match_numpy(case, kin, tol):
    s, A, B = case
    want = [_gmres(s.calculate_vector_b_tri, lambda v: _gmres(lambda z: A @ z, lambda z: z, v, kin)[0],
                   b, 90, tol)[1] for b in B[:2]]
    assert max(want) < 90
    for r in range(2):
        x, inf = s.gmres_run(B[r], tolerance=tol, use_initial_guess=False, near_field=True,
                             inner_iterations=kin)
        assert np.linalg.norm(B[r] - s.calculate_vector_b_tri(x)) <= 1.01 * tol * np.linalg.norm(B[r])
        assert abs(inf["iters"] - want[r]) <= 1, (kin, inf["iters"], want[r])
    bs = [DeviceBuffer(b.nbytes).upload(b) for b in B]
    xs = [DeviceBuffer(32 * s.N) for b in B]
    infos = s.gmres_run_batch_device([d.ptr for d in bs], [d.ptr for d in xs], tolerance=tol,
                                     use_initial_guess=False, near_field=True, inner_iterations=kin)
    for r in range(2):
        assert abs(infos[r]["iters"] - want[r]) <= 1, (kin, r, infos[r], want[r])


@pytest.fixture(scope="module")
def mixed(case):
    pp, tt = meshes.rough_surface(16, 16, 2.0, 2.0, 0.1, 0.5, 6, LAM)
    return SieTriMlfmm(LAM, 2.25, formulation="ICTF", normal_convention=2,
                       precision="mixed").precalculation_tri(pp, tt)


# 4 to 8 vectors take complex64 blocks, 9 and more the matrix-core products
@pytest.mark.parametrize("fmt,R,kin,tol", [
    ("fp8", 1, 1, 0.1), ("fp8", 1, 9, 1e-3), ("fp8", 1, 64, 1e-6), ("bf16", 1, 33, 1e-5),
    ("fp8", 3, 8, 1e-3), ("c64", 5, 9, 1e-3), ("c64", 5, 64, 1e-6), ("fp8", 10, 2, 0.03),
    ("fp8", 10, 33, 1e-6), ("bf16", 10, 33, 1e-6),
])
def test_low_precision_inner_steps_match_numpy(mixed, monkeypatch, fmt, R, kin, tol):
    s = mixed
    monkeypatch.setenv("SPK_NEAR_F8", "0" if fmt == "bf16" else "1")
    monkeypatch.setenv("SPK_RELAX", "0")

    def near(z):
        X = np.tile(z.astype(np.complex64), (R if R > 3 else 1, 1))
        return s.near_product_lowp(X, fmt, batched=R > 3)[0].astype(np.complex128)

    B = [s.get_vector_b_tri(*plane_wave(0.05 * r, 0.0, 2, "TM")) for r in range(R)]
    pick = sorted({0, R - 1})
    want = {r: _gmres(s.calculate_vector_b_tri, lambda v: _gmres(near, lambda z: z, v, kin)[0],
                      B[r], 90, tol)[1] for r in pick}
    bs = [DeviceBuffer(b.nbytes).upload(b) for b in B]
    xs = [DeviceBuffer(32 * s.N) for _ in B]
    kw = dict(tolerance=tol, use_initial_guess=False, near_field=True, inner_iterations=kin)
    infos = (s.gmres_run_batch_device([d.ptr for d in bs], [d.ptr for d in xs], **kw) if R > 1
             else [s.gmres_run_device(bs[0].ptr, xs[0].ptr, **kw)])
    for r in pick:
        x = xs[r].download()
        assert np.linalg.norm(B[r] - s.calculate_vector_b_tri(x)) <= 1.01 * tol * np.linalg.norm(B[r])
        assert abs(infos[r]["iters"] - want[r]) <= 1, (r, infos[r]["iters"], want[r])


def test_zero_right_hand_side_in_a_batch(case):
    s, _, B = case
    bs = [DeviceBuffer(b.nbytes).upload(b) for b in (B[0], np.zeros_like(B[0]), B[1])]
    xs = [DeviceBuffer(32 * s.N) for _ in bs]
    infos = s.gmres_run_batch_device([d.ptr for d in bs], [d.ptr for d in xs], tolerance=TOL,
                                     use_initial_guess=False, near_field=True)
    assert [i["info"] for i in infos][::2] == [0, 0] and infos[1]["iters"] == 0
