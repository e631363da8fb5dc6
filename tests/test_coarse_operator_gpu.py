"""The coarse grid as the whole preconditioner: below 2,048 rows there is one
level, so applying it solves [A + nugget I, P; P^T, 0] exactly. Sizes sit on
the edges of the 64-wide panels and 16-wide blocks of the dense factorisation,
inverse and operator. Calls go through the C ABI."""
import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,degree", [("bh3", 1), ("bh3", 0), ("exp", -1), ("exp", 0), ("th3", 2)])
@pytest.mark.parametrize("n", [12, 65, 68, 128 + 4, 129 + 10, 257, 700, 1537, 2047])
def test_one_level_preconditioner_solves_the_system(orc, kind, degree, n):
    print("coarse operator", kind, degree, n, flush=True)
    rng = np.random.default_rng(n)
    pts = rng.uniform(0, 1, (n, 3))
    rbf = {"bh3": pa.Biharmonic3D, "th3": pa.Triharmonic3D}.get(kind, lambda: pa.CovExponential([1.0, 0.5]))()
    nugget = 0.01
    pc = pa.RasPreconditioner(pa.Model(rbf, poly_degree=degree, nugget=nugget), pts)
    assert pc.n_levels() == 1
    # A vector is in the operator's range for any d; check the residual of the
    # dense system, scaled as for a backward stable solve: n ulps of |A| |x|.
    l = {-1: 0, 0: 1, 1: 4, 2: 10}[degree]
    d = np.concatenate([rng.normal(size=n), np.zeros(l)])
    x = pc.apply(d)
    r = np.linalg.norm(pts[:, None, :] - pts[None, :, :], axis=2)
    a = {"bh3": -r, "th3": r ** 3, "exp": np.exp(-6.0 * r)}[kind] + nugget * np.eye(n)
    cols = [np.ones(n), *pts.T] + [pts[:, i] * pts[:, j] for i in range(3) for j in range(i, 3)]
    p = np.array(cols[:l]).T.reshape(n, l)
    res = a @ x[:n] + p @ x[n:] - d[:n]
    # The weights' null-space form costs the condition of Q, below 1e3 here.
    scale = np.abs(a) @ np.abs(x[:n]) + np.abs(p) @ np.abs(x[n:])
    worst = np.max(np.abs(res) / scale.max())
    ortho = np.abs(p.T @ x[:n]).max() / max(np.abs(x[:n]).sum(), 1e-300) if l else 0.0
    print(f"  residual {worst:.2e}, P^T w {ortho:.2e}", flush=True)
    assert worst <= 1e3 * n * 2.2e-16
    assert ortho <= 1e3 * n * 2.2e-16
