"""The domain solves of the RAS preconditioner against dense solves. A vector
that is zero on the coarse grid passes the first coarse solve unchanged, so the
entries of one application outside the coarse grid are the fine domains' own
solutions (ras_preconditioner.hpp:191-250, fine_grid.hpp:97-142)."""
import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu


def monomials(degree, p):
    cols = [np.ones(len(p))] if degree >= 0 else []
    if degree >= 1:
        cols += list(p.T)
    if degree >= 2:
        x, y, z = p.T
        cols += [x * x, x * y, x * z, y * y, y * z, z * z]
    return np.stack(cols, 1) if cols else np.zeros((len(p), 0))


# Domain sizes that are and are not multiples of the solve's 32-wide blocks; the
# last one has more than 1,024 domains, which take a smaller workgroup and rows
# beyond those that it loads ahead.
@pytest.mark.parametrize("n,degree,fp32", [(2100, -1, True), (3000, 0, True), (5000, 1, False), (9000, 2, True),
                                           (12345, 0, False), (450_000, 0, True)])
def test_domain_solves(n, degree, fp32):
    print("domain solves", n, degree, fp32, flush=True)
    rng = np.random.default_rng(n)
    pts = rng.uniform(0, 1, (n, 3))
    nugget = 10.0
    rbf = pa.CovExponential([1.0, 0.5]) if degree < 1 else pa.Biharmonic3D()
    model = pa.Model(rbf, degree, nugget=nugget)
    l = model.poly_basis_size()
    ras = pa.RasPreconditioner(model, pts, pa.FitOptions(ras_fp32_factors=fp32))
    top = ras.n_levels() - 1
    if n < 20000:
        assert top == 1
    outside = np.ones(n, bool)
    for level in range(top):
        outside[ras.level_points(level)] = False
    doms = ras.domains(top)
    if n > 20000:
        assert len(doms) >= 1024
    # Non-zero outside the lower levels, and only on two domains' points, so
    # that the other levels' solves see zeros up to the last one.
    chosen = [0, len(doms) // 2]
    v = np.zeros(n + l)
    mask = np.zeros(n, bool)
    for k in chosen:
        mask[doms[k][0]] = True
    v[:n][mask & outside] = rng.normal(size=int((mask & outside).sum()))
    w = ras.apply(v)
    u = 2.0 ** -24 if fp32 else 2.0 ** -53
    diffs, at, bound = [], [], 0.0
    for k in chosen:
        idx, inner = doms[k]
        p = pts[idx]
        r = np.linalg.norm(p[:, None] - p[None], axis=2)
        a = np.exp(-3 * r / 0.5) if degree < 1 else -r
        a[np.diag_indices(len(idx))] += nugget
        q = monomials(degree, p)
        big = np.block([[a, q], [q.T, np.zeros((l, l))]])
        lam = np.linalg.solve(big, np.concatenate([v[idx], np.zeros(l)]))[:len(idx)]
        # the constraint eliminated through the first l points
        e = -np.linalg.solve(q[:l].T, q[l:].T) if l else np.zeros((0, len(idx)))
        z = np.vstack([e, np.eye(len(idx) - l)])
        cond = np.linalg.cond(z.T @ a @ z)
        own = inner & outside[idx]
        assert own.any()
        diffs.append(w[idx][own] - lam[own])
        at.append(p[own])
        b = len(idx) * u * cond * np.abs(lam).max()  # backward error n u of the factorisation
        print(f"  {len(idx)} points, cond {cond:.1e}, bound {b:.2e}", flush=True)
        bound = max(bound, b)
    # After the solve the sum is made orthogonal to the polynomials, which
    # subtracts one polynomial from all entries.
    diff, q = np.concatenate(diffs), monomials(degree, np.concatenate(at))
    if l:
        diff = diff - q @ np.linalg.lstsq(q, diff, rcond=None)[0]
    print(f"  error {np.abs(diff).max():.2e}", flush=True)
    assert np.abs(diff).max() <= bound
