"""The FP64 direct sums over every split of targets and sources (one target to
two per thread, one source to several chunks), against numpy; coincident
points, and distances whose squares overflow. Calls go through the C ABI."""
import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu

ANISO = np.array([[1.1, 0.2, 0.0], [0.0, 0.9, 0.1], [0.1, 0.0, 1.2]])


def make(kind):
    r = {"bh3": lambda: pa.Biharmonic3D([1.5, 0.0]), "bh3c": lambda: pa.Biharmonic3D([1.0, 0.2]),
         "th3": lambda: pa.Triharmonic3D([0.7, 0.0]), "exp": lambda: pa.CovExponential([1.2, 0.4])}[kind]()
    r.set_anisotropy(ANISO)
    return r


def terms(rbf, src, trg):
    """u = A (t - s), phi, grad factor f and Hessian coefficient t (H = f (I + t u u^T))."""
    u = (trg[:, None, :] - src[None, :, :]) @ rbf.anisotropy().T
    q = (u * u).sum(-1)
    p0, p1 = rbf.parameters()
    with np.errstate(all="ignore"):
        if rbf.short_name == "exp":
            r = np.sqrt(q)
            phi = p0 * np.exp(-3 * r / p1)
            f = -3 * phi / (p1 * r)
            t = -(1 + 3 * r / p1) / q
        else:
            rho2 = q + p1 * p1
            rho = np.sqrt(rho2)
            zero = rho == 0
            if rbf.short_name == "bh3":
                phi, f, t = -p0 * rho, np.where(zero, 0, -p0 / rho), np.where(zero, 0, -1 / rho2)
            else:
                phi, f, t = p0 * rho ** 3, 3 * p0 * rho, np.where(zero, 0, 1 / rho2)
    return u, phi, f, t


def close(y, ref, mag):
    # sums of n terms in some order, each term within a few ulp
    tol = 2.0 ** -52 * (8 + 4 * np.log2(len(mag) + 2)) * np.abs(mag).sum(0 if mag.ndim == 1 else 1) + 1e-300
    assert np.all(np.abs(y - ref) <= 64 * tol)


@pytest.mark.parametrize("kind", ["bh3", "bh3c", "th3", "exp"])
@pytest.mark.parametrize("n_trg,n_src", [(1, 1), (1, 1000), (2, 16385), (31, 257), (33, 513), (64, 4097), (65, 255),
                                         (257, 10_000), (32767, 65), (32768, 70), (33001, 1025)])
def test_values(kind, n_trg, n_src):
    print("direct values", kind, n_trg, n_src, flush=True)
    rng = np.random.default_rng(n_trg + n_src)
    src, trg, w = rng.uniform(0, 1, (n_src, 3)), rng.uniform(0, 1, (n_trg, 3)), rng.normal(size=n_src)
    k = min(n_src, n_trg) // 2
    trg[:k] = src[:k]
    rbf = make(kind)
    y = pa.direct_evaluate(rbf, src, w, trg)
    rows = np.unique(np.concatenate([np.arange(min(n_trg, 300)), np.arange(max(0, n_trg - 300), n_trg)]))
    _, phi, _, _ = terms(rbf, src, trg[rows])
    close(y[rows], phi @ w, phi * w)


@pytest.mark.parametrize("kind", ["bh3", "bh3c", "th3", "exp"])
@pytest.mark.parametrize("n_trg,n_src", [(1, 300), (63, 1), (257, 1500), (33_000, 300)])
def test_gradients_and_vector_weights(kind, n_trg, n_src):
    print("direct gradients", kind, n_trg, n_src, flush=True)
    rng = np.random.default_rng(n_trg + n_src)
    src, trg = rng.uniform(0, 1, (n_src, 3)), rng.uniform(0, 1, (n_trg, 3))
    w, w3 = rng.normal(size=n_src), rng.normal(size=(n_src, 3))
    if kind != "exp":  # its derivatives are undefined at the sources
        k = min(n_src, n_trg) // 2
        trg[:k] = src[:k]
    rbf = make(kind)
    rows = np.unique(np.concatenate([np.arange(min(n_trg, 200)), np.arange(max(0, n_trg - 200), n_trg)]))
    u, _, f, t = terms(rbf, src, trg[rows])
    g = np.einsum("ij,ijk->ijk", f, u) @ rbf.anisotropy()
    y = pa.direct_evaluate_gradient(rbf, src, w, trg)[rows]
    for c in range(3):
        close(y[:, c], g[:, :, c] @ w, g[:, :, c] * w)
    cfg = pa.FmmConfig("fp64", 10, -1, "direct")
    v = w3 @ rbf.anisotropy().T
    uv = np.einsum("ijk,jk->ij", u, v)
    ev = pa.make_fmm_gradient_evaluator(rbf)
    he = pa.make_fmm_hessian_evaluator(rbf)
    for e in (ev, he):
        e.set_config(cfg)
        e.set_source_points(src)
        e.set_weights(w3.ravel())
        e.set_target_points(trg)
    mag = np.abs(f) * np.sqrt((u * u).sum(-1)) * np.linalg.norm(v, axis=1)
    close(ev.evaluate()[rows], -(f * uv).sum(1), mag)
    h = -(f[:, :, None] * (v[None] + (t * uv)[:, :, None] * u)) @ rbf.anisotropy()
    hm = np.abs(f) * np.linalg.norm(v, axis=1) * (1 + np.abs(t) * (u * u).sum(-1)) * 2
    y = he.evaluate()[rows]
    assert he.stats()["direct"] == 1
    for c in range(3):
        close(y[:, c], h[:, :, c].sum(1), hm)


def test_columns_of_the_hessian_equal_the_vector_sum():
    rng = np.random.default_rng(9)
    src, trg, w = rng.uniform(0, 1, (700, 3)), rng.uniform(0, 1, (90, 3)), rng.normal(size=700)
    rbf = make("th3")
    for k in range(3):
        e3 = np.zeros((700, 3))
        e3[:, k] = w
        he = pa.make_fmm_hessian_evaluator(rbf)
        he.set_config(pa.FmmConfig("fp64", 10, -1, "direct"))
        he.set_source_points(src)
        he.set_weights(e3.ravel())
        he.set_target_points(trg)
        u, _, f, t = terms(rbf, src, trg)
        v = e3 @ rbf.anisotropy().T
        uv = np.einsum("ijk,jk->ij", u, v)
        h = -(f[:, :, None] * (v[None] + (t * uv)[:, :, None] * u)) @ rbf.anisotropy()
        np.testing.assert_allclose(he.evaluate(), h.sum(1), rtol=1e-11, atol=1e-11)


def test_overflowing_distances_keep_their_infinities():
    src = np.array([[0.0, 0.0, 0.0], [1e200, 0.0, 0.0]])
    trg = np.array([[1.0, 0.0, 0.0], [1e200, 0.0, 0.0], [3.0, 4.0, 0.0]])
    y = pa.direct_evaluate(pa.Biharmonic3D(), src, np.array([1.0, 1.0]), trg)
    assert np.array_equal(np.isinf(y), [True, True, True]) and np.all(y < 0)
    y = pa.direct_evaluate(pa.CovExponential([1.0, 1.0]), src, np.array([1.0, 1.0]), trg)
    np.testing.assert_allclose(y, [np.exp(-3.0), 1.0, np.exp(-15.0)], rtol=1e-14)
    y = pa.direct_evaluate(pa.Biharmonic3D(), src[:1], np.array([np.nan]), trg[:1])
    assert np.isnan(y[0])


@pytest.mark.parametrize("accuracy", [None, 1e-4])
@pytest.mark.parametrize("make_evaluator,per", [(pa.make_fmm_gradient_evaluator, 1), (pa.make_fmm_hessian_evaluator, 3)])
def test_first_sum_over_vector_weights_goes_the_way_of_the_next(make_evaluator, per, accuracy):
    """Without a fixed configuration the first evaluation chooses one; its
    values are the bits of the second's, and so are those after new points."""
    rng = np.random.default_rng(31)
    ev = make_evaluator(make("th3"))
    if accuracy is not None:
        ev.set_accuracy(accuracy)
    for n_src, n_trg in ((700, 900), (2500, 40)):
        src, trg = rng.uniform(0, 1, (n_src, 3)), rng.uniform(0, 1, (n_trg, 3))
        w = rng.normal(size=(n_src, 3))
        ev.set_source_points(src)
        ev.set_target_points(trg)
        ev.set_weights(w.ravel())
        first = ev.evaluate()
        assert ev.stats()["direct"] == 1
        np.testing.assert_array_equal(first, ev.evaluate())
        fixed = make_evaluator(make("th3"))
        fixed.set_config(pa.FmmConfig("fp64", 10, -1, "direct"))
        fixed.set_source_points(src)
        fixed.set_target_points(trg)
        fixed.set_weights(w.ravel())
        np.testing.assert_array_equal(first, fixed.evaluate())
