"""The near field alone: points inside the eight central leaves of a level-2
tree are all neighbours of each other, so no far field contributes. Sizes sit
on the edges of the mixed kernel's tiles (16 targets, 5 tiles per wave, 256
sources per chunk), the last one where the sources are shared out over several
workgroups. Calls go through the C ABI."""
import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu

KINDS = {"bh3": ("BH3", pa.Biharmonic3D, [1.5, 0.0]), "bh3c": ("BH3", pa.Biharmonic3D, [1.0, 0.03]),
         "th3": ("TH3", pa.Triharmonic3D, [0.7, 0.0]), "exp": ("EXP", pa.CovExponential, [1.2, 0.4])}
H = 1.01 / 4 / 2  # leaf half width


@pytest.mark.parametrize("precision", ["mixed", "mixed_comp"])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("n_src,n_trg", [(1, 1), (15, 17), (257, 16), (2048, 640), (2049, 81 * 8), (700, 2600),
                                         (5000, 3000), (20000, 120)])
def test_mixed_near_field_matches_direct_sum(orc, kind, precision, n_src, n_trg):
    print("near field", kind, precision, n_src, n_trg, flush=True)
    name, cls, params = KINDS[kind]
    rng = np.random.default_rng(n_src + n_trg)
    src = rng.uniform(0.25, 0.75, (n_src, 3))
    trg = rng.uniform(0.25, 0.75, (n_trg, 3))
    k = min(n_src, n_trg) // 2
    trg[:k] = src[:k]  # coincident pairs
    if n_trg > 1000:
        trg[k:k + 100] = src[:1] + rng.uniform(-1e-5, 1e-5, (100, 3))  # nearly coincident ones
    w = rng.normal(size=n_src)
    ev = pa.make_fmm_evaluator(cls(params), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig(precision, 4, 2, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    y = ev.evaluate()
    ref = orc.direct_rbf_sum(orc.make_rbf(getattr(orc, name), params), src, w, trg)
    # Per pair: r^2 in FP32 from exact splits (eight steps of the matrix unit
    # with roundings of up to 2^-21 together, observed 4.8e-7 of the largest
    # term), root, product and sums 2^-24 each along chains of n / 8; the
    # exponential turns a relative error of r into 3 r / range times as much.
    # Coordinates to 2^-32 H on each side: r to 2^-30 H.
    d = np.linalg.norm(trg[:, None, :] - src[None, :, :], axis=2)
    if kind in ("bh3", "bh3c"):
        phi, slope, grow = params[0] * np.sqrt(d * d + params[1] ** 2), params[0], 1.0
    elif kind == "th3":
        phi, slope, grow = params[0] * d ** 3, 0.0, 3.0
    else:
        phi, slope, grow = params[0] * np.exp(-3 * d / params[1]), 3 * params[0] / params[1], 1.0 + 3 * d / params[1]
    rel = 2.0 ** -21 * grow + 2.0 ** -24 * (2 + n_src / 8 ** 0.5 / 8)
    bound = (np.abs(w) * (phi * rel + slope * H * 2.0 ** -30 * (d > 0))).sum(axis=1) + 1e-12
    worst = np.max(np.abs(y - ref) / bound)
    print(f"  worst error / bound {worst:.3f}, rel {np.abs(y - ref).max() / np.abs(ref).max():.2e}", flush=True)
    assert worst <= 1.0


def single_pairs(rng, cls, params, precision, dist):
    """Values, exact values and distances of targets around single sources of
    weight 1, dist leaf half widths away; half of the sources sit so that
    leaves' common face lies between them and some of their targets."""
    out = []
    for k in range(8):
        s = rng.uniform(0.26, 0.74, 3)
        if k % 2:
            s[k // 2 % 3] = 0.5 - 0.3 * dist * H
        u = rng.normal(size=(300, 3))
        t = s + dist * H * u / np.linalg.norm(u, axis=1)[:, None]
        t = t[np.all((t > 0.25) & (t < 0.75), axis=1)]
        ev = pa.make_fmm_evaluator(cls(params), ((0, 0, 0), (1, 1, 1)))
        ev.set_config(pa.FmmConfig(precision, 4, 2, "fmm"))
        ev.set_source_points(s[None])
        ev.set_weights(np.ones(1))
        ev.set_target_points(t)
        y = ev.evaluate()
        assert ev.stats()["direct"] == 0
        out.append((y, np.linalg.norm(t - s, axis=1)))
    return [np.concatenate(a) for a in zip(*out)]


@pytest.mark.parametrize("precision", ["mixed", "mixed_comp"])
@pytest.mark.parametrize("k", range(0, 21, 2))
def test_mixed_near_field_of_one_close_pair(k, precision):
    print("close pair", k, precision, flush=True)
    y, r = single_pairs(np.random.default_rng(k), pa.Biharmonic3D, [1.0, 0.0], precision, 2.0 ** -k)
    # As above: 2^-21 of r, and each coordinate to 2^-32 H on each side.
    worst = np.max(np.abs(y + r) / (2.0 ** -21 * r + 2 * 3 ** 0.5 * 2.0 ** -32 * H))
    print(f"  worst error / bound {worst:.3f}, rms of r {np.sqrt(np.mean((y + r) ** 2 / r ** 2)):.1e}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("precision", ["mixed", "mixed_comp"])
def test_mixed_near_field_of_coincident_points_is_zero(precision):
    y, r = single_pairs(np.random.default_rng(1), pa.Biharmonic3D, [1.0, 0.0], precision, 0.0)
    assert not r.any() and not y.any()


@pytest.mark.parametrize("precision", ["mixed", "mixed_comp"])
@pytest.mark.parametrize("kind", ["bh3", "th3"])
@pytest.mark.parametrize("units2", [1e-9, 1e-3, 0.03, 0.3, 7.3, 1.3e4, 1.6e7, 1.7e7, 3e12])
def test_mixed_near_field_keeps_small_and_large_offsets(units2, kind, precision):
    """The kernels' offset, from far below the 2^-9 half widths that the
    coordinates are split at to far above the leaf, at close pairs."""
    print("offset", units2, kind, precision, flush=True)
    c = units2 ** 0.5 * H / 512
    _, cls, _ = KINDS[kind]
    for dist in (0.0, 2.0 ** -12, 2.0 ** -9, 0.3):
        y, r = single_pairs(np.random.default_rng(3), cls, [1.0, c], precision, dist)
        rho = np.sqrt(r * r + c * c)
        ref, grow = (-rho, 1.0) if kind == "bh3" else (rho ** 3, 3.0)
        # As for pairs without an offset; it is rounded to FP32 itself.
        off = 2.0 ** -21 + 2 * 3 ** 0.5 * 2.0 ** -32 * H * r / rho ** 2
        worst = np.max(np.abs(y - ref) / (np.abs(ref) * grow * off))
        print(f"  at {dist:.1e}: worst error / bound {worst:.3f}", flush=True)
        assert worst <= 1.0


@pytest.mark.parametrize("precision", ["mixed", "mixed_comp"])
@pytest.mark.parametrize("unit_weights", [True, False])
@pytest.mark.parametrize("width", [1e-12, 1e-10, 1e-9, 1.0, 1e9, 1e12])
def test_mixed_triharmonic_near_field_in_any_length_unit(width, unit_weights, precision):
    """Weights of about 1, and weights that give values of about 1."""
    print("width", width, unit_weights, precision, flush=True)
    rng = np.random.default_rng(17)
    src, trg = rng.uniform(0.25, 0.75, (2, 500, 3))
    w = rng.normal(size=500)
    ev = pa.make_fmm_evaluator(pa.Triharmonic3D([1.0, 0.0]), (np.zeros(3), np.full(3, width)))
    ev.set_config(pa.FmmConfig(precision, 4, 2, "fmm"))
    ev.set_source_points(width * src)
    ev.set_weights(w if unit_weights else w / width ** 3)
    ev.set_target_points(width * trg)
    y = ev.evaluate() / (width ** 3 if unit_weights else 1.0)
    assert ev.stats()["direct"] == 0
    term = w * np.linalg.norm(trg[:, None] - src[None], axis=2) ** 3
    # Three times the error of r, products, and sums along chains of 500 / 8.
    bound = np.abs(term).sum(1) * (3 * 2.0 ** -21 + 2.0 ** -24 * (2 + 500 / 8))
    worst = np.max(np.abs(y - term.sum(1)) / bound)
    print(f"  worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1.0


def test_mixed_near_field_is_the_same_on_either_stream():
    """One leaf of many targets next to leaves of few, with the near field
    beside the far field and after it."""
    rng = np.random.default_rng(3)
    src = rng.uniform(0.25, 0.75, (4000, 3))
    trg = np.concatenate([rng.uniform(0.26, 0.49, (2000, 3)), rng.uniform(0.51, 0.75, (37, 3))])
    w = rng.normal(size=4000)
    outs = []
    for overlap in (True, False):
        ev = pa.make_fmm_evaluator(pa.Biharmonic3D(), ((0, 0, 0), (1, 1, 1)))
        ev.set_config(pa.FmmConfig("mixed", 4, 2, "fmm"))
        ev.set_overlap(overlap)
        ev.set_source_points(src)
        ev.set_weights(w)
        ev.set_target_points(trg)
        outs.append(ev.evaluate())
    np.testing.assert_array_equal(outs[0], outs[1])


def pair_terms(kind, params, u, r2):
    """phi, f, t with grad phi = f u and H = f (I + t u u^T) of the isotropic kernels."""
    with np.errstate(divide="ignore", invalid="ignore"):
        if kind in ("bh3", "bh3c"):
            rho = np.sqrt(r2 + params[1] ** 2)
            return -params[0] * rho, np.where(rho > 0, -params[0] / rho, 0.0), np.where(rho > 0, -1.0 / rho ** 2, 0.0)
        if kind == "th3":
            rho = np.sqrt(r2)
            return params[0] * rho ** 3, 3 * params[0] * rho, np.where(rho > 0, 1.0 / r2, 0.0)
        r, c = np.sqrt(r2), 3.0 / params[1]
        e = params[0] * np.exp(-c * r)
        return e, -c * e / r, -(1.0 / r2 + c / r)


@pytest.mark.parametrize("mode", ["fp64 value", "fp64 gradient", "mixed gradient", "fp64 hessian", "mixed hessian"])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("n_src,n_trg", [(1, 1), (300, 4), (257, 33), (700, 129 * 8), (5000, 3000), (20000, 120)])
def test_near_field_on_the_vector_units(kind, mode, n_src, n_trg):
    """FP64 values, gradients and Hessian sums: 4, 8 or 16 target slots, up to
    8 (5) targets per thread, several passes, shared sources."""
    print("near field", kind, mode, n_src, n_trg, flush=True)
    _, cls, params = KINDS[kind]
    precision, what = mode.split()
    rng = np.random.default_rng(n_src + n_trg)
    src = rng.uniform(0.25, 0.75, (n_src, 3))
    trg = rng.uniform(0.25, 0.75, (n_trg, 3))
    if not (kind == "exp" and what != "value"):  # undefined at r = 0
        k = min(n_src, n_trg) // 2
        trg[:k] = src[:k]
    w = rng.normal(size=(n_src, 3) if what == "hessian" else n_src)
    make = {"value": pa.make_fmm_evaluator, "gradient": pa.make_fmm_gradient_transpose_evaluator,
            "hessian": pa.make_fmm_hessian_evaluator}[what]
    ev = make(cls(params), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig(precision, 4, 2, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w.ravel())
    ev.set_target_points(trg)
    y = ev.evaluate().reshape(n_trg, -1)
    assert ev.stats()["direct"] == 0
    rows = rng.permutation(n_trg)[:200]
    u = trg[rows][:, None, :] - src[None]
    r2 = (u * u).sum(-1)
    phi, f, t = pair_terms(kind, params, u, r2)
    r = np.sqrt(r2)
    if what == "value":
        term, mag = (w * phi)[..., None], np.abs(w * phi)
    elif what == "gradient":
        term, mag = (w * f)[..., None] * u, np.abs(w * f) * r
    else:
        uw = (u * w).sum(-1)
        term = -f[..., None] * (w + (t * uw)[..., None] * u)
        mag = np.abs(f) * np.linalg.norm(w, axis=1) * (1 + np.abs(t) * r2)
    # Sums: chains of at most n / 16 + 30 additions and products of half an ulp
    # each. Coordinates in the leaf frame: 2 ulp of the half width on each
    # side, so relative to r; the terms are of degree at most 3 in it.
    ulp = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    rel = ulp * (n_src / 16 + 30 + 12 * 3 ** 0.5 * H / np.maximum(r, ulp))
    bound = (mag * np.where(r > 0, rel, 0.0)).sum(1) + 1e-15 * (np.abs(w).max() * (1 + params[0]))
    if kind == "bh3c" or what == "value":
        bound += (mag * ulp * (n_src / 16 + 30)).sum(1)  # coincident pairs count
    if kind == "exp":
        bound *= 1 + 3 * np.sqrt(3) / params[1]  # degree of exp in r
    worst = np.max(np.abs(y[rows] - term.sum(1)) / bound[:, None])
    print(f"  worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("what,precision,many", [("value", "fp64", 600_001), ("gradient", "mixed", 600_001),
                                                 ("gradient", "fp64", 420_001), ("value", "mixed", 3_400_001)])
def test_very_many_targets_in_one_leaf(what, precision, many):
    """A zoom into one leaf: so many targets that their number times the
    number of passes over them does not fit 32 bits. 4,096 occupied leaves, so
    that no leaf is shared out to several workgroups."""
    print("many targets", what, precision, many, flush=True)
    rng = np.random.default_rng(many)
    width = 1.01 / 16
    centre = -0.005 + (np.arange(16) + 0.5) * width
    spots = centre[8] + rng.uniform(-0.49, 0.49, (1000, 3)) * width
    pick = rng.integers(0, 1000, many)
    grid = np.stack(np.meshgrid(centre, centre, centre, indexing="ij"), -1).reshape(-1, 3)
    src = centre[8] + rng.uniform(-1.49, 1.49, (300, 3)) * width  # in its neighbours: no far field
    w = rng.normal(size=300)
    make = pa.make_fmm_evaluator if what == "value" else pa.make_fmm_gradient_transpose_evaluator
    ev = make(pa.Biharmonic3D(), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig(precision, 3, 4, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(np.concatenate([grid, spots[pick]]))
    y = ev.evaluate().reshape(len(grid) + many, -1)[len(grid):]
    assert ev.stats()["n_trg_leaves"] == 4096
    u = spots[:, None, :] - src[None]
    r = np.linalg.norm(u, axis=2)
    term = -(w * r)[..., None] if what == "value" else -(w / r)[..., None] * u
    # Half an ulp per operation of a chain of at most 300 + 30, coordinates to
    # two ulp of the half width on each side.
    ulp = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    bound = (np.linalg.norm(term, axis=2) * ulp * (330 + 12 * 3 ** 0.5 * (width / 2) / r)).sum(1)
    worst = np.max(np.abs(y - term.sum(1)[pick]) / bound[pick, None])
    print(f"  worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1.0
