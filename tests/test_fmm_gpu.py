"""GPU parity of the FMM seam against the CPU oracle (FP64 direct summation),
bit-exact tree construction, and edge cases. Calls go through the C ABI."""
import sys

import numpy as np
import pytest

import polatory_amd as pa

pytestmark = pytest.mark.gpu


def log(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel_err(y, ref):
    return np.abs(y - ref).max() / np.abs(ref).max()


def make(kind, params=None, aniso=None):
    r = {"bh3": pa.Biharmonic3D, "th3": pa.Triharmonic3D, "exp": pa.CovExponential}[kind](
        params if params is not None else ([1.0, 2.0] if kind == "exp" else []))
    if aniso is not None:
        r.set_anisotropy(aniso)
    return r


def orc_rbf(orc, r):
    kind = {"bh3": orc.BH3, "th3": orc.TH3, "exp": orc.EXP}[r.short_name]
    return orc.make_rbf(kind, r.parameters(), r.anisotropy())


ANISO = np.array([[1.0, 0.1, 0.0], [0.0, 0.8, 0.2], [0.0, 0.0, 1.3]])


@pytest.mark.parametrize("kind", ["bh3", "th3", "exp"])
def test_gpu_direct_matches_oracle(orc, kind):
    log("direct", kind)
    rng = np.random.default_rng(11)
    src = rng.uniform(0, 1, (3000, 3))
    trg = rng.uniform(-0.1, 1.1, (2000, 3))
    w = rng.normal(size=3000)
    r = make(kind, aniso=ANISO)
    y = pa.direct_evaluate(r, src, w, trg)
    ref = orc.direct_rbf_sum(orc_rbf(orc, r), src, w, trg)
    assert rel_err(y, ref) < 1e-13


def _gpu_tree_vs_oracle(orc, ev, which, pts_raw, aniso, exact_order=True):
    """Codes, leaves and cells bit-exact against the oracle. exact_order=False:
    a tree cut back from a deeper level keeps its points sorted by the finer
    codes, so the permutation is compared as the set of points of each leaf."""
    info = ev.tree_info(which)
    L = info["level"]
    pts = orc.transform_points(aniso.reshape(-1), pts_raw)
    codes = orc.morton_codes(pts, info["lo"], info["inv_cell"], L)
    perm = orc.stable_sort_codes(codes)
    sorted_codes = codes[perm]
    gcodes, gperm, glc, gls = ev.export_tree(which)
    if exact_order:
        np.testing.assert_array_equal(gperm, perm)
    else:
        _, ls_ = orc.leaves(sorted_codes)
        for a, b in zip(ls_[:-1], ls_[1:]):
            np.testing.assert_array_equal(np.sort(gperm[a:b]), np.sort(perm[a:b]))
    np.testing.assert_array_equal(gcodes, sorted_codes)
    lc, ls = orc.leaves(sorted_codes)
    np.testing.assert_array_equal(glc, lc)
    np.testing.assert_array_equal(gls, ls)
    for l in range(L + 1):
        np.testing.assert_array_equal(ev.export_level(which, l), np.unique(lc >> np.uint64(3 * (L - l))))
    return L


@pytest.mark.parametrize("dist", ["uniform", "clustered", "aniso"])
def test_tree_and_lists_bit_exact(orc, dist):
    log("tree", dist)
    rng = np.random.default_rng(12)
    if dist == "clustered":
        src = np.concatenate([rng.normal(0.3, 0.02, (3000, 3)), rng.uniform(0, 1, (500, 3))])
        trg = np.concatenate([rng.normal(0.7, 0.05, (2000, 3)), rng.uniform(0, 1, (300, 3))])
    else:
        src = rng.uniform(0, 1, (4000, 3))
        trg = rng.uniform(0, 1, (2500, 3))
    aniso = ANISO if dist == "aniso" else np.eye(3)
    r = make("bh3", aniso=aniso)
    lo = np.minimum(src.min(0), trg.min(0))
    hi = np.maximum(src.max(0), trg.max(0))
    ev = pa.make_fmm_evaluator(r, (lo, hi))
    ev.set_config(pa.FmmConfig("mixed", 4, 4, "fmm"))
    ev.set_source_points(src)
    ev.set_target_points(trg)
    ev.set_weights(np.ones(len(src)))
    # the box follows src/fmm/utility.hpp:19-33
    c, w = orc.make_box(lo, hi, aniso)
    info = ev.tree_info(0)
    assert info["width"] == w
    np.testing.assert_array_equal(info["lo"], c - w / 2.0)
    L = _gpu_tree_vs_oracle(orc, ev, 0, src, aniso)
    _gpu_tree_vs_oracle(orc, ev, 1, trg, aniso)
    _, _, slc, _ = ev.export_tree(0)
    _, _, tlc, _ = ev.export_tree(1)
    np.testing.assert_array_equal(ev.export_p2p(), orc.p2p_lists(tlc, slc, L))
    for l in range(2, L + 1):
        tl = ev.export_level(1, l)
        sl = ev.export_level(0, l)
        np.testing.assert_array_equal(ev.export_m2l(l), orc.m2l_lists(tl, sl, l))


def test_adaptive_leaf_level_tree_matches_oracle(orc):
    """Automatic leaf level on a surface-like source set: the trees are built
    deeper and cut back to the level whose occupied leaves hold closest to
    0.8 P^3 points (100 at order 5); codes, leaves, cells and lists stay
    bit-exact."""
    log("adaptive leaf level")
    rng = np.random.default_rng(14)
    u = rng.normal(size=(60000, 3))
    src = 0.5 + 0.45 * u / np.linalg.norm(u, axis=1)[:, None]  # sphere surface
    trg = rng.uniform(0.05, 0.95, (20000, 3))
    r = make("bh3")
    ev = pa.make_fmm_evaluator(r, ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig("mixed", 5, -1, "fmm"))
    ev.set_source_points(src)
    ev.set_target_points(trg)
    ev.set_weights(np.ones(len(src)))
    L = _gpu_tree_vs_oracle(orc, ev, 0, src, np.eye(3), exact_order=False)
    assert _gpu_tree_vs_oracle(orc, ev, 1, trg, np.eye(3), exact_order=False) == L
    # uniform-density choice: round(log8(60000 / 100)) = 3; the shell's
    # occupied cells hold 268 points at level 3 and 66 at level 4
    assert L == 4
    _, _, slc, _ = ev.export_tree(0)
    _, _, tlc, _ = ev.export_tree(1)
    np.testing.assert_array_equal(ev.export_p2p(), orc.p2p_lists(tlc, slc, L))
    for l in range(2, L + 1):
        np.testing.assert_array_equal(ev.export_m2l(l), orc.m2l_lists(ev.export_level(1, l), ev.export_level(0, l), l))


# (kind, precision, order, tolerance on the relative L-inf error vs FP64 direct)
FMM_CASES = [
    ("bh3", "mixed", 4, 2e-4), ("bh3", "mixed", 6, 1e-5), ("bh3", "mixed", 8, 2e-6),
    ("bh3", "fp64", 6, 1e-5), ("bh3", "fp64", 10, 1e-8),
    ("th3", "mixed", 6, 1e-5), ("th3", "fp64", 8, 1e-7),
    ("exp", "mixed", 6, 1e-5), ("exp", "fp64", 8, 1e-7),
]


@pytest.fixture(scope="module")
def fmm_problem(orc):
    rng = np.random.default_rng(13)
    src = rng.uniform(0, 1, (20000, 3))
    trg = rng.uniform(0, 1, (12000, 3))
    w = rng.normal(size=20000)
    refs = {}
    for kind in ("bh3", "th3", "exp"):
        r = make(kind)
        refs[kind] = orc.direct_rbf_sum(orc_rbf(orc, r), src, w, trg)
    return src, trg, w, refs


@pytest.mark.parametrize("kind,prec,order,tol", FMM_CASES)
def test_fmm_matches_direct(fmm_problem, kind, prec, order, tol):
    log("fmm", kind, prec, order)
    src, trg, w, refs = fmm_problem
    ev = pa.make_fmm_evaluator(make(kind), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig(prec, order, 3, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    y = ev.evaluate()
    e = rel_err(y, refs[kind])
    log(f"  rel err {e:.3e} (tol {tol:.0e})")
    assert e < tol


def run_fmm(kind, cfg, src, w, trg):
    ev = pa.make_fmm_evaluator(make(kind), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(cfg)
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    y = ev.evaluate()
    return y, ev.stats()


@pytest.mark.parametrize("kind", ["bh3", "th3"])
def test_compressed_m2l(fmm_problem, kind):
    """Compressed transfers (the default at orders 7 and 8 for the homogeneous
    kernels): rank 128, the dense form's accuracy bound against the FP64 direct
    sum, and, at the largest rank (256), the FP64 dense result to 5e-9 (measured
    1.4e-9 for bh3, 9e-11 for th3): the basis is orthonormal and
    C_v = U^T K_v U is assembled correctly."""
    src, trg, w, refs = fmm_problem
    log("compressed m2l", kind)
    y_dense, st = run_fmm(kind, pa.FmmConfig("fp64", 7, 3, "fmm", svd_tol=0.0), src, w, trg)
    assert st["m2l_rank"] == 0
    y_full, st = run_fmm(kind, pa.FmmConfig("fp64", 7, 3, "fmm", svd_tol=1e-14), src, w, trg)
    assert st["m2l_rank"] == 256
    d = rel_err(y_full, y_dense)
    log(f"  rank 256 vs dense (FP64): {d:.2e}")
    assert d <= 5e-9
    for prec, tol in (("fp64", 1e-6), ("mixed", 2e-6)):
        y, st = run_fmm(kind, pa.FmmConfig(prec, 7, 3, "fmm"), src, w, trg)
        e = rel_err(y, refs[kind])
        log(f"  default {prec}: rank {st['m2l_rank']}, rel err {e:.2e} (dense FP64 {rel_err(y_dense, refs[kind]):.2e})")
        assert st["m2l_rank"] == 128
        assert e <= tol


def test_exponential_kernel_keeps_dense_m2l(fmm_problem):
    src, trg, w, refs = fmm_problem
    y, st = run_fmm("exp", pa.FmmConfig("mixed", 7, 3, "fmm"), src, w, trg)
    assert st["m2l_rank"] == 0
    assert rel_err(y, refs["exp"]) <= 1e-5


@pytest.mark.parametrize("prec,order,tol", [("mixed", 6, 1e-5), ("fp64", 10, 1e-8)])
def test_symmetric_fmm_matches_direct(orc, prec, order, tol):
    log("symmetric", prec, order)
    rng = np.random.default_rng(14)
    pts = rng.uniform(0, 1, (15000, 3))
    w = rng.normal(size=15000)
    r = make("th3", aniso=ANISO)
    ev = pa.make_fmm_symmetric_evaluator(r)
    ev.set_config(pa.FmmConfig(prec, order, 3, "fmm"))
    ev.set_points(pts)
    ev.set_weights(w)
    y = ev.evaluate()
    ref = orc.direct_rbf_sum(orc_rbf(orc, r), pts, w, pts)
    e = rel_err(y, ref)
    log(f"  rel err {e:.3e}")
    assert e < tol


def test_clustered_and_ragged_leaves(orc):
    log("clustered")
    rng = np.random.default_rng(15)
    src = np.concatenate([rng.normal(0.2, 0.01, (6000, 3)), rng.uniform(-1, 1, (2000, 3)),
                          np.array([[0.5, 0.5, 0.5]] * 50)])  # coincident points
    trg = np.concatenate([rng.normal(0.2, 0.05, (3000, 3)), rng.uniform(-1, 1, (1000, 3))])
    w = rng.normal(size=len(src))
    r = make("bh3")
    ev = pa.make_fmm_evaluator(r)
    ev.set_config(pa.FmmConfig("fp64", 8, 4, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    y = ev.evaluate()
    ref = orc.direct_rbf_sum(orc_rbf(orc, r), src, w, trg)
    assert rel_err(y, ref) < 1e-6


def test_weights_update_reuses_tree(orc):
    log("weights update")
    rng = np.random.default_rng(16)
    src = rng.uniform(0, 1, (9000, 3))
    trg = rng.uniform(0, 1, (9000, 3))
    r = make("bh3")
    ev = pa.make_fmm_evaluator(r)
    ev.set_config(pa.FmmConfig("mixed", 6, 3, "fmm"))
    ev.set_source_points(src)
    ev.set_target_points(trg)
    for seed in range(3):
        w = np.random.default_rng(seed).normal(size=9000)
        ev.set_weights(w)
        y = ev.evaluate()
        ref = orc.direct_rbf_sum(orc_rbf(orc, r), src, w, trg)
        assert rel_err(y, ref) < 1e-5


def test_small_and_empty_inputs(orc):
    log("small/empty")
    r = make("exp")
    ev = pa.make_fmm_evaluator(r)
    ev.set_source_points(np.zeros((1, 3)))
    ev.set_weights([2.0])
    ev.set_target_points(np.zeros((0, 3)))
    assert ev.evaluate().shape == (0,)
    ev.set_target_points(np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0]]))
    y = ev.evaluate()
    np.testing.assert_allclose(y, [2.0, 2.0 * np.exp(-1.5)], rtol=1e-14)
    with pytest.raises(ValueError):
        ev.set_weights([1.0, 2.0])


def test_accuracy_search_meets_accuracy(orc):
    log("accuracy search")
    rng = np.random.default_rng(17)
    src = rng.uniform(0, 1, (30000, 3))
    trg = rng.uniform(0, 1, (8000, 3))
    w = rng.normal(size=30000)
    r = make("bh3")
    ref = orc.direct_rbf_sum(orc_rbf(orc, r), src, w, trg)
    acc = 1e-6 * np.abs(ref).max()
    ev = pa.make_fmm_evaluator(r)
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    ev.set_accuracy(acc)
    y = ev.evaluate()
    log("  chosen", ev.config(), "err", np.abs(y - ref).max(), "acc", acc)
    # the search checks its sample (source points); targets may land slightly above
    assert np.abs(y - ref).max() < 3 * acc


@pytest.mark.parametrize("name", ["bh3", "th3", "exp"])
def test_fp64_near_field_alone_matches_direct(name):
    """All points in one leaf of a fixed level-2 tree: the FMM result is the
    FP64 near field alone, so it must equal the FP64 direct sum up to the
    summation order (this pins the near field's square root, refined from the
    hardware reciprocal square root, to a few ulp)."""
    rbf = {"bh3": pa.Biharmonic3D(), "th3": pa.Triharmonic3D(), "exp": pa.CovExponential([1.0, 0.3])}[name]
    rng = np.random.default_rng(61)
    src = rng.uniform(0.01, 0.24, (6000, 3))
    trg = rng.uniform(0.01, 0.24, (4000, 3))
    trg[:50] = src[:50]  # coincident pairs (zero distance)
    w = rng.normal(size=6000)
    ev = pa.FmmEvaluator(rbf, ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig("fp64", 10, 2, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    v = ev.evaluate()
    assert ev.stats()["direct"] == 0
    ref = pa.direct_evaluate(rbf, src, w, trg)
    err = np.abs(v - ref).max() / np.abs(ref).max()
    print(f"{name}: FP64 near field alone vs direct: {err:.2e}", flush=True)
    assert err <= 1e-13


def test_compensated_near_field_on_cancelling_weights():
    """Weights that cancel strongly (a large alternating pattern on a smooth
    field): the compensated mixed form is at least as accurate as the plain
    mixed form against the FP64 direct sum, and both run the FMM path. In the
    root mean square, where the squares of the near field's error and of the
    far field's, which the forms share, add up: the far field alone (FP64 form)
    is 2.96e-7 at its worst target and 4.8e-8 in the mean, and which form has
    the largest single error is chance (three of six seeds one way, three the
    other; in the mean 5.7e-8 against 7.1e-8, the same way for all six)."""
    rng = np.random.default_rng(71)
    src = rng.uniform(0, 1, (200_000, 3))
    trg = rng.uniform(0, 1, (20_000, 3))
    w = 1e4 * np.where(np.arange(200_000) % 2 == 0, 1.0, -1.0) * (1.0 + 1e-3 * rng.normal(size=200_000))
    rbf = pa.CovExponential([1.0, 0.5])
    ref = pa.direct_evaluate(rbf, src, w, trg[:2000])
    errs = {}
    for prec in ("mixed", "mixed_comp"):
        ev = pa.FmmEvaluator(rbf)
        ev.set_config(pa.FmmConfig(prec, 8, -1, "fmm"))
        ev.set_source_points(src)
        ev.set_weights(w)
        ev.set_target_points(trg)
        v = ev.evaluate()
        assert ev.stats()["direct"] == 0
        errs[prec] = np.sqrt(np.mean((v[:2000] - ref) ** 2)) / np.abs(ref).max()
    print(f"cancelling weights: mixed {errs['mixed']:.2e}, compensated {errs['mixed_comp']:.2e}", flush=True)
    assert errs["mixed_comp"] <= errs["mixed"]


def test_compensated_sums_of_the_near_field_alone():
    """The same pattern inside the eight central leaves, where there is no far
    field: the compensated sums are the more accurate ones at the worst target
    too (1.6e-7 against 5.9e-7)."""
    rng = np.random.default_rng(71)
    src = rng.uniform(0.25, 0.75, (20_000, 3))
    trg = rng.uniform(0.25, 0.75, (2000, 3))
    w = 1e4 * np.where(np.arange(20_000) % 2 == 0, 1.0, -1.0) * (1.0 + 1e-3 * rng.normal(size=20_000))
    rbf = pa.CovExponential([1.0, 0.5])
    ref = pa.direct_evaluate(rbf, src, w, trg)
    errs = {}
    for prec in ("mixed", "mixed_comp"):
        ev = pa.make_fmm_evaluator(rbf, ((0, 0, 0), (1, 1, 1)))
        ev.set_config(pa.FmmConfig(prec, 4, 2, "fmm"))
        ev.set_source_points(src)
        ev.set_weights(w)
        ev.set_target_points(trg)
        errs[prec] = np.abs(ev.evaluate() - ref).max() / np.abs(ref).max()
    print(f"cancelling weights, near field: mixed {errs['mixed']:.2e}, compensated {errs['mixed_comp']:.2e}", flush=True)
    assert errs["mixed_comp"] <= errs["mixed"]


@pytest.fixture(scope="module")
def headline_problem(orc):
    """The evaluation workload of the benchmark: 1,000,000 bh3 sources U[0,1]^3
    (seed 3) with N(0,1) weights (seed 4) at 1,000,000 targets U[0,1]^3
    (seed 6); the oracle's FP64 direct sum on 2,000 of the targets (seed 7)."""
    src = np.random.default_rng(3).uniform(0, 1, (1_000_000, 3))
    w = np.random.default_rng(4).normal(size=1_000_000)
    trg = np.random.default_rng(6).uniform(0, 1, (1_000_000, 3))
    sub = np.random.default_rng(7).permutation(1_000_000)[:2000]
    ref = orc.direct_rbf_sum(orc.make_rbf(orc.BH3), src, w, trg[sub])
    return src, w, trg, sub, ref


@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_headline_config_within_1e6_relative(headline_problem, prec):
    """bh3 at order 7 with the leaf level chosen by occupancy (the benchmark's
    configuration): relative L-inf error against the oracle's FP64 direct sum
    within 1e-6, with at least 150 sources per occupied leaf."""
    src, w, trg, sub, ref = headline_problem
    log("headline", prec)
    ev = pa.make_fmm_evaluator(make("bh3"), ((0, 0, 0), (1, 1, 1)))
    ev.set_config(pa.FmmConfig(prec, 7, -1, "fmm"))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    y = ev.evaluate()
    st = ev.stats()
    per_leaf = len(src) / st["n_src_leaves"]
    e = rel_err(y[sub], ref)
    log(f"  leaf level {st['leaf_level']}, {per_leaf:.0f} sources per leaf, M2L rank {st['m2l_rank']}, "
        f"rel err {e:.3e}")
    assert st["direct"] == 0
    assert per_leaf >= 150
    assert e <= 1e-6


def test_headline_accuracy_search_within_1e6_relative(headline_problem):
    """The accuracy search at 1e-6 x max|y| (absolute, as polatory's accuracy
    is) picks a configuration whose error at the benchmark's targets is within
    that accuracy."""
    src, w, trg, sub, ref = headline_problem
    acc = 1e-6 * np.abs(ref).max()
    ev = pa.make_fmm_evaluator(make("bh3"), ((0, 0, 0), (1, 1, 1)))
    ev.set_source_points(src)
    ev.set_weights(w)
    ev.set_target_points(trg)
    ev.set_accuracy(acc)
    y = ev.evaluate()
    e = np.abs(y[sub] - ref).max()
    log(f"  search chose {ev.config()}, abs err {e:.3e} (accuracy {acc:.3e})")
    assert e <= acc
