"""The evaluation with four waves per leaf: leaves of one target, of less than a wave, of a
power of two, of more than 64 and of more than 256 targets, every method, output and
precision, against the FP64 direct sums of the near field (one box, no far field), and plans
of few and of many leaves against the direct sums."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = (np.zeros(3), 1.0)


@pytest.mark.parametrize("n", [1, 2, 37, 64, 65, 200, 256, 257, 700])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-13), ("mixed", 1e-6)])
def test_one_leaf_vs_direct(n, precision, tol):
    """One leaf holding every point and target: the near field alone, so the direct sum."""
    import ffmm
    print(f"[eval wide] n={n} {precision}", flush=True)
    rng = np.random.default_rng(n)
    pts, tau, tgt = rng.random((n, 3)), rng.standard_normal(n), rng.random((2 * n + 1, 3))
    for m in (ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=4), ffmm.SphericalHarmonics(ffmm.Laplace3D(), p=4)):
        plan = ffmm.DevicePlan(m, pts, ppl=1000, bbox=BOX, precision=precision)
        assert plan.nnodes == 1
        u = plan.matvec(tau).cpu().numpy()
        v = plan.evaluate(tgt, ffmm.PotentialGradient).cpu().numpy()
        ud, vd = O.direct_self(pts, tau), O.direct(pts, tau, tgt)
        gd = O.direct(pts, tau, tgt, grad=True)
        if n > 1:
            assert np.linalg.norm(u - ud) < tol * np.linalg.norm(ud)
        else:
            assert u[0] == 0.0
        assert np.linalg.norm(v[:, 0] - vd) < tol * np.linalg.norm(vd)
        assert np.linalg.norm(v[:, 1:] - gd) < 10 * tol * np.linalg.norm(gd)


@pytest.mark.parametrize("n", [65, 257, 700])
@pytest.mark.parametrize("kind,p", [("yukawa", 10), ("yukawa", 13), ("yukawa", 14), ("stokes", 4)])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 2e-6)])
def test_one_leaf_harmonic_vs_direct(n, kind, p, precision, tol):
    """The same for Yukawa (potential and gradient; the weights of 256 lanes up to p = 13, one
    wave above) and Stokes (velocity and pressure).  FP32: a term's relative error is some ten
    roundings of 2^-24 and, in the exponential, kappa r < 9 of them: 2e-6."""
    import ffmm
    import harmonic as HO
    print(f"[eval wide] {kind} p={p} n={n} {precision}", flush=True)
    rng = np.random.default_rng(n + p)
    pts, tgt = rng.random((n, 3)), rng.random((n + 1, 3))
    me = np.arange(n)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)   # noqa: E731
    if kind == "yukawa":
        m, d = ffmm.SphericalHarmonics(ffmm.Yukawa3D(5.0), p=p), rng.standard_normal(n)
        outs = [(ffmm.Potential, 0), (ffmm.Gradient, 1), (ffmm.PotentialGradient, 2)]
    else:
        m, d = ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=p), rng.standard_normal((n, 9))
        outs = [(ffmm.Velocity, 0), (ffmm.Pressure, 3)]
    plan = ffmm.DevicePlan(m, pts, ppl=1000, bbox=BOX, precision=precision)
    assert plan.nnodes == 1
    for out, code in outs:
        ref = HO.direct(kind, pts, d, pts, code, kappa=5.0, skip=me)
        assert rel(plan.matvec(d, out).cpu().numpy().reshape(ref.shape), ref) < tol
        ref = HO.direct(kind, pts, d, tgt, code, kappa=5.0)
        assert rel(plan.evaluate(tgt, out).cpu().numpy().reshape(ref.shape), ref) < tol


@pytest.mark.parametrize("kernel,p,bound", [("cube", 8, 1e-6), ("yukawa", 12, 2e-4), ("stokes", 12, 2e-4)])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 1e-6)])
def test_few_leaves_vs_one_wave(kernel, p, bound, precision, tol):
    """The same sources evaluated at targets by a plan with few leaves of some 80 points (four
    waves) and by one with more than 16,384 leaves of one or two (one wave), both within the
    method's truncation (bound; the mixed form's FP32 besides) of the direct sum, the few-leaf
    plan at its sources too."""
    import ffmm
    import harmonic as HO
    rng = np.random.default_rng(3)
    n = 40_000
    pts = rng.random((n, 3))
    if kernel == "cube":
        m, d = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=p), rng.standard_normal(n)
    elif kernel == "yukawa":
        m, d = ffmm.SphericalHarmonics(ffmm.Yukawa3D(5.0), p=p), rng.standard_normal(n)
    else:
        m, d = ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=p), rng.standard_normal((n, 9))
    cache = ffmm.OperatorCache(m)
    print(f"[eval wide] {kernel} {precision}", flush=True)
    few = ffmm.DevicePlan(m, pts, ppl=200, bbox=BOX, cache=cache, precision=precision)
    many = ffmm.DevicePlan(m, pts, ppl=2, bbox=BOX, cache=cache, precision=precision)
    assert few.level_leaves.sum() < 6144 < 16384 < many.level_leaves.sum()
    tgt = rng.random((5000, 3))
    a, b = few.build_expansions(d).evaluate(tgt).cpu().numpy(), many.build_expansions(d).evaluate(tgt).cpu().numpy()
    kind = "laplace" if kernel == "cube" else kernel
    rows = rng.permutation(len(tgt))[:300]
    rel = lambda x, y: np.linalg.norm(x - y) / np.linalg.norm(y)   # noqa: E731
    limit = bound + (2e-6 if precision == "mixed" else 0.0)
    ref = HO.direct(kind, pts, d, tgt[rows], kappa=5.0)
    assert rel(a[rows], ref) < limit and rel(b[rows], ref) < limit
    rows = rng.permutation(n)[:300]
    u = few.evaluate_at_sources().cpu().numpy()
    assert rel(u[rows], HO.direct(kind, pts, d, pts[rows], kappa=5.0, skip=rows)) < limit
    # the same leaf's targets split over other tiles: each target's value does not depend on them
    order = rng.permutation(len(tgt))[:777]
    c = few.evaluate(tgt[order]).cpu().numpy()
    assert np.linalg.norm(c - a[order]) < tol * np.linalg.norm(a[order])


@pytest.mark.parametrize("n,ppl", [(1, 5), (90, 4), (600, 3), (2000, 3), (30_000, 40), (60_000, 2)])
@pytest.mark.parametrize("kernel,lo,hi", [("cube", 3600, 16384), ("yukawa", 450, 6144)])
def test_near_work_vs_tree(kernel, lo, hi, n, ppl):
    """The work that the evaluation's launch is chosen by against the downloaded tree: several
    blocks' leaves, empty ones; none where the number of leaves decides.  Whole numbers, so
    equal."""
    import ffmm
    rng = np.random.default_rng(n)
    pts = rng.random((n, 3))
    pts[: n // 3] = 0.4 + 0.01 * rng.random((n // 3, 3))
    m = (ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=2) if kernel == "cube"
         else ffmm.SphericalHarmonics(ffmm.Yukawa3D(5.0), p=2))
    plan = ffmm.DevicePlan(m, pts, ppl=ppl, bbox=BOX)
    t = plan.download_tree()
    leaf = (t.leaf != 0) & (t.ghost == 0)
    assert leaf.sum() == plan.level_leaves.sum()
    cnt = np.maximum(t.phi - t.plo + 1, 0).astype(np.int64)
    col = t.colleagues[leaf]
    q = cnt[leaf] * np.where(col >= 0, cnt[np.maximum(col, 0)], 0).sum(1)
    print(f"[eval wide] near work {kernel} n={n}: {leaf.sum()} leaves", flush=True)
    want = [q.sum(), q.max(), (cnt[leaf] > 0).sum()] if lo <= leaf.sum() < hi else [0, 0, 0]
    assert np.array_equal(plan.near_work(), np.array(want, dtype=np.float64))
