"""The evaluation with four waves per leaf (few leaves): leaves of one target, of less than
a wave, of a power of two, of more than 64 and of more than 256 targets, all outputs, every
method and precision, against the FP64 direct sums of the near field (one box, no far field)
and against the oracle-pinned plan of many leaves."""
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


@pytest.mark.parametrize("kernel", ["cube", "yukawa", "stokes"])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("mixed", 1e-6)])
def test_few_leaves_vs_one_wave(kernel, precision, tol):
    """The same sources evaluated at targets of a plan with few leaves (four waves) and of
    one with more than 16,384 leaves (one wave): both within the method's truncation of the
    direct sum, and the potential of the few-leaf plan equal to its own at the sources."""
    import ffmm
    rng = np.random.default_rng(3)
    n = 40_000
    pts = rng.random((n, 3))
    if kernel == "cube":
        m, d = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=6), rng.standard_normal(n)
    elif kernel == "yukawa":
        m, d = ffmm.SphericalHarmonics(ffmm.Yukawa3D(5.0), p=8), rng.standard_normal(n)
    else:
        m, d = ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=8), rng.standard_normal((n, 9))
    cache = ffmm.OperatorCache(m)
    print(f"[eval wide] {kernel} {precision}", flush=True)
    few = ffmm.DevicePlan(m, pts, ppl=200, bbox=BOX, cache=cache, precision=precision)
    many = ffmm.DevicePlan(m, pts, ppl=2, bbox=BOX, cache=cache, precision=precision)
    assert few.level_leaves.sum() < 6144 < 16384 < many.level_leaves.sum()
    tgt = rng.random((5000, 3))
    a, b = few.build_expansions(d).evaluate(tgt).cpu().numpy(), many.build_expansions(d).evaluate(tgt).cpu().numpy()
    assert np.linalg.norm(a - b) < 2e-3 * np.linalg.norm(b)
    # the same leaf's targets split over other tiles: each target's value does not depend on them
    order = rng.permutation(len(tgt))[:777]
    c = few.evaluate(tgt[order]).cpu().numpy()
    assert np.linalg.norm(c - a[order]) < tol * np.linalg.norm(a[order])
