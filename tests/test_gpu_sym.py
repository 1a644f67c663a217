"""The cube method's translations by symmetric blocks (csrc/sym.hip) against the oracle's
dense operators on the same tree: every even order the kernels take (1, 7, 19, 37 and 61
orbits: one to four row tiles, full and ragged), S2M as its own kernel and inside UC2E, both
precisions, workgroups with missing columns; an odd order keeps the dense operators."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = (np.zeros(3), 1.0)


@pytest.mark.parametrize("p,n,ppl,precision", [
    (2, 1500, 20, "f64"), (4, 3000, 20, "f64"), (5, 2000, 25, "f64"), (6, 3001, 30, "f64"), (8, 2500, 25, "f64"),
    (10, 2000, 40, "f64"), (4, 3000, 20, "mixed"), (6, 3001, 30, "mixed"), (8, 2500, 25, "mixed"),
    (4, 40_000, 4, "f64"), (6, 40_000, 4, "mixed")])
def test_blocks_vs_oracle(p, n, ppl, precision):
    """FP64: the oracle's rounding, 1e-11 (1e-10 at p = 10, whose pseudo-inverses are ten
    times worse conditioned); mixed: the FP32 M2L and evaluation, 2e-6."""
    import ffmm
    print(f"[sym] p={p} n={n} ppl={ppl} {precision}", flush=True)
    rng = np.random.default_rng(100 * p + ppl)
    pts = rng.random((n, 3))
    pts[: n // 3] = 0.4 + 0.05 * rng.random((n // 3, 3))
    tau = rng.standard_normal(n)
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=p)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=ppl, bbox=BOX, cache=cache, precision=precision)
    u = plan.matvec(tau).cpu().numpy()
    ref = O.FMM(cache.host_operators(), pts, ppl, BOX[0], BOX[1])
    u_ref = ref.matvec(tau)
    split = int(plan.level_s2m[2:].sum()) < 8192
    assert split == (n < 40_000)             # both forms of S2M are covered
    if precision == "mixed":
        assert np.linalg.norm(u - u_ref) < 2e-6 * np.linalg.norm(u_ref)
    else:
        assert np.max(np.abs(u - u_ref)) < (1e-10 if p == 10 else 1e-11) * np.max(np.abs(u_ref))


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_sources_beyond_the_lds_stage(precision):
    """1,350,000 uniform points with ppl = 110: the 32,768 boxes of level 5 are leaves of ~41
    sources, so workgroups of 16 of them hold more sources than the fused kernel stages in
    LDS (320 in FP64, 640 in FP32) and read them from global memory."""
    import ffmm
    n = 1_350_000
    print(f"[sym] heavy nodes {precision}", flush=True)
    rng = np.random.default_rng(5)
    pts, tau = rng.random((n, 3)), rng.standard_normal(n)
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=4)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=110, bbox=BOX, cache=cache, precision=precision)
    assert int(plan.level_s2m[2:].sum()) >= 8192 and plan.N / int(plan.level_s2m.sum()) > 40
    u = plan.matvec(tau).cpu().numpy()
    u_ref = O.FMM(cache.host_operators(), pts, 110, BOX[0], BOX[1]).matvec(tau)
    assert np.linalg.norm(u - u_ref) < (2e-6 if precision == "mixed" else 1e-11) * np.linalg.norm(u_ref)


@pytest.mark.parametrize("kernel,p", [("laplace", 2), ("laplace", 5), ("laplace", 10), ("yukawa", 7), ("laplace", 13),
                                      ("stokes", 3), ("stokes", 10), ("laplace", 16), ("laplace", 18), ("laplace", 19),
                                      ("stokes", 18), ("laplace", 20), ("stokes", 20)])
def test_harmonic_blocks_vs_oracle(kernel, p):
    """M2M and L2L by reflection parity against the harmonic oracle's dense operators on the
    same tree (1e-11, as tests/test_gpu_harmonic.py): one to four row tiles, expansions of
    one to seven chunks of 64 entries, one and four blocks, groups of 16 and of 4 columns with
    missing ones; p = 20, whose largest block has more than 64 entries, keeps the dense form."""
    import ffmm
    from test_gpu_harmonic import oracle_for
    print(f"[sym] harmonic {kernel} p={p}", flush=True)
    n = 1500
    rng = np.random.default_rng(10 * p)
    pts = rng.random((n, 3))
    pts[: n // 3] = 0.4 + 0.05 * rng.random((n // 3, 3))
    if kernel == "stokes":
        m, d = ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=p), rng.standard_normal((n, 9))
    else:
        K = ffmm.Laplace3D() if kernel == "laplace" else ffmm.Yukawa3D(5.0)
        m, d = ffmm.SphericalHarmonics(K, p=p), rng.standard_normal(n)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=10, bbox=BOX, cache=cache)
    u = plan.matvec(d).cpu().numpy()
    tree = plan.download_tree()
    u_ref = oracle_for(m, cache, pts, 10, tree.perm)[0].matvec(d)
    u_ref = u_ref.reshape(u.shape)
    assert np.max(np.abs(u - u_ref)) < 1e-11 * np.max(np.abs(u_ref))


def test_odd_order_of_many_check_points():
    """p = 9: 1,736 check points, more than one block of the general S2M; conditioned as p = 10."""
    import ffmm
    rng = np.random.default_rng(9)
    pts, tau = rng.random((1500, 3)), rng.standard_normal(1500)
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=9)
    cache = ffmm.OperatorCache(m)
    u = ffmm.DevicePlan(m, pts, ppl=25, bbox=BOX, cache=cache).matvec(tau).cpu().numpy()
    u_ref = O.FMM(cache.host_operators(), pts, 25, BOX[0], BOX[1]).matvec(tau)
    assert np.max(np.abs(u - u_ref)) < 1e-10 * np.max(np.abs(u_ref))


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("p,given", [(4, "scaled inverse"), (8, "regularised inverse"), (8, "scaled inverse down"),
                                     (4, "M2M of one child"), (8, "L2L of one child"), (8, "truncated"), (8, "odd pc")])
def test_given_operators_are_applied(p, given, precision):
    """Even orders whose operators are not those of the blocks (a scaled or regularised inverse
    of full rank, a truncated one, translations without the reflections' symmetry, check
    surfaces of an odd order) are applied as given: against the oracle with the same operators,
    to the tolerances of test_blocks_vs_oracle."""
    import ffmm
    print(f"[sym] given operators: {given} p={p} {precision}", flush=True)
    rng = np.random.default_rng(p)
    n = 2000
    pts = rng.random((n, 3))
    pts[: n // 3] = 0.4 + 0.05 * rng.random((n // 3, 3))
    tau = rng.standard_normal(n)
    kw = {"truncated": dict(pinv_rtol=1e-8), "odd pc": dict(pc=15)}.get(given, {})
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=p, **kw)
    cache = ffmm.OperatorCache(m)
    cache.fit_box(pts.min(0), pts.max(0), BOX)
    o = cache.host_operators()
    if given == "scaled inverse":
        o.P_up.invS *= 2.0
    elif given == "scaled inverse down":
        o.P_down.invS *= 0.5
    elif given == "regularised inverse":
        s = 1.0 / o.P_up.invS
        o.P_up.invS[:] = s / (s * s + (1e-6 * s[0]) ** 2)
    elif given == "M2M of one child":
        o.M2M[:, : o.nsmall] *= 1.25
    elif given == "L2L of one child":
        o.L2L[: o.nsmall] *= 1.25
    elif given == "truncated":
        assert o.P_up.rank < o.nsmall
    u = ffmm.DevicePlan(m, pts, ppl=20, bbox=BOX, cache=cache, precision=precision).matvec(tau).cpu().numpy()
    u_ref = O.FMM(o, pts, 20, BOX[0], BOX[1]).matvec(tau)
    if precision == "mixed":
        assert np.linalg.norm(u - u_ref) < 2e-6 * np.linalg.norm(u_ref)
    else:
        assert np.max(np.abs(u - u_ref)) < 1e-11 * np.max(np.abs(u_ref))


def _put_again(cache, monkeypatch):
    """Put the cache's host operators again into its device copy."""
    from ffmm import fmm as F
    h, call = cache.device(0), F.call

    def put(name, *args):
        if name == "ffmm_opcache_create":
            args[-1]._obj.value = h.value
        else:
            call(name, *args)
    cache._device.clear()
    monkeypatch.setattr(F, "call", put)
    cache.device(0)
    monkeypatch.setattr(F, "call", call)


def test_operators_put_again(monkeypatch):
    """Operators put again into a cache that a plan was made with: of the same form, the plan
    serves them; of the other form (here a scaled inverse, applied as given), the plan's
    passes, its evaluation and its captured replay are refused, and a new plan is right."""
    import ffmm
    rng = np.random.default_rng(4)
    pts, tau = rng.random((1500, 3)), rng.standard_normal(1500)
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=4)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=20, bbox=BOX, cache=cache).capture()
    u = plan.matvec(tau).cpu().numpy()
    cache.class_factors(0, 1e-6)
    _put_again(cache, monkeypatch)
    assert np.array_equal(plan.matvec(tau).cpu().numpy(), u)
    cache.host_operators().P_up.invS *= 2.0
    _put_again(cache, monkeypatch)
    for step in (plan.evaluate_at_sources, lambda: plan.replay(tau), lambda: plan.build_expansions(tau)):
        with pytest.raises(ffmm.DeviceError, match="replaced"):
            step()
    new = ffmm.DevicePlan(m, pts, ppl=20, bbox=BOX, cache=cache)
    v = new.matvec(tau).cpu().numpy()
    v_ref = O.FMM(cache.host_operators(), pts, 20, BOX[0], BOX[1]).matvec(tau)
    assert np.max(np.abs(v - v_ref)) < 1e-11 * np.max(np.abs(v_ref))
    new.set_tol(1e-6)            # factors put before keep the other form's order
    with pytest.raises(ffmm.DeviceError, match="replaced"):
        new.build_expansions(tau)


@pytest.mark.parametrize("p,pc,d,width", [(2, 4, 0.1, 1.0), (4, 8, 0.3, 0.7361), (6, 12, 0.1, 1e-5), (8, 16, 0.1, 1.0),
                                          (8, 16, 0.01, 3.3e4), (8, 24, 0.6, 1.0), (8, 8, 0.1, 0.3), (10, 20, 0.1, 1.0),
                                          (10, 20, 0.05, 17.0)])
def test_default_operators_take_the_blocks(p, pc, d, width, monkeypatch):
    """The library's own operators pass the checks of the blocks at every order, surface and
    width: a scaled inverse put afterwards is of the other form, which a plan of the first
    refuses."""
    import ffmm
    print(f"[sym] form of p={p} pc={pc} d={d} width={width}", flush=True)
    rng = np.random.default_rng(p)
    pts = width * rng.random((100, 3))
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=p, pc=pc, d=d)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=10, bbox=(np.zeros(3), width), cache=cache)
    plan.matvec(rng.standard_normal(100))
    cache.host_operators().P_up.invS *= 2.0
    _put_again(cache, monkeypatch)
    with pytest.raises(ffmm.DeviceError, match="replaced"):
        plan.evaluate_at_sources()
