"""The harmonic methods' class M2L in the mixed form at the edges of its tiles: orders of 1 to 4
blocks of 32 coefficients (N = 9 .. 121) and of more (the class GEMMs), both block counts, a
handful of pairs per class, ragged tiles, and chunks of one tile: the local expansions against
those of the FP64 plan, whose multipoles are the same.

Each operand is rounded to 24 bits and the sums of at most 121 terms are FP32, so a pair's
relative error is a few 2^-24 of its norm and a target's sum of up to 189 pairs no more:
10 x 2^-24 < 1e-6 bounds the ratio of the norms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BOX = (np.zeros(3), 1.0)


# the larger problem runs at two orders
@pytest.mark.parametrize("p,n,cap", [(p, n, cap) for p in (2, 4, 5, 7, 8, 9, 10, 11)
                                     for n, cap in ((70, None), (1500, None), (1500, "16"), (20000, None))
                                     if n < 20000 or p in (8, 10)])
@pytest.mark.parametrize("kind", ["laplace", "yukawa", "stokes"])
def test_mixed_class_m2l_vs_f64(kind, p, n, cap, monkeypatch):
    import ffmm
    print(f"[class M2L] {kind} p={p} n={n} cap={cap}", flush=True)
    rng = np.random.default_rng(p + n)
    pts = rng.random((n, 3)) ** 1.3
    m = {"laplace": lambda: ffmm.SphericalHarmonics(ffmm.Laplace3D(), p=p),
         "yukawa": lambda: ffmm.SphericalHarmonics(ffmm.Yukawa3D(5.0), p=p),
         "stokes": lambda: ffmm.StokesHarmonics(ffmm.Stokeslet3D(), p=p)}[kind]()
    d = rng.standard_normal((n, 9) if kind == "stokes" else n)
    cache = ffmm.OperatorCache(m)
    if cap:
        monkeypatch.setenv("FFMM_M2L_CHUNK_PAIRS", cap)
    out = []
    for prec in ("f64", "mixed"):
        plan = ffmm.DevicePlan(m, pts, ppl=5, bbox=BOX, cache=cache, precision=prec, m2l="dense")
        plan.build_expansions(d)
        out.append([np.asarray(x) for x in plan.download_expansions()[:2]])
    (M64, P64), (M32, P32) = out
    assert np.array_equal(M64, M32)
    assert np.linalg.norm(P64) > 0
    assert np.linalg.norm(P32 - P64) < 1e-6 * np.linalg.norm(P64)
