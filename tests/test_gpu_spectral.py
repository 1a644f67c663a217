"""The spectral M2L (csrc/spectral.hip) at its edges against the oracle's FP64 FMM on the same
tree: levels of a few sibling groups (partial tiles, one chunk of nodes), levels of several
chunks, tiles cut into halves and a half cut into quarters (sparse deepest levels), missing
colleagues and children without sources, both precisions."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BOX = (np.zeros(3), 1.0)


def _points(layout, n, rng):
    if layout == "uniform":
        return rng.random((n, 3))
    if layout == "quarters":    # a half of a tile names more than 192 boxes
        return np.random.default_rng(50).random((n, 3))
    if layout == "corner":      # one octant only: most colleagues are missing
        return 0.25 * rng.random((n, 3))
    v = rng.standard_normal((n, 3))
    s = 0.5 + 0.4 * v / np.linalg.norm(v, axis=1, keepdims=True)
    s[: n // 4] = 0.8 + 0.001 * rng.standard_normal((n // 4, 3))
    return s


def _largest_half(t):
    """The most distinct sourced colleagues that 8 consecutive sibling groups of a tile name."""
    most = 0
    for lo, hi in zip(t.level_start[2:-1], t.level_start[3:]):
        first = np.arange(lo, hi, 8)
        col = np.where(t.ghost[first][:, None] != 0, -1, np.delete(t.colleagues[t.parent[first]], 13, axis=1))
        ch = np.where(col >= 0, t.child_first[np.maximum(col, 0)], -1)
        sourced = (ch >= 0) & (t.has_source[np.maximum(ch, 0)[..., None] + np.arange(8) * (ch >= 0)[..., None]] != 0).any(-1)
        ch = np.where(sourced, ch, -1)
        most = max([most] + [np.sum(np.unique(ch[i:i + 8]) >= 0) for i in range(0, len(first), 8)])
    return most


@pytest.mark.parametrize("layout,n,ppl", [("uniform", 400, 4), ("uniform", 9000, 10), ("corner", 3000, 12),
                                          ("shell", 6000, 8), ("shell", 40_000, 12), ("uniform", 25_000, 3),
                                          ("quarters", 40_000, 2)])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-11), ("mixed", 2e-6)])
def test_spectral_vs_oracle(layout, n, ppl, precision, tol):
    import ffmm
    print(f"[spectral] {layout} n={n} ppl={ppl} {precision}", flush=True)
    rng = np.random.default_rng(n + ppl)
    pts, tau = _points(layout, n, rng), rng.standard_normal(n)
    m = ffmm.CubeKernelIndependent(ffmm.Laplace3D(), p=8)
    cache = ffmm.OperatorCache(m)
    plan = ffmm.DevicePlan(m, pts, ppl=ppl, bbox=BOX, cache=cache, precision=precision, m2l="spectral")
    staged, cut = plan.spectral_tiles()
    print(f"[spectral] tiles staged whole {staged.tolist()}, cut {cut.tolist()}", flush=True)
    assert staged.sum() > 0
    if layout == "quarters" or (n, ppl) == (25_000, 3):
        assert cut.sum() > 0
    if layout == "quarters":
        assert _largest_half(plan.download_tree()) > 192
    u = plan.matvec(tau).cpu().numpy()
    u_ref = O.FMM(cache.host_operators(), pts, ppl, *BOX).matvec(tau, m2l="spectral")
    assert np.max(np.abs(u - u_ref)) < tol * np.max(np.abs(u_ref))
