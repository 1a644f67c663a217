"""The circle method's M2L: circles of 4 to 64 points (with and without a remainder of the four
chains, a full wave), empty and ragged lists, against the oracle's FMM on the same tree
(1e-11: FP64 sums in another order, through the pseudo-inverses)."""
import numpy as np
import pytest

import circle2d as O2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ppl", [(150, 12), (2500, 9)])
@pytest.mark.parametrize("nequiv", [4, 7, 30, 61, 64])
def test_circle_m2l_vs_oracle(nequiv, n, ppl):
    import ffmm
    print(f"[circle2d M2L] nequiv={nequiv} n={n}", flush=True)
    rng = np.random.default_rng(nequiv + n)
    pts, tau = rng.random((n, 2)) ** 1.7, rng.standard_normal(n)
    m = ffmm.KernelIndependent(ffmm.Laplace2D(), nequiv=nequiv)
    cache = ffmm.CircleOperatorCache(m)
    plan = ffmm.CirclePlan(m, pts, ppl=ppl, bbox=((0.0, 0.0), 1.0), cache=cache)
    u = plan.matvec(tau).cpu().numpy()
    uo = O2.FMM2D(cache.operators, pts, ppl, (0.0, 0.0), 1.0).matvec(tau)
    uo = uo[0] if isinstance(uo, tuple) else uo
    assert np.max(np.abs(u - uo)) < 1e-11 * np.max(np.abs(uo))
