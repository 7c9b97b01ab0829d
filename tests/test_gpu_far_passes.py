"""P2L and M2P (the X and W lists) at the edges of their lane groupings: leaves of
1, 14, 15, 29 and 64 bodies and one larger than a workgroup, lists longer than
the staged entries, against the oracle; max relErr <= 1e-12, the agreement asked
of FP64 forces everywhere."""
import numpy as np
import pytest

import cabi

pytestmark = pytest.mark.gpu


def shells(n, seed):
    """Clumps at distances that halve towards a corner: deep beside shallow boxes, long W and X lists."""
    rng = np.random.default_rng(seed)
    k = rng.integers(0, 9, n)
    centre = np.exp2(-k.astype(float))[:, None] * np.array([1.0, 0.93, 0.87])
    return centre + 0.2 * np.exp2(-k.astype(float))[:, None] * rng.standard_normal((n, 3))


@pytest.mark.parametrize("cap", [1, 14, 15, 29, 64, 700])
@pytest.mark.parametrize("p", [1, 4, 8, 9, 13])
def test_far_passes_against_oracle(p, cap):
    n = {1: 400, 700: 6000}.get(cap, 2500)
    pos = shells(n, 10 * p + cap)
    m = np.random.default_rng(cap).uniform(0.5, 1.5, n) / n
    orc = cabi.oracle()
    ref, _ = orc.fmm(pos, m, 1.0, 1e-4, p, cap)
    s = cabi.product().AdaptiveFMM3D(G=1.0, eps=1e-4, p=p, threshold=cap)
    acc = s.computeAccelerations(pos, m)
    st = s.stats()
    mx, _ = cabi.rel_err(ref, acc)
    print(f"p={p} cap={cap}: W {st['n_w']} X {st['n_x']} largest leaf {st['max_leaf_occ']} max rel {mx:.2e}", flush=True)
    assert st["n_w"] > 0 and st["n_x"] > 0
    assert mx <= 1e-12
    s.set_overlap(False)  # the in-order passes: the same bits
    assert np.array_equal(s.computeAccelerations(pos, m), acc)
    acc2, phi = s.computeAccelerationsAndPotential(pos, m)
    assert np.array_equal(acc2, acc) and np.isfinite(phi).all()
    s.close()
