"""The reflection symmetry of the translation operators, which lets the kernels
apply one operator to all sources that are mirror images of each other.

  * CPU: the tables of every octant (and of every mirrored M2L offset) are the
    octant-0 (non-negative offset) table with the signs of the reflection on
    rows and columns, to the last bit;
  * GPU: forces against the oracle where the upward and downward kernels have
    partial tiles, single-child chains and one- to three-block row classes.
"""
import ctypes as C
import os

import numpy as np
import pytest

import cabi

DP = C.POINTER(C.c_double)


def classes(p):
    """Sign bits (1, 2, 4 for x, y, z) of each real coefficient."""
    out = []
    for n in range(p + 1):
        for a in range(n + 1):
            for im in range(2 if a else 1):
                out.append(((a & 1) ^ im) | (im << 1) | (((n + a) & 1) << 2))
    return np.array(out)


def signs(cls, s):
    return np.array([(-1.0) ** bin(s & c).count("1") for c in cls])


@pytest.mark.parametrize("p", [1, 4, 7])
def test_tables_are_reflections(p):
    lib = C.CDLL(os.path.join(cabi.ROOT, "tests", "model", "libmodel.so"))
    S = (p + 1) ** 2
    m2m, l2l, m2l = np.zeros((8, S, S)), np.zeros((8, S, S)), np.zeros((343, S, S))
    assert lib.model_tables(p, *(t.ctypes.data_as(DP) for t in (m2m, l2l, m2l))) == 0
    cls = classes(p)
    for s in range(8):
        d = signs(cls, s)
        for t in (m2m, l2l):
            assert np.array_equal(t[s], d[:, None] * t[0] * d[None, :]), s
        for o in np.ndindex(4, 4, 4):
            if max(o) < 2:
                continue
            r = [-v if s >> k & 1 else v for k, v in enumerate(o)]
            at = lambda v: (v[0] + 3) * 49 + (v[1] + 3) * 7 + v[2] + 3  # noqa: E731
            assert np.array_equal(m2l[at(r)], d[:, None] * m2l[at(o)] * d[None, :]), (o, s)


def cloud(kind, seed=4):
    rng = np.random.default_rng(seed)
    if kind == "pair":       # a chain of single-child boxes down to the eps floor
        return np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0], [1.0 - 1e-3, 1.0, 1.0]]), 1
    if kind == "octants":    # exactly 16 + 1 parents on one level
        g = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], float)
        pos = np.concatenate([c * 0.5 + 0.2 * rng.uniform(-1, 1, (12, 3)) for c in g])
        return np.concatenate([pos, 0.5 * g[:1] + 1e-3 * rng.uniform(-1, 1, (40, 3))]), 4
    return rng.standard_normal((1500, 3)) * np.array([1.0, 0.3, 0.05]), 9


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["pair", "octants", "slab"])
@pytest.mark.parametrize("p", [1, 2, 5, 8, 10, 13])
def test_forces_against_oracle(kind, p):
    """max relErr <= 1e-12, the agreement asked of FP64 forces everywhere."""
    pos, cap = cloud(kind)
    m = np.random.default_rng(1).uniform(0.5, 1.5, len(pos)) / len(pos)
    ref, _ = cabi.oracle().fmm(pos, m, 1.0, 0.004, p, cap)
    s = cabi.product().AdaptiveFMM3D(G=1.0, eps=0.004, p=p, threshold=cap)
    acc = s.computeAccelerations(pos, m)
    s.close()
    mx, _ = cabi.rel_err(ref, acc)
    print(f"{kind} p={p}: {mx:.2e}", flush=True)
    assert mx <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("p", [2, 4, 6, 8, 11, 16])
def test_batch_tiles_equal_alone(p):
    """A forest whose M2L runs full tiles gives each system the bits it has
    alone, where its few boxes run tiles of 16 targets over four waves."""
    rng = np.random.default_rng(p)
    sizes = [int(n) for n in rng.integers(1500, 4000, 70)]
    off = np.concatenate([[0], np.cumsum(sizes)])
    pos = rng.standard_normal((off[-1], 3))
    m = rng.uniform(0.5, 1.5, off[-1])
    s = cabi.product().AdaptiveFMM3D(G=1.0, eps=0.01, p=p, threshold=7)
    acc = s.computeBatch(pos, m, off)
    boxes = s.stats()["n_boxes"]
    assert boxes > 256 * 32  # more than fit tiles of 32 targets on the CUs
    for q in (0, 33, 69):
        sl = slice(off[q], off[q + 1])
        assert np.array_equal(acc[sl], s.computeAccelerations(pos[sl], m[sl])), q
    s.close()
    print(f"p={p}: {boxes} boxes", flush=True)
