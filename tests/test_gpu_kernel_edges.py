"""Kernels at the edges of their tiles and ranges, against the oracle or
against the general path of the same library."""
import sys

import numpy as np
import pytest

import oracle
from abyss_amd import regf, workloads

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("ref", [True, False])
@pytest.mark.parametrize("n,m", [(64, 64), (67, 1), (129, 65), (1025, 63), (1500, 1500)])
def test_derivs23_edges(n, m, ref):
    """Target blocks and j ranges that fill neither a wave nor a split, with
    a coincident pair and a particle whose r^2 overflows."""
    say(f"case: derivs23 n={n} m={m} reference_signs={ref}")
    js = workloads.plummer_equal(n, seed=4, k_nb=24)
    rng = np.random.default_rng(n + m)
    x, v = js.x.copy(), js.v.copy()
    x[n // 2] = x[n // 3]
    x[n - 1, 0] = 1.0e160
    a, ad = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    t = rng.permutation(n)[:m].astype(np.int32)
    t[0] = n // 2
    with regf.Context(device=0, cap=64) as c:
        c.upload_state(js.m, x, v, a, ad, np.zeros(n), js.r2)
        got = c.derivs23(t, reference_signs=ref)
    # the far particle and the others add nothing to each other (the oracle's
    # own products of 1e160 would overflow)
    want = np.zeros((m, 12))
    near, k = t != n - 1, n - 1
    want[near] = oracle.derivs23(x[:k], v[:k], a[:k], ad[:k], js.m[:k], js.r2[:k], t[near],
                                 ref_signs=ref)
    # each of the four parts of a row against its own largest entry; the
    # rounding of a row of n terms is below 1e-10 of it (n * 2^-53 times the
    # ratio of the largest term to the sum, at most ~1e4 here)
    scale = np.abs(want).reshape(-1, 2, 6).max(axis=2, keepdims=True) + 1e-300
    err = np.abs(got - want).reshape(-1, 2, 6) / scale
    say(f"  max err = {err.max():.3e}")
    assert np.isfinite(got).all() and err.max() <= 1e-10
