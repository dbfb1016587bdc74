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


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED, regf.PREC_REFINED])
@pytest.mark.parametrize("n,m", [(1025, 300), (2049, 2049), (10007, 777), (16385, 4096),
                                 (65536, 64)])
def test_short_spans_equal_long_ones(n, m, prec):
    """A launch of few workgroups takes more, shorter j-splits; with at least
    four tiles per split the same launch gives the same lists, and sums that
    differ by the order of their FP64 partials."""
    say(f"case: spans n={n} m={m} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=2, k_nb=40)
    t = np.random.default_rng(m).permutation(n)[:m].astype(np.int32)
    with regf.Context(device=0, cap=64, precision=prec) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        got = [a.copy() for a in c.query(t)]
        p = c.plan()
        c.set_tuning(0, max(1, n // 1024), 0, p["lanes_per_target"])
        want = c.query(t)
        say(f"  plan {p}, long spans: {c.plan()['j_splits']} splits")
    assert np.array_equal(got[2], want[2]) and np.array_equal(got[3], want[3])
    for a, b in zip(got[:2], want[:2]):
        # the sums have the same FP32 runs and at most 128 + 64 FP64 partials
        # (200 * 2^-53 of the largest partial, whose ratio to the sum is below
        # 1e4); a target whose flag changes moves by the checked tolerance
        rel = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
        bad = rel > 1e-9
        assert rel.max() <= 1e-6 and bad.sum() <= (1 if prec == regf.PREC_CHECKED else 0)


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
@pytest.mark.parametrize("n,m", [(1024, 300), (4096, 600), (16385, 601), (65536, 300)])
def test_noalloc_bad_targets_in_every_merge(n, m, prec):
    """One split, and the merges of up to 8, up to 16 and more splits: bad
    targets get NaN and INT_MIN and are not recomputed, the others are as on
    a list that holds target 0 in their place."""
    from .test_zz_no_alloc import Hip, assert_same, context_query, device_jset, noalloc_query
    js = workloads.plummer_kroupa(n, seed=2, k_nb=40)
    t = np.random.default_rng(m).permutation(n)[:m].astype(np.int32)
    bad = np.array([0, 5, 17, m - 1])
    t[bad] = [n, -1, np.iinfo(np.int32).min, np.iinfo(np.int32).max]
    hip = Hip()
    try:
        got = noalloc_query(hip, device_jset(hip, js), n, t, 64, prec)
    finally:
        hip.free()
    t0 = t.copy()
    t0[bad] = 0
    assert np.isnan(got[0][bad]).all() and np.isnan(got[1][bad]).all()
    assert (got[2][bad] == np.iinfo(np.int32).min).all()
    good = np.setdiff1d(np.arange(m), bad)
    assert_same(got, context_query(js, t0, 64, prec), 64, prec, rows=good)


@pytest.mark.parametrize("n,m,cap,k_nb", [
    (1024, 1, 256, 48),        # one split, results written in place
    (1000, 64, 64, 20),        # the same, the most targets
    (1500, 65, 64, 20),        # more targets than that
    (4096, 4096, 30, 40),      # mirrored merge, overflowed lists
    (20000, 3001, 256, 64),    # mirrored query against a fetch in chunks
    (20000, 6007, 300, 200),   # several chunks both ways
    (9000, 4097, 1000, 90)])   # first block above the mirrored ones
@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
def test_query_equals_launch_and_fetch(n, m, cap, k_nb, prec):
    """The routes of results to the host give the same bytes and leave the
    rows past each count alone, also after blocks of other sizes."""
    say(f"case: results n={n} m={m} cap={cap} precision={prec}")
    js = workloads.plummer_equal(n, seed=6, k_nb=k_nb)
    t = np.random.default_rng(m).permutation(n)[:m].astype(np.int32)
    with regf.Context(device=0, cap=cap, precision=prec) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        got = [a.copy() for a in c.query(t)]
        small = [a.copy() for a in c.query(t[:1])]
        c.set_targets(t)
        c.launch()
        want = c.fetch()
        again = c.query(t)
    for a, b, d in zip(got, want, again):
        assert np.array_equal(a, b) and np.array_equal(a, d)
    assert small[2][0] == got[2][0] and np.array_equal(small[3][0], got[3][0])
    filled = np.arange(cap)[None, :] < np.minimum(np.abs(got[2]), cap)[:, None]
    assert (got[3][~filled] == -1).all() and (got[3][filled] >= 0).all()
    assert (got[2] < 0).any() == (cap < k_nb)


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_MIXED, regf.PREC_REFINED])
@pytest.mark.parametrize("n,cap,k_nb,splits", [
    (5, 8, 3, 1), (256, 64, 40, 1), (257, 64, 40, 1), (1000, 20, 40, 1), (1279, 64, 40, 3),
    (4099, 400, 350, 2), (32768, 64, 40, 7), (32769, 64, 40, 7)])
def test_lists_by_tile_equal_lists_by_step(n, cap, k_nb, splits, prec):
    """Four lanes per target list a tile at a time (up to 32768 particles, and
    in FP64 terms on any), sixteen a step at a time: the same lists, with own
    targets, partial tiles, overflow and coincident particles in the way."""
    say(f"case: lists n={n} cap={cap} splits={splits} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=8, k_nb=min(k_nb, n - 2))
    x = js.x.copy()
    x[n // 2] = x[0]
    t = np.random.default_rng(n).permutation(n)[:min(n, 2000)].astype(np.int32)
    out = []
    with regf.Context(device=0, cap=cap, precision=prec) as c:
        c.upload(js.m, x, js.v, js.r2)
        for lanes in (4, 16):
            c.set_tuning(0, splits, 0, lanes)
            out.append([a.copy() for a in c.query(t)])
            assert c.plan()["lanes_per_target"] == lanes
    a, b = out
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])
    assert (np.abs(a[2]) > 0).any()
    # sums: FP64 terms differ by the order of n additions (n * 2^-53 of the
    # largest partial, at most 1e4 times the sum), FP32 runs by the rounding
    # of their 64 terms (64 * 2^-24), both of the whole array
    tol = 1e-10 if prec != regf.PREC_SPLIT else 4e-6
    for p, q in zip(a[:2], b[:2]):
        assert np.linalg.norm(p - q) <= tol * np.linalg.norm(q)


@pytest.mark.parametrize("nt", [1, 3, 4, 5, 16384, 16385])
def test_list_kernels_from_mapped_memory(nt):
    """Up to 16384 targets the list kernels read their inputs in place and in
    any case write their results in place, four targets a workgroup: each
    target's values equal those of a call by 777 others, bit for bit; the
    gather records written by a prediction equal those packed from a j-set."""
    say(f"case: list kernels targets={nt}")
    n, t_new = 20000, 2.0 ** -7
    js = workloads.plummer_kroupa(n, seed=4, k_nb=40)
    rng = np.random.default_rng(nt)
    t = rng.permutation(n)[:nt].astype(np.int32)
    dt = rng.uniform(1e-3, 1e-2, nt)
    a_old = rng.normal(size=(nt, 6))
    parts = [slice(k, min(k + 777, nt)) for k in range(0, nt, 777)]
    every = np.arange(n, dtype=np.int32)
    with regf.Context(device=0, cap=200) as c, regf.Context(device=0, cap=200) as d:
        for k in (c, d):
            k.upload(js.m, js.x, js.v, js.r2)
            k.keep_lists()
            k.query(every)
        acc, adot = c.irregular(t)
        for s in parts:
            p, q = d.irregular(t[s])
            assert np.array_equal(acc[s], p) and np.array_equal(adot[s], q)
        # c: records of the prediction; d: records packed from an uploaded j-set
        z = np.zeros((n, 3))
        c.upload_state(js.m, js.x, js.v, z, z, np.zeros(n), js.r2)
        c.predict(t_new)
        c.query(every)
        d.upload(js.m, js.x + t_new * js.v, js.v, js.r2)
        d.query(every)
        acc, adot = c.irregular(t)
        out = c.regular_step(t, dt, a_old)[4]
        for s in parts:
            p, q = d.irregular(t[s])
            assert np.array_equal(acc[s], p) and np.array_equal(adot[s], q)
        for s in parts:
            assert np.array_equal(out[s][:, 12:], d.regular_step(t[s], dt[s], a_old[s])[4][:, 12:])


@pytest.mark.parametrize("count", [1, 63, 64, 65, 1500])
def test_updates_and_calls_that_do_not_wait(count):
    """Records that reach the state by way of LDS, two updates one after the
    other, and steps queued behind an update and a prediction: the same bytes
    as from a j-set uploaded at once."""
    say(f"case: updates count={count}")
    n, t_new, cap = 3000, 2.0 ** -6, 150
    js = workloads.plummer_kroupa(n, seed=12, k_nb=30)
    rng = np.random.default_rng(count)
    m, x, v, r2 = js.m.copy(), js.x.copy(), js.v.copy(), js.r2.copy()
    zero = np.zeros((n, 3))
    with regf.Context(device=0, cap=cap) as c, regf.Context(device=0, cap=cap) as d:
        c.upload_state(m, x, v, zero, zero, np.zeros(n), r2)
        c.keep_lists()
        for nt in (70, 3, 64, 65, 900, n, 1, 300):
            for _ in range(2):
                i = rng.permutation(n)[:count].astype(np.int32)
                x[i] += 1e-3 * rng.normal(size=(count, 3))
                v[i] *= 1.01
                m[i] *= 0.99
                r2[i] *= 1.02
                z = zero[:count]
                c.update_state(i, m[i], x[i], v[i], z, z, np.zeros(count), r2[i])
            c.predict(t_new)
            t = rng.permutation(n)[:nt].astype(np.int32)
            if nt % 2:
                got = c.regular_step(t, np.full(nt, 1e-3), np.zeros((nt, 6)))[:4]
            else:
                got = c.query(t)
            d.upload(m, x + t_new * v, v, r2)
            want = d.query(t)
            for p, q in zip(got, want):
                assert np.array_equal(p, q)


@pytest.mark.parametrize("tiles", [7, 8, 9])
def test_spans_around_the_priority_rule(tiles):
    """Four lanes per target above 32768 particles: workgroups of few tiles
    keep equal wave priorities, from 8 tiles on they do not.  Same lists as
    with 16 lanes per target; the FP32 runs are one tile each in both kernels,
    so only the order of the FP64 partials differs."""
    say(f"case: spans tiles={tiles}")
    n, cap = 40000, 200
    js = workloads.plummer_kroupa(n, seed=3, k_nb=80)
    t = np.random.default_rng(tiles).permutation(n)[:300].astype(np.int32)
    whole = (n + 255) // 256
    out = []
    with regf.Context(device=0, cap=cap, precision=regf.PREC_SPLIT) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        for splits, lanes in ((-(-whole // tiles), 4), (1, 4), (1, 16)):
            c.set_tuning(0, splits, 0, lanes)
            out.append([a.copy() for a in c.query(t)])
    for o in out[1:]:
        assert np.array_equal(out[0][2], o[2]) and np.array_equal(out[0][3], o[3])
    # 157 partials, the largest up to 1e4 times their sum
    tol = whole * 2.0 ** -53 * 1e4
    for p, q in zip(out[0][:2], out[1][:2]):
        assert np.linalg.norm(p - q) <= tol * np.linalg.norm(q)


@pytest.mark.parametrize("n,m,cap,k_nb", [
    (20000, 4097, 256, 64),      # first block whose rows leave early
    (20000, 20000, 256, 64),     # several chunks
    (20000, 4097, 30, 40),       # rows small enough for one copy: not early
    (20000, 5000, 100, 110),     # overflow
    (9000, 4500, 1000, 5)])
def test_rows_sent_beside_the_recomputation(n, m, cap, k_nb):
    """A checked query of more than 4096 targets sends its list rows while the
    flagged targets are recomputed; launch and fetch send them afterwards."""
    say(f"case: rows early n={n} m={m} cap={cap}")
    js = workloads.plummer_kroupa(n, seed=5, k_nb=k_nb)
    rng = np.random.default_rng(m)
    with regf.Context(device=0, cap=cap, precision=regf.PREC_CHECKED) as c:
        for f in (1.0, 0.0, 1.3):   # also no neighbour at all
            c.upload(js.m, js.x, js.v, js.r2 * f)
            t = rng.permutation(n)[:m].astype(np.int32)
            for _ in range(2):
                got = [a.copy() for a in c.query(t)]
                status, flagged = c.last_status, c.last_recheck()
                c.set_targets(t)
                c.launch()
                want = c.fetch()
                assert status == c.last_status and flagged == c.last_recheck()
                for p, q in zip(got, want):
                    assert np.array_equal(p, q)
        # a launch after a query, and the list kernels behind a step
        c.keep_lists()
        step = c.regular_step(t, np.full(m, 1e-3), np.zeros((m, 6)))
        for p, q in zip(step[:4], want):
            assert np.array_equal(p, q)
    assert flagged > 0


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED, regf.PREC_REFINED])
@pytest.mark.parametrize("n,lanes", [(1024, 0), (3000, 16), (9000, 64)])
def test_small_blocks_as_arguments(n, lanes, prec):
    """A query of up to 64 targets passes them to the kernel, a launch leaves
    them in memory, where a later block of the same size is found."""
    say(f"case: small blocks n={n} lanes={lanes} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=2, k_nb=20)
    rng = np.random.default_rng(n)
    with regf.Context(device=0, cap=64, precision=prec) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        c.set_tuning(0, 0, 0, lanes)
        for nt in (1, 63, 64, 65, 64, 2, 3):
            t = rng.permutation(n)[:nt].astype(np.int32)
            got = [a.copy() for a in c.query(t)]
            c.set_targets(t)
            c.launch()
            want = c.fetch()
            again = c.query(t)
            for p, q, r in zip(got, want, again):
                assert np.array_equal(p, q) and np.array_equal(p, r)
            assert (got[2] != 0).any()


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED, regf.PREC_MIXED,
                                  regf.PREC_REFINED, regf.PREC_FP64])
@pytest.mark.parametrize("n,m,cap,k_nb", [(67, 65, 64, 20), (300, 300, 64, 20),
                                          (1024, 257, 30, 40), (1900, 1900, 256, 40)])
def test_one_split_through_the_merge(n, m, cap, k_nb, prec):
    """A query of one split and more than 64 targets merges it into host
    memory, a launch leaves it where the kernel wrote it: the same bytes, and
    the same behind a step of resident lists."""
    say(f"case: one split n={n} m={m} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=9, k_nb=k_nb)
    t = np.random.default_rng(m).permutation(n)[:m].astype(np.int32)
    with regf.Context(device=0, cap=cap, precision=prec) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        c.set_tuning(0, 1, 0, 0)
        got = [a.copy() for a in c.query(t)]
        status, flagged = c.last_status, c.last_recheck()
        assert c.plan()["j_splits"] == 1
        c.set_targets(t)
        c.launch()
        want = c.fetch()
        assert status == c.last_status and flagged == c.last_recheck()
        c.keep_lists()
        step = c.regular_step(t, np.full(m, 1e-3), np.zeros((m, 6)))
        acc, adot = c.irregular(t)
    for p, q, r in zip(got, want, step):
        assert np.array_equal(p, q) and np.array_equal(p, r)
    assert np.array_equal(step[4][:, 12:15], acc) and np.array_equal(step[4][:, 15:], adot)
    assert (got[2] < 0).any() == (cap < k_nb)


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
def test_one_split_at_the_scratch_limit(prec):
    """A query whose one split does not fit the scratch limit leaves it where
    the kernel wrote it: the same bytes."""
    say(f"case: scratch limit precision={prec}")
    n, m = 1000, 700
    js = workloads.plummer_kroupa(n, seed=9, k_nb=40)
    t = np.random.default_rng(1).permutation(n)[:m].astype(np.int32)
    out = []
    for limit in (2 << 30, 1):
        with regf.Context(device=0, cap=100, precision=prec) as c:
            c.set_scratch_limit(limit)
            c.upload(js.m, js.x, js.v, js.r2)
            c.set_tuning(0, 1, 0, 16)
            out.append([a.copy() for a in c.query(t)])
            assert c.plan()["j_splits"] == 1
    for p, q in zip(*out):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("cap", [1, 17, 18, 700, 2030, 2031, 2048, 2049])
def test_regular_step_around_the_staged_lists(cap):
    """The corrector stages the old and new list of a target in LDS when both
    fit the workgroup's share, where the target's results follow them; lists of
    other strides are read where they are: the same bytes, and the irregular
    force of the step is that over the new lists, also overflowed ones."""
    say(f"case: staged lists cap={cap}")
    n, m = 4000, 70
    js = workloads.plummer_kroupa(n, seed=11, k_nb=300)
    rng = np.random.default_rng(11)
    t = rng.permutation(n)[:m].astype(np.int32)
    dt, a_old = rng.uniform(1e-3, 1e-2, m), rng.normal(size=(m, 6))
    z, out = np.zeros((n, 3)), []
    for stride in (cap, 701):
        with regf.Context(device=0, cap=stride) as c:
            c.upload_state(js.m, js.x, js.v, z, z, np.zeros(n), js.r2)
            c.keep_lists()
            c.query(t)
            c.predict(2.0 ** -5)   # other neighbours
            out.append(c.regular_step(t, dt, a_old))
            acc, adot = c.irregular(t)
            assert np.array_equal(out[-1][4][:, 12:15], acc)
            assert np.array_equal(out[-1][4][:, 15:], adot)
    if cap < 700:
        return
    for k in (0, 1, 2, 4):
        assert np.array_equal(out[0][k], out[1][k])
    assert np.array_equal(out[0][3][:, :700], out[1][3][:, :700]) and (out[0][2] > 0).all()


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
@pytest.mark.parametrize("n,cap,k_nb", [(4099, 64, 40), (4099, 20, 40), (32768, 64, 40)])
def test_shapes_list_by_tile_alike(n, cap, k_nb, prec):
    """Four lanes per target on a j-set of at most 32768 particles: every tile
    and workgroup gives the bits of 256 j and 4 waves, with own targets in full
    and partial tiles and overflowed lists."""
    say(f"case: shapes by tile n={n} cap={cap} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=13, k_nb=k_nb)
    rng = np.random.default_rng(n + cap)
    t = np.concatenate([np.arange(n - 5, n), rng.permutation(n - 5)[:600]]).astype(np.int32)
    with regf.Context(device=0, cap=cap, precision=prec) as c:
        c.upload(js.m, js.x, js.v, js.r2)
        for splits in (1, 3):
            c.set_tuning(0, splits, 0, 4)
            base = None
            for tile, waves in [(256, 4), (128, 4), (64, 4), (128, 2), (64, 2), (64, 1)]:
                c.set_shape(tile, waves)
                got = [a.copy() for a in c.query(t)] + [c.last_recheck()]
                p = c.plan()
                assert (p["tile"], p["waves_per_block"], p["lanes_per_target"]) == (tile, waves, 4)
                base = base or got
                for a, b in zip(got, base):
                    assert np.array_equal(a, b)
            # and the lists are those of sixteen lanes, found a step at a time
            c.set_shape()
            c.set_tuning(0, splits, 0, 16)
            want = c.query(t)
            assert np.array_equal(base[2], want[2]) and np.array_equal(base[3], want[3])
            assert (base[2] < 0).any() == (cap < k_nb)
