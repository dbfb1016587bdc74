"""Launches recorded into a HIP graph by the caller (abyss_ctx_stream) and
replayed between other calls on the context: every replay leaves what an
eager launch of the same targets on the same j-set leaves."""
import ctypes
import sys

import numpy as np
import pytest

from abyss_amd import regf, workloads

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


class Graph:
    """What a `with` block enqueues on a context's stream, as a graph."""

    def __init__(self, ctx):
        self.lib = ctypes.CDLL("libamdhip64.so")
        self.stream = ctypes.c_void_p(ctx.stream)
        self.graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()

    def __enter__(self):
        # the default mode: calls that may wait or allocate are refused
        assert self.lib.hipStreamBeginCapture(self.stream, 0) == 0
        return self

    def __exit__(self, kind, *a):
        rc = self.lib.hipStreamEndCapture(self.stream, ctypes.byref(self.graph))
        if kind is None:
            assert rc == 0
            assert self.lib.hipGraphInstantiate(ctypes.byref(self.exec), self.graph, None, None,
                                                ctypes.c_size_t(0)) == 0

    def replay(self):
        assert self.lib.hipGraphLaunch(self.exec, self.stream) == 0

    def free(self):
        self.lib.hipStreamSynchronize(self.stream)
        if self.exec:
            self.lib.hipGraphExecDestroy(self.exec)
        if self.graph:
            self.lib.hipGraphDestroy(self.graph)


def same(a, b):
    return all(np.array_equal(p, q) for p, q in zip(a, b))


@pytest.mark.parametrize("n,nt,prec", [
    (n, nt, p) for n, nt in ((1024, 1), (1024, 64), (20000, 16), (20000, 300))
    for p in (regf.PREC_SPLIT, regf.PREC_CHECKED)])
def test_replays_between_other_calls(n, nt, prec):
    """One split and several, lists of up to 64 targets and longer ones (a
    checked block of 300 with the count of its recomputation on the device)."""
    say(f"case: replay n={n} targets={nt} precision={prec}")
    js = [workloads.plummer_kroupa(n, seed=s, k_nb=30) for s in (1, 2)]
    rng = np.random.default_rng(n + nt)
    pick = [rng.permutation(n)[:nt].astype(np.int32) for _ in range(4)]
    with regf.Context(device=0, cap=64, precision=prec) as c, \
            regf.Context(device=0, cap=64, precision=prec) as d:
        want = {}
        for k, s in enumerate(js):
            d.upload(s.m, s.x, s.v, s.r2)
            for i, t in enumerate(pick):
                want[k, i] = [a.copy() for a in d.query(t)]
        c.upload(js[0].m, js[0].x, js[0].v, js[0].r2)
        c.set_targets(pick[0])
        c.launch()
        assert same(c.fetch(), want[0, 0])
        g = Graph(c)
        with g:
            c.launch()
        for i in (1, 2, 3):
            c.set_targets(pick[i])
            g.replay()
            assert same(c.fetch(), want[0, i])
            # a query of the same targets, then a replay on another j-set
            assert same(c.query(pick[i]), want[0, i])
            c.upload(js[1].m, js[1].x, js[1].v, js[1].r2)
            g.replay()
            assert same(c.fetch(), want[1, i])
            c.upload(js[0].m, js[0].x, js[0].v, js[0].r2)
        g.free()


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
@pytest.mark.parametrize("n", [1024, 20000])
def test_first_launch_of_a_context_recorded(n, prec):
    """A block's first launch allocates nothing, so it can be recorded."""
    say(f"case: first launch recorded n={n} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=3, k_nb=30)
    rng = np.random.default_rng(n)
    with regf.Context(device=0, cap=64, precision=prec) as c, \
            regf.Context(device=0, cap=64, precision=prec) as d:
        for k in (c, d):
            k.upload(js.m, js.x, js.v, js.r2)
        c.set_targets(rng.permutation(n)[:16].astype(np.int32))
        g = Graph(c)
        with g:
            c.launch()
        for _ in range(3):
            t = rng.permutation(n)[:16].astype(np.int32)
            c.set_targets(t)
            g.replay()
            assert same(c.fetch(), d.query(t))
        g.free()


@pytest.mark.parametrize("prec", [regf.PREC_SPLIT, regf.PREC_CHECKED])
@pytest.mark.parametrize("n", [1024, 20000])
def test_replay_after_a_query_of_more_rows(n, prec):
    """Queries of up to 4096 targets within the context's capacity, also with
    more than 1 MB of list rows, leave the buffers of a recorded launch of 16
    targets where they are."""
    say(f"case: replay after larger queries n={n} precision={prec}")
    js = workloads.plummer_kroupa(n, seed=4, k_nb=30)
    rng = np.random.default_rng(n)
    sizes = (min(n, 4096), 900, min(n, 2500), 64)
    with regf.Context(device=0, cap=400, precision=prec) as c, \
            regf.Context(device=0, cap=400, precision=prec) as d:
        for k in (c, d):
            k.upload(js.m, js.x, js.v, js.r2)
        # the scratch and outputs of every block, before anything is recorded
        for nt in sizes:
            c.set_targets(np.arange(nt, dtype=np.int32))
            c.launch()
            c.fetch()
        c.set_targets(rng.permutation(n)[:16].astype(np.int32))
        g = Graph(c)
        with g:
            c.launch()
        for nt in sizes[1:] + sizes[:1]:
            big = rng.permutation(n)[:nt].astype(np.int32)
            assert same(c.query(big), d.query(big))
            t = rng.permutation(n)[:16].astype(np.int32)
            c.set_targets(t)
            g.replay()
            assert same(c.fetch(), d.query(t))
        g.free()


def test_calls_that_wait_are_refused_and_leave_nothing_behind():
    """Under a capture the calls that wait for their results, and updates of the
    state, fail; the capture goes on, and the context holds what it held."""
    say("case: calls refused under a capture")
    n, cap = 5000, 128
    js = workloads.plummer_kroupa(n, seed=5, k_nb=30)
    rng = np.random.default_rng(5)
    a, ad = 0.1 * rng.normal(size=(n, 3)), 0.1 * rng.normal(size=(n, 3))
    t, other = (rng.permutation(n)[:300].astype(np.int32) for _ in range(2))
    dt, a_old = np.full(300, 1e-3), np.zeros((300, 6))
    with regf.Context(device=0, cap=cap) as c, regf.Context(device=0, cap=cap) as d:
        for k in (c, d):
            k.upload_state(js.m, js.x, js.v, a, ad, np.zeros(n), js.r2)
            k.keep_lists()
            k.query(np.arange(n, dtype=np.int32))
            k.irregular(t)
            # gather records of the positions before, not of these
            k.upload_state(js.m, 1.01 * js.x, js.v, a, ad, np.zeros(n), js.r2)
        held = [p.copy() for p in c.query(t)]
        d.query(t)
        g = Graph(c)
        with g:
            for call in (lambda: c.query(other), lambda: c.irregular(other),
                         lambda: c.regular_step(other, dt, a_old),
                         lambda: c.update_state(other, js.m[other], 2 * js.x[other], js.v[other],
                                                a[other], ad[other], np.zeros(300),
                                                js.r2[other])):
                with pytest.raises(regf.AbyssError) as e:
                    call()
                assert e.value.code == regf.ERR_HIP
        assert same(c.fetch(), held)
        assert same(c.irregular(t), d.irregular(t))
        for k in (c, d):
            k.predict(2.0 ** -7)
        assert same(c.irregular(other), d.irregular(other))
        assert same(c.regular_step(other, dt, a_old), d.regular_step(other, dt, a_old))
        g.free()


def test_recorded_predictions_and_the_irregular_force():
    """A prediction that is recorded but not run leaves the j-set, and what the
    irregular force reads of it, as uploaded; each replay moves both."""
    say("case: recorded predictions")
    n, t_new = 5000, 2.0 ** -6
    js = workloads.plummer_kroupa(n, seed=7, k_nb=30)
    rng = np.random.default_rng(7)
    a, ad = 0.1 * rng.normal(size=(n, 3)), 0.1 * rng.normal(size=(n, 3))
    t = rng.permutation(n)[:500].astype(np.int32)
    with regf.Context(device=0, cap=128) as c, regf.Context(device=0, cap=128) as d:
        for k in (c, d):
            k.upload_state(js.m, js.x, js.v, a, ad, np.zeros(n), js.r2)
            k.keep_lists()
            k.query(np.arange(n, dtype=np.int32))
            k.irregular(t)
            # gather records of the positions before, not of these
            k.upload_state(js.m, 1.01 * js.x, js.v, a, ad, np.zeros(n), js.r2)
        g = Graph(c)
        with g:
            c.predict(t_new)
        assert same(c.irregular(t), d.irregular(t))
        for factor in (1.01, 1.02):
            g.replay()
            d.predict(t_new)
            assert same(c.irregular(t), d.irregular(t))
            for k in (c, d):
                k.upload_state(js.m, factor * js.x, js.v, a, ad, np.zeros(n), js.r2)
            assert same(c.irregular(t), d.irregular(t))
        g.free()
