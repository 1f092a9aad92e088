"""The resident step of small systems (up to 256 slices of 64 rows, lists of
at most 120 bonds) against the oracle, bit for bit: row counts at the edges
of a unit, of a slice, of the lane counts 32 / 16 / 8 and of its range,
lists broken in the middle and to the end, both integrators and operators,
specimens, and a wait that runs out."""
import ctypes
import sys
import threading
import time

import numpy as np
import pytest

import oracle as orc
from pdhelpers import (compare_specimens, lattice, make_pair, make_system, material,
                       specimen_pair)

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def pair(n, pull=6.0, factor=3.0):
    """n rows of a jittered lattice, the first layer fixed, the last pulled."""
    w = 4 if n < 2000 else 12
    x4 = lattice(w, w, -(-n // (w * w)), 0.01, 0.05, n)[:n]
    k = np.arange(n) // (w * w)
    bc = ((k == 0) | (k == k[-1])).astype(np.int32) if n > w * w else np.zeros(n, np.int32)
    vbc = np.zeros((n, 4))
    vbc[(k == k[-1]) & (bc == 1), 2] = pull
    return make_pair(x4, [material(0.01, factor)], v4=vbc.copy(), bc=bc, vbc=vbc)


def compare(S, ctx, steps, **kw):
    broken = 0
    for k in range(1, steps + 1):
        p = dict(dict(dt=1e-4, clock_scale=min(k, 10) / 10.0, precond=1, rtol=1e-8), **kw)
        so = S.step(orc.make_params(**p))
        sg = ctx.step(pds.make_params(**p))
        assert (so.cg_iterations, so.broken_bonds) == (sg.cg_iterations, sg.broken_bonds), k
        for f, want in (("position", S.x), ("velocity", S.v), ("new_stretch", S.s)):
            got = ctx.download("stretch" if f == "new_stretch" else f)
            same = np.array_equal(got[:, :3], want[:, :3]) if got.ndim > 1 else np.array_equal(got, want)
            assert same, (f, k)
        broken += sg.broken_bonds
    assert np.array_equal(ctx.download("bond_top"), S.top)
    return broken


# 1, 63..65: a slice's edge; 4096 / 4097 and 8192 / 8193: the lane counts;
# 16384 / 16385: the last resident size and the first general one
@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 257, 1000, 4096, 4097, 8192, 8193, 16384, 16385])
def test_sizes_match_oracle(n):
    say("case small n", n)
    S, ctx = pair(n)
    broken = compare(S, ctx, 12 if n < 4000 else 6)
    say(dict(n=n, broken=broken))
    ctx.close()


@pytest.mark.parametrize("kw", [dict(matrix_free=1), dict(matrix_free=2), dict(precond=0),
                                dict(integrator=1), dict(max_iter=3), dict(rtol=1e10),
                                dict(graph=1)])
def test_options_match_oracle(kw):
    say("case small", kw)
    S, ctx = pair(900)
    o = {k: v for k, v in kw.items() if k not in ("matrix_free", "graph")}
    for k in range(1, 25):
        p = dict(dict(dt=1e-4, clock_scale=min(k, 10) / 10.0, precond=1, rtol=1e-8), **o)
        so = S.step(orc.make_params(**p))
        sg = ctx.step(pds.make_params(**dict(p, **kw)), allow_fail=True)
        assert (so.cg_iterations, bool(so.converged), so.broken_bonds) == \
            (sg.cg_iterations, bool(sg.converged), sg.broken_bonds), k
        assert np.array_equal(ctx.download("position")[:, :3], S.x[:, :3]), k
    ctx.close()


@pytest.mark.parametrize("factor", [2.5, 3.1, 3.3])
def test_list_lengths(factor):
    """Longest lists below and above the 120 blocks a row's lanes hold, and
    rows that lose most of their bonds."""
    say("case small horizon", factor)
    S, ctx = pair(1700, pull=12.0, factor=factor)
    say(dict(longest=int(ctx.download("bond_top").max()) + 1))
    assert compare(S, ctx, 20) > 0
    ctx.close()


def test_wait_that_runs_out_falls_back():
    """A wait limit of zero: every workgroup gives up at its first wait and
    the general kernels solve the step, with the same results."""
    say("case small wait limit")
    L = pds.lib()
    L.pd_set_wait_limit.argtypes = [ctypes.c_void_p, ctypes.c_double]
    S, ctx = pair(8000)
    assert L.pd_set_wait_limit(ctx._h, 0.0) == pds.PD_OK
    compare(S, ctx, 2)
    assert L.pd_set_wait_limit(ctx._h, 2.0) == pds.PD_OK
    compare_from = S.x.copy()
    for k in range(3, 6):
        p = dict(dt=1e-4, clock_scale=k / 10.0, precond=1, rtol=1e-8)
        S.step(orc.make_params(**p))
        ctx.step(pds.make_params(**p))
    assert np.array_equal(ctx.download("position")[:, :3], S.x[:, :3])
    assert not np.array_equal(compare_from, S.x)
    assert L.pd_set_wait_limit(ctx._h, -1.0) == pds.PD_ERR_ARG
    ctx.close()


def test_operands_out_of_range_take_ieee_forms():
    """A coordinate outside the shared-reciprocal range: IEEE quotients."""
    say("case small range flag")
    x4 = lattice(6, 6, 8, 0.01, 0.0, 3)
    x4[:, :3] -= x4[0, :3]
    x4[5, 1] = 1e-200
    S, ctx = make_pair(x4, [material(0.01)])
    compare(S, ctx, 6)
    ctx.close()


# 32, 16 and 8 lanes per row; rows of padding before the first specimen
@pytest.mark.parametrize("lead", [0, 256, 512])
@pytest.mark.parametrize("sizes", [(300, 700), (2500, 3000), (5000, 1, 4000)])
def test_specimens_match_oracle(sizes, lead):
    """Every specimen as if alone, in one resident launch (one wait a step)."""
    say("case small specimens", sizes, lead)
    first, alone, ctx = specimen_pair(sizes, lead)
    syncs = []

    def step(q):
        sg = ctx.step(pds.make_params(**q))
        syncs.append(sg.host_syncs)
        return sg

    broken = compare_specimens(first, alone, ctx, step, {}, 12)
    say(dict(broken=broken, syncs=syncs))
    assert broken > 0 and syncs == [1] * 12
    ctx.close()


def test_limit_counts_from_each_wait():
    """A solve that makes progress outlasts the limit and is not given up,
    also while another context's kernels slow some of its workgroups down:
    40,000 iterations of 8 us or more, 0.1 s a wait."""
    say("case small long solve")
    L = pds.lib()
    L.pd_set_wait_limit.argtypes = [ctypes.c_void_p, ctypes.c_double]

    def bar(n, w):
        x4 = lattice(w, w, -(-n // (w * w)), 0.01, 0.05, n)[:n]
        v4 = np.zeros((n, 4))
        v4[:, :3] = np.random.default_rng(n).uniform(-1, 1, (n, 3))
        ctx = pds.Context(n, [material(0.01)])
        pds.load_state(ctx, x4, v4, np.full(n, 1e9))
        ctx.build_bonds()
        return ctx

    other, stop = bar(100000, 40), threading.Event()

    def load():
        while not stop.is_set():
            other.step(pds.make_params(dt=1e-6, matrix_free=1, rtol=1e-12))

    out = []
    for limit in (2.0, 0.1):
        ctx = bar(13225, 4)
        assert L.pd_set_wait_limit(ctx._h, limit) == pds.PD_OK
        stop.clear()
        t = threading.Thread(target=load)
        t.start()
        try:
            st = ctx.step(pds.make_params(dt=1.0, precond=0, rtol=0.0, max_iter=40000),
                          allow_fail=True)
        finally:
            stop.set()
            t.join()
        out.append((st.cg_iterations, st.host_syncs, st.residual_norm,
                    ctx.download("position").tobytes()))
        ctx.close()
    other.close()
    say([o[:3] for o in out])
    assert out[0][0] == 40000 and out[0][1] == 1
    assert out[0] == out[1]


@pytest.mark.parametrize("kw", [dict(matrix_free=0), dict(matrix_free=1), dict(matrix_free=2),
                                dict(matrix_free=1, integrator=1), dict(precond=0),
                                dict(matrix_free=0, graph=1), dict(rtol=1e10)])
@pytest.mark.parametrize("lead", [0, 256])
def test_fallback_matches_oracle(lead, kw):
    """A limit of zero gives the solve up before its first iteration, also one
    that would end there: that step and the next ones come from the general
    kernels (more than one host wait; a general step after that has the
    previous one's count), a new limit takes the resident solve up again."""
    say("case small fallback", lead, kw)
    first, alone, ctx = specimen_pair((300, 700), lead)
    syncs = []

    def step(q):
        if len(syncs) == 3:
            ctx.set_wait_limit(0.0)
        if len(syncs) == 6:
            ctx.set_wait_limit(2.0)
        sg = ctx.step(pds.make_params(**q))
        syncs.append(sg.host_syncs)
        return sg

    compare_specimens(first, alone, ctx, step, kw, 9)
    say(syncs)
    assert syncs[:3] == [1] * 3 and syncs[6:] == [1] * 3
    assert syncs[3] > 1
    with pytest.raises(pds.PDError):
        ctx.set_wait_limit(-1.0)
    ctx.close()


def test_contexts_step_side_by_side():
    """A short system's steps end while another context's long solve (126 of the
    256 workgroups, 40,000 iterations) is still under way, each with the bits
    of a run of its own."""
    say("case small side by side")

    def bar(n, seed):
        x4 = lattice(4, 4, -(-n // 16), 0.01, 0.05, seed)[:n]
        v4 = np.zeros((n, 4))
        v4[:, :3] = np.random.default_rng(seed).uniform(-1, 1, (n, 3))
        ctx = pds.Context(n, [material(0.01)])
        pds.load_state(ctx, x4, v4, np.full(n, 1e9))
        ctx.build_bonds()
        return ctx

    def long_solve(ctx):
        st = ctx.step(pds.make_params(dt=100.0, precond=0, rtol=0.0, max_iter=40000),
                      allow_fail=True)
        say(dict(iterations=st.cg_iterations))
        assert st.cg_iterations > 30000 and st.host_syncs == 1

    def short_steps(ctx):
        for _ in range(20):
            ctx.step(pds.make_params(dt=1e-4))

    want = []
    for n, work in ((2000, long_solve), (300, short_steps)):
        ctx = bar(n, n)
        work(ctx)
        want.append(ctx.download("position"))
        ctx.close()
    a, b = bar(2000, 2000), bar(300, 300)
    errors = []

    def run():
        try:
            long_solve(a)
        except Exception as e:  # noqa: BLE001 -- told to the test's thread
            errors.append(e)

    t = threading.Thread(target=run)
    t.start()
    time.sleep(0.05)  # the long solve (0.3 s) has its workgroups
    t0 = time.perf_counter()
    short_steps(b)
    spent = time.perf_counter() - t0
    still = t.is_alive()
    t.join()
    say(dict(short=spent, still=still))
    assert not errors and still
    assert np.array_equal(a.download("position"), want[0])
    assert np.array_equal(b.download("position"), want[1])
    a.close()
    b.close()


def listed_pair(x4, counts, lists, factor, s0, **kw):
    """make_pair with the lists given (counts, padded rows)."""
    mats = [material(0.01, factor)]
    S = make_system(x4, mats, s0=s0, lists=(counts, lists), **kw)
    ctx = pds.Context(len(x4), mats)
    pds.load_state(ctx, x4, S.v, S.s00, bc=kw.get("bc"), vbc=kw.get("vbc"))
    ctx.set_bonds(counts, lists)
    return S, ctx


def compare_limited(S, ctx, steps, **kw):
    """compare() of solves that may end at the iteration limit (a list cut off
    leaves no symmetric matrix); returns the first step's host waits."""
    syncs = []
    for k in range(1, steps + 1):
        p = dict(dict(dt=1e-4, clock_scale=k / 10.0, precond=1, rtol=1e-8, max_iter=30), **kw)
        so = S.step(orc.make_params(**p))
        sg = ctx.step(pds.make_params(**p), allow_fail=True)
        syncs.append(sg.host_syncs)
        assert so.cg_iterations > 1
        assert (so.cg_iterations, so.broken_bonds, so.residual_norm) == \
            (sg.cg_iterations, sg.broken_bonds, sg.residual_norm), k
        assert np.isfinite(S.x).all()
        assert np.array_equal(ctx.download("position")[:, :3], S.x[:, :3]), k
    assert np.array_equal(ctx.download("bond_top"), S.top)
    return syncs[0]


# 32, 16 and 8 lanes per row
@pytest.mark.parametrize("layers", [7, 90, 180])
@pytest.mark.parametrize("longest", [119, 120, 121, 128, 129])
def test_longest_list(layers, longest):
    """Lists of exactly the longest that the resident step takes, one fewer and
    more (rows well inside the lattice have 146 neighbours, cut off here)."""
    say("case small longest list", layers, longest)
    x4 = lattice(7, 7, layers, 0.01, 0.01, layers)
    n = len(x4)
    counts, lists, _ = orc.bonds_brute(x4, [0.0324])
    assert counts.max() == 146
    counts = np.minimum(counts, longest).astype(np.int32)
    k = np.arange(n) // 49
    bc = ((k == 0) | (k == layers - 1)).astype(np.int32)
    vbc = np.zeros((n, 4))
    vbc[k == layers - 1, 2] = 12.0
    S, ctx = listed_pair(x4, counts, lists[:, :longest], 3.24, 0.02, v4=vbc.copy(), bc=bc, vbc=vbc)
    first = compare_limited(S, ctx, 6)
    say(dict(waits=first, broken=int(counts.sum() - (S.top + 1).sum())))
    assert (first == 1) == (longest <= 120)
    ctx.close()


@pytest.mark.parametrize("others", [1823, 1824])
def test_neighbours_of_a_unit(others):
    """Eight lanes per row: rows 64 .. 127 have this many neighbours outside;
    with themselves and one more the first are the 1888 that the solve holds in
    LDS, the second one too many."""
    say("case small neighbours of a unit", others)
    n = 8256
    x4 = lattice(12, 12, 58, 0.01, 0.05, 3)[:n]
    rows = [[q for q in (p - 1, p + 1) if 0 <= q < n] for p in range(n)]
    for i in range(64):
        rows[64 + i] = list(range(128 + i, 128 + others, 64))
    counts = np.array([len(r) for r in rows], np.int32)
    lists = np.zeros((n, counts.max()), np.int32)
    for p, r in enumerate(rows):
        lists[p, :len(r)] = r
    v4 = np.zeros((n, 4))
    v4[:, :3] = np.random.default_rng(n).uniform(-1, 1, (n, 3))
    S, ctx = listed_pair(x4, counts, lists, 3.0, 1e9, v4=v4)
    first = compare_limited(S, ctx, 3)
    say(dict(waits=first))
    assert (first == 1) == (others == 1823)
    ctx.close()
