"""The matrix-free product with eight lanes per row (up to 512 slices of 64
rows) and with four (up to 1536), on systems that do not take the resident
step (here because they are timed, solved on their own or too large for it):
row counts at the edges of a wave's rows, a slice, a tile and of the ranges,
lists of every remainder by its 16 slots and longer than the resident step's,
specimens and a range flag."""
import sys

import numpy as np
import pytest

import oracle as orc
from pdhelpers import compare_specimens, lattice, make_pair, material, specimen_pair
from test_gpu_small import compare, pair

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def general(S, ctx, steps, **kw):
    """compare() with the step timed, so that it takes the general kernels."""
    broken = 0
    for k in range(1, steps + 1):
        p = dict(dict(dt=1e-4, clock_scale=min(k, 10) / 10.0, precond=1, rtol=1e-8), **kw)
        so = S.step(orc.make_params(**p))
        sg = ctx.step(pds.make_params(matrix_free=1, timing=1, **p))
        assert (so.cg_iterations, so.broken_bonds, so.residual_norm) == \
            (sg.cg_iterations, sg.broken_bonds, sg.residual_norm), k
        for f, want in (("position", S.x), ("velocity", S.v)):
            assert np.array_equal(ctx.download(f)[:, :3], want[:, :3]), (f, k)
        broken += sg.broken_bonds
    assert np.array_equal(ctx.download("bond_top"), S.top)
    return broken


@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 255, 257, 1000, 8193])
def test_sizes_match_oracle(n):
    say("case lanes n", n)
    S, ctx = pair(n)
    say(dict(broken=general(S, ctx, 8 if n < 4000 else 4)))
    ctx.close()


@pytest.mark.parametrize("factor", [1.1, 1.8, 2.3, 2.9, 4.2])
def test_list_lengths(factor):
    say("case lanes factor", factor)
    S, ctx = pair(1000, pull=2.0, factor=factor)
    say(dict(longest=int(S.top.max()) + 1, broken=general(S, ctx, 4, precond=0)))
    ctx.close()


def test_first_size_past_the_resident_step():
    say("case lanes 16385")
    S, ctx = pair(16385)
    compare(S, ctx, 3, matrix_free=1)
    ctx.close()


def test_operands_out_of_range_take_ieee_forms():
    say("case lanes range flag")
    x4 = lattice(6, 6, 8, 0.01, 0.0, 3)
    x4[:, :3] -= x4[0, :3]
    x4[5, 1] = 1e-200
    S, ctx = make_pair(x4, [material(0.01)])
    general(S, ctx, 4)
    ctx.close()


@pytest.mark.parametrize("n,factor", [(32768, 3.0), (32769, 3.0), (40001, 2.3), (98304, 1.8),
                                      (98305, 1.8)])
def test_ends_of_the_ranges_equal_stored(n, factor):
    """The last size with eight lanes, the first with four, the last with four
    and the first with one, against the stored blocks."""
    say("case lanes n", n, factor)
    x4 = lattice(48, 48, -(-n // 2304), 0.01, 0.05, n)[:n]
    v4 = np.zeros((n, 4))
    v4[:, 2] = np.linspace(-1, 1, n)
    out = []
    for mode in (0, 1):
        ctx = pds.Context(n, [material(0.01, factor)])
        pds.load_state(ctx, x4, v4, np.full(n, 0.02))
        ctx.build_bonds()
        st = [ctx.step(pds.make_params(dt=1e-4, precond=1, rtol=1e-8, matrix_free=mode))
              for _ in range(3)]
        out.append(([(s.cg_iterations, s.broken_bonds, s.residual_norm) for s in st],
                    ctx.download("position"), ctx.download("velocity")))
        ctx.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("mode", [0, 1])
def test_captured_steps_equal_eager(mode):
    """Past the resident step, captured: the folds inside the direction update
    and the per-slice partials on every replay."""
    say("case lanes captured", mode)
    n = 17000
    ends = []
    for graph in (0, 1):
        x4 = lattice(26, 26, 26, 0.01, 0.05, n)[:n]
        k = np.arange(n) // 676
        bc = ((k == 0) | (k == k[-1])).astype(np.int32)
        vbc = np.zeros((n, 4))
        vbc[k == k[-1], 2] = 6.0
        ctx = pds.Context(n, [material(0.01)])
        pds.load_state(ctx, x4, vbc.copy(), np.full(n, 0.01), bc=bc, vbc=vbc)
        ctx.build_bonds()
        out = []
        for step in range(1, 9):
            st = ctx.step(pds.make_params(dt=1e-4, clock_scale=step / 8.0, precond=1, rtol=1e-8,
                                          matrix_free=mode, graph=graph))
            out.append((st.cg_iterations, st.broken_bonds, st.live_bonds, st.residual_norm))
            if step % 3 == 0:
                ctx.download("velocity")  # the program's own work between replays
        ends.append((out, ctx.download("position"), ctx.download("bond_top")))
        ctx.close()
    say(dict(its=[o[0] for o in ends[0][0]], broken=sum(o[1] for o in ends[0][0])))
    assert ends[0][0] == ends[1][0]
    assert np.array_equal(ends[0][1], ends[1][1]) and np.array_equal(ends[0][2], ends[1][2])


# 18,176 rows, the first tile padding: eight lanes per row; 34,304: four
@pytest.mark.parametrize("sizes,lead", [((300, 9000, 8000), 256), ((9000, 1, 8500, 16000), 0)])
def test_specimens_match_oracle(sizes, lead):
    """Specimens past the resident step, stored and recomputed, eager and
    captured: each as if alone in the oracle, also beside ones that have ended."""
    say("case lanes specimens", sizes, lead)
    first, alone, ctx = specimen_pair(sizes, lead, pull=9.0)
    others = [(dict(matrix_free=m, graph=g), specimen_pair(sizes, lead, pull=9.0)[2])
              for m, g in ((0, 1), (1, 0), (1, 1))]
    ends = set()

    def step(q):
        sg = ctx.step(pds.make_params(**q))
        per = ctx.specimen_stats(len(sizes))
        ends.add(tuple(s["cg_iterations"] for s in per))
        for kw, o in others:
            so = o.step(pds.make_params(**dict(q, **kw)))
            assert (so.cg_iterations, so.broken_bonds, so.live_bonds) == \
                (sg.cg_iterations, sg.broken_bonds, sg.live_bonds), kw
            assert o.specimen_stats(len(sizes)) == per, kw
            for f in ("position", "velocity", "bond_top"):
                assert np.array_equal(o.download(f), ctx.download(f)), (f, kw)
        return sg

    broken = compare_specimens(first, alone, ctx, step, {}, 10)
    say(dict(broken=broken, iterations=sorted(ends)))
    assert broken > 0 and any(len(set(e)) > 1 for e in ends)
    for c in [ctx] + [o for _, o in others]:
        c.close()
