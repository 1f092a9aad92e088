"""The bond lists against the all-pairs build: group and wave edges, lists at
the longest length of the group kernel (128) and past it, several bodies with
their own horizons, invisible particles, pairs at the horizon exactly and
horizons whose square leaves the normal range."""
import numpy as np
import pytest

import oracle as orc
from pdhelpers import lattice

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


def check(x4, horizons, body=None, act=None):
    n = x4.shape[0]
    ctx = pds.Context(n, [(h, 0.1 * h, 1.0, 1.0) for h in horizons])
    pds.load_state(ctx, x4, np.zeros((n, 4)), np.full(n, 0.02), body=body, act=act)
    st = ctx.build_bonds()
    got_n, got = ctx.get_bonds()
    ctx.close()
    # invisible particles bond with nobody: a body of their own each
    b = np.zeros(n, np.int32) if body is None else body.copy()
    hs = list(horizons)
    if act is not None:
        gone = np.flatnonzero(act == 3)
        b[gone] = len(hs) + np.arange(len(gone))
        hs += [hs[0]] * len(gone)
    counts, lists, total = orc.bonds_brute(x4, hs, body=b)
    assert np.array_equal(got_n, counts) and st.total_bonds == total
    for p in range(n):
        assert np.array_equal(got[p, :counts[p]], np.sort(lists[p][:counts[p]])), p
    return int(counts.max())


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 129, 1000])
@pytest.mark.parametrize("factor", [1.0, 1.8, 3.0, 3.015])
def test_sizes(n, factor):
    print("case build", n, factor, flush=True)
    x4 = lattice(9, 9, 13, 0.01, 0.05 if factor != 1.0 else 0.0, n)[:n]
    check(x4, [factor * 0.01])


@pytest.mark.parametrize("n", [128, 129, 130, 200])
def test_longest_lists(n):
    """Everyone within everyone's horizon: lists of n - 1."""
    print("case build longest", n, flush=True)
    x4 = np.zeros((n, 4))
    x4[:, :3] = np.random.default_rng(n).uniform(-1, 1, (n, 3))
    assert check(x4, [10.0]) == n - 1


def test_bodies_and_invisible_particles_in_any_order():
    print("case build bodies", flush=True)
    rng = np.random.default_rng(3)
    x4 = lattice(10, 10, 9, 0.01, 0.2, 5)
    x4 = x4[rng.permutation(900)]
    act = np.where(rng.random(900) < 0.1, 3, 0).astype(np.int32)
    check(x4, [0.03, 0.021, 0.012], body=rng.integers(0, 3, 900).astype(np.int32), act=act)


@pytest.mark.parametrize("h", [1.0, 3.0, 2.0 ** 0.5, 0.1, 1e-170, 1e155])
def test_pairs_at_the_horizon(h):
    """Pairs at distance h times 1 - 4 ulp .. 1 + 4 ulp along an axis and on
    the diagonal of a square."""
    print("case build at the horizon", h, flush=True)
    k = 1.0 + np.arange(-8, 9) * 2.0 ** -53
    x4 = np.zeros((1 + 2 * len(k), 4))
    x4[1:1 + len(k), 0] = h * k
    x4[1 + len(k):, 1] = x4[1 + len(k):, 2] = -h * k / 2.0 ** 0.5
    check(x4, [h])
