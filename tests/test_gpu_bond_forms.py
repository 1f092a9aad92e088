"""Bond lengths at the floor (float)1e-10 that the unit vector divides by: the
shared-reciprocal forms leave out the floor and are taken only when every
bond is longer, the others go through IEEE division.  Lengths on both sides
of it, against the oracle bit for bit."""
import sys

import numpy as np
import pytest

import oracle as orc
from pdhelpers import deformed_pair

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")

FLOOR = np.float32(1e-10)
LENGTHS = [0.0, 1e-290, 5e-11, float(FLOOR), float(np.nextafter(FLOOR, np.float32(1))), 2e-10,
           1e-3]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("length", LENGTHS)
def test_short_bond_matches_oracle(length):
    say("case short bond", length)
    S, ctx = deformed_pair(s_fixed=10.0)
    S.x[0, :3] = 0.0
    S.x[1, :3] = (length, 0.0, 0.0)  # a lattice neighbour of particle 0
    ctx.upload("position", S.x)
    S.assemble(orc.make_params())
    x = np.zeros((S.n, 4))
    x[:, :3] = np.random.default_rng(5).normal(size=(S.n, 3))
    want = S.spmv(x)[:, :3]
    assert np.isnan(want).any() == (length * length == 0.0)
    for mode in (0, 1):
        ctx.assemble(pds.make_params(matrix_free=mode))
        assert np.array_equal(ctx.spmv(x)[:, :3], want, equal_nan=True), mode
    ctx.close()


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("length", LENGTHS[1:])
def test_short_bond_solve_matches_oracle(length, mode):
    """Three iterations of the stored and of the recomputing solve."""
    say("case short bond solve", length, mode)
    kw = dict(dt=2e-6, precond=0, rtol=0.0, max_iter=3)
    S, ctx = deformed_pair(s_fixed=10.0)
    S.x[0, :3] = 0.0
    S.x[1, :3] = (length, 0.0, 0.0)
    ctx.upload("position", S.x)
    S.assemble(orc.make_params(**kw))
    S.cg(orc.make_params(**kw))
    ctx.assemble(pds.make_params(matrix_free=mode, **kw))
    with pytest.raises(pds.PDError, match="iteration limit"):
        ctx.solve(pds.make_params(matrix_free=mode, **kw))
    assert np.array_equal(ctx.download("solution")[:, :3], S.sol[:, :3], equal_nan=True)
    ctx.close()
