"""The general solve's folds at the edges of their loads: tiles at one load
per thread, eight, and past them, and around the size where the direction
update stops folding for itself.  Stored against recomputed blocks, whose
products differ in kernel and partials but not in bits, and against the oracle
where it is quick."""
import numpy as np
import pytest

import oracle as orc
from pdhelpers import lattice, make_pair, material

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


def run(n, mode, steps):
    w = 64
    x4 = lattice(w, w, -(-n // (w * w)), 0.01, 0.05, n)[:n]
    v4 = np.zeros((n, 4))
    v4[:, :3] = np.random.default_rng(n).uniform(-1, 1, (n, 3))
    ctx = pds.Context(n, [material(0.01, 1.2)])
    pds.load_state(ctx, x4, v4, np.full(n, 0.02))
    ctx.build_bonds()
    st = [ctx.step(pds.make_params(dt=1e-4, precond=1, rtol=1e-9, matrix_free=mode, timing=1))
          for _ in range(steps)]
    out = ([(s.cg_iterations, s.broken_bonds, s.residual_norm) for s in st],
           ctx.download("position"))
    ctx.close()
    return out


# 256 tiles, 257; 1024 tiles (the last to fold in every workgroup), 1025; 2049
@pytest.mark.parametrize("n", [65536, 65537, 262144, 262145, 524289])
def test_sizes_agree(n):
    print("case fold", n, flush=True)
    a, b = run(n, 0, 2), run(n, 1, 2)
    assert a[0] == b[0] and a[0][0][0] > 1
    assert np.array_equal(a[1], b[1])


def test_end_at_the_iteration_limit():
    """The limit, not the tolerance, ends the solve: the same count and x."""
    print("case fold limit", flush=True)
    kw = dict(dt=2e-4, precond=1, rtol=0.0, max_iter=5)
    S, ctx = make_pair(lattice(8, 8, 9, 0.01, 0.05, 1), [material(0.01)],
                       v4=np.pad(np.random.default_rng(0).uniform(-1, 1, (576, 3)), ((0, 0), (0, 1))))
    S.assemble(orc.make_params(**kw))
    S.cg(orc.make_params(**kw))
    ctx.assemble(pds.make_params(**kw))
    with pytest.raises(pds.PDError, match="iteration limit"):
        ctx.solve(pds.make_params(**kw))
    assert np.array_equal(ctx.download("solution")[:, :3], S.sol[:, :3])
    ctx.close()
