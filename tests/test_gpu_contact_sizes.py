"""The contact phase at the edges of its kernels: particle counts around a
tile of 256 and around the 4096 tiles up to which the selection adds up the
tiles' counts in place, bodies from two to eight, and dense neighbourhoods of
many chunks of 64 members."""
import numpy as np
import pytest

import oracle as orc
from pdhelpers import lattice, make_pair, material

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


def kwargs(rc):
    return dict(contact_radius=rc, contact_stiffness=2.5e8, contact_volume=1.0, contact_cell=rc)


def forces(x4, body, mats, kw):
    n = x4.shape[0]
    ctx = pds.Context(n, mats)
    pds.load_state(ctx, x4, np.zeros((n, 4)), np.full(n, 0.02), body=body)
    ctx.build_bonds()
    ctx.assemble(pds.make_params(**kw))
    fc = ctx.download("contact_force")
    ctx.close()
    return fc


@pytest.mark.parametrize("n,nbody", [(2, 2), (255, 2), (256, 3), (257, 2), (511, 8), (1025, 5),
                                     (3000, 8)])
def test_sizes_match_oracle(n, nbody):
    print("case contact", n, nbody, flush=True)
    rng = np.random.default_rng(n)
    x4 = np.zeros((n, 4))
    x4[:, :3] = rng.uniform(0.0, 0.1, (n, 3))
    if n == 2:
        x4[1, :3] = x4[0, :3] + 0.001
    body = (np.arange(n) % nbody).astype(np.int32)
    mats = [material(0.01, horizon_factor=0.05)] * nbody
    kw = kwargs(0.02 if n < 3000 else 0.035)  # up to 27 cells of 130 members
    S, ctx = make_pair(x4, mats, body=body)
    S.contact(orc.make_params(**kw))
    ctx.assemble(pds.make_params(**kw))
    fc = ctx.download("contact_force")
    ctx.close()
    assert np.abs(S.fc).max() > 0
    assert np.array_equal(fc[:, :3], S.fc[:, :3])


def test_selection_past_4096_tiles():
    """The same contacts behind a filler that ends with the 4096th tile, or one
    particle later: counts added up in place, or scanned."""
    print("case contact tiles", flush=True)
    a = lattice(8, 8, 4, 0.01, 0.05, 1)
    b = lattice(4, 4, 4, 0.0047, 0.05, 2, origin=(0.02, 0.02, 0.0335))
    total = 4096 * 256 + 1
    far = lattice(103, 102, 100, 0.01, 0.0, 3, origin=(1.0, 1.0, 1.0))[:total - len(a) - len(b)]
    assert len(a) + len(b) + len(far) == total
    x4 = np.concatenate([a, far[:500000], b, far[500000:]])
    body = np.zeros(total, np.int32)
    body[len(a) + 500000:len(a) + 500000 + len(b)] = 1
    mats = [material(0.01, horizon_factor=0.5)] * 2  # no bonds
    f1 = forces(x4, body, mats, kwargs(0.0075))
    f0 = forces(x4[:-1], body[:-1], mats, kwargs(0.0075))
    S = make_pair(np.concatenate([a, b]), mats,
                  body=np.repeat([0, 1], [len(a), len(b)]).astype(np.int32))[0]
    S.contact(orc.make_params(**kwargs(0.0075)))
    at = np.r_[0:len(a), len(a) + 500000:len(a) + 500000 + len(b)]
    assert np.abs(S.fc).max() > 0
    for f in (f0, f1):
        assert np.array_equal(f[at, :3], S.fc[:, :3])
        assert not f[np.setdiff1d(np.arange(len(f)), at)].any()
