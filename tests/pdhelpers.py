"""Small input builders shared by the tests (no reference code involved)."""
import numpy as np

import oracle as orc


def lattice(nx, ny, nz, h, jitter, seed, origin=(0.0, 0.0, 0.0)):
    """x-fastest simple-cubic lattice with uniform jitter in +-jitter*h."""
    rng = np.random.default_rng(seed)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    g = np.stack([i, j, k], -1).reshape(-1, 3).astype(np.float64) * h
    g += rng.uniform(-1, 1, g.shape) * jitter * h
    g += np.asarray(origin)
    x4 = np.zeros((g.shape[0], 4))
    x4[:, :3] = g
    return x4


def material(h, horizon_factor=3.0, stiffness=1e4, mass=1e-3):
    """(horizon, radius, c_bond, mass) for spacing h: r = h/2, c = k h."""
    return (horizon_factor * h, 0.5 * h, stiffness * h, mass)


def make_system(x4, materials, body=None, s0=0.02, seed=1973, v4=None, lists=None, **kw):
    n = x4.shape[0]
    hs = [m[0] for m in materials]
    if lists is None:
        counts, lists, total = orc.bonds_brute(x4, hs, body=body)
        assert total >= 0
    else:  # (counts, padded rows)
        counts, lists = lists
    rs, col = orc.lists_to_csr(counts, lists)
    s00 = orc.stretch_init(n, s0, seed)
    v4 = np.zeros((n, 4)) if v4 is None else v4
    return orc.OracleSystem(x4, v4, s00, rs, col, materials, body=body, **kw)


def make_pair(x4, materials, body=None, s0=0.02, seed=1973, v4=None, bc=None, vbc=None,
              act=None):
    """The same initial state in the oracle and in a GPU context (bonds built
    on the GPU); returns (oracle_system, gpu_context)."""
    import pdsolver as pds
    n = x4.shape[0]
    sys_ = make_system(x4, materials, body=body, s0=s0, seed=seed, v4=v4, bc=bc, vbc=vbc,
                       act=act)
    ctx = pds.Context(n, materials)
    pds.load_state(ctx, x4, sys_.v, sys_.s00, body=body, act=act, bc=bc, vbc=vbc)
    ctx.build_bonds()
    return sys_, ctx


def config0_state(nx=20, ny=20, nz=20, h=0.01, jitter=0.05, seed=1973, top_speed=1.0):
    """Tension specimen: x-fastest jittered lattice, bottom z-layer fixed,
    top z-layer moved at +top_speed along z."""
    x4 = lattice(nx, ny, nz, h, jitter, seed)
    n = x4.shape[0]
    k = np.arange(n) // (nx * ny)
    bc = ((k == 0) | (k == nz - 1)).astype(np.int32)
    vbc = np.zeros((n, 4))
    vbc[k == nz - 1, 2] = top_speed
    v4 = vbc.copy()
    return x4, bc, vbc, v4


def deformed_pair(nx=10, ny=9, nz=8, amp=0.03, seed=0, s_fixed=0.02):
    """Oracle / GPU pair on a jittered lattice with random velocities and a
    random displacement of amp * spacing; stretch limits set to s_fixed."""
    h = 0.01
    x4 = lattice(nx, ny, nz, h, 0.05, seed)
    rng = np.random.default_rng(seed + 1)
    v4 = np.zeros_like(x4)
    v4[:, :3] = rng.uniform(-1, 1, (x4.shape[0], 3))
    sys_, ctx = make_pair(x4, [material(h)], v4=v4)
    disp = rng.uniform(-1, 1, (x4.shape[0], 3)) * amp * h
    sys_.x[:, :3] += disp
    ctx.upload("position", sys_.x)
    if s_fixed is not None:
        sys_.s[:] = s_fixed
        ctx.upload("stretch", sys_.s)
    return sys_, ctx


def specimen_pair(sizes, lead=0, pull=6.0, factor=3.0, s0=0.02):
    """Independent tension specimens in one GPU context, `lead` rows of
    INVISIBLE padding before the first, and each of them alone in the oracle;
    returns (first rows, oracle systems, gpu context)."""
    import pdsolver as pds
    mats = [material(0.01, factor)]
    far = np.array([[-1.0, -1.0, -1.0, 0.0]])
    parts, first, alone = [], [], []

    def padding(m):
        return (np.tile(far, (m, 1)), np.zeros((m, 4)), np.zeros(m, np.int32), np.full(m, s0),
                np.full(m, 3, np.int32))

    if lead:
        parts.append(padding(lead))
    row = lead
    for i, n in enumerate(sizes):
        w = 4 if n < 2000 else 12
        x4 = lattice(w, w, -(-n // (w * w)), 0.01, 0.05, 7 * n + i, origin=(0.5 * i, 0.0, 0.0))[:n]
        k = np.arange(n) // (w * w)
        bc = ((k == 0) | (k == k[-1])).astype(np.int32)
        vbc = np.zeros((n, 4))
        vbc[k == k[-1], 2] = pull * (1.0 + 0.3 * i)
        sys_ = make_system(x4, mats, s0=s0, seed=11 + i, v4=vbc.copy(), bc=bc, vbc=vbc)
        parts.append((x4, vbc, bc, sys_.s00.copy(), np.zeros(n, np.int32)))
        alone.append(sys_)
        first.append(row)
        pad = -n % 256
        if pad:
            parts.append(padding(pad))
        row += n + pad
    x4, vbc, bc, s00, act = (np.concatenate(c) for c in zip(*parts))
    ctx = pds.Context(row, mats)
    pds.load_state(ctx, x4, vbc.copy(), s00, act=act, bc=bc, vbc=vbc)
    ctx.build_bonds()
    ctx.set_specimens(np.array(first, np.int32), np.array(sizes, np.int32))
    return first, alone, ctx


def compare_specimens(first, alone, ctx, step, kw, steps):
    """Steps the context by step(kw) and every specimen alone in the oracle:
    the same bits, counts and residuals; returns the broken bonds."""
    broken = 0
    for k in range(1, steps + 1):
        q = dict(dict(dt=1e-4, clock_scale=min(k, 10) / 10.0, precond=1, rtol=1e-8), **kw)
        o = {a: b for a, b in q.items() if a not in ("matrix_free", "graph", "timing")}
        sg = step(q)
        per = ctx.specimen_stats(len(alone))
        xg, vg = ctx.download("position"), ctx.download("velocity")
        tops = ctx.download("bond_top")
        br = 0
        for i, (f, S) in enumerate(zip(first, alone)):
            so = S.step(orc.make_params(**o))
            br += so.broken_bonds
            assert per[i]["cg_iterations"] == so.cg_iterations, (k, i)
            assert per[i]["residual_norm"] == so.residual_norm, (k, i)
            assert np.array_equal(xg[f:f + S.n, :3], S.x[:, :3]), (k, i)
            assert np.array_equal(vg[f:f + S.n, :3], S.v[:, :3]), (k, i)
            assert np.array_equal(tops[f:f + S.n], S.top), (k, i)
        assert sg.broken_bonds == br, k
        broken += br
    return broken
