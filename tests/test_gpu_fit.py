"""The trainer's fold of the per-wave losses and gradients over batches whose
wave count is no multiple of its 256-wave trips or its 16-term steps: the
first step's loss, at a learning rate of zero, against the numpy restatement
of the network over the same drawn samples."""
import sys

import numpy as np
import pytest

import oracle as orc
from pdhelpers import deformed_pair
from test_gpu_learned import blocks, mix64, mlp

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")


@pytest.mark.parametrize("batch", [128, 640, 8192, 8320, 16512])
def test_loss_of_every_wave(batch):
    print("case fit batch", batch, flush=True)
    sys.stdout.flush()
    sys_, ctx = deformed_pair(amp=0.05, s_fixed=0.01)
    kw = dict(dt=1e-4, precond=1, rtol=1e-8)
    sys_.assemble(orc.make_params(**kw))
    ctx.assemble(pds.make_params(**kw))
    tr = pds.Trainer(1000, seed=3)
    count = tr.add(ctx, seed=11, stride=1)
    smp = tr.samples(0, count)
    loss = tr.fit(1, batch=batch, lr=0.0, seed=21)[0]
    net = tr.params()
    with np.errstate(over="ignore"):
        draw = mix64(np.uint64(21) ^ mix64(np.arange(batch, dtype=np.uint64))) % np.uint64(count)
    d = smp[:, 16:22].astype(np.float64)
    diag = d[:, [0, 1, 2, 1, 3, 4, 2, 4, 5]]
    M = blocks(net, mlp(net, smp[:, :16]), diag).reshape(-1, 3, 3)
    r = (M @ smp[:, 22:25, None].astype(np.float64))[:, :, 0] - smp[:, 25:28]
    want = (r ** 2).sum(1)[draw.astype(np.int64)].mean()
    print(dict(batch=batch, samples=count, loss=float(loss), restated=float(want)), flush=True)
    # BF16 activations: 2^-8 relative each, averaged over the batch; a lost
    # wave changes the sum by 1 / waves >= 2e-3
    assert abs(loss - want) <= 1e-3 * want
    assert np.array_equal(net[:5760], pds.Trainer(1, seed=3).params()[:5760])
    tr.close()
    ctx.close()
