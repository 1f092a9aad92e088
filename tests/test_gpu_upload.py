"""Vector fields are stored with a zero fourth component, whatever the caller's
array holds there, and the caller's array is left alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
pds = pytest.importorskip("pdsolver")

from pdhelpers import material  # noqa: E402


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_upload_clears_the_fourth_component(n):
    print("case upload", n, flush=True)
    ctx = pds.Context(n, [material(0.01)])
    a = np.random.default_rng(n).normal(size=(n, 4))
    a[0, 3] = np.nan
    for f in ("position", "velocity", "bc_velocity", "solution"):
        sent = a.copy()
        ctx.upload(f, sent)
        got = ctx.download(f)
        assert np.array_equal(got[:, :3], a[:, :3]) and np.all(got[:, 3] == 0.0), f
        assert np.array_equal(sent, a, equal_nan=True), f
    ctx.close()
