"""Waves per work item in a batch that fills the GPU (more than 8192 work
items): small frames by the batch's rule, frames
that ask for a count by theirs, every instance bit for bit as alone (MI355X
only)."""
import numpy as np
import pytest

import test_gpu_batch as tb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [0, 2, 8])
def test_batch_waves(fd, wl, monkeypatch, waves):
    monkeypatch.setattr(tb, "MIX", [(640, 512, 4, (0.2, 0.1, 6.0), 0), (512, 512, 8, (1.0, -1.0, 5.0), 0),
                                    (96, 96, 32, (0.5, -0.3, 5.0), 8), (64, 65, 33, (0.0, 0.0, 6.0), 0)])
    print(f"[batch waves] {waves}", flush=True)
    scene, ctx, items, keep = tb._setup(fd, wl)
    alone = [tb._alone(fd, wl, scene, it) for it in items]
    items[2]["waves"] = waves
    stream = fd.Stream()
    b = fd.Batch(ctx, items)
    b.launch(stream.handle)
    stream.sync()
    for k, it in enumerate(items):
        (sh, mk), _ = alone[k]
        assert np.array_equal(it["shadow"].download(np.float32).view(np.uint32), np.asarray(sh).ravel().view(np.uint32)), k
        assert np.array_equal(it["masks"].download(np.uint32).ravel(), np.asarray(mk).ravel().view(np.uint32)), k
    b.close()
    stream.close()
    ctx.close()
