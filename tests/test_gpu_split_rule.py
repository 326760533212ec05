"""The automatic list split on both sides of its lines (triangles per bin 16
and 512, work items 256): the same bits as whole lists (MI355X only)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w", [40, 112])   # 8 x 8 bins: 90 and 261 work items at most
@pytest.mark.parametrize("ntris", [1023, 1024, 32767, 32768])
def test_split_rule(fd, wl, w, ntris):
    print(f"[split rule] {w} {ntris}", flush=True)
    frame = wl.Frame("split", wl.tris_uniform(ntris, 5), wl.receivers_plane(w, w, 4.0),
                     wl.LightDesc(0.5, 0.5, (0.1, -0.2, 4.0), res_w=12, res_h=12), backface_cull=0, grid_log2=3)
    out = []
    for split in (0, 1):
        frame.list_split = split
        fr = fd.FrameRunner(frame)
        rc, st = fr.run()
        assert rc == 0 and st.exit_code == 0
        out.append(fr.outputs())
        fr.close()
    assert np.array_equal(np.asarray(out[0][0]).view(np.uint32), np.asarray(out[1][0]).view(np.uint32))
    assert np.array_equal(out[0][1], out[1][1])
    assert 0.0 < np.asarray(out[0][0]).mean()
