"""The bounce's stage queues in one launch: odd lane sizes, and grids of fewer workgroups than the
queues fill (the launch strides over the rest). Bit for bit against the oracle, as the other
wavefront tests."""
import numpy as np
import pytest

from raccoongpurender_amd import render_scenes as R
from tests import wf_helpers as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paths,queue_blocks", [(1, 0), (255, 0), (257, 1), (1283, 1), (4099, 3)])
def test_odd_lanes_and_small_grids(ctx, paths, queue_blocks):
    sd = R.material_test_scene(24, 20)
    g = W.gpu_lane(ctx, sd, paths, queue_blocks=queue_blocks)
    o = W.oracle_lane(sd, paths)
    for s in range(8):
        g.step()
        o.step()
        cg, pg = g.queue_counts()
        co, po = o.queue_counts()
        assert np.array_equal(cg, co) and pg == po, s
        sg, so = g.state(), o.state()
        mm = W.state_mismatches(sg, so)
        assert all(v == 0 for v in mm.values()), (s, mm)
        for k in range(7):
            assert np.array_equal(sg["items"][k, :cg[k]], so["items"][k, :co[k]]), (s, k)
