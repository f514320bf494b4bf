"""The queue compaction at the edges of its rule: up to 1024 blocks of 256 slots the scatter sums the
blocks before it itself, 256 totals a read; more blocks are scanned by a launch of their own. Queue
lengths, items and the sample cursor equal the oracle's, bit for bit."""
import numpy as np
import pytest

from raccoongpurender_amd import render_scenes as R
from tests import wf_helpers as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 255 * 256 + 1, 256 * 256 + 1, 260 * 256 - 3, 1024 * 256 - 255, 1024 * 256,
                               1024 * 256 + 1])
def test_queues_equal_the_oracles(ctx, n):
    print(f"case queues of {n} slots", flush=True)
    sd = R.material_test_scene(24, 16, volume=True)
    g, o = W.gpu_lane(ctx, sd, n), W.oracle_lane(sd, n)
    for step in range(3):
        g.step()
        o.step()
        cg, pg = g.queue_counts()
        co, po = o.queue_counts()
        assert np.array_equal(cg, co) and pg == po, (step, cg, co)
        ig, io = g.state()["items"], o.state()["items"]
        for k in range(7):
            assert np.array_equal(ig[k, :cg[k]], io[k, :co[k]]), (step, k)
    g.close()
