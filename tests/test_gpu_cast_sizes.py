"""The persistent cast's waves by batch size (64 rays a wave, 4 to 7 waves per SIMD): at the edges of
the rule every ray's hit is the one-thread-per-ray kernel's, bit for bit."""
import numpy as np
import pytest

from raccoongpurender_amd import _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", ["stackless", "threaded", "threaded_single"])
def test_hits_at_the_edges(ctx, variant):
    v, f = scenes.displaced_icosphere(level=4)
    scene = _lib.Scene(ctx, _lib.BVH(v, f))
    rng = np.random.default_rng(12)
    n = 425985
    rays = np.zeros(n, _lib.RAY_DTYPE)
    o = rng.normal(size=(n, 3))
    rays["ro"] = 2.0 * o / np.linalg.norm(o, axis=1, keepdims=True)
    d = rng.normal(size=(n, 3)) * 0.5 - rays["ro"]
    rays["rd"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmax"] = np.float32(3.4e38)
    one = _lib.trace(ctx, scene, rays, variant=variant, block=64)
    assert (one["prim"] >= 0).mean() > 0.2
    # (65,536 rays are one wave per SIMD's worth; the counts of waves change at k + 1/2 of them)
    for k in (1, 7169, 294911, 294912, 360447, 360448, 425983, 425984, n):
        print(f"case {variant} {k} rays", flush=True)
        hits = _lib.trace(ctx, scene, rays[:k], variant=variant, block=0)
        assert np.array_equal(hits.view(np.uint32), one[:k].view(np.uint32))
