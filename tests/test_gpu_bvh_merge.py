"""The chunked bottom-up merge of the LBVH boxes at the edges of its chunks of 1024 leaves:
boxes, then pairs and segment hits (which read the traversal records the merge writes)
against the FP32-strict oracle, bit for bit, after a build, a refit and an update."""
import numpy as np
import pytest

from oracle import oracle as orc
from xrtailor_amd import scenes
from xrtailor_amd.bvh import BVH, Traverse

pytestmark = pytest.mark.gpu


def _same_boxes(g, o):
    hg, ho = g.host(), o.host()
    np.testing.assert_array_equal(hg["nodes"], ho["nodes"])
    np.testing.assert_array_equal(hg["aabbs"], ho["aabbs"])


@pytest.mark.parametrize("nf", [1, 2, 3, 1023, 1024, 1025, 1026, 2047, 2048, 2049, 5000, 20001])
def test_merge_at_chunk_edges(nf):
    print(f"case chunked merge, {nf} faces", flush=True)
    rng = scenes.Rng(nf)
    n = 102
    pos, tris = scenes.grid(n, 1.0)
    pos = (pos + 2e-3 * rng.normal(pos.size).reshape(-1, 3)).astype(np.float32)
    pos[:, 1] += 0.05 * np.sin(25.0 * pos[:, 0])
    order = np.argsort(rng.uniform(len(tris)))     # faces from all over the sheet
    tris = np.ascontiguousarray(tris[order[:nf]])
    g, o = BVH(), orc.Bvh()
    for t in (g, o):
        t.Build(pos[::-1].copy(), tris)             # an earlier tree of the same handle
        t.Build(pos, tris)
    _same_boxes(g, o)
    x1 = (pos + 3e-3 * rng.normal(pos.size).reshape(-1, 3)).astype(np.float32)
    n1 = orc.vertex_normals(pos, scenes.grid(n, 1.0)[1])
    for t in (g, o):
        t.RefitMidstep(x1, n1, 0.002)
    _same_boxes(g, o)
    for t in (g, o):
        t.Update(pos, x1, ccd=True)
    _same_boxes(g, o)
    np.testing.assert_array_equal(Traverse(g, g, 1e-4), orc.traverse(o, o, 1e-4))
    p0 = (rng.uniform(3 * 300).reshape(-1, 3) - 0.5).astype(np.float32) * np.array([1, 0.2, 1], np.float32)
    p1 = (p0 + 0.03 * rng.normal(3 * 300).reshape(-1, 3)).astype(np.float32)
    for a, b in zip(g.Query(p0, p1), o.Query(p0, p1)):
        np.testing.assert_array_equal(a, b)
