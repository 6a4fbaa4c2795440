"""Self-contact pairs visited once per couple of faces (batched) against the directed pairs of
the plain path: the same states, records and pair counts, bit for bit, with the stage and the
lists within their sizes and beyond them."""
import numpy as np
import pytest

from gpu_helpers import free_device_memory
from xrtailor_amd import scenes
from xrtailor_amd._ffi import XrtError
from xrtailor_amd.solver import build_solver, make_params

pytestmark = pytest.mark.gpu


def _crumpled(n, seed, noise):
    """a sheet of n x n vertices of 1 m, every vertex moved by `noise` faces of random offset"""
    rng = scenes.Rng(seed)
    pos, tris = scenes.grid(n, 1.0)
    x0 = (pos + noise / n * rng.normal(pos.size).reshape(-1, 3)).astype(np.float32)
    return scenes.ClothSpec(pos, tris, np.zeros(0, np.int32), 1e-8, 1e-4, x0)


# noise 3: some hundred pairs a face, more than the 64 couples of a leaf's stage (found again);
# the capacities: ample, lists too short (pairs stored), pairs lost.  listed: all instances on
# the item path
@pytest.mark.parametrize("noise,cap,items,lost,listed",
                         [(0.2, 128, 128, False, True), (3.0, 2048, 4096, False, True),
                          (3.0, 2048, 60, False, False), (0.2, 9, 128, True, False),
                          (3.0, 100, 64, True, False)])
def test_couples_match_plain(noise, cap, items, lost, listed):
    print(f"case couples noise={noise} cap={cap} items={items}", flush=True)
    specs = [_crumpled(n, 5 + n, noise) for n in (3, 17, 24)]
    xp = make_params(bend_model=1, enable_self_contact=1, ground_height=-1.0, num_substeps=2,
                     num_iterations=3, num_collision_passes=3, pair_update_interval=2,
                     pair_capacity_per_face=cap,
                     repulsion_vf_items_per_face=items, repulsion_ee_items_per_face=items)
    a, ia = build_solver(specs, xp, seed=3)
    b, ib = build_solver(specs, xp, seed=3)
    on_items = []
    for _ in range(2):
        n = a.time_repulsion(1)[1]                  # a batched substep, and what its lists hold
        print("  ", n, flush=True)
        on_items.append(n["item_path_instances"])
        for j in ib:
            b.SubstepPlain(j)
    assert all(n == len(specs) for n in on_items) if listed else all(n < len(specs) for n in on_items)
    for s in (a, b):
        if lost:                                    # the first pairs were kept
            with pytest.raises(XrtError, match="overflow"):
                s.sync()
        else:
            s.sync()
    per_face = []
    for i, j, sp in zip(ia, ib, specs):
        for u, v in zip(a.GetState(i), b.GetState(j)):
            np.testing.assert_array_equal(u, v)
        ca, cb = a.Contacts(i), b.Contacts(j)
        assert ca["pairs"] == cb["pairs"]
        per_face.append(ca["pairs"] / len(sp.tris))
    print("  pairs per face", per_face, flush=True)
    if noise > 1:  # a face's pair with itself and two for each couple: some leaf has over 64
        assert max(per_face) > 1 + 2 * 64
    assert lost == (max(per_face) > cap)


# an obstacle of 2^16 vertices (items listed by 16-bit vertex ids) and one of more (by edges)
@pytest.mark.parametrize("side", [256, 257])
def test_large_obstacle_matches_plain(side):
    print(f"case obstacle of {side} x {side} vertices", flush=True)
    pos, tris = scenes.grid(side, 1.5)
    pos = pos.astype(np.float32)
    pos[:, 1] = -0.001 + 0.0005 * np.sin(40.0 * pos[:, 0])
    sp = _crumpled(17, 4, 0.05)
    sp = scenes.ClothSpec(sp.pos, sp.tris, sp.pinned, 1e-8, 1e-4, sp.x0, (pos, tris))
    xp = make_params(bend_model=1, enable_self_contact=1, enable_obstacle_contact=1,
                     ground_height=-1.0, num_substeps=2, num_iterations=3, num_collision_passes=3,
                     pair_update_interval=2, pair_capacity_per_face=4096,
                     repulsion_vf_items_per_face=4096, repulsion_ee_items_per_face=8192)
    a, ia = build_solver([sp], xp, seed=3)
    b, ib = build_solver([sp], xp, seed=3)
    for _ in range(2):
        a.SubstepBatched()
        b.SubstepPlain(ib[0])
    a.sync()
    for u, v in zip(a.GetState(ia[0]), b.GetState(ib[0])):
        np.testing.assert_array_equal(u, v)
    c = a.Contacts(ia[0])
    assert c["pairs"] == b.Contacts(ib[0])["pairs"] and c["obs_pairs"] > 1000


def test_lists_without_room_for_vertex_ids_match_small_ones():
    """Item lists of 0.7 of the free memory: their 16-bit vertex ids do not fit beside all of them."""
    n = 17
    faces = 2 * (n - 1) ** 2
    cap = (2 ** 31 - 1) // (9 * faces)              # pairs a face: the largest with lists on
    free = free_device_memory()
    k = int(0.7 * free / (8 * 13 * cap * faces))    # pairs, 3 VF and 9 EE items each
    print(f"case lists of {k} x {8e-9 * 13 * cap * faces:.1f} GB of {1e-9 * free:.0f} GB",
          flush=True)
    assert k >= 1
    specs = [_crumpled(n, 40 + j, 0.2) for j in range(k)]
    runs = []
    for kw in (dict(pair_capacity_per_face=cap, repulsion_vf_items_per_face=3 * cap,
                    repulsion_ee_items_per_face=9 * cap), dict(pair_capacity_per_face=128)):
        s, ids = build_solver(specs, make_params(bend_model=1, enable_self_contact=1,
                                                 ground_height=-1.0, num_substeps=2,
                                                 num_iterations=3, **kw), seed=3)
        s.FramesBatched(2)
        s.sync()
        runs.append([a for i in ids for a in s.GetState(i)])
        s.close()
        print("  ran", flush=True)
    for a, b in zip(*runs):
        np.testing.assert_array_equal(a, b)


def test_lists_that_cannot_be_resized_are_empty():
    """Capacities beyond the device's memory are refused.  The instance that met the limit then runs
    without lists (without a pair list its pairs are reported as lost) until others are set."""
    n = 17
    faces = 2 * (n - 1) ** 2
    cap = (2 ** 31 - 1) // (9 * faces)
    k = int(1.3 * free_device_memory() / (8 * 13 * cap * faces)) + 1
    print(f"case resize of {k} x {8e-9 * 13 * cap * faces:.1f} GB", flush=True)
    specs = [_crumpled(n, 60 + j, 0.2) for j in range(k)]
    small = dict(bend_model=1, enable_self_contact=1, ground_height=-1.0, num_substeps=2,
                 num_iterations=3, pair_capacity_per_face=128)
    large = dict(small, pair_capacity_per_face=cap, repulsion_vf_items_per_face=3 * cap,
                 repulsion_ee_items_per_face=9 * cap)
    s, ids = build_solver(specs, make_params(**small), seed=3)
    with pytest.raises(XrtError, match="memory"):
        s.set_params(make_params(**large))
    print("  refused", flush=True)
    s.FramesBatched(1)
    try:
        s.sync()
    except XrtError as e:                           # not even its pairs fit
        assert "overflow" in str(e)
    s.set_params(make_params(**small))
    for i, sp in zip(ids, specs):
        s.SetState(i, sp.x0, np.zeros_like(sp.x0))
    r, jds = build_solver(specs, make_params(**small), seed=3)
    for c, cids in ((s, ids), (r, jds)):
        c.FramesBatched(1)
        c.sync()
    for i, j in zip(ids, jds):
        for u, v in zip(s.GetState(i), r.GetState(j)):
            np.testing.assert_array_equal(u, v)
