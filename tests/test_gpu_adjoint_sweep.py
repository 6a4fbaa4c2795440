"""The reverse sweep (every color of an iteration in one launch, adjoints in LDS) against one
launch per color: the same gradients, bit for bit.  A fan of triangles with more edge colors
than a sweep holds makes its whole context run per color."""
import numpy as np
import pytest

from gpu_helpers import free_device_memory
from xrtailor_amd import scenes
from xrtailor_amd.solver import ClothSolver, make_params

pytestmark = pytest.mark.gpu


def _fan(n=160):
    a = 2 * np.pi * np.arange(n) / n
    pos = np.concatenate([[[0, 0, 0]], np.stack([np.cos(a), 0 * a, np.sin(a)], 1)])
    i = np.arange(n)
    return pos, np.stack([0 * i, 1 + i, 1 + (i + 1) % n], 1).astype(np.int32)


def _grad(sides, per_color, xp, lra):
    s = ClothSolver(params=xp)
    rng = scenes.Rng(7)
    ids, x0, v0, seeds = [], [], [], []
    for n in sides:
        pos, tris = scenes.grid(n, 1.0)
        i = s.AddCloth(pos, tris, 1e-6, 1e-3)
        s.Pin(i, np.array([0, n - 1], np.int32))
        if lra:
            s.AddLraSlots(i, np.array([0, n - 1], np.int32))
        ids.append(i)
        x0.append((pos + 1e-3 * rng.normal(pos.size).reshape(-1, 3)).astype(np.float32))
        v0.append((0.2 * rng.normal(pos.size)).reshape(-1, 3).astype(np.float32))
        seeds.append(rng.normal(pos.size).reshape(-1, 3).astype(np.float32))
    if per_color:
        s.AddCloth(*_fan(), 1e-6, 1e-3)
    s.Start(3)
    for i, x, v in zip(ids, x0, v0):
        s.SetState(i, x, v)
    got = []
    for seed in (1.0, -2.0):                     # the second pass reuses the buffers
        s.AdjointBegin(2, 1)
        patches, cut = s.sweep_patches()["adjoint"], sum(n * n > 1200 for n in sides)
        assert patches == 0 if per_color else patches >= len(sides) + cut
        for i, g in zip(ids, seeds):
            s.AdjointSeed(i, seed * g, 0.01 * g)
        s.AdjointBackward()
        for i in ids:
            got += [*s.GradCompliance(i), *s.GradState(i)]
    s.close()
    return got


@pytest.mark.parametrize("sides,iters,bending,lra", [((2, 3), 3, 1, False), ((34, 35), 4, 1, True),
                                                     ((70,), 3, 1, False), ((48, 20), 2, 0, False)])
def test_sweep_matches_launch_per_color(sides, iters, bending, lra):
    print(f"case reverse sweep sides={sides} iterations={iters} bending={bending}", flush=True)
    xp = make_params(bend_model=1, solve_bending=bending, ground_height=-0.01, ground_friction=0.3,
                     num_substeps=2, num_iterations=iters)
    a, b = _grad(sides, False, xp, lra), _grad(sides, True, xp, lra)
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
    assert any(np.abs(x).max() > 0 for x in a)


def test_backward_takes_no_memory():
    """What the reverse sweep needs is there when AdjointBegin returns (a second context, so that
    the runtime has taken its own memory for these kernels)."""
    print("case reverse sweep: memory after AdjointBegin", flush=True)
    xp = make_params(bend_model=1, ground_height=-0.01, num_substeps=2, num_iterations=2)
    pos, tris = scenes.grid(400, 1.0)
    taken = []
    for _ in range(2):
        s = ClothSolver(params=xp)
        i = s.AddCloth(pos, tris, 1e-6, 1e-3)
        s.Start(3)
        s.AdjointBegin(1, 1)
        s.AdjointSeed(i, np.ones_like(pos, dtype=np.float32), None)
        before = free_device_memory()
        s.AdjointBackward()
        s.sync()
        taken.append(before - free_device_memory())
        s.close()
    print("  bytes", taken, flush=True)
    assert taken[1] == 0
