"""Shared helpers of the GPU parity tests: build a solver and the oracle cloth that
mirrors an instance (same topology, colors, LRA CSR and FP32-rounded state)."""
from __future__ import annotations

import ctypes as C

import numpy as np

from oracle import oracle as orc
from xrtailor_amd import _ffi
from xrtailor_amd.solver import ClothSolver, build_solver, make_params  # noqa: F401


def rel_err(x, ref) -> float:
    """||x - ref||_inf / max(||ref||_inf, 1 m)"""
    x = np.asarray(x, np.float64)
    ref = np.asarray(ref, np.float64)
    return float(np.abs(x - ref).max() / max(np.abs(ref).max(), 1.0))


def free_device_memory() -> int:
    """Free bytes of the device, from the HIP runtime that the library is linked with."""
    free, total = C.c_size_t(), C.c_size_t()
    assert _ffi.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def build(specs, params, seed=0):
    return build_solver(specs, params, seed=seed)


def oracle_of(solver: ClothSolver, inst: int, stretch_compliance, bend_compliance,
              x0=None, v=None) -> orc.Cloth:
    """Oracle cloth with the instance's constraints and colors, and its current device state
    (or the given x0 / v).  stretch_compliance: scalar or per-edge array (edge order of
    solver.edges)."""
    n = solver.counts(inst)
    edges, rest, scol = solver.edges(inst)
    bends, theta, bcol = solver.bends(inst)
    if x0 is None or v is None:
        gx0, gv = solver.GetState(inst)
        x0 = gx0 if x0 is None else x0
        v = gv if v is None else v
    w = solver.inv_mass(inst)
    s_comp = np.broadcast_to(np.asarray(stretch_compliance, np.float64), (n.n_edges,)).copy()
    b_comp = np.full(n.n_bends, float(bend_compliance))
    kw = {}
    if n.lra_slots:
        sv, ptr, sl, rs = solver.lra(inst)
        kw = dict(slot_vert=sv, lra_ptr=ptr, lra_slot=sl, lra_rest=rs.astype(np.float64))
    return orc.Cloth(np.asarray(x0, np.float64), np.asarray(v, np.float64), w.astype(np.float64),
                     edges, rest.astype(np.float64), s_comp, scol, n.stretch_colors,
                     bends, theta.astype(np.float64), b_comp, bcol, n.bend_colors, **kw)
