"""Box kernels (tensor-product blocks, csrc/box.h) against the oracle and the general kernels.

FP64: RHS and advance within 1e-12 of the oracle (max-normalised per component, the bar of
the general kernels).  FP32-bulk: RHS within 2e-6 of the unfused general kernels on the same
mesh (the bar between the two general forms).  Sizes lie around the 15 x 16 tile: one tile and
less, one row or column more, the smallest block (3 cells), partial last tiles.  Wall-modelled
faces on every axis.  A mesh that is a box but for one node moved by 1e-6 of a cell takes the
general kernels.
"""
import numpy as np
import pytest

import cases
import golden_io
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402

HYB = {"kind": "Hybrid", "central": {"kind": "KEP", "order": 4}}
HYB_KEEP = {"kind": "Hybrid", "central": {"kind": "KEEP", "order": 2},
            "upwind": {"kind": "MUSCLHLLC", "limiter": "minmod"}}
WM = {"kind": "WallModel", "T_wall": 290.0, "n_match": 1}
WM3 = {"kind": "WallModel", "T_wall": None, "n_match": 3}
SLIP, NOSLIP = {"kind": "SlipWall"}, {"kind": "NoSlipWall", "T_wall": 310.0}


def box_spec(n, walls, scheme, sgs, move=0.0):
    """Stretched tensor-product block; walls[d]: None (periodic) or the BC of both faces."""
    axes = []
    for d, (k, le) in enumerate(zip(n, cases.L)):
        s = np.linspace(0.0, 1.0, k + 1)
        axes.append(le * (s if walls[d] is None else s + (0.05 + 0.03 * d) * np.sin(2 * np.pi * s)))
    nodes = np.stack(np.meshgrid(*axes, indexing="ij"))
    if move:
        nodes[0, 1, 1, 1] += move * cases.L[0] / n[0]
    connect, bcs = [], []
    for d, (lo, hi) in enumerate((("imin", "imax"), ("jmin", "jmax"), ("kmin", "kmax"))):
        if walls[d] is None:
            shift = [0.0, 0.0, 0.0]
            shift[d] = -cases.L[d]
            connect.append(["all", lo, "all", hi, shift])
        else:
            bcs += [["all", lo, dict(walls[d])], ["all", hi, dict(walls[d])]]
    spec = {"name": "box", "blocks": ["all"], "ng": 3, "connect": connect, "bcs": bcs, "scheme": scheme,
            "sgs": sgs, "sgs_kwargs": {}, "cfl": 0.5, "constraints": [], "sources": [], "gas": {}}
    return spec, {"nodes_all": nodes}


def state(mesh, s):
    Q = s.init_state(cases.prim_fn)
    return cases.interior_noise(mesh.blocks, [np.asarray(q.cpu()) for q in Q], 3, amp=0.05)


def gradient_launches(s, Q):
    s.profile(("grad",))
    s.rhs(Q)
    torch.cuda.synchronize()
    n = s.profile_read().get("grad", (0.0, 0))[1]
    s.profile(())
    return n


PARAMS = [((3, 3, 3), (None, WM, None), HYB, "vreman"),
          ((4, 15, 16), (None, WM, None), {"kind": "KEP", "order": 2}, "wale"),
          ((5, 16, 17), (WM3, SLIP, NOSLIP), {"kind": "MUSCLHLLC", "limiter": "minmod"}, "smagorinsky"),
          ((7, 14, 33), (NOSLIP, WM3, WM), {"kind": "KEEP", "order": 4}, "none"),
          ((9, 31, 15), (SLIP, None, WM3), HYB_KEEP, "vreman"),
          ((33, 47, 35), (None, WM3, None), {"kind": "KEP", "order": 4}, "wale"),
          ((70, 30, 32), (WM, WM, WM), HYB, "smagorinsky")]


@pytest.mark.parametrize("n,walls,scheme,sgs", PARAMS)
def test_fp64_box_matches_the_oracle(n, walls, scheme, sgs):
    spec, arrays = box_spec(n, walls, scheme, sgs)
    print(f"[box fp64] {n}", flush=True)
    mesh, s = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    Q = state(mesh, s)
    assert gradient_launches(s, Q) == 0          # the box kernels form the gradients themselves
    blk, ng = mesh.blocks[0], 3
    R = s.rhs(Q)[0].cpu().numpy()
    assert golden_io.rel_err(blk.interior(R), blk.interior(ref.rhs(Q)[0])) <= 1e-12
    assert np.all(R[:, :ng] == 0.0) and np.all(R[:, :, :, -ng:] == 0.0)
    dt = float(s.max_dt(Q))
    A, B = s.advance(Q, dt)[0].cpu().numpy(), ref.advance(Q, dt)[0]
    assert golden_io.rel_err(A, B) <= 1e-12
    for ci in (1, 2, n[0]):                      # every chunk length gives the same cells
        s.set_tiling(ci, 1)
        assert torch.equal(s.rhs(Q)[0], torch.as_tensor(R, device="cuda"))


@pytest.mark.parametrize("n,walls,scheme,sgs", PARAMS)
def test_fp32_box_matches_the_general_kernels(n, walls, scheme, sgs):
    spec, arrays = box_spec(n, walls, scheme, sgs)
    print(f"[box fp32] {n}", flush=True)
    mesh, s = cases.build(wmx, spec, arrays, solver_kwargs={"precision": "fp32", "gauge": (1e5, 290.0)})
    Q = state(mesh, s)
    blk = mesh.blocks[0]
    R = blk.interior(s.rhs(Q)[0])
    q1 = s.advance(Q, 1e-6)[0]
    s.set_fused_gradients(False)
    G = blk.interior(s.rhs(Q)[0])
    assert golden_io.rel_err(R.cpu().numpy(), G.cpu().numpy()) <= 2e-6
    assert golden_io.rel_err(q1.cpu().numpy(), s.advance(Q, 1e-6)[0].cpu().numpy()) <= 2e-8


def test_a_mesh_that_is_nearly_a_box_takes_the_general_kernels():
    spec, arrays = box_spec((8, 16, 17), (None, WM, None), HYB, "vreman", move=1e-6)
    mesh, s = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    Q = state(mesh, s)
    blk = mesh.blocks[0]
    R = s.rhs(Q)[0].cpu().numpy()
    assert golden_io.rel_err(blk.interior(R), blk.interior(ref.rhs(Q)[0])) <= 1e-12


@pytest.mark.parametrize("n", [(3, 3, 3), (8, 16, 8), (11, 31, 13)])
def test_box_cfl_step_is_the_oracles(n):
    """The filtered CFL minimum of a box block (less than, exactly and several workgroups of
    1024 cells): fields with one fastest cell at either end, equal cells, and states whose
    minimum is no number, zero or negative."""
    spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman")
    mesh, s = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    blk = mesh.blocks[0]
    noise = state(mesh, s)[0]
    prim = np.array([1.2, 0.0, 0.0, 0.0, 1e5])
    flat = np.asarray(s.init_state(lambda xc: prim[:, None, None, None] + 0.0 * xc[:1])[0].cpu())
    tests = {"noise": noise, "equal cells": flat}
    for name, at, v, val in (("first", 0, 4, 2e6), ("last", -1, 4, 2e6), ("nan", -1, 2, np.nan), ("inf", 0, 4, np.inf),
                             ("negative density", 0, 0, -1.0), ("negative pressure", -1, 4, -1.0),
                             ("huge", 0, 1, 1e200), ("zero density", -1, 0, 0.0)):
        q = noise.copy()
        blk.interior(q)[(v,) + (at,) * 3] = val
        tests[name] = q
    for name, q in tests.items():
        with np.errstate(all="ignore"):
            want = float(np.asarray(ref.max_dt([q])))
        got = float(s.max_dt([q]))
        assert got == want or (np.isnan(got) and np.isnan(want)) or abs(got - want) <= 1e-13 * abs(want), (name, got, want)
