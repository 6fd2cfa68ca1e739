"""How the library takes a program's steps (mw_pass_plan; needs no GPU), and what the
benchmark calls the launches it times."""

import ctypes

import pytest

from witwin_maxwell_amd import build as mwbuild
from witwin_maxwell_amd.fdtd import native


@pytest.fixture(scope="module")
def lib():
    import os
    if not os.path.exists(mwbuild.library_path()):
        mwbuild.build()
    return native.load_library()


def _program(nodes, pml, z_planes=0, lossy=False, dft=0, plane_wave=False):
    """A single-pass program of that grid with `z_planes` flux planes (six observed
    (component, column) planes each), and a workspace; buffers are never read."""
    fake = ctypes.c_void_p(4096)
    p, w = native.MwProgram(), native.MwWorkspace()
    p.grid.nx, p.grid.ny, p.grid.nz = nodes
    p.fused, p.total_steps, p.dt = 1, 1000, 1.0
    for q in range(6):
        p.coeffs.decay_value[q] = p.coeffs.curl_value[q] = 1.0
    for q in range(3):
        p.coeffs.curl[q] = fake
        p.coeffs.decay[q] = fake if lossy else None
    for a in range(3):
        p.grid.inv_e[a] = p.grid.inv_h[a] = fake
        p.grid.bc_lo[a] = p.grid.bc_hi[a] = 1 if pml else 4
    if pml:
        p.cpml.enabled = 1
        axes = (1, 2, 0, 2, 0, 1)  # the derivative axis of each psi array, E then H
        for q in range(12):
            n = nodes[axes[q % 6]] - (q >= 6)
            p.cpml.psi_low[q], p.cpml.psi_high_start[q], p.cpml.psi_high_len[q] = pml, n - pml, pml
    planes = []
    for i in range(z_planes):
        k = int(nodes[2] * (0.35 + 0.33 * i))
        planes += [native.MwPlaneObs(c, 2, k - d, 0, fake, fake) for c, d in ((0, 0), (1, 0), (3, 0), (3, 1), (4, 0), (4, 1))]
    keep = (native.MwPlaneObs * max(1, len(planes)))(*planes)
    p.planes = ctypes.cast(keep, ctypes.POINTER(native.MwPlaneObs))
    p.n_planes, p.nf_obs, p.nf_dft = len(planes), 8, dft
    terms = []
    if plane_wave:  # the two sheets of a soft +z plane wave
        for c in (0, 4):
            t = native.MwTerm()
            t.component, t.kind, t.patch, t.delay, t.values = c, 1, fake, fake, fake
            for a in range(3):
                t.offset[a] = pml + 3
                t.shape[a] = 1 if a == 2 else nodes[a] - 2 * (pml + 3)
            terms.append(t)
        held = [(native.MwTerm * 1)(t) for t in terms]
        p.n_e_terms = p.n_h_terms = 1
        p.e_terms, p.h_terms = (ctypes.cast(h, ctypes.POINTER(native.MwTerm)) for h in held)
        keep = (keep, held)
    for q in range(6):
        w.psi_e_alt[q] = fake
    w.line_history, w.term_steps = fake, 2
    w.stage, w.stage_depth, w.stage_floats = fake, 32, 32 * 6 * 2 * nodes[0] * nodes[1]
    return p, w, keep


def _pass_plan(lib, *args, workspace=True, **kw):
    p, w, _keep = _program(*args, **kw)
    out = (ctypes.c_int32 * 3)()
    native.check(lib.mw_pass_plan(ctypes.byref(p), ctypes.byref(w) if workspace else None, out), lib)
    return tuple(out)


def test_pass_plan_reports_the_route(lib):
    steps, blocks, chunk = _pass_plan(lib, (257, 257, 257), 0)
    assert steps == 2 and blocks > 0 and chunk > 0
    steps, blocks, chunk = _pass_plan(lib, (121, 121, 121), 12)  # costlier tiles get shorter chunks
    assert steps == 2 and 0 < blocks <= 256 and chunk == 0
    steps, blocks, chunk = _pass_plan(lib, (281, 281, 281), 12)
    assert steps == 2 and chunk == 16
    assert _pass_plan(lib, (121, 121, 121), 12, workspace=False) == (0, 0, 0)
    p, w, _keep = _program((121, 121, 121), 12)
    out = (ctypes.c_int32 * 3)()
    for field, value in (("z_tiling", 3), ("fused", 0), ("n_points", 65)):
        old = getattr(p, field)
        setattr(p, field, value)
        native.check(lib.mw_pass_plan(ctypes.byref(p), ctypes.byref(w), out), lib)
        assert out[0] == 0, field
        setattr(p, field, old)
    assert lib.mw_pass_plan(None, None, out) == -1
    p.n_planes = 17
    assert lib.mw_pass_plan(ctypes.byref(p), ctypes.byref(w), out) == -1


@pytest.mark.parametrize("plan,kernel,steps", [((2, 256, 0), "MARCH_KERNEL", 2), ((0, 0, 0), "STEP_KERNEL", 1)])
def test_benchmark_names_the_launches_a_run_takes(plan, kernel, steps):
    """Also where the tiling is the library's own and the march refuses the scene."""
    import bench

    class Run:
        def pass_plan(self):
            return plan
    assert bench.step_launches(Run()) == (getattr(bench, kernel), steps)


@pytest.mark.parametrize("nodes,pml,z_planes,lossy,dft,steps,chunk", [
    # measured on both sides (us a step, two-step passes / separate launches), a tenth
    # or more apart
    ((401, 65, 125), 8, 2, False, 0, 0, 0),     # 118 / 95
    ((161, 161, 161), 12, 2, False, 0, 2, 0),   # 108 / 148
    ((281, 105, 105), 12, 2, False, 0, 2, 0),   # 93 / 116
    ((185, 185, 185), 12, 0, False, 0, 2, 0),   # 172 / 195
    ((185, 185, 185), 12, 0, True, 0, 0, 0),    # 244 / 209
    ((201, 101, 67), 12, 0, True, 0, 0, 0),     # 86 / 64
    ((121, 121, 121), 12, 0, True, 0, 2, 0),    # 64 / 73
    ((225, 225, 225), 12, 2, False, 0, 2, 0),   # by weight 227, blocks of sixteen planes 324
    ((249, 249, 249), 12, 2, False, 0, 2, 16),  # 400 and 379
    ((189, 197, 311), 8, 0, False, 0, 2, 16),   # 273 and 234
    ((121, 121, 121), 10, 0, False, 1, 2, 0),   # running sums: 57 / 88
    ((193, 193, 193), 0, 2, True, 0, 2, None),  # no layers: 153 / 200
])
def test_route_follows_the_cost_of_both_sides(lib, nodes, pml, z_planes, lossy, dft, steps, chunk):
    got = _pass_plan(lib, nodes, pml, z_planes, lossy, dft, plane_wave=pml == 12)
    assert got[0] == steps
    if chunk is not None:
        assert got[2] == chunk
