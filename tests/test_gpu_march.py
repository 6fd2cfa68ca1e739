"""The tile march (single-pass steps taken one or two at a time by one kernel) vs the
float64 oracle where its tiles, chunks and stages end.

Shapes are node counts around a tile's own 60 (two steps) and 62 (one step) columns and
12 / 14 rows, all in equal blocks for passes of two steps.  Runs are split so that single steps, pairs of two-step passes and stage blocks
begin at odd places.  Tolerance 1e-5 of a family's peak: about ten roundings of 2^-24
per sample and step over 22 steps."""

import numpy as np
import pytest
import torch

import witwin_maxwell_amd as mw
from witwin_maxwell_amd import configs
from witwin_maxwell_amd.fdtd.plan import compile_plan

from test_gpu_parity import _check_fields, _check_monitors, _check_psi

pytestmark = pytest.mark.gpu

SHAPES = [(12, 16, 64), (13, 17, 65), (10, 29, 125), (31, 30, 126), (70, 77, 130)]
FACES = [dict(default="pml"), dict(default="pml", x_low="pec", y_high="pmc", z_low="none"), dict(default="pec")]


def _scene(nodes, faces, lossy):
    dx = configs.DX
    pads = [[4 if faces.get(f"{a}_{s}", faces["default"]) == "pml" else 0 for s in ("low", "high")] for a in "xyz"]
    cells = [n - 1 - sum(p) for n, p in zip(nodes, pads)]
    h = [0.5 * (n - 0.01) * dx for n in cells]  # the grid rounds up to whole cells
    scene = mw.Scene(domain=mw.Domain(tuple((-x, x) for x in h)), grid=mw.GridSpec.uniform(dx),
                     boundary=mw.BoundarySpec.faces(num_layers=4, **faces), device="cuda")
    scene.add_structure(mw.Structure(mw.Box((0.1 * h[0], -0.2 * h[1], 0.3 * h[2]), (h[0], h[1], 0.8 * h[2])),
                                     mw.Material(eps_r=3.0, sigma_e=0.05 if lossy else 0.0)))
    scene.add_source(mw.PointDipole((0.2 * dx, 0.3 * dx, -0.4 * dx), (0.5, 0.3, 1.0), profile="ideal",
                                    source_time=mw.CW(configs.F0)))
    freqs = (0.9 * configs.F0, 1.1 * configs.F0)
    for axis, q in zip("xyz", range(3)):
        scene.add_monitor(mw.PlaneMonitor(axis, axis=axis, position=0.25 * h[q], fields=("Ez", "Hy"),
                                          frequencies=freqs))
    scene.add_monitor(mw.PointMonitor("p", (0.0, 0.0, 0.0), fields=("Ey", "Hz"), frequencies=freqs))
    return scene, freqs


@pytest.mark.parametrize("faces", FACES, ids=["pml", "mixed", "pec"])
@pytest.mark.parametrize("nodes", SHAPES, ids=str)
def test_march_matches_oracle_at_tile_edges(nodes, faces):
    from oracle.driver import OracleRun
    from witwin_maxwell_amd.fdtd.runtime import DeviceRun
    print(f"case: march {nodes} {faces}", flush=True)
    scene, freqs = _scene(nodes, faces, lossy=nodes[0] % 2 == 0)
    plan = compile_plan(scene, frequencies=freqs, time_steps=22, window="none")
    assert tuple(plan.shape) == nodes
    ref, dev = OracleRun(plan).run(), DeviceRun(plan, "cuda", plane_stage_depth=8)
    for end in (1, 12, 15, 22):
        dev.run(end - dev.step_index)
    torch.cuda.synchronize()
    _check_fields(ref, dev)
    _check_psi(plan, ref, dev)
    _check_monitors(ref, dev)
    whole = DeviceRun(plan, "cuda").run()  # the same bits wherever a run is split
    for c, t in whole.fields.items():
        assert torch.equal(t, dev.fields[c]), c
    for a, b in zip(whole.plane_re + [whole.point_re], dev.plane_re + [dev.point_re]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("nf", [1, 2, 3])
def test_full_field_sums_match_oracle(nf):
    """Running sums of all E, read in groups of two frequencies: whole and odd groups,
    on a grid whose tiles and planes end inside."""
    from oracle.driver import OracleRun
    from witwin_maxwell_amd.fdtd.runtime import DeviceRun
    print(f"case: march full-field sums, {nf} frequencies", flush=True)
    scene, _ = _scene((13, 17, 65), FACES[1], lossy=False)
    scene.monitors.clear()
    freqs = tuple(np.linspace(0.9, 1.1, nf) * configs.F0)
    plan = compile_plan(scene, frequencies=freqs, time_steps=22, window="none", full_field_dft=True)
    ref, dev = OracleRun(plan).run(), DeviceRun(plan, "cuda").run()
    torch.cuda.synchronize()
    assert len(plan.dft_frequencies) == nf
    for part, sums in enumerate((dev.dft_re, dev.dft_im)):
        want = {c: np.asarray(ref.dft[c][part]) for c in sums}
        scale = max(float(np.max(np.abs(v))) for v in want.values())
        for c, t in sums.items():
            assert np.max(np.abs(t.double().cpu().numpy() - want[c])) <= 1e-5 * scale, (c, part)
