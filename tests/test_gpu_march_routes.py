"""Each way the library takes a run's steps, named by the library and held to the
float64 oracle: passes in blocks listed by cost, in blocks of sixteen planes, and the
separate launches of a run that keeps every step to itself.  Tolerance 1e-5 of a
family's peak: about ten roundings of 2^-24 per sample and step over 22 steps."""

import ctypes

import numpy as np
import pytest
import torch

from witwin_maxwell_amd.fdtd import native as nat
from witwin_maxwell_amd.fdtd.plan import compile_plan

from test_gpu_march import FACES, _scene
from test_gpu_parity import _check_fields, _check_monitors, _check_psi

pytestmark = pytest.mark.gpu

LISTED = (90, 77, 130)  # 3 x 7 tiles of 90 planes: two-step passes list their blocks from 1536 on


def _run(plan, splits, **kw):
    from witwin_maxwell_amd.fdtd.runtime import DeviceRun
    dev = DeviceRun(plan, "cuda", **{k: v for k, v in kw.items() if k != "xchunk"})
    dev.set_tiling(kw.get("xchunk", 0), 0, 0)
    route = dev.pass_plan()
    for end in splits:
        dev.run(end - dev.step_index)
    dev.run()
    torch.cuda.synchronize()
    return dev, route


@pytest.mark.parametrize("faces", FACES[:2], ids=["pml", "mixed"])
@pytest.mark.parametrize("nodes,xchunk", [(LISTED, 0), (LISTED, 16), ((31, 30, 126), 16)],
                         ids=["listed", "sixteen", "sixteen-remainder"])
def test_passes_match_oracle(nodes, xchunk, faces):
    """x, y and z planes and a point, split so that single steps and pairs of passes
    begin at odd places."""
    from oracle.driver import OracleRun
    print(f"case: march {nodes} xchunk {xchunk} {faces}", flush=True)
    scene, freqs = _scene(nodes, faces, lossy=False)
    plan = compile_plan(scene, frequencies=freqs, time_steps=22, window="none")
    assert tuple(plan.shape) == nodes
    ref = OracleRun(plan).run()
    dev, route = _run(plan, (1, 12, 15), plane_stage_depth=8, xchunk=xchunk)
    assert route[0] == 2 and route[2] == xchunk, route
    _check_fields(ref, dev)
    _check_psi(plan, ref, dev)
    _check_monitors(ref, dev)


@pytest.mark.parametrize("faces", FACES, ids=["pml", "mixed", "pec"])
@pytest.mark.parametrize("nodes", [(12, 16, 64), (31, 30, 126)], ids=str)
def test_separate_launches_match_oracle(nodes, faces):
    """The separate launches at the library's own tiling, lossy and not."""
    from oracle.driver import OracleRun
    print(f"case: separate launches {nodes} {faces}", flush=True)
    scene, freqs = _scene(nodes, faces, lossy=nodes[0] % 2 == 0)
    plan = compile_plan(scene, frequencies=freqs, time_steps=22, window="none")
    ref = OracleRun(plan).run()
    dev, route = _run(plan, (1, 12, 15), plane_stage_depth=8, multi_step=False)
    assert route == (0, 0, 0)
    _check_fields(ref, dev)
    _check_psi(plan, ref, dev)
    _check_monitors(ref, dev)


@pytest.mark.parametrize("depth", [0, 3, 8, 32])
def test_staged_sums_equal_per_step_sums(depth):
    """Planes of the three axes sampled in two-step passes and folded a block at a time
    give, to the bit, the sums of adding each step's plane after that step."""
    print(f"case: staged against per-step sums, depth {depth}", flush=True)
    scene, freqs = _scene((13, 29, 65), FACES[0], lossy=False)
    plan = compile_plan(scene, frequencies=freqs, time_steps=37, window="none")
    dev, route = _run(plan, (9, 10), plane_stage_depth=depth)
    assert route[0] == 2
    from witwin_maxwell_amd.fdtd.runtime import DeviceRun
    step = DeviceRun(plan, "cuda")
    step.program.n_planes = step.program.n_points = 0
    nf = len(freqs)
    weights = [torch.as_tensor(np.ascontiguousarray(w, dtype=np.float32), device="cuda") for w in plan.obs_weights]
    sums = [(torch.zeros_like(re), torch.zeros_like(re)) for re in dev.plane_re]
    for n in range(plan.time_steps):
        step.run(1)
        for (comp, axis, index), (re, im) in zip(plan.observers.planes, sums):
            wc, ws = weights[:2] if comp[0] == "E" else weights[2:]
            f = step.fields[comp]
            nat.check(step.lib.mw_accumulate_plane(
                nat.ptr(f), *f.shape, "xyz".index(axis), index, nf, ctypes.c_void_p(wc[n].data_ptr()),
                ctypes.c_void_p(ws[n].data_ptr()), nat.ptr(re), nat.ptr(im), nat.current_stream()), step.lib)
    torch.cuda.synchronize()
    for (re, im), a, b in zip(sums, dev.plane_re, dev.plane_im):
        assert float(a.abs().max()) > 0
        assert torch.equal(re, a) and torch.equal(im, b)
