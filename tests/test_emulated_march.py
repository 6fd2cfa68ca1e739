"""The tile march compiled for the host (tests/emu: a block's sixteen wavefronts in
lockstep at its barriers) with every address and every array index checked, against
the float64 oracle: tile edges, grids far smaller than a tile, every face mode,
coefficient mode and kind of source term, staged planes and points under split calls,
blocks of equal and of weighted length.  Tolerance 1e-5 of a family's peak (about ten
roundings of 2^-24 per sample and step over at most 15 steps)."""

import os
import subprocess
import sys

import pytest

from test_emulated_kernels import CSRC, EMU, ROOT, _asan_runtime

GROUPS = ("march", "march_terms", "march_blocks", "stage_rows", "scratch")


@pytest.fixture(scope="module")
def checked_library(tmp_path_factory):
    asan = _asan_runtime()
    if asan is None:
        pytest.skip("g++ with AddressSanitizer is not available")
    out = tmp_path_factory.mktemp("emu_march")
    src = out / "maxwell_fdtd_emu.cpp"
    src.write_text(open(os.path.join(CSRC, "maxwell_fdtd.hip")).read())
    lib = out / "libmaxwell_fdtd_emu.so"
    cmd = ["g++", "-std=c++20", "-O1", "-g", "-fPIC", "-shared", "-fsanitize=address,bounds",
           "-fno-sanitize-recover=bounds", "-w", "-I", EMU, "-I", os.path.join(ROOT, "include"), "-I", CSRC, str(src),
           os.path.join(EMU, "emu_globals.cpp"), "-o", str(lib)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-4000:]
    return str(lib), asan


def test_march_matches_oracle_under_emulation(checked_library):
    lib, asan = checked_library
    env = dict(os.environ, LD_PRELOAD=asan, ASAN_OPTIONS="detect_leaks=0", OMP_NUM_THREADS="1")
    procs = {g: subprocess.Popen([sys.executable, os.path.join(EMU, "run_case.py"), lib, g], stdout=subprocess.PIPE,
                                 stderr=subprocess.PIPE, text=True, env=env) for g in GROUPS}
    failed = []
    for g, proc in procs.items():
        out, err = proc.communicate(timeout=900)
        print(out)
        if proc.returncode != 0 or not out.strip().endswith("OK"):
            failed.append((g, out[-3000:], err[-3000:]))
    assert not failed, failed
