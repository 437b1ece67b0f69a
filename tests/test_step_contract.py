"""What step libraries and the runtime have to agree on.

  * A library built for other structures is refused, and creating its program
    fails saying so, also where a built-in program has its name (CPU).
  * build.sh builds anew when a header of the runtime is newer than its outputs
    (CPU, with compilers that only write their output files).
  * Steps that add and remove write their flags for every agent; a step program
    whose source an earlier compiler wrote sets them only, and runs alike (GPU:
    both against the model stepped in Python).
"""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EARLIER = os.path.join(REPO, "oracle", "_build", "libsteps_births_earlier.so")
CELL = [("pos", "float2"), ("life", "int"), ("age", "int")]

REFUSED = """
import ctypes as C
from openabl_amd import load_library
lib = load_library()
n = lib.abl_hip_program_count()
reg = getattr(lib, "_ZN3abl16register_programEPKNS_11ProgramDescE")  # the symbol older libraries call
reg.argtypes, reg.restype = [C.c_void_p], C.c_bool
keep = []
for name in (b"older", b"circle"):
    desc = (C.c_char_p * 64)(name)
    keep.append(desc)
    assert not reg(desc)
    h = C.c_void_p()
    assert lib.abl_hip_create(name, 0, C.byref(h)) == 1
    assert b"built for another version" in lib.abl_hip_last_error(), lib.abl_hip_last_error()
    b = C.c_size_t()
    assert lib.abl_hip_estimate_footprint(name, 0, 0, None, None, 10, 10, C.byref(b)) == 1
assert lib.abl_hip_program_count() == n
assert lib.abl_hip_create(b"nobody", 0, C.byref(h)) == 1
assert b"unknown program nobody" in lib.abl_hip_last_error()
print("refused")
"""


def test_library_of_another_version_is_refused():
    r = subprocess.run([sys.executable, "-c", REFUSED], cwd=REPO, capture_output=True, text=True)
    assert r.returncode == 0 and "refused" in r.stdout, r.stderr


def test_build_script_looks_at_the_runtimes_headers(tmp_path):
    from openabl_amd import codegen
    gen, root, bin_ = tmp_path / "gen", tmp_path / "root", tmp_path / "bin"
    (root / "include").mkdir(parents=True)
    (root / "openabl_amd" / "csrc").mkdir(parents=True)
    bin_.mkdir()
    headers = [root / "include" / "abl_hip.h", root / "openabl_amd" / "csrc" / "abl_runtime.hpp"]
    for h in headers:
        h.write_text("")
    for cc in ("hipcc", "g++"):  # writes what follows -o
        (bin_ / cc).write_text('#!/bin/sh\nwhile [ "$1" != -o ]; do shift; done\n'
                               f': > "$2"\necho {cc} >> "{tmp_path}/calls"\n')
        (bin_ / cc).chmod(0o755)
    codegen.generate(codegen.model_path("births"), str(gen))
    calls = tmp_path / "calls"

    def build():
        calls.write_text("")
        env = dict(os.environ, ABL_HIP_ROOT=str(root), PATH=f"{bin_}:{os.environ['PATH']}")
        subprocess.run(["./build.sh"], cwd=gen, check=True, env=env)
        for f in ("libsteps.so", "main"):  # older than what is touched below, newer than the sources
            os.utime(gen / f, (2e9, 2e9))
        return calls.read_text().split()

    assert build() == ["hipcc", "g++"]
    assert build() == []
    for h in headers + [gen / "steps.hip"]:
        os.utime(h, (2e9 + 1, 2e9 + 1))
        assert build() == ["hipcc", "g++"], h
        os.utime(h, (1e9, 1e9))
        assert build() == []


def stepped(n, steps):
    """births.abl in Python: [(pos, life, age)] in id order."""
    cells = [((float(i % 100), float(i // 100 % 100)), 2 + i % 13, i % 7) for i in range(n)]
    for _ in range(steps):
        cells = [(p, life - 1, age + 1) for p, life, age in cells]
        cells += [(p, 3 + age, 0) for p, _, age in cells if age % 4 == 0]
        cells = [c for c in cells if c[1] >= 1]
        born = [(p, 6, 1) for p, _, age in cells if age > 9]
        cells = [c for c in cells if c[2] <= 9] + born
    return cells


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["births", "births_earlier"])
@pytest.mark.parametrize("n", [1, 257, 3000, 40000])
def test_flags_of_steps_that_add_and_remove(form, n):
    """One agent, two tiles of removals, and the populations on either side of
    the limit up to which a block counts the flags before its tile itself."""
    from openabl_amd import Simulation, codegen, load_library, record_dtype
    print(f"case step contract {form} {n}", flush=True)
    name = form if form == "births_earlier" else "model_births"
    if form == "births_earlier":
        if not os.path.exists(EARLIER):
            pytest.skip("libsteps_births_earlier.so not built")
        load_library()
        keep = C.CDLL(EARLIER)  # noqa: F841 (registers its program)
    else:
        codegen.load_program(codegen.program_dir(name))
    dt = record_dtype(CELL, "f64")
    start = stepped(n, 0)
    rec = np.zeros(n, dt)
    rec["pos"], rec["life"], rec["age"] = ([c[k] for c in start] for k in range(3))
    sim = Simulation(name, "f64")
    sim.upload(rec)
    for upto in (1, 4, 9):
        sim.simulate(upto - {1: 0, 4: 1, 9: 4}[upto])
        got, want = sim.download(dt), stepped(n, upto)
        assert len(got) == len(want), upto
        assert np.array_equal(got["pos"], np.array([c[0] for c in want]).reshape(-1, 2)), upto
        assert got["life"].tolist() == [c[1] for c in want], upto
        assert got["age"].tolist() == [c[2] for c in want], upto
    sim.close()
