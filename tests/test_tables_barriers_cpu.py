"""The barriers of the table step that wait for no stores (csrc/tables_gfx950.hip), in the compiler's intermediate form: each is
handed the tables.  They are a ``__restrict__`` argument, so loads and stores of them may move across an asm statement that
does not name them, whatever it says that it clobbers."""
import importlib.util
import os
import re
import subprocess

import pytest

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lingbot-map_amd")


def test_bare_barriers_are_handed_the_tables():
    spec = importlib.util.spec_from_file_location("_lbm_build_flags", os.path.join(PACKAGE, "lingbot_map_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc here")
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-shared")]
    ir = subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-S", "-emit-llvm", "-o", "-",
                         os.path.join(build.CSRC, "tables_gfx950.hip")], stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True, check=True).stdout
    kernels = [f for f in re.findall(r"^define [^\n]*lbm_tables_kernel.*?^}", ir, re.M | re.S)]
    assert len(kernels) == 4
    for k in kernels:
        barriers = re.findall(r'asm sideeffect "s_barrier", "([^"]*)"\(([^)]*)\)', k)
        assert len(barriers) == 2 or "noalias" not in k.split("\n", 1)[0]
        for constraints, operands in barriers:
            assert "~{memory}" in constraints and operands.startswith("ptr")
