"""The check of tests/test_isa_hazards_cpu.py on the tile kernels of gemm_mid.hpp: no instruction touches a register of a hand-issued
LDS read before the wait that covers it.  One instantiation file per way of reading weights; the accumulators must be AGPRs that the
loop never moves (the compiler spends 300 moves per k-tile if they are left to it)."""
import os
import re
import subprocess

import pytest

from tests.test_isa_hazards_cpu import _build_recipe, hazards


@pytest.mark.parametrize("src", ["gemm_mid_tiled_192.hip", "gemm_mid_nk_128.hip"])
def test_no_register_is_touched_before_its_read_has_landed(tmp_path, src):
    recipe = _build_recipe()
    if not os.path.exists(recipe.HIPCC):
        pytest.skip("no hipcc in this image")
    out = str(tmp_path / "out.s")
    subprocess.run([recipe.HIPCC] + recipe.HIP_FLAGS + ["-S", "--cuda-device-only", os.path.join(recipe.CSRC, src), "-o", out],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.PIPE)
    text = open(out).read()
    kernels, reads, found = hazards(text)
    assert kernels > 0 and reads > 100 and not found, found[:3]
    for body in re.findall(r"^_ZN2lg12gemm_f16_mid\w+:[^\n]*\n(.*?)s_endpgm", text, re.S | re.M):
        loop = max(re.split(r"^\.LBB\w+:", body, flags=re.M), key=lambda b: b.count("v_mfma"))
        assert loop.count("v_mfma") > 0 and "v_accvgpr" not in loop
