"""What the compiler does not know about the hand-issued instructions of gemm_mid.hpp, checked in the gfx950 assembly of every
instantiation: no instruction touches a register of a hand-issued LDS read before the wait that covers it (the check of
tests/test_isa_hazards_cpu.py); no instruction touches an accumulator between the last matrix instruction and the nops after which its
result is there; and the accumulators are AGPRs that the loop never moves (the compiler spends 300 moves per k-tile if they are left to it)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from tests.test_isa_hazards_cpu import _build_recipe, hazards


def _kernels(text):
    return re.findall(r"^(_ZN2lg12gemm_f16_mid\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.S | re.M)


def early_accumulator_uses(body):
    """Instructions that name an AGPR after the last matrix instruction of a kernel and before its first `s_nop 15`."""
    lines = [l.split(";")[0].strip() for l in body.splitlines()]
    drain = next(i for i, l in enumerate(lines) if l.startswith("s_nop 15"))
    last = max(i for i in range(drain) if lines[i].startswith("v_mfma"))
    return [l for l in lines[last + 1:drain] if re.search(r"\ba\[?\d", l)]


def test_an_accumulator_read_before_the_drain_is_seen():
    body = "v_mfma_f32_16x16x32_f16 a[0:3], v[0:3], v[4:7], a[0:3]\n%s\ts_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15\n\tv_accvgpr_read_b32 v0, a0\n"
    assert early_accumulator_uses(body % "") == []
    assert len(early_accumulator_uses(body % "\tscratch_store_dwordx4 off, a[192:195], off offset:8 ; 16-byte Folded Spill\n")) == 1
    assert len(early_accumulator_uses(body % "\tv_accvgpr_read_b32 v9, a3\n")) == 1


def test_nothing_touches_a_register_whose_value_is_still_on_its_way(tmp_path):
    recipe = _build_recipe()
    if not os.path.exists(recipe.HIPCC):
        pytest.skip("no hipcc in this image")
    sources = [s for s in recipe.HIP_SOURCES if '#include "gemm_mid.hpp"' in open(os.path.join(recipe.CSRC, s)).read()]

    def to_asm(src):
        out = str(tmp_path / (src + ".s"))
        subprocess.run([recipe.HIPCC] + recipe.HIP_FLAGS + ["-S", "--cuda-device-only", os.path.join(recipe.CSRC, src), "-o", out],
                       check=True, stdout=subprocess.PIPE, stderr=subprocess.PIPE)
        return src, open(out).read()

    with ThreadPoolExecutor(max_workers=4) as ex:
        results = [(src, text) for src, text in ex.map(to_asm, sources) if _kernels(text)]
    assert len(results) == 9     # three layouts, three widths (the 96-wide tiles share a file with the 128-wide ones)
    for src, text in results:
        kernels, reads, found = hazards(text)
        assert kernels > 0 and reads > 100 and not found, (src, found[:3])
        for name, body in _kernels(text):
            assert early_accumulator_uses(body) == [], (src, name)
            loop = max(re.split(r"^\.LBB\w+:", body, flags=re.M), key=lambda b: b.count("v_mfma")).rpartition("v_mfma")[0]
            assert loop.count("v_mfma") > 0 and "v_accvgpr" not in loop, (src, name)
