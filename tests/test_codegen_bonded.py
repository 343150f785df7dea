"""No bonded kernel that an ordinary step launches touches scratch memory. (test_codegen allows up to 72 bytes to some of them, which once
spilled; none does now, so a spill that came back would pass there. The per-atom variants may use scratch, as there.)"""
import os
import re

import pytest

import test_codegen as tc


@pytest.mark.skipif(not os.path.exists(tc.HIPCC), reason="hipcc not installed")
def test_no_scratch_in_bonded_kernels(tmp_path):
    asm = tc._asm("k_bonded.hip", str(tmp_path / "k_bonded.s"))
    names = [m for m in re.findall(r"\.amdhsa_kernel (\S+)", asm) if m.startswith("_ZN3rxa")]
    short = {n: re.sub(r"^\d+", "", re.sub(r"(ENS_|EvNS_).*", "", n.replace("_ZN3rxa12_GLOBAL__N_1", ""))) for n in names}
    ordinary = [n for n in names if not tc.PERATOM.match(short[n])]
    assert len(ordinary) > 30 and sum(short[n] in tc.ALLOWED for n in ordinary) >= 10   # the names still match
    assert not [short[n] for n in ordinary if tc._touches_scratch(asm, n)]
