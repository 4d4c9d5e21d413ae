"""The fp32 attention backward kernels that leave dS in memory need no more registers for it, in the built library, than costs
them a wave of a SIMD or makes them spill where they did not."""
import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin/"
NAME = re.compile(r"attn_f32_bwd_dkdv(?:_pair)?_kernelILi\d+E(?:Lb[01]ELi[12]E)?Lb([01])EE")


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-readelf"), reason="no reader of its notes here")
def test_saving_scores_costs_no_waves(ffk, tmp_path):
    shutil.copy(ffk.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([LLVM + "llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    found = {False: {}, True: {}}
    for path in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", path], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n  - (?=\.agpr_count)", notes)[1:]:
            value = dict(re.findall(r"^ *\.(name|vgpr_count|vgpr_spill_count|sgpr_spill_count): +(\S+)$", kernel, re.M))
            m = NAME.search(value["name"])
            if m:
                form = value["name"][:m.start(1)]
                found[m.group(1) == "1"][form] = [int(value[k]) for k in ("vgpr_count", "vgpr_spill_count", "sgpr_spill_count")]
    assert len(found[True]) == 8 and set(found[True]) == set(found[False])
    for form, (registers, spilled, scalars) in found[True].items():
        without, spilled_without, _ = found[False][form]
        waves = [512 // -(-n // 8 * 8) for n in (registers, without)]
        print(form, found[True][form], found[False][form], waves)
        assert waves[0] == waves[1] and scalars == 0, form
        # the form that spills anyway (head sizes from 132 on, through registers): a few more
        assert spilled <= (0 if spilled_without == 0 else spilled_without + 8), form
