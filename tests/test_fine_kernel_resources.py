"""Register budgets of the neighbour kernels that take several lanes per particle, read from the
gfx950 assembly (no GPU needed). VGPRs come from 512 per lane in granules of 8, so 7 waves per
SIMD need at most 72, 6 at most 80 and 5 at most 96. Density and a single scene's force keep 7,
energy the 6 that its LDS (24,064 bytes of 160 KiB per block) allows, a batch's kernels, whose
lanes each hold their scene's parameters, 6 and (force) 5. None may spill: the launches are bound
by the latency of their chains, which scratch loads would lengthen, with the same results.
"""
import os
import re
import shutil
import subprocess

import pytest

from sca2012_amd import build as sbuild

# kernel, batched -> max VGPRs
BUDGET = {("k_density_fine", 0): 72, ("k_force_fine", 0): 72, ("k_energy_fine", 0): 80,
          ("k_density_fine", 1): 80, ("k_force_fine", 1): 96, ("k_energy_fine", 1): 80}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not (os.path.exists(sbuild.HIPCC) or shutil.which(sbuild.HIPCC)):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / "sph_fine.s")
    cmd = [sbuild.HIPCC] + sbuild.FLAGS + ["--cuda-device-only", "-S",
                                           os.path.join(sbuild.CSRC, "sph_fine.hip"), "-o", out]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    with open(out) as f:
        return f.read()


@pytest.mark.parametrize("stem, batched", sorted(BUDGET))
def test_registers_and_scratch(assembly, stem, batched):
    found = {}
    for m in re.finditer(r"^(_Z\w+\d%sILi(\d)ELb%dE\w+):" % (stem, batched), assembly, re.M):
        meta = assembly[assembly.find(".Lfunc_end", m.end()):][:4000]
        found[m.group(1)] = [int(re.search(k + r":\s*(\d+)", meta).group(1))
                             for k in ("NumSgprs", "NumVgprs", "ScratchSize")]
    assert len(found) == (2 if batched else 3), sorted(found)  # 3D-2 and 3D-4, and 2D
    over = {n: r for n, r in found.items() if r[0] > 102 or r[1] > BUDGET[stem, batched] or r[2] > 0}
    assert not over, over
