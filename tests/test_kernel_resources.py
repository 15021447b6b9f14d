"""The build refuses a kernel with register spills: one instance of the relaxation kernel
that spilled has faulted the GPU (the spill was stored with the execution mask still off)."""
import os
import re

import pytest

from firecore_amd import build as fb

REMARK = """a.hip:118:1: remark: Function Name: {name} [-Rpass-analysis=kernel-resource-usage]
  118 | kernel(int a) {{
      | ^
a.hip:118:1: remark:     TotalSGPRs: 106 [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     VGPRs: 168 [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     ScratchSize [bytes/lane]: {scratch} [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     Dynamic Stack: False [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     SGPRs Spill: 162 [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     VGPRs Spill: {spill} [-Rpass-analysis=kernel-resource-usage]
a.hip:118:1: remark:     LDS Size [bytes/block]: 48 [-Rpass-analysis=kernel-resource-usage]
"""


def test_spills_are_refused():
    clean = REMARK.format(name="clean", scratch=0, spill=0)
    res = fb.kernel_resources(clean)
    assert res["clean"]["VGPRs"] == 168 and res["clean"]["LDS Size"] == 48
    fb.check_scratch(res)
    for scratch, spill in [(16, 0), (0, 1), (80, 20)]:
        with pytest.raises(RuntimeError, match="spilling"):
            fb.check_scratch(fb.kernel_resources(clean + REMARK.format(name="spilling", scratch=scratch, spill=spill)))
    with pytest.raises(RuntimeError, match="no resource-usage remarks"):
        fb.check_scratch(fb.kernel_resources("warning: something else"))


def test_built_kernels_have_no_scratch():
    if not os.path.exists(fb.RESOURCES):
        pytest.skip("library built elsewhere")
    res = fb.resources()
    assert sum("relax_persistent_kernel" in k for k in res) == 32
    fb.check_scratch(res)


def test_inline_assembly_restores_the_execution_mask():
    """Assembly that narrows exec puts back what it found: a constant would turn on the lanes
    of a caller in divergent code."""
    for name in os.listdir(fb.CSRC):
        with open(os.path.join(fb.CSRC, name)) as f:
            assert not re.search(r"exec(_lo|_hi)?, *-?\d", f.read()), name
