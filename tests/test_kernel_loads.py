"""How many values a compiled kernel's lanes load."""
import os
import re
import shutil
import subprocess
import tempfile

import pytest

from conftest import ROOT


def test_parameter_kernel_loads_only_its_parcel():
    """Per lane params_kernel loads 9 + 9 + 2 values of its parcel, and not the
    630 values of the a2 and a4 maps, which are the same for all."""
    from specfab_amd import build
    if not shutil.which(build.HIPCC):
        pytest.skip("no hipcc")
    out = os.path.join(tempfile.gettempdir(), "sfg_kernels_%d.s" % os.getpid())
    subprocess.check_call([build.HIPCC] + build.HIPFLAGS + ["-I", build.CSRC, "--cuda-device-only", "-S",
                                                            os.path.join(build.CSRC, "sfg_kernels.hip"), "-o", out],
                          stderr=subprocess.DEVNULL)
    text = open(out).read()
    os.remove(out)
    body = re.search(r"^_ZN3sfg13params_kernel\w+:.*?\.end_amdhsa_kernel", text, re.S | re.M).group(0)
    loads = re.findall(r"^\s+(?:global|flat)_load_dword(x[24])?", body, re.M)
    words = sum({"": 1, "x2": 2, "x4": 4}[x] for x in loads)
    assert 0 < words <= 2 * (9 + 9 + 2), (len(loads), words)
    assert not re.search(r"^\s+scratch_", body, re.M)
