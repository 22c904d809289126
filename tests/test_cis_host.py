"""The sine/cosine polynomials of the kernels (csrc/sarf_cis.hpp), compiled for the
host and compared with libm in long double over a revolution.  CPU only."""
import os
import shutil
import subprocess

import pytest

from uncc_sar_focusing_amd._build import CSRC, HIPCC

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not available")


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cis") / "cis_check")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--offload-host-only", f"-I{CSRC}",
                    os.path.join(HERE, "host", "cis_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, check=True)
    return {k: float(v) for k, v in (ln.split() for ln in r.stdout.splitlines())}


def test_fp64(errors):
    """The polynomial's last step rounds by half an ulp of a number below 8, times x
    = 1/8, the product by half an ulp of a number below 1, and the steps before
    by less: 4.4e-16 in all, the terms left out 5e-17."""
    assert errors["cis_rev64"] <= 4.4e-16


def test_fp32(errors):
    """The last sum rounds by half an ulp of a number below 1 (3e-8), the squared
    argument and the product added to it by as much relative to 0.3: 3.6e-8."""
    assert errors["cis_rev"] <= 6.6e-8
