"""The INT4 prefill GEMM's stores do not wait for each other.  Loads and stores
share one counter on gfx950, so a store whose address comes from a vector load
waits for every store issued before that load returned: with each output tile's
segment read by vector loads, the stores of a workgroup ran one after the other
(8 us a round of workgroups at 128 rows by 17 tiles).  Compiles one
kernel of csrc/pf4_kernel.h to assembly; CPU only."""
import os
import re
import shutil
import subprocess

import pytest

from breeze_amd import _build

SRC = """#include "pf4_kernel.h"
namespace bq { template __global__ void pf4_kernel<%s, %s, 5, 4>(Pf4Args); }
"""


@pytest.mark.skipif(shutil.which(_build.HIPCC) is None, reason="no hipcc")
@pytest.mark.parametrize("two_pass,zeros", [("false", "false"), ("true", "true")])
def test_stores_do_not_wait(tmp_path, two_pass, zeros):
    src, out = tmp_path / "one.hip", tmp_path / "one.s"
    src.write_text(SRC % (two_pass, zeros))
    subprocess.run([_build.HIPCC, "-x", "hip", *_build.FLAGS, *_build.DEVICE_FLAGS, "-I", _build.CSRC,
                    "--offload-device-only", "-S", str(src), "-o", str(out)], check=True, capture_output=True)
    lines = [s.strip() for s in out.read_text().splitlines()]
    code = [s for s in lines if s and not s.startswith((";", ".")) and not re.match(r"^[\w$.]+:", s)]
    stores = [i for i, s in enumerate(code) if s.startswith("global_store_dword")]
    assert len(stores) >= 32
    assert not any(s.startswith("flat_store") for s in code)
    # Between two stores of one group (addresses apart by adds only) no wait.
    waits = [i for i in stores if any("vmcnt" in s for s in code[max(0, i - 4):i])]
    assert len(waits) <= len(stores) // 8, f"{len(waits)} of {len(stores)} stores wait"
