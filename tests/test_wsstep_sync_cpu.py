"""The single-launch optimiser step hands tiles from workgroup to workgroup
through flags (rvgp_amd/csrc/wsstep.hip).  A flag raised before the producer's
L2 write-back has finished lets a consumer read the previous step's tile, which
no test of results shows reliably; so the compiled kernel is read instead: every
L2 write-back is followed by a wait for it before anything else is stored."""
import os
import re
import shutil
import subprocess

import pytest

from rvgp_amd import _build


def test_every_l2_write_back_is_waited_for(tmp_path):
    if not os.path.exists(_build.HIPCC) and shutil.which("hipcc") is None:
        pytest.skip("hipcc not available")
    out = str(tmp_path / "wsstep.s")
    cmd = [_build.HIPCC, *_build.FLAGS, "--cuda-device-only", "-S",
           os.path.join(_build.CSRC, "wsstep.hip"), "-o", out]
    subprocess.run(cmd, check=True, capture_output=True)
    with open(out) as fh:
        code = [line.strip() for line in fh if line.startswith("\t") and not line.startswith("\t.")]
    backs = [i for i, line in enumerate(code) if line.startswith("buffer_wbl2")]
    for i in backs:
        rest = [line for line in code[i + 1:i + 40] if not line.startswith(";")]
        wait = next(k for k, line in enumerate(rest) if line.startswith("s_waitcnt") and "vmcnt(0)" in line)
        store = next((k for k, line in enumerate(rest)
                      if line.startswith(("global_store", "flat_store", "buffer_store", "global_atomic"))), len(rest))
        assert wait < store, code[i:i + store + 2]


def test_there_is_a_write_back_for_every_flag(tmp_path):
    """The test above says nothing of a write-back that is not there: each of the
    two kernels has at least one for every task that raises a flag."""
    if not os.path.exists(_build.HIPCC) and shutil.which("hipcc") is None:
        pytest.skip("hipcc not available")
    src, out = os.path.join(_build.CSRC, "wsstep.hip"), str(tmp_path / "wsstep.s")
    subprocess.run([_build.HIPCC, *_build.FLAGS, "--cuda-device-only", "-S", src, "-o", out], check=True,
                   capture_output=True)
    with open(src) as fh:
        sites = fh.read().count("publish(sync + ") + 1  # and the filter's, publish(a.sync + ...)
    with open(out) as fh:
        kernels = re.findall(r"^(\w*ws_step_kernel\w*):(.*?)^\.Lfunc_end", fh.read(), re.S | re.M)
    assert len(kernels) == 2 and sites == 7
    backs = sorted(len(re.findall(r"^\tbuffer_wbl2\b", body, re.M)) for _, body in kernels)
    assert backs[0] >= sites - 1 and backs[1] >= sites, backs  # the first has no residual task
