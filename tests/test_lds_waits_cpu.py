"""Loads into LDS behind reads of the same bytes: the wait for the reads is stated, not left to where the instructions that use them happen to stand (the device assembly, no GPU)."""
import re
import shutil
import subprocess

import pytest

from koifish_amd import build as B


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_small_batch_products_wait_for_their_reads_before_the_loads_that_overwrite_them(tmp_path):
    """a wave's LDS is its own, so no barrier stands between a turn's reads and the next rows' loads, and the compiler's own waits order no LDS read in front of an LDS-writing load"""
    out = tmp_path / "gemm.s"
    src = "%s/kf_gemm.hip" % B.CSRC
    r = subprocess.run([B.HIPCC] + B.HIP_FLAGS + B.HIP_FILE_FLAGS.get("kf_gemm.hip", []) + ["-w", "--cuda-device-only", "-S", src, "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    kernels = re.findall(r"^(_ZN2kf\w*gemm_direct\w*):.*?\n(.*?)^\.Lfunc_end", out.read_text(), re.M | re.S)
    loading = 0
    for name, body in kernels:
        pending = stated = loads = 0
        for line in body.splitlines() * 2:   # (twice: the loop's end in front of its beginning)
            op = line.split(";")[0].strip()
            if "#ASMSTART" in line or "#ASMEND" in line:
                stated = "#ASMSTART" in line
            elif op.startswith("ds_read"):
                pending = 1
            elif stated and re.match(r"s_waitcnt .*lgkmcnt\(0\)", op):
                pending = 0
            elif op.startswith("buffer_load") and op.endswith(" lds"):
                loads += 1
                assert not pending, "%s: %s" % (name, op)
        loading += loads > 0
    assert loading >= 16, (loading, [n for n, _ in kernels])   # six storages by 32 and 64 rows and their pairs, blocks of 16 weight rows
