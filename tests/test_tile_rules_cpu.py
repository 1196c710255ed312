"""Which tile a launch takes, where both sides were timed: the rules of the headers as the host compiler evaluates them (no GPU)."""
import shutil
import subprocess

import pytest

from koifish_amd import build as B

# (rows of the weight, token rows, K, us on 256 x 256 tiles, us on 192 x 256 tiles)
TIMED = [(6144, 1900, 1024, 37.9, 31.7), (6144, 1900, 12288, 262.0, 240.9), (6144, 2608, 2048, 102.2, 83.2), (8704, 1971, 25600, 1259.3, 1001.3), (10240, 3500, 4096, 280.2, 238.4), (5120, 4096, 12288, 542.5, 518.3),
         (12288, 5888, 1024, 179.6, 171.1), (12288, 6912, 2048, 331.9, 312.4), (12288, 5888, 4096, 486.1, 497.7), (12288, 6912, 4096, 585.3, 605.7), (8704, 8000, 8192, 934.7, 978.7),
         (12288, 11008, 1024, 325.5, 362.6), (12288, 11008, 2048, 514.5, 561.5), (12288, 11008, 4096, 884.9, 952.2)]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_the_faster_of_the_big_tiles_is_taken(tmp_path):
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm3_tile.h"\n' % B.CSRC + "".join("static_assert(kf::g3_prefer_wide(%d, %d, %d) == %s);\n" % (m, n, k, "true" if wide < big else "false") for m, n, k, big, wide in TIMED))
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
