"""Where lanes of one wave exchange values through LDS without a barrier, the compiler is told the order: it sees one lane's addresses, and may swap a lane's load with a store that only other lanes' loads
depend on.  No run can show the difference (a build that happens to keep the order gives the same bits), so the device code's unoptimised IR is read, which hipcc writes from source without a GPU."""
import os
import re
import shutil
import subprocess

import pytest

from koifish_amd import build as B

ORDER = {'fence syncscope("wavefront") release': "release", "@llvm.amdgcn.wave.barrier": "barrier", 'fence syncscope("wavefront") acquire': "acquire"}


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_token_rows_of_decode_products_are_turned_in_order(tmp_path):
    out = tmp_path / "rb.ll"
    subprocess.check_call([B.HIPCC] + B.HIP_FLAGS + ["-w", "--cuda-device-only", "-emit-llvm", "-S", "-Xclang", "-disable-llvm-passes", os.path.join(B.CSRC, "kf_rb_linear.hip"), "-o", str(out)])
    functions = {m.group(1): m.group(2) for m in re.finditer(r"^define [^@]*@([\w$]+)\(.*?\{\n(.*?)^\}", out.read_text(), re.M | re.S)}

    def marks(name, deep=True):
        found = []
        for line in functions[name].splitlines():
            found += [v for k, v in ORDER.items() if k in line]
            call = re.search(r"call .*@(\w+)\(", line)
            if deep and call and call.group(1) in functions:
                found += marks(call.group(1), False)
        return found
    turns = [n for n in functions if "RbTokens" in n and "4turn" in n]
    assert len(turns) == 4                                                    # 16, 32, 48, 64 columns
    for name in turns:
        assert marks(name) == ["release", "barrier", "acquire"] * 2, name     # the run before has been read | these rows are stored
