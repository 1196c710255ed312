"""The workspace of a prompt's launches (Fish::PrefillScratch), on the CPU: the host library over an ABI of empty functions whose allocator keeps a log and can refuse."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "koifish_amd", "libkf_host.so")
ALLOC = """
#include <stdlib.h>
#include <string.h>
typedef unsigned long size_t_;
size_t_ stub_limit = ~0ul, stub_copies = 0, stub_stacked = 0, stub_matrix = 0, stub_scratch = 0;
size_t_ stub_size[4096]; void* stub_at[4096]; int stub_n = 0; size_t_ stub_live = 0, stub_peak = 0;
const char* kf_last_error(void) { return ""; }
int kf_init(int device, void* stream, void** out) { *out = calloc(1, 4096); return 0; }
int kf_malloc(void* c, size_t_ bytes, void** out) {
    if (bytes >= stub_limit) return OOM;
    *out = malloc(16), stub_at[stub_n] = *out, stub_size[stub_n++] = bytes, stub_live += bytes;
    if (stub_live > stub_peak) stub_peak = stub_live;
    return 0;
}
int kf_free(void* c, void* p) {
    for (int i = 0; i < stub_n; i++) if (stub_at[i] == p) stub_live -= stub_size[i], stub_at[i] = 0;
    return 0;
}
int kf_set_scratch(void* c, void* p, size_t_ bytes) { stub_scratch = bytes; return 0; }
size_t_ kf_layer_copies_bytes(void) { return stub_copies; }
size_t_ kf_linear_multi_scratch_bytes(void) { return stub_stacked; }
size_t_ kf_linear_scratch_bytes(void) { return stub_matrix; }
size_t_ kf_resident_scratch_bytes(void) { return 4096; }
"""
CHILD = """
import ctypes as C, os, sys
here = sys.argv[1]
hip, host = C.CDLL(os.path.join(here, "libkf_hip.so"), C.RTLD_GLOBAL), C.CDLL(os.path.join(here, "libkf_host.so"))
val = lambda n: C.c_ulong.in_dll(hip, n)
host.kfh_create.restype, rc = C.c_void_p, C.c_int(0)
MB = 1 << 20

def model(matrix=0):
    val("stub_copies").value, val("stub_stacked").value, val("stub_matrix").value, val("stub_limit").value = 1000 * MB, 300 * MB, matrix, (1 << 64) - 1
    h = C.c_void_p(host.kfh_create(0, None, 256, 2, 4, 2, 64, 512, 512, 2048, C.c_float(1e-6), C.c_float(1e-6), C.c_float(1e6), C.byref(rc)))
    assert h.value, rc.value
    keep = (C.c_char * 4096)()
    for layer in range(2):
        for slot, (m, k) in enumerate([(256, 256), (128, 256), (128, 256), (256, 256), (512, 256), (512, 256), (256, 512)]):
            assert host.kfh_set_weight(h, layer, slot, 14, m, k, keep, C.c_size_t(m * k // 2 + (m + k + m * k // 64) * 2), C.c_size_t(m * k // 2), 1, 128, 0, 15, 8) == 0
        for slot in range(4):
            assert host.kfh_set_norm(h, layer, slot, keep, 64, 1) == 0
    assert host.kfh_set_weight(h, -1, 0, 3, 512, 256, keep, C.c_size_t(512 * 256 * 2), C.c_size_t(512 * 256 * 2), 1, 128, 0, 15, 8) == 0
    assert host.kfh_tie_head(h) == 0 and host.kfh_set_norm(h, -1, 0, keep, 256, 1) == 0
    return h, keep

def prefill(h):
    return host.kfh_prefill(h, (C.c_int * 8)(), 8, 0)

def largest():
    n = C.c_int.in_dll(hip, "stub_n").value
    return max((C.c_ulong * 4096).in_dll(hip, "stub_size")[:n])

case = sys.argv[2]
h, keep = model(matrix=200 * MB if case == "peak" else 0)
base = val("stub_live").value
if case == "room":
    assert prefill(h) == 0 and val("stub_scratch").value == 1000 * MB
if case == "no room":          # the copies only save time: the block without them
    val("stub_limit").value = 900 * MB
    assert prefill(h) == 0 and val("stub_scratch").value == 300 * MB
    val("stub_limit").value = (1 << 64) - 1
    assert prefill(h) == 0 and val("stub_scratch").value == 300 * MB   # not tried again at every prompt
if case == "no room at all":
    val("stub_limit").value = 200 * MB
    assert prefill(h) < 0
    val("stub_limit").value = (1 << 64) - 1
    assert prefill(h) == 0 and val("stub_scratch").value == 1000 * MB
if case == "resident":         # the copies of a layer are never made beside resident ones
    host.kfh_set_prefill_resident(h, 1, C.c_size_t(1 << 34))
    assert prefill(h) == 0 and val("stub_scratch").value == 300 * MB and largest() < 1000 * MB
    host.kfh_set_prefill_resident(h, 0, C.c_size_t(0))
    assert prefill(h) == 0 and val("stub_scratch").value == 1000 * MB
if case == "peak":             # the block of the single matrices' routes goes before the larger one is taken
    assert val("stub_scratch").value == 200 * MB
    assert prefill(h) == 0 and val("stub_scratch").value == 1000 * MB and val("stub_peak").value < base - 200 * MB + 1100 * MB
print("ok")
"""


@pytest.fixture(scope="module")
def libs(tmp_path_factory):
    if not os.path.exists(HOST):
        pytest.skip("libkf_host.so is not built")
    d = tmp_path_factory.mktemp("stub")
    with open(os.path.join(ROOT, "include", "kf_abi.h")) as f:
        oom = next(line.split()[2] for line in f if line.startswith("#define KF_OUTOF_GPUMEMORY"))
    need = {line.split()[-1] for line in subprocess.check_output(["nm", "-D", "--undefined-only", HOST], text=True).splitlines() if line.split()[-1].startswith("kf")}
    own = {w for w in need if w + "(" in ALLOC}
    src = ALLOC + "".join("int %s(void) { return 0; }\n" % n for n in sorted(need - own))
    (d / "stub.c").write_text(src)
    subprocess.check_call(["gcc", "-O1", "-w", "-shared", "-fPIC", "-DOOM=" + oom, "-Wl,-soname,libkf_hip.so", "-o", str(d / "libkf_hip.so"), str(d / "stub.c")])
    os.symlink(HOST, d / "libkf_host.so")
    return d


@pytest.mark.parametrize("case", ["room", "no room", "no room at all", "resident", "peak"])
def test_workspace_of_a_prompt(libs, case):
    r = subprocess.run([sys.executable, "-c", CHILD, str(libs), case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
