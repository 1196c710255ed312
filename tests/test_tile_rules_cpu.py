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


# (rows of the weight, token rows, K, a tile within a tenth of the fastest of the five as timed; the last: fewer than 256 tokens take no 256-token tile)
PICKED = [(6144, 515, 1024, "DUO"), (6144, 1030, 1024, "HALF"), (6144, 2047, 1024, "WIDE"), (6144, 2608, 1024, "SMALL"), (12288, 515, 2048, "SMALL"), (12288, 1030, 2048, "BIG"), (12288, 6000, 2048, "WIDE"),
          (24576, 700, 5120, "WIDE"), (24576, 2047, 5120, "BIG"), (2048, 2608, 6144, "HALF"), (5120, 2608, 8192, "BIG"), (1600, 8192, 1600, "BIG"), (6400, 8192, 1600, "BIG"), (151936, 200, 1024, "SMALL")]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_one_round_of_tiles_is_taken_where_there_is_one(tmp_path):
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm3_tile.h"\n' % B.CSRC + "".join("static_assert(kf::g3_pick(%d, %d, %d, true) == kf::G3_%s);\n" % (m, n, k, t) for m, n, k, t in PICKED))
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]


# (rows, token rows, either operand k-major or one, the tile): as timed, and at the edges of the rule
KM_PICKED = [(1600, 6400, True, "SLIM"), (6400, 1600, True, "FLAT"), (4096, 2560, True, "FLAT"), (3000, 3000, True, "FLAT"), (1600, 5120, False, "SLIM"), (6400, 3000, False, "SLIM"), (2048, 5120, False, "FLAT"),
             (1600, 8192, False, "BIG"), (6400, 8192, False, "BIG"), (4800, 5120, False, "BIG"), (2048, 4096, True, "BIG"), (2049, 4096, True, "FLAT"), (1608, 6400, True, "BIG")]

# the same with K: up to the longest that was timed
KM_PICKED_LONG = [(1600, 6400, 8192, True, "SLIM"), (4096, 2560, 8256, True, "BIG"), (3000, 3000, 16384, True, "BIG"), (1600, 5120, 8192, False, "SLIM"), (1600, 5120, 50304, False, "BIG"), (6400, 3000, 8256, False, "BIG")]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_tiles_of_160_are_taken_where_they_need_no_more_rounds(tmp_path):
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm3_tile.h"\n' % B.CSRC + "".join("static_assert(kf::g3_km_pick(%d, %d, 1600, %s, %d, %d) == kf::G3_%s);\n" % (m, n, str(b).lower(), m, n if b else 0, t) for m, n, b, t in KM_PICKED)
                   + "".join("static_assert(kf::g3_km_pick(%d, %d, %d, %s, %d, %d) == kf::G3_%s);\n" % (m, n, k, str(b).lower(), m, n if b else 0, t) for m, n, k, b, t in KM_PICKED_LONG))
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]


# (rows of the image, the longest k-row in reach): the last byte that a base's scalar and lane offsets name lies below the descriptor's end, with eight values more it does not
KM_REACH = [(128, 2 ** 26 - 8), (160, 2 ** 24 - 8), (256, 2 ** 27 - 8)]


def _last_byte(rows, ld):
    """of the loads that share a base, as g3_src_km deals them: chunk by chunk along the k-rows, 64 lanes an instruction, eight waves of 160 rows (20 instructions), else four instructions a wave"""
    chunks, end = rows // 8, 0
    for i in range(20 if rows == 160 else 4):
        scalar = (i // 5) * 16 if rows == 160 else i * (64 // chunks)
        for lane in range(64):
            kr = ((i % 5) * 64 + lane) // chunks if rows == 160 else lane // chunks
            assert scalar + kr == (i * 64 + lane) // chunks
            end = max(end, scalar * 2 * ld + kr * 2 * ld + (ld - 8) * 2 + 16)
    return end


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_k_rows_are_in_reach_of_the_offsets_of_their_tile(tmp_path):
    """and a longer row than the 160-row tiles reach takes the big tiles: transposed it would be a product that the other kernels refuse (2^24 x 2048: 2^32 pieces of eight)"""
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm3_tile.h"\n' % B.CSRC + "".join("static_assert(kf::g3_km_reach<%d>(%d) && !kf::g3_km_reach<%d>(%d));\n" % (r, ld, r, ld + 8) for r, ld in KM_REACH)
                   + "static_assert(kf::g3_km_pick(1600, 6400, 1600, true, 1600, 6400) == kf::G3_SLIM && kf::g3_km_pick(1600, 6400, 1600, true, 1 << 24, 6400) == kf::G3_BIG && kf::g3_km_pick(6400, 1600, 1600, true, 6400, 1 << 24) == kf::G3_BIG);\n"
                   + "static_assert(kf::g3_km_pick(1 << 24, 300, 1600, true, 1 << 24, 300) == kf::G3_FLAT);\n")
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    for rows, ld in KM_REACH:
        assert _last_byte(rows, ld) <= 0x7FFFFFF0 < _last_byte(rows, ld + 8)


# (big tiles of the launch, K, us cut in owners and tails, us whole)
TAILS = [(150, 2048, 63.6, 52.0), (150, 2048, 64.4, 53.1), (175, 2560, 80.1, 61.9), (144, 4096, 95.3, 90.0), (144, 4096, 88.6, 88.3), (160, 4096, 94.6, 90.8), (160, 4096, 93.3, 92.3), (140, 6400, 112.1, 119.1),
         (160, 8192, 154.7, 167.7), (160, 8192, 149.6, 161.1), (175, 8192, 167.0, 166.2)]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_tails_of_big_tiles_are_cut_off_where_that_was_the_faster(tmp_path):
    """within 1.5 %, what two runs of one side differ by"""
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm3_tile.h"\nstatic_assert(kf::g3_tails_from(128) == 2048 / 64);\n' % B.CSRC
                   + "static_assert(kf::g3_km_pick(1608, 6400, 4160, true, 1608, 6400) == kf::G3_BIG && 4160 / 64 >= kf::g3_tails_from(256));\n"   # the GPU test of repeated runs has this shape for its tails
                   + "".join("static_assert(%d / 64 %s kf::g3_tails_from(256));\n" % (k, ">=" if cut < whole else "<") for _, k, cut, whole in TAILS if abs(cut - whole) > 0.015 * whole))
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]


# (storage, matrices in the launch, token rows, blocks of 32 weight rows, 64 token rows a workgroup): 4 bits as timed in prompts; the others, whose rounds were not timed, only several matrices from 256 such workgroups on
WIDE = [("Q4", 1, 128, 96, True), ("Q4", 1, 256, 96, False), ("Q4", 1, 256, 64, True), ("Q4", 3, 64, 256, True), ("Q4", 1, 32, 1280, False), ("Q4", 1, 33, 132, True), ("Q4", 1, 64, 132, True), ("Q4", 1, 64, 128, False), ("Q4", 1, 64, 288, False)] + \
       [(f, *c) for f in ("BF16", "F8", "Q4R", "Q2", "Q1") for c in ((1, 64, 132, False), (1, 256, 160, False), (3, 192, 128, True), (3, 64, 256, True), (3, 63, 512, False), (2, 64, 255, False))]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_64_token_rows_a_workgroup_where_that_was_timed(tmp_path):
    src = tmp_path / "rules.hip"
    src.write_text('#include "%s/kf_gemm.hip"\n' % B.CSRC + "".join("static_assert(kf::gd_wide(kf::FMT_%s, %d, %d, %d) == %s);\n" % (f, j, n, rb, str(w).lower()) for f, j, n, rb, w in WIDE))
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]


# (pieces of 8 weights, matrices interleaved, offsets of the copy in 32 bits): gate and up of 65552 x 16384 lie in 4 296 015 872 bytes
REACH = [(65552 * 16384 // 8, 1, True), (65552 * 16384 // 8, 2, False), (65536 * 16384 // 8 - 1, 2, True), ((1 << 28) - 1, 1, True), (1 << 28, 1, False), ((1 << 31) - 1, 2, False)]


@pytest.mark.skipif(not shutil.which(B.HIPCC), reason="no hipcc")
def test_offsets_of_dequantised_copies_are_bounded_where_they_end(tmp_path):
    src = tmp_path / "reach.hip"
    src.write_text('#include "%s/kf_kernels.h"\n' % B.CSRC + "".join("static_assert(kf::deq4_in_reach(%dull, %d) == %s && kf::deq4_counted(%dull, %d));\n" % (n, i, "true" if r else "false", n, i) for n, i, r in REACH)
                   + "static_assert(!kf::deq4_counted(1ull << 31, 1) && !kf::deq4_counted(0x7FFFFFFFull, 3));\n")
    r = subprocess.run([B.HIPCC, "--cuda-host-only", "-fsyntax-only", "-std=c++17", "-w", str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
