"""CPU-side checks of the C ABI: the library loads, exports every symbol the
header declares, validates arguments without touching a GPU, and its host-side
weight repack is byte-identical to the oracle's."""
import ctypes as C
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name", ["a81w41", "a81w41_model", "a81w41_dense"])
def test_exports_every_declared_symbol(pkg, name):
    L, signatures, also = {"a81w41": (pkg.capi.lib(), pkg.capi.SIGNATURES, set()),
                           "a81w41_model": (pkg.capi.core(), pkg.capi.CORE_SIGNATURES, {"a81w41_status_string", "a81w41_last_error"}),
                           "a81w41_dense": (pkg.capi.dense(), pkg.capi.DENSE_SIGNATURES, set())}[name]
    header = open(os.path.join(ROOT, "include", name + ".h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)   # declarations only, not prose
    declared = set(re.findall(r"\b(a81w41_[A-Za-z0-9_]+)\s*\(", header)) | also
    assert declared, "no declarations parsed"
    for symbol in sorted(declared):
        assert hasattr(L, symbol), f"library lacks {symbol}"
    assert declared == set(signatures), declared ^ set(signatures)


def test_blob_sizes(pkg):
    L = pkg.capi.lib()
    assert L.a81w41_weight_blob_bytes(4096, 4096, 0) == 32768 * 320
    assert L.a81w41_weight_blob_bytes(4096, 4096, 1) == 32768 * 384
    assert L.a81w41_act_blob_bytes(4096, 0) == 64 * 72
    assert L.a81w41_act_blob_bytes(322 * 4096, 1) == 20608 * 80
    assert L.a81w41_weight_blob_bytes(4095, 4096, 0) == 0   # K % 64 != 0
    assert L.a81w41_act_blob_bytes(100, 0) == 0


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("N,K", [(8, 64), (24, 320), (1024, 4096)])
def test_host_repack_matches_oracle(pkg, ora, synth, fp32, N, K):
    w4, scale, offset = synth.weight_files(N, K, seed=61)
    scale = scale * np.float32(1.2345)      # not fp16-representable: exercises the rounding
    got = pkg.ops.repack_w81_weight(K, N, scale, offset, w4, fp32)
    assert np.array_equal(got, ora.repack(w4, scale, offset, K, N, fp32))


def test_argument_errors(pkg):
    L = pkg.capi.lib()
    buf = np.zeros(4096, np.uint8)
    p = buf.ctypes.data_as(C.c_void_p)
    assert L.a81w41_repack_w81_weight_fp16(100, 8, 32, p, p, p, p) == 1
    assert b"K % 64" in L.a81w41_last_error()
    assert L.a81w41_repack_w81_weight_fp16(64, 8, 16, p, p, p, p) == 1
    assert L.a81w41_repack_w81_weight_fp32(64, 8, 32, None, p, p, p) == 1
    assert L.a81w41_quantize_row_q8_1_repack_fp16(p, p, 100, None) == 1
    assert L.a81w41_quantize_row_q8_1_repack_fp16(p, p, 0, None) == 0      # empty input is a no-op
    assert L.a81w41_gemv_repack_A81W41_fp16(p, p, p, 1, 12, 64, None) == 1  # N % 8
    assert L.a81w41_gemm_repack_A81W41_fp32(p, p, p, 0, 8, 64, None) == 1   # M < 1
    h = C.c_void_p()
    assert L.a81w41_context_create(0, 64, C.byref(h)) == 1
    assert L.a81w41_linear_forward(None, p, 1, p, None) == 1
    assert L.a81w41_status_string(1) == b"invalid argument"


def test_no_gpu_is_reported_not_faked(pkg):
    """Without a device the compute entry points must fail loudly (no CPU path)."""
    import torch

    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    L = pkg.capi.lib()
    buf = np.zeros(4096, np.uint8)
    p = buf.ctypes.data_as(C.c_void_p)
    assert L.a81w41_quantize_row_q8_1_repack_fp32(p, p, 64, None) == 4
    assert L.a81w41_gemv_repack_A81W41_fp16(p, p, p, 1, 8, 64, None) == 4


def test_gemm_schedule_covers_every_tile_and_chunk_once(pkg):
    """The work list of the 64 x 64-tile kernel (persistent grid, last round cut along K): walked on the host for
    the shapes and row counts the layer sees and for odd ones, on the real chip size and on smaller ones.
    Every tile and every K chunk exactly once, tile numbering one-to-one, no partial tile shared."""
    L = pkg.capi.lib()
    shapes = [(4096, 4096), (4096, 1024), (4096, 12288), (12288, 4096), (4096, 6144), (4096, 24576),
              (512, 256), (4096, 8), (256, 4104), (64, 64), (1024, 40)]
    rows = [9, 33, 64, 65, 128, 322, 512, 640, 832, 1024, 2048, 4096]
    used_split = 0
    for K, N in shapes:
        for M in rows:
            for resident, cus in ((1024, 256), (512, 256), (768, 256), (16, 4), (3, 3)):
                got = L.a81w41_gemm_schedule_selfcheck(M, N, K, resident, cus)
                assert got >= 0, (M, N, K, resident, cus, got)
                assert got <= 4096
                used_split += got > 0
    assert used_split > 20      # the K split really is exercised
    assert L.a81w41_gemm_schedule_selfcheck(0, 64, 64, 1024, 256) < 0   # argument errors are negative too


def test_gemm_schedule_follows_the_teams(pkg):
    """Few tiles go to teams of waves on a tile: the check walks their shares, from one super-block of K on, with K that no ring or
    part divides, and reports the partial tiles of that plan and not of the list that is not launched."""
    L = pkg.capi.lib()
    for K in (64, 128, 192, 256, 320, 704, 1408, 1472, 2048, 2112, 3712, 4096, 4160, 6144, 12288, 12352):
        for N in (8, 72, 1024, 2504, 4096, 12288):
            for M in (33, 40, 64, 65, 90, 120, 180, 250, 322):
                for cus in (256, 64, 4):
                    got = L.a81w41_gemm_schedule_selfcheck(M, N, K, 4 * cus, cus)
                    assert 0 <= got <= 4096, (M, N, K, cus, got)
    # 128 tiles: two parts of four teams, not the list's four; 64: four parts; 192 over 4608: none; K that is no multiple of 512: none
    for M, N, K, parts in ((128, 4096, 4096, 256), (57, 4096, 12288, 256), (192, 4096, 4608, 0), (40, 2504, 3712, 0)):
        assert L.a81w41_gemm_schedule_selfcheck(M, N, K, 1024, 256) == parts, (M, N, K)


# Which tiles of a launch are cut on 256 CUs, by parts (0: none).  T tiles of 64 x 64, K in super-blocks of 64.
@pytest.mark.parametrize("M,N,K,parts", [
    # up to two a CU: whole up to 16 super-blocks (T = 257, 427), halves of all beyond
    (33, 16392, 1024, 0), (420, 3904, 1024, 0), (420, 3904, 1536, 854),
    # up to two and a half (T = 640): whole up to 24, beyond two a CU and the other 128 in halves
    (640, 4096, 1536, 0), (640, 4096, 2048, 256), (600, 4096, 2560, 256),
    # up to three (T = 649, 767): whole below 192
    (641, 3720, 4096, 0), (641, 3720, 11776, 0), (641, 3720, 12288, 274), (830, 3776, 2048, 0),
    # a few more than three (T = 816, 845, 870): three a CU and the rest cut
    (709, 4304, 2048, 192), (780, 4104, 2048, 308), (780, 4104, 512, 154), (950, 3712, 1024, 408),
    # up to three and a half (T = 880, 882, 888, 891, 896): whole up to 16 only
    (868, 3976, 1024, 0), (350, 9464, 1024, 0), (529, 6304, 1536, 246), (691, 5120, 4608, 224), (868, 4096, 2560, 256), (868, 4096, 11264, 512),
    # up to four (T = 897, 912, 1024): whole below 192
    (830, 4416, 4096, 0), (1024, 3592, 11776, 0), (1024, 4096, 512, 0),
    # more: cut where the last round has few (126, 191 tiles), whole where it has more (146, 192), cut over long ranges: 192 in quarters, 256 in halves
    (1472, 3200, 512, 252), (1100, 4136, 512, 0), (960, 5184, 1024, 764), (1030, 4096, 1024, 256), (1160, 4096, 1024, 0), (1216, 4096, 4096, 768),
    (1280, 4096, 4096, 512)])
def test_gemm_schedule_cuts_what_it_should(pkg, M, N, K, parts):
    assert pkg.capi.lib().a81w41_gemm_schedule_selfcheck(M, N, K, 1024, 256) == parts


def test_gemm_schedule_of_a_layer_cuts_ranges_that_no_ring_divides(pkg):
    """Between one and two tiles a CU a layer object's launch is cut from 40 super-blocks on, in halves and from 192 on in quarters, with remainders
    of one to three; the check walks it and reports -8 if it was left whole."""
    L = pkg.capi.lib()
    for blocks in (41, 42, 43, 58, 61, 190, 191, 193, 194, 195, 209, 301):
        for cus in (256, 64):
            for M in (33, 70, 330, 1000, 2047):
                rows = -(-M // 64)
                for tiles in {cus // rows + 1, 3 * cus // (2 * rows), 2 * cus // rows}:
                    # 0: a call without a layer does not cut them
                    assert L.a81w41_gemm_schedule_selfcheck(M, 64 * tiles - 8, 64 * blocks, 4 * cus, cus) == 0, (M, tiles, blocks, cus)


def test_block_scaled_gemm_plan_covers_every_unit_once(pkg):
    """The layer object's M > 32 kernel cuts the (tile, 32-block) units of a launch into equal contiguous runs:
    walked on the host for the layer's shapes and odd ones, for several device sizes."""
    L = pkg.capi.lib()
    shapes = [(4096, 4096), (4096, 1024), (4096, 12288), (12288, 4096), (4096, 6144), (4096, 24576), (4096, 151936),
              (512, 256), (4096, 8), (256, 4104), (64, 64), (1024, 40)]
    shared = 0
    for K, N in shapes:
        for M in (33, 64, 65, 128, 129, 322, 512, 640, 1024, 2048, 4096):
            for slots in (512, 256, 8, 3, 1):
                got = L.a81w41_gemm_fp6_plan_selfcheck(M, N, K, slots)
                assert got >= 0, (M, N, K, slots, got)
                shared += got > 0
    assert shared > 50
    assert L.a81w41_gemm_fp6_plan_selfcheck(0, 64, 64, 512) < 0


@pytest.mark.parametrize("room", [0, 5000, 1 << 20, 20 << 20, 1 << 40])
def test_weights_read_ahead_stay_in_the_matrix(pkg, room):
    """A one-token pass reads weights of later launches beside its attention: inside the matrix and within the room given, and all of
    what a launch reads first where there is room for it."""
    L = pkg.capi.lib()
    end = C.c_longlong()
    for K, N in [(4096, 4096), (4096, 24576), (64, 64), (64, 8), (512, 256), (12288, 4096), (1024, 40), (4096, 1088), (1536, 192), (192, 151936)]:
        for gate_up in (0, 1):
            got = L.a81w41_gemv_ahead_selfcheck(N, K, gate_up, room, C.byref(end))
            assert 0 <= got <= room and got <= end.value <= N // 8 * (K // 64) * 320, (K, N, gate_up)
            if room == 1 << 40 and N % 64 == 0:
                assert got == N // 8 * (K // 64) * 320, (K, N, gate_up)
    D = pkg.capi.dense()
    for ld, rows in [(2048, 2048), (64, 1), (64, 300), (768, 3072), (1024, 17), (6144, 2048), (2048, 40), (576, 255)]:
        for bf16 in (0, 1):
            for gate_up in (0, 1):
                got = D.a81w41_dense_ahead_selfcheck(rows, ld, gate_up, room, bf16, C.byref(end))
                whole = (32 * ((rows + 15) // 16) if gate_up else rows) * ld * (2 if bf16 else 4)
                assert 0 <= got <= room and got <= end.value and end.value <= whole, (ld, rows, bf16, gate_up)
                if room == 1 << 40 and rows % 512 == 0:
                    assert got == whole
    assert L.a81w41_gemv_ahead_selfcheck(7, 64, 0, 0, C.byref(end)) < 0
    # gate and up whose output is no product in one launch (sizes that are no multiple of 64, rows too long for its prologue): the plain launch's
    for N, K in [(80, 64), (2 * 3112, 1024), (2 * 1000, 4096), (8192, 65536)]:
        plain, paired = ((L.a81w41_gemv_ahead_selfcheck(N, K, gate_up, room, C.byref(end)), end.value) for gate_up in (0, 1))
        assert plain == paired, (N, K)


def test_strides_past_32_bit_offsets_have_a_kernel(pkg):
    """Tiles up to 256 rows copy by 32-bit offsets; strides with which a tile's rows reach 4 GB go to the kernel with 64-bit ones."""
    form = pkg.capi.dense().a81w41_dense_form_selfcheck
    for bf16, step, size in ((0, 32, 4), (1, 64, 2)):
        for rows in (1, 65, 256, 4000):
            last = ((1 << 32) // size // min(rows, 256) - 1) // step * step   # the widest stride whose rows end before 4 GB
            last = min(last, (1 << 31) - step)                              # strides are ints
            for more, far in ((0, False), (step, min(rows, 256) * (last + step) * size >= 1 << 32)):
                if last + more < 1 << 31:
                    assert (form(rows, 8, step, last + more, step, bf16) == 7) == far, (bf16, rows, more)
                    assert (form(8, rows, step, step, last + more, bf16) == 7) == far, (bf16, rows, more)
    assert form(1, 1, 64, 100, 64, 1) < 0
