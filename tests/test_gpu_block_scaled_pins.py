"""Three pins of the block-scaled (fp6 matrix op) kernel that its fp32 outputs on zero-mean activations do not give.

1. Its block dots are the reference's integers (quantized_gemx_kernels.cc:430-457,509: int32 dot, then
   cvtepi32_ps).  The kernel never holds them as integers, so they are made visible: weight scale 1, min 0,
   activation blocks with d = 1 and exactly one live 32-block per row -- then C[m][n] IS float(idot) and must
   equal the oracle's block dot bit for bit, over the whole int8 range incl. the extremes 15 x -127 x 32 =
   -60 960 and q = -128 (high piece -8), with ragged M and N.
2. Its min terms fma(mW, sA, acc) (quantized_gemx_kernels.cc:509-512) run on bf16 pieces (three for the
   scaled sum, two for the min).  With zero-mean weights (min = -7.5 scale) and rows that are not zero-mean the min
   term is far larger than the result it cancels down to; the error must stay inside the path's 1e-4 bar
   with room to spare.
3. The order of its sums: a product's K slot in the min terms' matrix op decides how they are rounded (2e-7 of a call), and a prompt
   whose rows are rounded to 8 bits ahead of every linear makes 1e-2 of that.  A call's bits are held."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blocks80(q: np.ndarray, d: np.ndarray) -> np.ndarray:
    """Hand-made q8_repack_1x2_fp32 rows: q int8 [M][K], d fp32 [M][K/32]; scaled sum = d * sum(q) in fp32."""
    M, K = q.shape
    blob = np.zeros((M, K // 64, 80), np.uint8)
    par = np.zeros((M, K // 64, 4), np.float32)
    d2 = d.reshape(M, K // 64, 2)
    sums = q.reshape(M, K // 64, 2, 32).astype(np.int32).sum(axis=3).astype(np.float32)
    par[:, :, 0:2] = d2
    par[:, :, 2:4] = d2 * sums
    blob[:, :, :16] = par.view(np.uint8).reshape(M, K // 64, 16)
    blob[:, :, 16:] = q.reshape(M, K // 64, 64).view(np.uint8)
    return blob.reshape(-1)


@pytest.mark.parametrize("M,N,K", [(37, 40, 256), (130, 264, 512), (322, 512, 1024)])
def test_block_dots_are_the_reference_integers(pkg, ora, synth, M, N, K):
    import torch

    rng = np.random.default_rng(900 + M)
    nb = K // 32
    codes = rng.integers(0, 16, size=(N, K), dtype=np.uint8)
    codes[1, :] = 15                               # the largest code everywhere
    codes[2, :] = 0
    w4 = (codes.reshape(N, K // 64, 2, 32)[:, :, 0, :] | (codes.reshape(N, K // 64, 2, 32)[:, :, 1, :] << 4)).reshape(N, K // 2)
    scale = np.ones((N, nb), np.float32)
    offset = np.zeros((N, nb), np.float32)
    q = np.zeros((M, K), np.int8)
    d = np.zeros((M, nb), np.float32)
    live = rng.integers(0, nb, size=M)
    for m in range(M):
        b = live[m]
        row = rng.integers(-128, 128, size=32).astype(np.int8)
        if m == 0:
            row[:] = -127                          # 15 * -127 * 32 = -60 960 against column 1
        elif m == 1:
            row[:] = -128                          # the corner x86's out-of-range conversion produces: high piece -8
        elif m == 2:
            row[:] = 127
        elif m == 3:
            row[:] = np.where(np.arange(32) % 2 == 0, -128, 127)
        q[m, 32 * b:32 * b + 32] = row
        d[m, b] = 1.0
    blob = _blocks80(q, d)
    b32 = ora.repack(w4, scale, offset, K, N, True)
    ctx = pkg.ops.Context(max_rows=M, max_cols=K)
    layer = pkg.Linear.from_blobs(None, b32, N, K, ctx)
    idot = ora.block_idot(blob, True, b32, True, M, N, K)                  # [M][N][K/32] int32
    want = idot[np.arange(M), :, live].astype(np.float32)                  # the live block of each row
    assert want[0, 1] == -60960.0 and want[1, 1] == -61440.0
    assert np.array_equal(ora.gemm_fp32(blob, b32, M, N, K), want)         # the oracle's GEMM says the same
    a_dev = torch.from_numpy(blob).cuda()
    for kernel in ("block_scaled", "int8"):
        layer.set_kernel(kernel)
        got = layer.forward_quantized(a_dev, M).cpu().numpy()
        assert np.array_equal(got, want), kernel


@pytest.mark.parametrize("name,N,K", [("gate", 12288, 4096), ("down", 4096, 12288)])
@pytest.mark.parametrize("rows", ["abs_normal", "constant_plus_noise"])
def test_min_terms_with_zero_mean_weights_and_biased_rows(pkg, ora, synth, name, N, K, rows):
    import torch

    M = 322
    w4, scale, _ = synth.weight_files(N, K, 930)
    offset = (np.float32(-7.5) * scale).astype(np.float32)     # codes 0..15 around 7.5: zero-mean weights
    x = synth.activations(M, K, 931)
    x = np.abs(x) if rows == "abs_normal" else (np.float32(3.0) + np.float32(0.25) * x)
    b16, b32 = ora.repack(w4, scale, offset, K, N, False), ora.repack(w4, scale, offset, K, N, True)
    want = ora.linear_forward_fast(x, b16, b32, N)
    ctx = pkg.ops.Context(max_rows=M, max_cols=K)
    layer = pkg.Linear.from_blobs(None, b32, N, K, ctx)
    xd = torch.from_numpy(x).cuda()
    errs = {}
    for kernel in ("block_scaled", "int8"):
        layer.set_kernel(kernel)
        got = layer.forward(xd).cpu().numpy()
        errs[kernel] = float(np.max(np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)))
    # how much larger the min term is than what is left of it: the cancellation the pieces' precision has to survive
    blob = ora.quantize(x, True).reshape(M, K // 64, 80)
    s_a = blob[:, :, 8:16].copy().view(np.float32).reshape(M, K // 32).astype(np.float64)
    min_term = s_a[:8] @ offset.astype(np.float64).T
    ratio = float(np.median(np.linalg.norm(min_term, axis=1) / np.linalg.norm(want[:8], axis=1)))
    print(f"\n[{name}, {rows}: min term = {ratio:.0f} x result; max row error block-scaled {errs['block_scaled']:.2e}, "
          f"int8 {errs['int8']:.2e}]")
    assert errs["int8"] <= 1e-5
    assert errs["block_scaled"] <= 4e-5          # the path's bar is 1e-4: a factor 2.5 in hand (observed 2.0e-5 .. 2.6e-5)


# Of sums on 256 CUs (the cut of the work into runs goes by them).  Runs of one to four blocks past a multiple of four and of many, tiles of one run
# and of several, one panel and ragged ones.
@pytest.mark.parametrize("M,N,K,bits", [(33, 8, 64, 1823667629), (130, 136, 448, 2408502087), (65, 1000, 2048, 2921864782),
                                        (100, 512, 12288, 529302396), (322, 1024, 4096, 2724076504)])
def test_sums_keep_their_order(pkg, synth, M, N, K, bits):
    import torch

    w4, scale, _ = synth.weight_files(N, K, M + N)
    layer = pkg.Linear.from_arrays(w4, scale * np.float32(1.0371), np.float32(-7.3) * scale, N=N, K=K)
    layer.set_kernel("block_scaled")
    x = torch.from_numpy(np.float32(0.5) + synth.activations(M, K, K + 1)).cuda()
    assert zlib.crc32(layer.forward(x).cpu().numpy().tobytes()) == bits
