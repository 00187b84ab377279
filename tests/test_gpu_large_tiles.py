"""The large bf16 and int8 tiles of k_pp.hip: every tile shape at its edges
(ragged rows and columns, one k-block, odd and even block counts, a k tail
inside a block, k-splits, padded strides whose padding holds NaN), and the
calls that must keep other kernels.  bf16 within the fp32 bound of _util.py
against the fp64 product of the operands, int8 bit-exact."""

import numpy as np
import pytest

import _util as u

torch = pytest.importorskip("torch")

TILES = [(256, 256), (256, 192), (256, 128), (128, 128), (128, 256), (128, 192), (256, 64)]
BF16_FIRST, S8_FIRST = 51, 30  # TILE_CFG / S8_CFG of TILES[0]


def dev_copy(x, device):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def stream():
    return torch.cuda.current_stream().cuda_stream


# M, N, K, pad of A's and B's rows, splits, alpha, beta
SHAPES = [(9, 2, 8, 0, 1, 1.0, 0.0), (255, 257, 64, 2, 1, 0.5, 1.0), (257, 130, 200, 4, 1, 1.0, 0.0),
          (300, 515, 72, 0, 2, -2.0, 0.25), (128, 63, 320, 2, 3, 1.0, 1.0), (511, 449, 136, 6, 1, 1.0, 0.0)]


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("tb", [0, 1])
def test_bf16_tiles(lib, orc, dev, tile, tb):
    for M, N, K, pad, splits, alpha, beta in SHAPES:
        lda, ldb = K + pad, (K + pad if tb else N + N % 2 + pad)
        A = u.bf16_bits(orc, u.normal(orc, M * K, 1)).reshape(M, K)
        B = u.bf16_bits(orc, u.normal(orc, N * K, 2, 0, 0.02)).reshape((N, K) if tb else (K, N))
        C0 = u.uniform(orc, M * N, 3).reshape(M, N)
        sa, sb = np.full((M, lda), 0x7FC0, np.uint16), np.full((B.shape[0], ldb), 0x7FC0, np.uint16)
        sa[:, :K], sb[:, :B.shape[1]] = A, B
        want, scale = u.exact(u.bf16_value(A), u.bf16_value(np.ascontiguousarray(B.T if tb else B)), alpha, beta, C0)
        dA, dB = dev_copy(sa.view(np.int16), dev), dev_copy(sb.view(np.int16), dev)
        got = []
        for _ in range(2):
            dC = dev_copy(C0 if beta else np.full_like(C0, np.nan), dev)
            with lib.tunables(TILE_CFG=BF16_FIRST + tile, TILE_SPLITS=splits):
                p = lib.plan_bf16_ex(M, N, K, transB=tb)
                # (the plan query has packed strides: odd rows of a K x N B are not on 4-byte boundaries)
                assert (N % 2 and not tb) or (p["rows"], p["cols"], p["block"]) == (*TILES[tile], 512), p
                lib.gemm_bf16_ex(M, N, K, alpha, dA, lda, dB, ldb, beta, dC, N, transB=tb, stream=stream())
            got.append(host(dC))
        u.assert_fp32_close(got[0], want, scale, K, f"{TILES[tile]} tb={tb} {M}x{N}x{K} splits={splits}")
        u.assert_bits_equal(got[0], got[1], "repeated call")


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("scaled", [0, 1])
def test_s8_tiles(lib, orc, dev, tile, scaled):
    for M, N, K, pad, splits, _, _ in SHAPES:
        K = 16 * ((K + 15) // 16) * (2 if K > 64 else 1)  # up to several blocks of 128
        ld = K + 4 * pad
        A, B = u.ints8(orc, M * K, 1).reshape(M, K), u.ints8(orc, N * K, 2).reshape(N, K)
        sa, sb = np.full((M, ld), 77, np.int8), np.full((N, ld), 77, np.int8)
        sa[:, :K], sb[:, :K] = A, B
        acc = A.astype(np.int64) @ B.astype(np.int64).T
        scale = u.uniform(orc, N, 4, 1e-3, 2e-3)
        dA, dB = dev_copy(sa, dev), dev_copy(sb, dev)
        with lib.tunables(S8_CFG=S8_FIRST + tile, S8_SPLITS=splits):
            p = lib.plan_s8(M, N, K, with_scale=scaled)
            assert (p["rows"], p["cols"], p["block"]) == (*TILES[tile], 512), p
            if scaled:
                dC = torch.full((M, N), float("nan"), device=dev)
                lib.gemm_s8s8f32_colscale(M, N, K, dA, ld, dB, ld, dev_copy(scale, dev), dC, N, stream=stream())
                u.assert_bits_equal(host(dC), acc.astype(np.float32) * scale, f"{TILES[tile]} {M}x{N}x{K}")
            else:
                dC = torch.full((M, N), -1, dtype=torch.int32, device=dev)
                lib.gemm_s8s8s32(M, N, K, dA, ld, dB, ld, dC, N, stream=stream())
                assert np.array_equal(host(dC), acc.astype(np.int32)), (TILES[tile], M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_s8_tiles_dynamic_scale(lib, orc, dev, tile):
    """The dequantizing epilogue of the fp32-input int8 GEMM on these tiles
    (quantized copies of both operands): the oracle's bits."""
    for M, N, K, _, splits, _, _ in SHAPES:
        M, K = max(M, 9), 16 * ((K + 15) // 16) * (2 if K > 64 else 1)
        A, B, C0 = u.uniform(orc, M * K, 1), u.uniform(orc, K * N, 2), u.uniform(orc, M * N, 3)
        for beta in (0.0, 0.5):
            want = C0.copy()
            orc.orc_gemm_int8(M, N, K, 0.75, u.ptr(A), K, u.ptr(B), N, beta, u.ptr(want), N)
            dC = dev_copy(C0 if beta else np.full_like(C0, np.nan), dev)
            with lib.tunables(Q8B=0, S8_CFG=S8_FIRST + tile, S8_SPLITS=splits):
                p = lib.plan_s8(M, N, K, with_scale=1)
                assert (p["rows"], p["cols"], p["block"]) == (*TILES[tile], 512), p
                lib.gemm_int8_f32(M, N, K, 0.75, dev_copy(A, dev), K, dev_copy(B, dev), N, beta, dC, N, stream=stream())
            u.assert_bits_equal(host(dC), want, f"{TILES[tile]} {M}x{N}x{K} beta={beta}")


def test_planned_by_size_and_k_alignment(lib):
    """Many-row shapes take the large tiles (bf16 2048 x 11008 x 4096 225 ->
    171 us, int8 1024 x 11008 x 4096 100 -> 49 us on MI355X); a K off whole
    16-byte chunks, and a forced choice of them there, keep the other tiles."""
    large = set(TILES)
    for tb in (0, 1):
        p = lib.plan_bf16_ex(2048, 11008, 4096, transB=tb)
        assert (p["rows"], p["cols"], p["block"]) in {(*t, 512) for t in large}, p
        for cfg in (0, BF16_FIRST):
            with lib.tunables(TILE_CFG=cfg):
                p = lib.plan_bf16_ex(2048, 11008, 4100, transB=tb)
                assert (p["rows"], p["cols"], p["block"]) not in {(256, 256, 512), (256, 192, 512), (256, 128, 512)}, p
    p = lib.plan_s8(1024, 11008, 4096)
    assert (p["rows"], p["cols"]) in large, p
    for cfg in (-1, S8_FIRST):
        with lib.tunables(S8_CFG=cfg):
            p = lib.plan_s8(1024, 11008, 4104)
            assert (p["rows"], p["cols"]) not in large, p


def test_plans_name_the_kernel(lib):
    """A plan's name is the kernel's, not that of the kernel it stands in for."""
    assert lib.plan_bf16_ex(2048, 11008, 4096, transB=1)["name"] == "dnnopt_tile_bf16_dma_pp"
    assert lib.plan_bf16_copies(1024, 11008, 4096)["name"] == "dnnopt_tile_bf16_dma_pp"
    assert lib.plan_s8(1024, 11008, 4096)["name"] == "dnnopt_s8_dma_pp"
    with lib.tunables(TILE_CFG=33, S8_CFG=29):
        assert lib.plan_bf16_ex(2048, 11008, 4096, transB=1)["name"] == "dnnopt_tile_bf16_dma"
        assert lib.plan_s8(1024, 11008, 4096)["name"] == "dnnopt_s8_dma"


@pytest.mark.parametrize("M,N,K", [(4096, 4096, 8400000), (2048, 1024, 8400000), (1024, 1024, 17000000),
                                   (256, 64, 8388608), (2048, 4096, 16777200), (128, 128, 16777216)])
def test_int8_long_rows_keep_tiles(lib, M, N, K):
    """Tiles of 128 and 256 rows cannot reach rows of 8.4 M or 16.8 M bytes with
    32-bit offsets; the lower int8 tiles can, and such a call stays on tiles,
    also when a large tile is forced."""
    b = u.binding()
    for cfg in (-1, S8_FIRST):
        with lib.tunables(S8_CFG=cfg):
            p = lib.plan_s8(M, N, K)
            assert p["kernel"] == b.K_MFMA_S8, p
            assert p["rows"] * K + K < 2**31 - 1 and p["cols"] * K + K < 2**31 - 1, p


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "s8"])
def test_wide_c_stride_keeps_other_tiles(lib, orc, dev, kind):
    """256 rows of C that span 2^31 bytes or more (ldc = 2^21) are past the
    large tiles' 32-bit offsets: the call takes other tiles, also when one is
    forced, and writes nothing between C's rows."""
    M, N, K, ldc = 300, 512, 256, 1 << 21
    dC = torch.full(((M - 1) * ldc + N,), -7, dtype=torch.float32 if kind == "bf16" else torch.int32, device=dev)
    if kind == "bf16":
        A, B = u.bf16_bits(orc, u.normal(orc, M * K, 1)).reshape(M, K), u.bf16_bits(orc, u.normal(orc, N * K, 2)).reshape(N, K)
        with lib.tunables(TILE_CFG=BF16_FIRST):
            lib.gemm_bf16_ex(M, N, K, 1.0, dev_copy(A.view(np.int16), dev), K, dev_copy(B.view(np.int16), dev), K, 0.0, dC,
                             ldc, transB=1, stream=stream())
        want, scale = u.exact(u.bf16_value(A), u.bf16_value(np.ascontiguousarray(B.T)))
        u.assert_fp32_close(host(torch.as_strided(dC, (M, N), (ldc, 1))), want, scale, K, "ldc 2^21")
    else:
        A, B = u.ints8(orc, M * K, 1).reshape(M, K), u.ints8(orc, N * K, 2).reshape(N, K)
        with lib.tunables(S8_CFG=S8_FIRST):
            lib.gemm_s8s8s32(M, N, K, dev_copy(A, dev), K, dev_copy(B, dev), K, dC, ldc, stream=stream())
        want = A.astype(np.int64) @ B.astype(np.int64).T
        assert np.array_equal(host(torch.as_strided(dC, (M, N), (ldc, 1))), want)
    assert bool((torch.as_strided(dC, (M - 1, ldc - N), (ldc, 1), N) == -7).all())
