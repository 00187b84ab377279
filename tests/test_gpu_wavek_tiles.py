"""fp32 tiles whose waves split k (k_wavek.hip): every tile shape and both
layouts of B at its edges -- ragged rows and columns, one k-block, a number of
blocks that is and is not a multiple of the ring's four stages, a k tail inside
a wave's 16 k and inside a 16-byte chunk, k-splits, padded strides whose padding
holds NaN, beta and the hook's bias -- within the fp32 bound of _util.py."""

import numpy as np
import pytest

import _util as u

torch = pytest.importorskip("torch")

TILES = [(96, 48), (64, 64), (64, 48), (48, 48), (64, 32), (32, 48), (32, 64)]
FIRST = 58  # TILE_CFG of TILES[0]


def dev_copy(x, device):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def stream():
    return torch.cuda.current_stream().cuda_stream


# M, N, K, pad, splits, alpha, beta
SHAPES = [(33, 65, 1, 0, 1, 1.0, 0.0), (97, 70, 64, 1, 1, 0.5, 1.0), (64, 130, 250, 3, 1, 1.0, 0.0),
          (100, 97, 321, 2, 1, -2.0, 0.25), (50, 67, 515, 0, 3, 1.0, 1.0), (200, 64, 1024, 4, 2, 1.0, 0.0),
          (34, 193, 83, 1, 1, 1.0, 1.0)]


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("tb", [0, 1])
def test_tiles(lib, orc, dev, tile, tb):
    for M, N, K, pad, splits, alpha, beta in SHAPES:
        A = u.normal(orc, M * K, 1).reshape(M, K)
        B = u.normal(orc, N * K, 2).reshape((N, K) if tb else (K, N))
        sa, sb = np.full((M, K + pad), np.nan, np.float32), np.full((B.shape[0], B.shape[1] + pad), np.nan, np.float32)
        sa[:, :K], sb[:, :B.shape[1]] = A, B
        C0 = u.uniform(orc, M * N, 3).reshape(M, N)
        want, scale = u.exact(A, np.ascontiguousarray(B.T if tb else B), alpha, beta, C0)
        got = []
        for _ in range(2):
            dC = dev_copy(C0 if beta else np.full_like(C0, np.nan), dev)
            with lib.tunables(TILE_CFG=FIRST + tile, TILE_SPLITS=splits):
                p = lib.plan_sgemm(M, N, K, transB=tb)
                assert (p["rows"], p["cols"], p["block"]) == (*TILES[tile], 256), p
                lib.sgemm(M, N, K, alpha, dev_copy(sa, dev), K + pad, dev_copy(sb, dev), B.shape[1] + pad, beta, dC, N,
                          transB=tb, stream=stream())
            got.append(host(dC))
        u.assert_fp32_close(got[0], want, scale, K, f"{TILES[tile]} tb={tb} {M}x{N}x{K} splits={splits}")
        u.assert_bits_equal(got[0], got[1], "repeated call")


@pytest.mark.gpu
def test_hook_bias_is_its_own_rounding(lib, orc, dev):
    """The bias is added to the finished output as a separate rounding (alpha =
    1/3 with exact integer sums), on the plan of 384 x 3072 x 768."""
    M, N, K = 384, 3072, 768
    p = lib.plan_sgemm(M, N, K, transB=1)
    assert (p["rows"], p["cols"], p["block"]) in {(*t, 256) for t in TILES}, p
    A, B = u.small_ints(orc, M * K, 1).reshape(M, K), u.small_ints(orc, N * K, 2).reshape(N, K)
    bias = u.uniform(orc, N, 4)
    dC = torch.full((M, N), float("nan"), device=dev)
    lib.ext_sgemm("T", "N", N, M, K, 1 / 3, dev_copy(B, dev), K, dev_copy(A, dev), K, 0.0, dC, N, bias=dev_copy(bias, dev),
                  stream=stream())
    acc = (A.astype(np.float64) @ B.T.astype(np.float64)).astype(np.float32)
    u.assert_bits_equal(host(dC), np.float32(1 / 3) * acc + bias, "bias")


def test_planned_where_they_balance(lib):
    """384 x 3072: 256 equal 96 x 48 tiles (20.6 us against 23.9 on MI355X); up
    to 32 rows, a stored K x M A and K x N weights from 4096 rows keep other
    tiles."""
    p = lib.plan_sgemm(384, 3072, 768, transB=1)
    assert (p["rows"], p["cols"], p["grid_x"], p["splits"]) == (96, 48, 256, 1), p
    for args, kw in (((32, 3072, 768), {"transB": 1}), ((384, 3072, 768), {"transA": 1}), ((384, 3072, 4096), {})):
        p = lib.plan_sgemm(*args, **kw)
        assert (p["rows"], p["cols"], p["block"]) not in {(*t, 256) for t in TILES if t != (64, 64)}, p
