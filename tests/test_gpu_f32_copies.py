"""The fp32-input bf16 GEMM on operands rounded ahead into workspace: A alone,
or both (many rows), against the fp64 product of the bf16-rounded operands;
ragged sizes, padded strides with NaN in the padding, beta, rounding ties and
special values; calls under graph capture, which keep to the direct tiles."""

import numpy as np
import pytest

import _util as u

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev_copy(x, device):
    return torch.from_numpy(np.ascontiguousarray(x)).to(device)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def stream():
    return torch.cuda.current_stream().cuda_stream


# The models round A alone on some of these (tests/test_copies_routes.py says which),
# the others keep the tiles that round while staging.
SHAPES = [(200, 9000, 1000, 0, 1.0, 0.0), (380, 10007, 777, 3, 0.5, 1.0), (513, 2500, 1501, 1, -2.0, 0.25),
          (1024, 4100, 520, 2, 1.0, 0.0), (1030, 2049, 1003, 5, 1.0, 1.0), (300, 500, 129, 1, 1.0, 0.0),
          (65, 130, 64, 0, 1.0, 1.0)]


@pytest.mark.parametrize("M,N,K,pad,alpha,beta", SHAPES)
def test_against_rounded_operands(lib, orc, dev, M, N, K, pad, alpha, beta):
    A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
    sa, sb = np.full((M, K + pad), np.nan, np.float32), np.full((K, N + pad), np.nan, np.float32)
    sa[:, :K], sb[:, :N] = A, B
    C0 = u.uniform(orc, M * N, 3).reshape(M, N)
    want, scale = u.exact(u.bf16_value(u.bf16_bits(orc, A)), u.bf16_value(u.bf16_bits(orc, B)), alpha, beta, C0)
    dA, dB = dev_copy(sa, dev), dev_copy(sb, dev)
    got = []
    for _ in range(2):
        dC = dev_copy(C0 if beta else np.full_like(C0, np.nan), dev)
        lib.gemm_bf16_f32in(M, N, K, alpha, dA, K + pad, dB, N + pad, beta, dC, N, stream=stream())
        got.append(host(dC))
    u.assert_fp32_close(got[0], want, scale, K, f"{M}x{N}x{K}")
    u.assert_bits_equal(got[0], got[1], "repeated call")


@pytest.mark.parametrize("M,N,K", [(256, 9000, 1024), (1024, 4096, 512)])
def test_rounding_and_special_values(lib, orc, dev, M, N, K):
    """One nonzero of A per row (1.0): C's row is a row of B, rounded.  Ties,
    subnormals, infinities and NaNs of B come out as the rounding formula
    leaves them."""
    rng = np.random.default_rng(5)
    B = rng.integers(0, 1 << 32, (K, N), dtype=np.uint64).astype(np.uint32)
    B[:, ::3] = (B[:, ::3] & 0xFFFF0000) | 0x8000  # ties
    B &= 0xBFFFFFFF  # finite (exponents below 2^0) ...
    B[:, 7] = 0x7F800000  # ... but for a column each of inf and NaN
    B[:, 11] = 0x7FC00000
    A = np.zeros((M, K), np.float32)
    pick = rng.integers(0, K, M)
    A[np.arange(M), pick] = 1.0
    dC = torch.full((M, N), float("nan"), device=dev)
    lib.gemm_bf16_f32in(M, N, K, 1.0, dev_copy(A, dev), K, dev_copy(B.view(np.float32), dev), N, 0.0, dC, N, stream=stream())
    got = host(dC)
    want = u.bf16_value(u.bf16_bits(orc, np.ascontiguousarray(B.view(np.float32)[pick])))
    cols = np.ones(N, bool)
    cols[[7, 11]] = False  # 0 * inf and 0 * NaN of the other rows make NaN there
    # the matrix cores flush no bf16 operand, but a product below the fp32 normals may differ
    normal = np.abs(want[:, cols]) >= 2.0 ** -126
    assert np.array_equal(got[:, cols][normal], want[:, cols][normal])
    assert np.isnan(got[:, [7, 11]]).all()


def test_under_graph_capture(lib, orc, dev):
    """A captured call rounds while staging (a graph must not keep the address
    of workspace that a later call may free), whether or not its stream has
    workspace already; replays between eager calls, one of which grows the
    workspace, stay within the bound."""
    M, N, K = 512, 8192, 512
    A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
    want, scale = u.exact(u.bf16_value(u.bf16_bits(orc, A)), u.bf16_value(u.bf16_bits(orc, B)))
    dA, dB = dev_copy(A, dev), dev_copy(B, dev)
    for warm in (False, True):
        s = torch.cuda.Stream()
        dC, dE = torch.full((M, N), float("nan"), device=dev), torch.full((M, N), float("nan"), device=dev)
        torch.cuda.synchronize()
        if warm:
            lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dE, N, stream=s.cuda_stream)
            torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, stream=s.cuda_stream)
        for rep in range(3):
            dC.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            u.assert_fp32_close(host(dC), want, scale, K, f"replay {rep}, warm={warm}")
            lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dE, N, stream=s.cuda_stream)
            u.assert_fp32_close(host(dE), want, scale, K, f"eager {rep}, warm={warm}")
            if rep == 0:  # a larger call on the same stream
                big = torch.zeros((2048, 4096), device=dev)
                lib.gemm_bf16_f32in(2048, 4096, 2048, 1.0, torch.zeros((2048, 2048), device=dev), 2048,
                                    torch.zeros((2048, 4096), device=dev), 4096, 0.0, big, 4096, stream=s.cuda_stream)
                torch.cuda.synchronize()


def test_captured_after_a_warm_call(lib, orc, dev):
    """Eager calls take the rounded copies, a captured one the split tiles: its
    split-k workspace is there after the warm-up call on the same stream."""
    M, N, K = 284, 2304, 3904
    assert lib.plan_bf16(M, N, K, fp32_inputs=1)["splits"] > 1
    A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
    want, scale = u.exact(u.bf16_value(u.bf16_bits(orc, A)), u.bf16_value(u.bf16_bits(orc, B)))
    dA, dB = dev_copy(A, dev), dev_copy(B, dev)
    dC = torch.full((M, N), float("nan"), device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    call = lambda: lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, stream=s.cuda_stream)
    call()
    torch.cuda.synchronize()
    u.assert_fp32_close(host(dC), want, scale, K, "warm-up")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call()
    for rep in range(3):
        dC.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        u.assert_fp32_close(host(dC), want, scale, K, f"replay {rep}")


# TILE_CFG of a launch on copies -> (operands copied, rows, columns, TILE_CFG of the direct tiles with its blocks of k)
FORCED = {65: (1, 128, 96, 20), 66: (1, 256, 96, 40), 51: (2, 256, 256, 40), 52: (2, 256, 192, 40),
          53: (2, 256, 128, 40), 54: (2, 128, 128, 40), 55: (2, 128, 256, 40), 56: (2, 128, 192, 40), 57: (2, 256, 64, 40)}


@pytest.mark.parametrize("cfg", sorted(FORCED))
@pytest.mark.parametrize("splits", [1, 2])
def test_every_tile_on_copies(lib, orc, dev, cfg, splits):
    """Each tile that reads copies, at its edges (a k tail, odd strides, one
    block of k, odd and even block counts): within the fp32 bound, and the bits
    of the tiles that round while staging, with the same k-splits."""
    operands, rows, cols, direct = FORCED[cfg]
    for M, N, K, pad, alpha, beta in [(9, 64, 5, 1, 1.0, 0.0), (129, 97, 64, 0, 0.5, 1.0), (255, 193, 200, 3, 1.0, 0.0),
                                      (257, 300, 391, 2, -2.0, 0.25), (300, 515, 1001, 0, 1.0, 1.0)]:
        A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
        sa, sb = np.full((M, K + pad), np.nan, np.float32), np.full((K, N + pad), np.nan, np.float32)
        sa[:, :K], sb[:, :N] = A, B
        C0 = u.uniform(orc, M * N, 3).reshape(M, N)
        want, scale = u.exact(u.bf16_value(u.bf16_bits(orc, A)), u.bf16_value(u.bf16_bits(orc, B)), alpha, beta, C0)
        dA, dB = dev_copy(sa, dev), dev_copy(sb, dev)
        got = []
        for c in (cfg, direct):
            dC = dev_copy(C0 if beta else np.full_like(C0, np.nan), dev)
            with lib.tunables(TILE_CFG=c, TILE_SPLITS=splits):
                p = lib.plan_bf16_copies(M, N, K)
                if c == cfg:
                    assert (p["operands"], p["rows"], p["cols"], p["block"]) == (operands, rows, cols, 512), p
                else:
                    assert p["operands"] == 0, p
                lib.gemm_bf16_f32in(M, N, K, alpha, dA, K + pad, dB, N + pad, beta, dC, N, stream=stream())
            got.append(host(dC))
        u.assert_fp32_close(got[0], want, scale, K, f"{cfg} {M}x{N}x{K} splits={splits}")
        u.assert_bits_equal(got[0], got[1], f"{cfg} and {direct} {M}x{N}x{K} splits={splits}")


CAPTURED = [(284, 2304, 3904), (512, 8192, 512), (200, 9000, 1000), (1024, 4100, 520), (1000, 2048, 4096),
            (700, 1024, 4096), (846, 7552, 3840), (571, 2731, 3648), (640, 2714, 3170), (976, 3648, 1243),
            (176, 8384, 3392)]


@pytest.mark.parametrize("M,N,K", CAPTURED)
def test_captured_bits_are_eager_bits(lib, orc, dev, M, N, K):
    """The route (on copies, or under capture while staging) changes no bit."""
    A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
    dA, dB = dev_copy(A, dev), dev_copy(B, dev)
    dC, dE = torch.full((M, N), float("nan"), device=dev), torch.full((M, N), float("nan"), device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dE, N, stream=s.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, stream=s.cuda_stream)
    want = host(dE)
    for rep in range(3):
        dC.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        u.assert_bits_equal(host(dC), want, f"replay {rep}")


def test_workspace_grows_in_powers_of_two(lib, dev):
    """Sizes that creep up reallocate the copies' workspace a few times in all."""
    s = torch.cuda.Stream()
    N, K = 4096, 4096
    plans = {M: lib.plan_bf16_copies(M, N, K) for M in range(960, 8192, 256)}
    rows = [M for M, p in plans.items() if p["operands"] == 2 and p["splits"] == 1]
    assert len(rows) > 8 and plans[rows[-1]]["workspace_bytes"] > 80 << 20, plans
    B = torch.zeros((K, N), device=dev)
    held = []
    A, C = torch.zeros((max(rows), K), device=dev), torch.zeros((max(rows), N), device=dev)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for M in rows:
        lib.gemm_bf16_f32in(M, N, K, 1.0, A, K, B, N, 0.0, C, N, stream=s.cuda_stream)
        torch.cuda.synchronize()
        held.append(before - torch.cuda.mem_get_info()[0])
        assert held[-1] >= plans[M]["workspace_bytes"]
    assert len(set(held)) <= 3, held  # up to 128 MiB from 32 MiB at the least


@pytest.mark.parametrize("M,N,K", [(9, 64, 1), (32, 70, 1023), (31, 4096, 1024), (16, 16384, 1024), (33, 130, 1152),
                                   (64, 8192, 1300)])
@pytest.mark.parametrize("splits", [1, 2])
def test_32_row_tiles_rounding_early_or_late(lib, orc, dev, M, N, K, splits):
    """The 32 x 64 tiles round an operand when it arrives (TILE_CFG 19) or when
    it is written to LDS (67): the same bits, on both sides of the rule that
    picks between them (a CU to every workgroup, 8 blocks of 128 k or more)."""
    A, B = u.normal(orc, M * K, 1).reshape(M, K), u.normal(orc, K * N, 2, 0, 0.02).reshape(K, N)
    dA, dB = dev_copy(A, dev), dev_copy(B, dev)
    got = []
    for cfg in (19, 67):
        dC = torch.full((M, N), float("nan"), device=dev)
        with lib.tunables(TILE_CFG=cfg, TILE_SPLITS=splits):
            p = lib.plan_bf16(M, N, K, fp32_inputs=1)
            assert (p["rows"], p["cols"], p["block"]) == (32, 64, 256), p
            lib.gemm_bf16_f32in(M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, stream=stream())
        got.append(host(dC))
    want, scale = u.exact(u.bf16_value(u.bf16_bits(orc, A)), u.bf16_value(u.bf16_bits(orc, B)))
    u.assert_fp32_close(got[1], want, scale, K, f"{M}x{N}x{K} splits={splits}")
    u.assert_bits_equal(got[0], got[1], f"{M}x{N}x{K} splits={splits}")
