"""Which calls of the fp32-input bf16 GEMM round operands ahead into workspace,
and on which tiles (host only)."""
import random

import pytest


# M, N, K: operands rounded ahead, and the tile and k-splits on the copies
ROUTES = [((200, 9000, 1000), (1, 128, 96, 1)), ((380, 10007, 777), (1, 256, 96, 1)), ((284, 2304, 3904), (1, 128, 96, 3)),
          ((512, 11008, 4096), (1, 256, 96, 1)), ((1024, 11008, 4096), (2, 256, 192, 1)), ((640, 2714, 3170), (2, 64, 128, 1)),
          ((976, 3648, 1243), (2, 128, 128, 1)), ((300, 500, 129), (0, 32, 64, 1)), ((65, 130, 64), (0, 32, 64, 1))]


@pytest.mark.parametrize("size,want", ROUTES)
def test_route_by_size(lib, size, want):
    p = lib.plan_bf16_copies(*size)
    assert (p["operands"], p["rows"], p["cols"], p["splits"]) == want, p


def test_copies_keep_the_splits(lib):
    """Copies are made for tiles with the k-splits of the launch that a captured
    call makes, so that both sum k in the same ranges."""
    rng = random.Random(1)
    size = lambda lo, hi: int(lo * (hi / lo) ** rng.random())
    made = 0
    for _ in range(3000):
        M, N, K = size(9, 2048), size(768, 11008), size(768, 4096)
        p = lib.plan_bf16_copies(M, N, K)
        made += p["operands"] > 0
        assert p["splits"] == lib.plan_bf16(M, N, K, fp32_inputs=1)["splits"], (M, N, K, p)
    assert made > 300


def test_scratch_of_a_launch_on_copies(lib):
    """The workspace of a launch on copies holds its split-k partials too, and
    all of it stays within 256 MiB."""
    rng = random.Random(2)
    size = lambda lo, hi: int(lo * (hi / lo) ** rng.random())
    pad = lambda v, n: (v + n - 1) // n * n
    split = 0
    for _ in range(3000):
        M, N, K = size(65, 8192), size(768, 16384), size(768, 8192)
        p = lib.plan_bf16_copies(M, N, K)
        if not p["operands"]:
            continue
        copies = 2 * pad(K, 8) * (M + (pad(N, 8) if p["operands"] == 2 else 0))
        tiles = pad(M, p["rows"]) * pad(N, p["cols"])
        partials = 4 * p["splits"] * tiles if p["splits"] > 1 else 0
        split += partials > 0
        assert copies + partials <= p["workspace_bytes"] <= 256 << 20, (M, N, K, p)
        assert p["workspace_bytes"] - copies - partials < (2 << 20), (M, N, K, p)
    assert split > 50
