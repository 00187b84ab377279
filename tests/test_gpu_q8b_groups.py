"""The fp32-input int8 GEMM's 64 x 32 tiles with one or two wave groups sharing
k: bit-equal to the oracle at the edges of the groups' blocks of 128 k, of the
tile, and on both sides of one tile per CU."""
import numpy as np
import pytest
import torch

import _util as u

from test_gpu_parity import dev_copy, host, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(9, 1), (64, 32), (65, 33), (40, 100)])
@pytest.mark.parametrize("K", [1, 100, 128, 129, 256, 257, 384, 385, 640, 1000])
def test_blocks_of_k(lib, orc, dev, M, N, K):
    check(lib, orc, dev, M, N, K, 2)


@pytest.mark.parametrize("M,N,K,groups", [(128, 4096, 300, 2), (129, 4096, 300, 1), (64, 8192, 200, 2),
                                          (64, 8193, 200, 1), (1024, 512, 513, 2)])
def test_one_tile_per_cu(lib, orc, dev, M, N, K, groups):
    check(lib, orc, dev, M, N, K, groups)


def check(lib, orc, dev, M, N, K, groups):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus == 256:
        assert lib.plan_int8_f32(M, N, K)["block"] == 256 * groups
    A, B, C0 = u.uniform(orc, M * K, 1), u.uniform(orc, K * N, 2), u.uniform(orc, M * N, 3)
    for beta in (0.0, 0.5):
        want = C0.copy()
        orc.orc_gemm_int8(M, N, K, 0.75, u.ptr(A), K, u.ptr(B), N, beta, u.ptr(want), N)
        dC = dev_copy(C0, dev)
        lib.gemm_int8_f32(M, N, K, 0.75, dev_copy(A, dev), K, dev_copy(B, dev), N, beta, dC, N, stream=stream())
        assert np.array_equal(host(dC).view(np.uint32), want.view(np.uint32)), beta
