"""The maxima pass of the fp32-input int8 GEMM (dnnopt_absmax_part) takes four,
two or one row of an operand at a time: the largest element is found wherever
it stands, at the edges of those steps, and padding is not read."""
import numpy as np
import pytest
import torch

import _util as u

from test_gpu_parity import dev_copy, host, stream

pytestmark = pytest.mark.gpu


# (M, N, K): K columns of A and N of B on both sides of 1024, 2048 and 4096;
# row counts that are no multiple of the step, and blocks of several steps.
@pytest.mark.parametrize("M,N,K,pad", [
    (5, 1024, 1025, 0), (9, 1025, 1024, 3), (10, 2048, 2049, 0), (11, 2049, 2047, 4), (3, 4096, 4097, 1),
    (13, 4100, 1023, 0), (130, 5, 7, 0), (1, 1, 1, 0), (67, 515, 2050, 2),
])
def test_largest_element_anywhere(lib, orc, dev, M, N, K, pad):
    A0, B0 = u.uniform(orc, M * K, 1).reshape(M, K), u.uniform(orc, K * N, 2).reshape(K, N)
    lda, ldb = K + pad, N + pad
    edge = lambda n: sorted({0, min(255, n - 1), min(1023, n - 1), min(1024, n - 1), n // 2, n - 1})
    spots = [(r, c) for r in (0, M // 2, M - 1) for c in edge(K)][::2] + [(M - 1, K - 1)]
    spots_b = [(r, c) for r in (0, K // 2, K - 1) for c in edge(N)][::2] + [(K - 1, N - 1)]
    for i in range(max(len(spots), len(spots_b))):
        A, B = A0.copy(), B0.copy()
        A[spots[i % len(spots)]] = -37.5
        B[spots_b[i % len(spots_b)]] = 61.25
        want = np.zeros((M, N), np.float32)
        orc.orc_gemm_int8(M, N, K, 1.0, u.ptr(A), K, u.ptr(B), N, 0.0, u.ptr(want), N)
        Ap, Bp = np.full((M, lda), np.inf, np.float32), np.full((K, ldb), np.inf, np.float32)
        Ap[:, :K], Bp[:, :N] = A, B
        dC = torch.full((M, N), float("nan"), device=dev)
        lib.gemm_int8_f32(M, N, K, 1.0, dev_copy(Ap, dev), lda, dev_copy(Bp, dev), ldb, 0.0, dC, N, stream=stream())
        assert np.array_equal(host(dC).view(np.uint32), want.view(np.uint32)), (i, spots[i % len(spots)])
