"""One-pass slicing of operands read along columns whose rows are not 16-byte aligned, against the
CPU implementation: strips at the right edge, k panels partly past K, both strip forms."""
import pytest
import torch

import bit_reproducible_training_amd as rg

pytestmark = pytest.mark.gpu


def _operand(rows, cols, offset):
    """A contiguous [rows, cols] GPU tensor that starts `offset` floats into an allocation."""
    return torch.randn(rows * cols + offset, device="cuda")[offset:].view(rows, cols)


# M, N past the one-launch kernel; K <= 256 takes a strip per wavefront, more a strip per block.
@pytest.mark.parametrize("M,N", [(521, 601), (1001, 515), (517, 640), (513, 1030)])
@pytest.mark.parametrize("K", [1, 7, 33, 64, 255, 257, 300, 769, 2049])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_unaligned_column_operands(M, N, K, offset):
    torch.manual_seed(M + N + K + offset)
    A, B = _operand(K, M, offset), _operand(K, N, offset)
    A[:, M - 1] *= 1e-3
    A[K - 1, 0] = 7.0
    B[K // 2, N - 1] = -1e4
    if K > 8:
        A[3, 5] = float("nan")
        B[K - 2, 9] = float("inf")
    want = rg.gemm(A.cpu(), B.cpu(), M, N, K, True, False)
    got = rg.gemm(A, B, M, N, K, True, False).cpu()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
