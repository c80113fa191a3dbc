"""The default tile shape of a batch's transforms (CPU only: no kernel runs)."""
import pytest

from fribois2d_amd import gpu

DIRECT = 1 | 2 | 8 | 16   # the shapes that load straight into LDS: 16-byte aligned operands only


# below 96 tiles of 64x64 | from there on | from 192 tiles of 96x128 on
@pytest.mark.parametrize("M,N,shape", [(48, 64, 0), (512, 704, 0), (512, 768, 1), (1440, 1536, 1), (1536, 1536, 3)])
def test_default_shape_is_one_every_instance_can_run(M, N, shape):
    pick = gpu.load().fribo_test_gemm_pick
    assert pick(M, N, 31) == shape
    assert pick(M, N, 4) == 2
    for mask in range(32):
        mask |= 4
        assert (mask >> pick(M, N, mask)) & 1
    assert pick(M, N, 31 & ~(1 << shape)) == 2
    assert pick(M, N, DIRECT | 4) == shape
