"""Which products of an FC layer the runtime gives to its own GEMM kernels (tkm_gemm_mfma_preferred): those
that its kernels were measured slower at than the library stay with the library, on either side of each
line of the rule, and operands that the kernels cannot read are refused.  No GPU: the rule is host code."""
import ctypes

import pytest

from test_gemm_gpu import Problem
from tokamak_amd import runtime as R


def problem(M, N, K, weight_grad=0, ptr=1 << 20):
    """weight_grad: in^T dout, M x N from K rows; else rows M, stored along k."""
    return Problem(ptr, ptr, ptr, M, N, K, M if weight_grad else K, N if weight_grad else K, N, 0)


def preferred(M, N, K, weight_grad=0, **kw):
    return R.lib().tkm_gemm_mfma_preferred(ctypes.byref(problem(M, N, K, weight_grad, **kw)), weight_grad)


# M x N x K of products at which the library was faster: large ones (4096 x 8192 x 512: 46 us against 63), long
# sums of few tiles (256 x 1024 x 4096: 12 against 20)
@pytest.mark.parametrize("shape", ((4096, 8192, 512), (8192, 768, 2304), (2048, 4096, 4096), (8192, 4096, 4096),
                                   (16384, 1024, 4096), (256, 512, 8192), (256, 1024, 4096), (256, 1024, 2816),
                                   (64, 1024, 3080), (512, 1024, 4096), (2048, 2048, 2048), (4096, 512, 2864),
                                   (128, 28672, 4096)))
def test_library_keeps_what_it_is_faster_at(shape):
    assert not preferred(*shape)
    assert R.lib().tkm_gemm_mfma_supported(ctypes.byref(problem(*shape)), 0)


# the layers of the small decoders, at the most rows and at few, and of a large one at few rows (128 x 4096 x 14336:
# 74 us against the library's 123)
@pytest.mark.parametrize("shape", ((4096, 1536, 512), (4096, 512, 2752), (4096, 2752, 512), (2048, 512, 2752),
                                   (64, 512, 1536), (16, 512, 2048), (2048, 384, 128), (2048, 128, 704), (8, 8, 8),
                                   (128, 4096, 4096), (128, 4096, 14336), (2048, 1024, 2048)))
def test_own_kernels_keep_small_layers(shape):
    assert preferred(*shape)


@pytest.mark.parametrize("shape,own", (((512, 8192, 4096), 1), ((2048, 2048, 16384), 1), ((2752, 512, 64), 1),
                                       ((2048, 2056, 64), 0), ((3072, 3072, 2048), 0), ((4096, 4096, 8192), 0)))
def test_weight_gradients_by_size_of_result(shape, own):
    assert preferred(*shape, weight_grad=1) == own


@pytest.mark.parametrize("field", ("A", "B", "C"))
def test_unaligned_operands_are_refused(field):
    for weight_grad in (0, 1):
        p = problem(256, 256, 256, weight_grad)
        assert R.lib().tkm_gemm_mfma_supported(ctypes.byref(p), weight_grad)
        setattr(p, field, (1 << 20) + 8)
        assert not R.lib().tkm_gemm_mfma_supported(ctypes.byref(p), weight_grad)
        assert not R.lib().tkm_gemm_mfma_preferred(ctypes.byref(p), weight_grad)
