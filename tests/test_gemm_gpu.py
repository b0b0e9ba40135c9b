"""The runtime's own GEMM kernels (tokamak_amd/csrc/tkm_gemm_mfma.hip) alone, on every operand form and
tile size, against a float64 product of the same 16-bit operands.

Bounds: an fp32 sum of K products carries at most K * 2^-24 of the sum of the products' magnitudes
(each partial sum rounds once); a 16-bit result adds its unit roundoff, 2^-11 of the value in fp16 (11
significant bits) and 2^-8 in bf16 (8)."""
import ctypes

import pytest

from attn_cases import log

pytestmark = pytest.mark.gpu

TILES = {"auto": -1, "256x128": 0, "128x128": 1, "128x64": 2, "64x64": 3, "128x64 split": 4, "64x64 split": 5}


class Problem(ctypes.Structure):
    _fields_ = [("A", ctypes.c_void_p), ("B", ctypes.c_void_p), ("C", ctypes.c_void_p), ("M", ctypes.c_int),
                ("N", ctypes.c_int), ("K", ctypes.c_int), ("lda", ctypes.c_int), ("ldb", ctypes.c_int),
                ("ldc", ctypes.c_int), ("tile0", ctypes.c_longlong)]


def lib():
    from tokamak_amd import runtime as R
    L = R.lib()
    L.tkm_gemm_mfma_tiles.restype = ctypes.c_longlong
    L.tkm_gemm_mfma_group.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_int,
                                      ctypes.c_void_p]
    return L


def guarded(shape, dtype, fill=float("nan")):
    """A tensor of `shape` between 256 NaN elements on either side (and the whole, to check them)."""
    import torch
    n = shape[0] * shape[1]
    whole = torch.full((n + 512,), float("nan"), dtype=dtype, device="cuda")
    t = whole[256:256 + n].view(shape)
    t.fill_(fill)
    return t, whole


def check(name, got, whole, ref, mag, K, bits):
    import torch
    assert torch.isnan(whole[:256]).all() and torch.isnan(whole[-256:]).all(), f"{name}: wrote outside C"
    err = (got.double() - ref).abs()
    bound = K * 2.0 ** -24 * mag + (ref.abs() * 2.0 ** -bits + 2.0 ** -24 if bits < 24 else 0)
    bad = int((~(err <= bound)).sum())
    log(f"    {name}: max err {float(err.max()):.3e}, {bad} past the bound")
    assert bad == 0


# rows, then the two layer sizes: single rows and chunks, tiles less and more one chunk, partial
# k-steps, k shorter than the pipeline
SHAPES = [(1, 8, 8), (65, 72, 40), (127, 136, 200), (128, 128, 64), (129, 264, 328), (300, 520, 136), (520, 64, 576)]
# sizes on either side of the lines of the tile's rule: 64x64 and its split form (K 768), the split 128x64, 128x128
LONG = [(200, 64, 328), (200, 64, 760), (200, 64, 776), (70, 72, 2056), (4090, 384, 1032), (2560, 512, 1032),
        (2552, 1656, 72)]


@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("bf16", (0, 1))
@pytest.mark.parametrize("b_along_k,accumulate", ((0, 0), (1, 0), (1, 1)))
def test_layer_products(gpu, tile, bf16, b_along_k, accumulate):
    """out = in W and din (+)= dout W^T; operands between NaN guards, so a read outside them shows."""
    import torch
    L = lib()
    dt = torch.bfloat16 if bf16 else torch.float16
    for M, N, K in SHAPES + (LONG if tile == "auto" else []):
        log(f"[case] tile {tile} bf16={bf16} b_along_k={b_along_k} acc={accumulate} {M}x{N}x{K}")
        torch.manual_seed(M + N + K)
        A, _ = guarded((M, K), dt)
        B, _ = guarded((N, K) if b_along_k else (K, N), dt)
        A.copy_(torch.randn(M, K, device="cuda"))
        B.copy_(torch.randn(B.shape, device="cuda"))
        C, whole = guarded((M, N), dt)
        Bd = (B.T if b_along_k else B).double()
        ref, mag = A.double() @ Bd, A.double().abs() @ Bd.abs()
        if accumulate:
            C.copy_(torch.randn(M, N, device="cuda"))
            ref, mag = ref + C.double(), mag + C.double().abs()
        p = Problem(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, K, B.shape[1], N, 0)
        assert L.tkm_gemm_mfma_supported(ctypes.byref(p), 0)
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert L.tkm_gemm_mfma_run(ctypes.byref(p), b_along_k, bf16, TILES[tile], accumulate, st) == 0
        torch.cuda.synchronize()
        check("C", C, whole, ref, mag, K + 1, 8 if bf16 else 11)


@pytest.mark.parametrize("tile", ("256x128", "128x128", "64x64"))
@pytest.mark.parametrize("bf16", (0, 1))
def test_weight_gradient_group(gpu, tile, bf16):
    """dW = in^T dout of several layers in one launch (any number of rows)."""
    import torch
    L = lib()
    dt = torch.bfloat16 if bf16 else torch.float16
    shapes = [(72, 136, 77), (8, 8, 1), (264, 64, 300), (128, 320, 64), (520, 136, 130)]
    probs, keep, t0 = [], [], 0
    for K, N, rows in shapes:
        torch.manual_seed(K + N + rows)
        X, _ = guarded((rows, K), dt)
        Y, _ = guarded((rows, N), dt)
        X.copy_(torch.randn(rows, K, device="cuda"))
        Y.copy_(torch.randn(rows, N, device="cuda"))
        C, whole = guarded((K, N), torch.float32)
        p = Problem(X.data_ptr(), Y.data_ptr(), C.data_ptr(), K, N, rows, K, N, N, t0)
        assert L.tkm_gemm_mfma_supported(ctypes.byref(p), 1)
        t0 += L.tkm_gemm_mfma_tiles(ctypes.byref(p), TILES[tile])
        probs.append(bytes(p))
        keep.append((X, Y, C, whole))
    table = torch.frombuffer(bytearray(b"".join(probs)), dtype=torch.uint8).cuda()
    log(f"[case] dW group tile {tile} bf16={bf16}: {t0} tiles")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert L.tkm_gemm_mfma_group(ctypes.c_void_p(table.data_ptr()), len(probs), t0, bf16, TILES[tile], st) == 0
    torch.cuda.synchronize()
    for (K, N, rows), (X, Y, C, whole) in zip(shapes, keep):
        check(f"dW {K}x{N} rows {rows}", C, whole, X.double().T @ Y.double(), X.double().abs().T @ Y.double().abs(),
              rows + 1, 24)
