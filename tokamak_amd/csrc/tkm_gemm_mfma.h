// tkm_gemm_mfma.h -- C entry points of the runtime's own GEMM kernels (tkm_gemm_mfma.hip).
#ifndef TKM_GEMM_MFMA_H
#define TKM_GEMM_MFMA_H

#ifdef __cplusplus
extern "C" {
#endif

#define TKM_GEMM_MFMA_API __attribute__((visibility("default")))   /* for the tests of the kernels alone */

/* C[M][N] = A(m, k) B(k, n), row-major, leading dimensions in elements.  A and B are 16-bit; how each
 * is stored is the entry point's: along k ([index][k]) or along its output index ([k][index]).
 * Pointers are 16-byte aligned. */
typedef struct {
    const void *A, *B;
    void *C;
    int M, N, K;
    int lda, ldb, ldc;
    long long tile0;             /* grouped launches: the problem's first tile */
} TkmGemmProblem;

enum { TKM_GEMM_TILE_AUTO = -1, TKM_GEMM_TILE_256x128 = 0, TKM_GEMM_TILE_128x128 = 1, TKM_GEMM_TILE_128x64 = 2,
       TKM_GEMM_TILE_64x64 = 3,
       /* two groups of waves on alternate k-steps; tkm_gemm_mfma_run only */
       TKM_GEMM_TILE_128x64_SPLIT = 4, TKM_GEMM_TILE_64x64_SPLIT = 5 };

/* Whether the kernels take the shape: stored rows in multiples of 8 elements, aligned pointers, offsets within
 * a tile in 32 bits.  weight_grad: the operands of tkm_gemm_mfma_group (any K), else of tkm_gemm_mfma_run. */
TKM_GEMM_MFMA_API int tkm_gemm_mfma_supported(const TkmGemmProblem *p, int weight_grad);

/* Whether they also are the faster ones for it, against hipBLASLt: the runtime's choice. */
TKM_GEMM_MFMA_API int tkm_gemm_mfma_preferred(const TkmGemmProblem *p, int weight_grad);

/* A along k; B along k (b_along_k = 1) or along n.  16-bit C, written or (accumulate = 1) added to in
 * fp32.  tile: TKM_GEMM_TILE_*. */
TKM_GEMM_MFMA_API int tkm_gemm_mfma_run(const TkmGemmProblem *p, int b_along_k, int bf16, int tile, int accumulate,
                                        void *stream);

/* Weight gradients: A along m, B along n, fp32 C written.  `table` (device memory) holds n problems
 * with their first tiles; tile is not 128x64 or a split one, tiles the total of tkm_gemm_mfma_tiles. */
TKM_GEMM_MFMA_API long long tkm_gemm_mfma_tiles(const TkmGemmProblem *p, int tile);
TKM_GEMM_MFMA_API int tkm_gemm_mfma_group(const TkmGemmProblem *table, int n, long long tiles, int bf16, int tile,
                                          void *stream);

#ifdef __cplusplus
}
#endif

#endif /* TKM_GEMM_MFMA_H */
