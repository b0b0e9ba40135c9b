// tkm_gemm_mfma.hip -- the runtime's FC GEMMs on gfx950 matrix cores.
//
//   C[m][n] = sum_k A(m, k) B(k, n)  (+ C[m][n]),  fp32 accumulation, row-major C
//
// for the three products of an FC layer, none of which needs a transposed copy:
//   forward  out[rows][N] = in[rows][K] W[K][N]        A along k (KC), B along n (NC)
//   dX       din[rows][K] = dout[rows][N] W[K][N]^T    A along k,      B along k
//   dW       dW[K][N]     = in[rows][K]^T dout[rows][N] A along m (NC), B along n
// An operand stored along k ("KC", [index][k]) is read from LDS 16 bytes per lane, the MFMA's own
// layout; one stored along its output index ("NC", [k][index]) is read with the transposing
// ds_read_b64_tr_b16.  Tiles go HBM -> LDS by DMA and are swizzled as the attention kernels'
// (attn_common.h), which keeps both kinds of reads free of bank conflicts.
//
// What bounds them: with 4096 rows and K, N of 512 to 2752 a 128x128 tile runs 8 to 43 steps of 64 k, so
// the latency of the first loads and the fill of the chip by few tiles weigh as much as the matrix rate;
// and the transposing reads deliver half the bytes per cycle, so dW (both operands NC) is bound by LDS
// reads.  Hence several tile sizes (pick_tile), STAGES k-steps of LDS with STAGES - 1 in flight, a fixed
// place for every LDS read and request between the MFMAs (in one burst they hold the wave's issue: dW of
// 4096 rows, 512 x 8192: 65 -> 46 us).
// Measured in bf16 at rows 4096 from a captured graph, operands out of cache, against hipBLASLt's first choice:
//   forward  N 1536, K 512 : 14.9 us (17.2)     dX  N 512, K 1536 : 15.1 us (17.4)
//            N 512,  K 512 :  7.4 us (11.6)         N 512, K 512  :  7.3 us (11.0)
//            N 2752, K 512 : 24.8 us (28.9)         N 512, K 2752 : 22.3 us (26.2)
//            N 512, K 1376 : 15.3 us (19.9)         N 1376, K 512 : 13.9 us (19.6)
// and 8192 x 4096 x 4096 in 272 us, 1.01 PFLOP/s (256x128), where the library takes 176: tkm_gemm_mfma_preferred
// has the line between the two.  The 8-layer decoder's training step, one runtime: 3690 us with hipBLASLt,
// 2750 with these kernels and the attention kernels' wave groups.  A tile of one wave group sums over k in order
// (its outputs equalled the library's bit for bit); two groups each sum every other k-step.
//
// A workgroup is 4 waves in a 2 x 2 grid, or two such groups that take the k-steps in turn and add their
// sums through LDS (pick_tile).  The product is formed transposed (the B operand's columns
// are the MFMA's rows), so a lane holds one row of C and 4 consecutive columns per register quad;
// the tile leaves through LDS as fp32 rows, read back as whole 16-byte groups of columns.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attn_common.h"
#include "tkm_gemm_mfma.h"

namespace {

using namespace tkm;

constexpr int BK = 64, KST = BK / 16;   // k of one step, its MFMA k-groups

// Descriptor of what is left of an operand (0 bytes or less: every request is out of range).
__device__ __forceinline__ u32x4 desc(const char* base, long long bytes) {
    return make_rsrc(base, bytes <= 0 ? 0u : (bytes > 0x7fffffffll ? 0x7fffffffu : (uint32_t)bytes));
}

// Until at most N of this wave's DMA requests are in flight and its LDS reads are done, then the
// workgroup's barrier: after it every wave's share of the awaited tile is in LDS.
template <int N>
__device__ __forceinline__ void wait_step() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// LDS layout of one operand tile.  KC: IDX rows of BK values; NC: BK rows of IDX values.
template <bool KC, int IDX>
struct Operand {
    static constexpr int ROWS = KC ? IDX : BK, COLS = KC ? BK : IDX;
    static constexpr int ROWB = COLS * 2, CPR = COLS / 8, BYTES = ROWS * ROWB;
    static constexpr int RPI = 64 / CPR, NI = ROWS / RPI / 4;   // rows per DMA request, requests per wave
    static_assert(COLS == 64 || COLS == 128 || COLS == 256, "tile rows of 128, 256 or 512 bytes");
    static __device__ __forceinline__ int swizzle(int r) { return swz<(COLS > 128 ? 128 : COLS)>(r); }
};

template <int DT, bool AKC, bool BKC, int BM, int BN, int STAGES, bool OUT32, int GROUPS = 1>
struct Gemm {
    using TA = Operand<AKC, BM>;
    using TB = Operand<BKC, BN>;
    static constexpr int WM = BM / 2, WN = BN / 2, MB = WM / 32, NB = WN / 32;
    static constexpr int NDMA = TA::NI + TB::NI;
    static constexpr int STAGE_BYTES = TA::BYTES + TB::BYTES;
    static constexpr int EPITCH = WN + 4;                       // fp32 staging row
    static constexpr int EPI_BYTES = GROUPS * 4 * 32 * EPITCH * 4;
    // the groups' exchange of partial sums: of each 4-wave group's MB blocks of rows, those the other stores
    static constexpr int OWN = GROUPS == 2 && MB > 1 ? MB / 2 : MB;
    static constexpr int XCH_BYTES = GROUPS == 2 ? 8 * OWN * NB * 4096 : 0;
    static constexpr int TILE_BYTES = GROUPS * STAGES * STAGE_BYTES;
    static constexpr int LDS_BYTES = TILE_BYTES > EPI_BYTES + XCH_BYTES ? TILE_BYTES : EPI_BYTES + XCH_BYTES;
    static_assert(GROUPS == 1 || GROUPS == 2, "one or two wave groups");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS of one CU");

    // LDS reads of one MFMA operand (32 indices from idx0, 16 k of step ks): one of 16 bytes per lane
    // (KC) or two transposing ones of 8 (NC).
    template <bool KC>
    static constexpr int PIECES = KC ? 1 : 2;
    template <class T, bool KC>
    static __device__ __forceinline__ void piece(u32x4& x, const char* t, int idx0, int ks, int tt, int lane) {
        const int l32 = lane & 31, hi = lane >> 5;
        if constexpr (KC) {
            const int r = idx0 + l32;
            x = ld_lds16((const uint16_t*)(t + r * T::ROWB + (((ks * 2 + hi) ^ T::swizzle(l32)) << 4)));
        } else {
            const int row = ks * 16 + hi * 8 + tt * 4 + ((lane & 15) >> 2);
            const int col = idx0 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
            const u32x2 v = ld_lds_tr(t + row * T::ROWB + (((col >> 3) ^ T::swizzle(row)) << 4) + (col & 7) * 2);
            x[2 * tt] = v[0];
            x[2 * tt + 1] = v[1];
        }
    }

    static __device__ __forceinline__ void run(const TkmGemmProblem& p, int tm, int tn, int accumulate, char* smem) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3, grp = GROUPS == 1 ? 0 : wave8 >> 2;
        const int m0 = tm * BM, n0 = tn * BN;
        const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
        const int nt = ((p.K + BK - 1) / BK + GROUPS - 1) / GROUPS;   // steps of each group
        char* const tiles = smem + grp * STAGES * STAGE_BYTES;
        const uint32_t lds0 = lds_addr(smem) + (uint32_t)(grp * STAGES * STAGE_BYTES);

        // Bytes from one k-step's tile to the next, and from the tile's first byte to the tensor's end.
        const long long pa = 2ll * p.lda, pb = 2ll * p.ldb;
        const char* abase = (const char*)p.A + (AKC ? (long long)m0 * pa : 2ll * m0);
        const char* bbase = (const char*)p.B + (BKC ? (long long)n0 * pb : 2ll * n0);
        const long long aend = AKC ? (p.M - 1ll - m0) * pa + 2ll * p.K : (p.K - 1ll) * pa + 2ll * (p.M - m0);
        const long long bend = BKC ? (p.N - 1ll - n0) * pb + 2ll * p.K : (p.K - 1ll) * pb + 2ll * (p.N - n0);
        const long long astep = AKC ? 2ll * BK : BK * pa, bstep = BKC ? 2ll * BK : BK * pb;

        // This lane's global offset for each of its wave's requests, and its chunk's first k (KC).
        uint32_t va[TA::NI], vb[TB::NI];
        const int ra = lane / TA::CPR, ca = lane % TA::CPR, rb = lane / TB::CPR, cb = lane % TB::CPR;
#pragma unroll
        for (int i = 0; i < TA::NI; ++i) {
            const int r = (wave * TA::NI + i) * TA::RPI + ra;
            va[i] = (uint32_t)r * (uint32_t)pa + (uint32_t)((ca ^ TA::swizzle(r)) << 4);
        }
#pragma unroll
        for (int i = 0; i < TB::NI; ++i) {
            const int r = (wave * TB::NI + i) * TB::RPI + rb;
            vb[i] = (uint32_t)r * (uint32_t)pb + (uint32_t)((cb ^ TB::swizzle(r)) << 4);
        }

        // The requests of one step's tile, one at a time (q = 0 .. NDMA - 1).
        struct Tile {
            u32x4 da, db;
            uint32_t lds;
            int left;       // k left from this step on (chunks past K come from out of range, as zeros)
        };
        auto tile_at = [&](int step, int buf) __attribute__((always_inline)) {
            const int t = step * GROUPS + grp;      // the groups take the k-steps in turn
            return Tile{desc(abase + t * astep, aend - t * astep), desc(bbase + t * bstep, bend - t * bstep),
                        lds0 + (uint32_t)(buf * STAGE_BYTES), p.K - t * BK};
        };
        auto request = [&](const Tile& x, int q) __attribute__((always_inline)) {
            if (q < TA::NI) {
                uint32_t v = va[q];
                if constexpr (AKC) {
                    const int r = (wave * TA::NI + q) * TA::RPI + ra;
                    if (x.left < BK) v = ((ca ^ TA::swizzle(r)) << 3) < x.left ? v : 0x80000000u;
                }
                dma16_ready(x.da, x.lds + (wave * TA::NI + q) * 1024, v);
            } else {
                const int i = q - TA::NI;
                uint32_t v = vb[i];
                if constexpr (BKC) {
                    const int r = (wave * TB::NI + i) * TB::RPI + rb;
                    if (x.left < BK) v = ((cb ^ TB::swizzle(r)) << 3) < x.left ? v : 0x80000000u;
                }
                dma16_ready(x.db, x.lds + TA::BYTES + (wave * TB::NI + i) * 1024, v);
            }
        };

        f32x16 acc[MB][NB];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = f32x16{};

        // Operands of one k-step in registers.  Those of (step t + 1, k-group g) are read from LDS once the
        // MFMAs of (t, g) have gone out, 2 to 3 k-groups ahead of their use, into the same registers.  A
        // wave issues in order and stalls while the LDS or request queues are full, so the reads and the
        // DMA requests are dealt out between the MFMAs, slot by slot.
        u32x4 xa[KST][MB], xb[KST][NB];
        constexpr int PA = PIECES<AKC>, PB = PIECES<BKC>, NRK = MB * PA + NB * PB;   // reads per k-group
        constexpr int KSLOT = MB * NB, NSLOT = KST * KSLOT;                          // MFMAs per k-group, per step
        constexpr int MEET = KSLOT + (KSLOT + 1) / 2, REST = NSLOT - MEET;           // slot of the barrier, slots after
        auto read = [&](int stage, int ks, int q) __attribute__((always_inline)) {
            const char* at = tiles + stage * STAGE_BYTES;
            if (q < MB * PA) piece<TA, AKC>(xa[ks][q / PA], at, wm + (q / PA) * 32, ks, q % PA, lane);
            else {
                const int u = q - MB * PA;
                piece<TB, BKC>(xb[ks][u / PB], at + TA::BYTES, wn + (u / PB) * 32, ks, u % PB, lane);
            }
        };

#pragma unroll
        for (int t = 0; t < STAGES; ++t) {
            const Tile tl = tile_at(t, t);
            dma_ready(tl.da, tl.db);
#pragma unroll
            for (int q = 0; q < NDMA; ++q) request(tl, q);
        }
        wait_step<(STAGES - 1) * NDMA>();
#pragma unroll
        for (int r = 0; r < (KST - 1) * NRK; ++r) read(0, r / NRK, r % NRK);
        // Past the last step the requests are out of range (zeros into a stage nobody reads) and the
        // reads unused: every step has the same instructions and the same number in flight.
        int buf = 0;
        for (int t = 0; t < nt; ++t) {
            const int next = buf + 1 == STAGES ? 0 : buf + 1;
            const Tile tl = tile_at(t + STAGES, buf);
            dma_ready(tl.da, tl.db);
#pragma unroll
            for (int s = 0; s < NSLOT; ++s) {
                const int ks = s / KSLOT, i = (s / NB) % MB, j = s % NB;
                // every wave has read stage t, and tile t + 1 is in LDS
                if (s == MEET) wait_step<(STAGES - 2) * NDMA>();
                acc[i][j] = mfma32<DT>(xb[ks][j], xa[ks][i], acc[i][j]);
                if (s < KSLOT) {
#pragma unroll
                    for (int r = s * NRK / KSLOT; r < (s + 1) * NRK / KSLOT; ++r) read(buf, KST - 1, r);
                }
                if (s >= MEET) {
                    const int u = s - MEET;
                    constexpr int NR = (KST - 1) * NRK;
#pragma unroll
                    for (int r = u * NR / REST; r < (u + 1) * NR / REST; ++r) read(next, r / NRK, r % NRK);
#pragma unroll
                    for (int q = u * NDMA / REST; q < (u + 1) * NDMA / REST; ++q) request(tl, q);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            buf = next;
        }
        wait_step<0>();

        // Two groups: each hands the other the sums of the rows that the other stores (one block of rows:
        // group 0 stores them all), lane by lane, past the staging rows.
        const int own0 = GROUPS == 2 && MB > 1 ? grp * OWN : 0;
        if constexpr (GROUPS == 2) {
            float* xch = reinterpret_cast<float*>(smem + EPI_BYTES);
            if (MB > 1 || grp == 1) {
#pragma unroll
                for (int i = 0; i < OWN; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        const f32x16 give = MB > 1 && grp == 1 ? acc[i][j] : acc[MB - OWN + i][j];
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            *reinterpret_cast<f32x4*>(xch + ((((wave8 * OWN + i) * NB + j) * 4 + q) * 64 + lane) * 4) =
                                f32x4{give[q * 4], give[q * 4 + 1], give[q * 4 + 2], give[q * 4 + 3]};
                    }
            }
            __syncthreads();
            if (MB == 1 && grp == 1) return;
#pragma unroll
            for (int i = 0; i < OWN; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    f32x16 keep = MB > 1 && grp == 1 ? acc[MB - OWN + i][j] : acc[i][j];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f32x4 x = *reinterpret_cast<const f32x4*>(
                            xch + (((((wave8 ^ 4) * OWN + i) * NB + j) * 4 + q) * 64 + lane) * 4);
#pragma unroll
                        for (int e = 0; e < 4; ++e) keep[q * 4 + e] += x[e];
                    }
                    acc[i][j] = keep;
                }
        }

        // acc[i][j]: lane row wm + (own0 + i)*32 + l32, columns wn + j*32 + g4*8 + hi*4 + 0..3 of register quad g4.
        const int l32 = lane & 31, hi = lane >> 5;
        float* st = reinterpret_cast<float*>(smem) + wave8 * 32 * EPITCH;
        constexpr int VEC = OUT32 ? 4 : 8, CPW = WN / VEC, RPP = 64 / CPW;   // columns a lane stores, lanes per row
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4)
                    *reinterpret_cast<f32x4*>(st + l32 * EPITCH + j * 32 + g4 * 8 + hi * 4) =
                        f32x4{acc[i][j][g4 * 4], acc[i][j][g4 * 4 + 1], acc[i][j][g4 * 4 + 2], acc[i][j][g4 * 4 + 3]};
            // one wave's LDS operations complete in order: its own rows need no wait beyond the reads'
#pragma unroll
            for (int q = 0; q < 32 / RPP; ++q) {
                const int r = q * RPP + lane / CPW, c = (lane % CPW) * VEC;
                const int m = m0 + wm + (own0 + i) * 32 + r, n = n0 + wn + c;
                const f32x4 x = *reinterpret_cast<const f32x4*>(st + r * EPITCH + c);
                if constexpr (OUT32) {
                    if (m < p.M && n < p.N) *reinterpret_cast<f32x4*>((float*)p.C + (size_t)m * p.ldc + n) = x;
                } else {
                    const f32x4 y = *reinterpret_cast<const f32x4*>(st + r * EPITCH + c + 4);
                    if (m < p.M && n < p.N) {
                        uint16_t* cp = (uint16_t*)p.C + (size_t)m * p.ldc + n;
                        float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                        if (accumulate) {
                            const u32x4 old = ld_global16(cp);
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                const uint32_t o = old[w];
                                v[2 * w] += to_f32<DT>((uint16_t)(o & 0xffffu));
                                v[2 * w + 1] += to_f32<DT>((uint16_t)(o >> 16));
                            }
                        }
                        *reinterpret_cast<u32x4*>(cp) = u32x4{pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3]),
                                                              pack2<DT>(v[4], v[5]), pack2<DT>(v[6], v[7])};
                    }
                }
            }
        }
    }
};

// Workgroup w runs on XCD w % 8: each XCD takes a contiguous run of tiles, so the tiles that share an
// operand's rows share one L2.
__device__ __forceinline__ int xcd_tile(int w, int n) {
    const int x = w & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (w >> 3);
}

template <int DT, bool AKC, bool BKC, int BM, int BN, int STAGES, bool OUT32, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, GROUPS == 2 || BM * BN * STAGES < 65536 ? 2 : 1)
void k_gemm(TkmGemmProblem p, int accumulate) {
    using G = Gemm<DT, AKC, BKC, BM, BN, STAGES, OUT32, GROUPS>;
    __shared__ __attribute__((aligned(1024))) char smem[G::LDS_BYTES];
    const int tiles_n = (p.N + BN - 1) / BN;
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    G::run(p, t / tiles_n, t % tiles_n, accumulate, smem);
}

// Several weight gradients in one launch: the table gives each problem's first tile.
template <int DT, int BM, int BN, int STAGES>
__global__ __launch_bounds__(256, BM * BN * STAGES >= 65536 ? 1 : 2)
void k_gemm_group(const TkmGemmProblem* __restrict__ table, int np) {
    using G = Gemm<DT, false, false, BM, BN, STAGES, true>;
    __shared__ __attribute__((aligned(1024))) char smem[G::LDS_BYTES];
    const int w = xcd_tile(blockIdx.x, gridDim.x);
    int lo = 0, hi = np - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (table[mid].tile0 <= w) lo = mid; else hi = mid - 1;
    }
    const TkmGemmProblem p = table[lo];
    const int t = w - p.tile0, tiles_n = (p.N + BN - 1) / BN;
    G::run(p, t / tiles_n, t % tiles_n, 0, smem);
}

long long tiles_of(const TkmGemmProblem& p, int bm, int bn) {
    return (long long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
}

int status() { return hipGetLastError() == hipSuccess ? 0 : -1; }

template <int DT, bool BKC, int BM, int BN, int STAGES, int GROUPS = 1>
int launch_t(const TkmGemmProblem& p, int accumulate, hipStream_t s) {
    hipLaunchKernelGGL((k_gemm<DT, true, BKC, BM, BN, STAGES, false, GROUPS>), dim3((unsigned)tiles_of(p, BM, BN)),
                       dim3(256 * GROUPS), 0, s, p, accumulate);
    return status();
}

// Tile of one product, measured at rows 4096 in bf16, in cache (us at 256x128, 128x128, 128x64, 64x64):
//   N 8192, K 512 : 57, 64, 66, 95      four tiles of 256x128 a CU: the LDS reads of a larger wave
//   N 2752, K 512 : 22, 19, 22, 29      tile (128x64) are the cheapest
//   N 1536, K 512 : 13, 12, 13, 17      fewer tiles than that leave CUs idle in the last round
//   N 512, K 2752 : 33, 30, 18, 21      128 tiles of 128x128 leave half the chip idle
//   N 512, K 512  : 11, 7.4, 6.5, 7.0
// and rows 256, N 512, K 2752 (where a step's latency counts): 32, 21, 18, 15.
// With one workgroup a CU (the smaller tiles) a step takes about 900 cycles where its LDS reads need 384:
// one wave a SIMD waits for each barrier.  Two wave groups that take the k-steps in turn fill those waits,
// for one merge through LDS at the end.  A layer's operands come from other CUs' writes and from memory, so
// the lines are set by operands out of cache and by whole steps (us, one group / two; in cache):
//   128x64, rows 4096, N 512:  K 1376 15.6 / 15.7 (11.8 / 12.1)   K 1536 15.2 / 15.6 (11.8 / 10.9)
//                              K 2752 23.2 / 23.0 (19.7 / 18.2)   the decoder's step at 4096 rows 2770 / 2751
//   64x64, rows 2048, N 512:   K 512 5.7 / 6.1 (5.5 / 5.5)        K 1376 10.8 / 11.2 (9.9 / 8.5)
//                              K 1536 11.2 / 11.3 (10.4 / 8.7)    K 2752 16.1 / 16.2 (14.7 / 12.4)
//          rows 256, N 512:    K 512 5.4 / 5.8 (5.2 / 5.2)        K 1376 9.6 / 8.7 (9.4 / 8.0)
//                              K 1536 9.1 / 8.5 (9.2 / 7.9)       K 2752 14.0 / 12.0 (14.5 / 11.6)
// A 64x64 form of two groups with two stages each, two workgroups of which fit a CU, led in cache up to K 1376
// (rows 2048, K 1376: 8.0) and lost out of it, for want of loads in flight (13.0; K 2752: 22.1): the
// decoder's step without it went from 1831 to 1788 us at 1024 rows and from 1541 to 1476 at 64.  The
// lines of 256 tiles of 128x128 and of 160 of 128x64 are from the same runs (512 x 2752 x 512: 8.5 us at 64x64,
// 6.5 at 128x64; 2048 x 2304 x 768: 19.9 at 128x64, 17.2 at 128x128).
int pick_tile(const TkmGemmProblem& p) {
    if (tiles_of(p, 256, 128) >= 512) return TKM_GEMM_TILE_256x128;
    if (tiles_of(p, 128, 128) >= 256) return TKM_GEMM_TILE_128x128;
    const long long n = tiles_of(p, 128, 64);
    if (n >= 160) return p.K >= 1024 && n <= 256 ? TKM_GEMM_TILE_128x64_SPLIT : TKM_GEMM_TILE_128x64;
    return p.K < 768 || tiles_of(p, 64, 64) > 256 ? TKM_GEMM_TILE_64x64 : TKM_GEMM_TILE_64x64_SPLIT;
}

template <int DT, bool BKC>
int launch_tile(const TkmGemmProblem& p, int tile, int accumulate, hipStream_t s) {
    switch (tile < 0 ? pick_tile(p) : tile) {
        case TKM_GEMM_TILE_256x128: return launch_t<DT, BKC, 256, 128, 3>(p, accumulate, s);
        case TKM_GEMM_TILE_128x128: return launch_t<DT, BKC, 128, 128, 2>(p, accumulate, s);
        case TKM_GEMM_TILE_128x64: return launch_t<DT, BKC, 128, 64, 3>(p, accumulate, s);
        case TKM_GEMM_TILE_128x64_SPLIT: return launch_t<DT, BKC, 128, 64, 3, 2>(p, accumulate, s);
        case TKM_GEMM_TILE_64x64_SPLIT: return launch_t<DT, BKC, 64, 64, 4, 2>(p, accumulate, s);
        default: return launch_t<DT, BKC, 64, 64, 4>(p, accumulate, s);
    }
}

template <int DT>
int launch_group(const TkmGemmProblem* d, int n, long long tiles, int tile, hipStream_t s) {
    if (tile == TKM_GEMM_TILE_256x128)
        hipLaunchKernelGGL((k_gemm_group<DT, 256, 128, 3>), dim3((unsigned)tiles), dim3(256), 0, s, d, n);
    else if (tile == TKM_GEMM_TILE_128x128)
        hipLaunchKernelGGL((k_gemm_group<DT, 128, 128, 4>), dim3((unsigned)tiles), dim3(256), 0, s, d, n);
    else
        hipLaunchKernelGGL((k_gemm_group<DT, 64, 64, 4>), dim3((unsigned)tiles), dim3(256), 0, s, d, n);
    return status();
}

}  // namespace

extern "C" {

int tkm_gemm_mfma_supported(const TkmGemmProblem* p, int weight_grad) {
    if (p->M < 1 || p->N < 1 || p->K < 1 || p->N % 8 || p->lda % 8 || p->ldb % 8 || p->ldc % 8) return 0;
    if (weight_grad ? p->M % 8 : p->K % 8) return 0;
    if (((uintptr_t)p->A | (uintptr_t)p->B | (uintptr_t)p->C) & 15u) return 0;
    const long long lim = 1ll << 30;    // offsets of 256 stored rows, formed in 32 bits
    return 512ll * p->lda < lim && 512ll * p->ldb < lim && tiles_of(*p, 64, 64) < (1ll << 31);
}

// Measured in bf16 from a captured graph, operands out of cache, us of these kernels / of hipBLASLt:
//   M x N x K
//   4096 x 8192 x 512 :  63 / 46       4096 x 512 x 2752 : 22 / 26     4096 x 2752 x 512  : 25 / 29
//   8192 x 2048 x 512 :  30 / 25       4096 x 1024 x 512 : 12 / 14     8192 x 768 x 2304  : 41 / 35
//   2048 x 4096 x 4096:  77 / 70       2048 x 2048 x 2048: 29 / 26     8192 x 4096 x 4096 : 272 / 176
// so large products, where its kernels' higher rate counts, are the library's from 6e9 multiply-adds on, of few
// rows (bound by reading the other operand) later:
//   128 x 4096 x 4096 :  24 / 39       128 x 4096 x 14336: 74 / 123    128 x 28672 x 4096 : 74 / 56
// and long sums of few tiles, which it splits further:
//   256 x 512 x 8192  :  35 / 15       256 x 1024 x 4096 : 20 / 12     512 x 1024 x 4096  : 21 / 16
//   256 x 1024 x 2816 :  16 / 10       256 x 768 x 2304  : 11 / 9      512 x 1024 x 2816  : 16 / 15
// Weight gradients by the size of the result:
//   512 x 8192, rows 4096: 50 / 53     2048 x 2048: 45 / 52            3072 x 3072, rows 2048: 65 / 52
int tkm_gemm_mfma_preferred(const TkmGemmProblem* p, int weight_grad) {
    if (!tkm_gemm_mfma_supported(p, weight_grad)) return 0;
    if (weight_grad) return (long long)p->M * p->N <= 1ll << 22;
    const long long n = tiles_of(*p, 64, 64);
    if ((p->K > 2048 && n <= 64) || (p->K > 3072 && p->M > 128 && n <= 128)) return 0;
    return (double)p->M * p->N * p->K < (p->M <= 128 ? 10e9 : 6e9);
}

int tkm_gemm_mfma_run(const TkmGemmProblem* p, int b_along_k, int bf16, int tile, int accumulate, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (bf16)
        return b_along_k ? launch_tile<DT_BF16, true>(*p, tile, accumulate, s)
                         : launch_tile<DT_BF16, false>(*p, tile, accumulate, s);
    return b_along_k ? launch_tile<DT_F16, true>(*p, tile, accumulate, s)
                     : launch_tile<DT_F16, false>(*p, tile, accumulate, s);
}

long long tkm_gemm_mfma_tiles(const TkmGemmProblem* p, int tile) {
    return tile == TKM_GEMM_TILE_256x128   ? tiles_of(*p, 256, 128)
           : tile == TKM_GEMM_TILE_128x128 ? tiles_of(*p, 128, 128)
                                           : tiles_of(*p, 64, 64);
}

int tkm_gemm_mfma_group(const TkmGemmProblem* table, int n, long long tiles, int bf16, int tile, void* stream) {
    if (n <= 0 || tiles <= 0) return 0;
    return bf16 ? launch_group<DT_BF16>(table, n, tiles, tile, (hipStream_t)stream)
                : launch_group<DT_F16>(table, n, tiles, tile, (hipStream_t)stream);
}

}  // extern "C"
