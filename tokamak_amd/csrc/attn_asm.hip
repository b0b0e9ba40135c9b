// attn_asm.hip -- host side of the hand-scheduled gfx950 assembly kernels, generated by
// tokamak_amd/asmgen and embedded in this library as code objects:
//
//   tkm_fa_fwd_d128_f16        forward, fp16    (asmgen/attn_fwd.py)
//   tkm_fa_fwd_d128_bf16       forward, bf16    (asmgen/attn_fwd.py, P as two bf16 halves)
//   tkm_fa_bwd_dkdv_d128_f16   backward dK, dV, fp16  (asmgen/attn_dkdv.py)
//   tkm_fa_bwd_dkdv_d128_bf16  backward dK, dV, bf16  (P and dS as two bf16 halves)
//   tkm_fa_bwd_dq_d128_f16     backward dQ (and D), fp16  (asmgen/attn_dq.py)
//   tkm_fa_bwd_dq_d128_bf16    backward dQ (and D), bf16  (dS as two bf16 halves)
//
// The code objects are loaded per device by tkm_attn_init (the runtime calls it at ignite,
// before any capture), or else by the first launch on that device.  A first launch inside a
// stream capture loads them with the thread's capture mode relaxed, so the load is never
// recorded into the graph.  Kernels are launched with hipModuleLaunchKernel on the caller's
// stream; a launch allocates nothing.
//
// They serve D = 128, fp16 and bf16, where the rules of attn_launch.h (pick_rows_form, pick_keys_form) give
// them the call -- grids that their 256-row items fill, and the smallest calls -- and the offsets fit
// their 32-bit buffer offsets; every other configuration goes to the HIP kernels (attn_fwd.hip,
// attn_bwd.hip).  On a gfx950 device a failed load is an error (kAsmLoadError), never a silent
// switch to the HIP kernels.
#include <mutex>
#include <stdio.h>
#include <stdint.h>
#include <string.h>

#include <hip/hip_runtime.h>

#include "attn_launch.h"

extern "C" {
extern const unsigned char tkm_fa_fwd_d128_f16_co[];
extern const unsigned char tkm_fa_fwd_d128_bf16_co[];
extern const unsigned char tkm_fa_bwd_dkdv_d128_f16_co[];
extern const unsigned char tkm_fa_bwd_dkdv_d128_bf16_co[];
extern const unsigned char tkm_fa_bwd_dq_d128_f16_co[];
extern const unsigned char tkm_fa_bwd_dq_d128_bf16_co[];
}

namespace tkm {

namespace {

constexpr int kMaxDevices = 64;

enum AsmKernel {
    kFwd = 0, kBwdDkdv = 1, kBwdDq = 2, kFwdBf16 = 3, kBwdDkdvBf16 = 4, kBwdDqBf16 = 5, kNumAsm = 6
};

struct AsmImage {
    const unsigned char* code;
    const char* name;
};
const AsmImage kImages[kNumAsm] = {
    {tkm_fa_fwd_d128_f16_co, "tkm_fa_fwd_d128_f16"},
    {tkm_fa_bwd_dkdv_d128_f16_co, "tkm_fa_bwd_dkdv_d128_f16"},
    {tkm_fa_bwd_dq_d128_f16_co, "tkm_fa_bwd_dq_d128_f16"},
    {tkm_fa_fwd_d128_bf16_co, "tkm_fa_fwd_d128_bf16"},
    {tkm_fa_bwd_dkdv_d128_bf16_co, "tkm_fa_bwd_dkdv_d128_bf16"},
    {tkm_fa_bwd_dq_d128_bf16_co, "tkm_fa_bwd_dq_d128_bf16"},
};

std::mutex g_mu;
hipFunction_t g_fn[kMaxDevices][kNumAsm];
int g_state[kMaxDevices];  // 0 not loaded, 1 loaded, 2 not gfx950 (no assembly path), -1 failed
int g_n_cu[kMaxDevices];   // compute units (workgroups of a persistent launch)
char g_load_err[kMaxDevices][160];

// Loads the code objects on device `dev` (current); g_mu held.
int load_device_locked(int dev) {
    if (g_state[dev] != 0) return g_state[dev];
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) {
        snprintf(g_load_err[dev], sizeof g_load_err[dev], "hipGetDeviceProperties: %s",
                 hipGetErrorString(e));
        return g_state[dev] = -1;
    }
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) return g_state[dev] = 2;
    g_n_cu[dev] = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 1;
    hipFunction_t fn[kNumAsm] = {};
    for (int k = 0; k < kNumAsm; ++k) {
        hipModule_t mod = nullptr;
        e = hipModuleLoadData(&mod, kImages[k].code);
        if (e == hipSuccess) {
            e = hipModuleGetFunction(&fn[k], mod, kImages[k].name);
            if (e != hipSuccess) (void)hipModuleUnload(mod);
        }
        if (e != hipSuccess) {
            snprintf(g_load_err[dev], sizeof g_load_err[dev], "loading %s: %s", kImages[k].name,
                     hipGetErrorString(e));
            return g_state[dev] = -1;
        }
    }
    for (int k = 0; k < kNumAsm; ++k) g_fn[dev][k] = fn[k];  // modules stay loaded until exit
    return g_state[dev] = 1;
}

int current_device(int* dev) {
    if (hipGetDevice(dev) != hipSuccess || *dev < 0 || *dev >= kMaxDevices) return -1;
    return 0;
}

// Kernel k of the current device, loading the code objects on first use.  Returns the
// function, or nullptr with *status = 1 (not gfx950: no assembly path) or -2 (load failed).
hipFunction_t function_for_current_device(AsmKernel k, void* stream, int* status) {
    int dev = -1;
    if (current_device(&dev)) {
        *status = -2;
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_state[dev] == 0) {
        // A first launch inside a capture: load with this thread's capture mode relaxed so
        // that the module load is neither refused nor recorded.
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        (void)hipStreamIsCapturing((hipStream_t)stream, &cs);
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        const bool relax = cs == hipStreamCaptureStatusActive;
        if (relax) (void)hipThreadExchangeStreamCaptureMode(&mode);
        load_device_locked(dev);
        if (relax) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    if (g_state[dev] == 1) return g_fn[dev][k];
    *status = g_state[dev] == 2 ? 1 : -2;
    return nullptr;
}

int n_cu_current_device() {
    int dev = -1;
    if (current_device(&dev)) return 1;
    std::lock_guard<std::mutex> lock(g_mu);
    return g_n_cu[dev] > 0 ? g_n_cu[dev] : 1;
}

// m = ceil(2^32 / d) when mulhi(x, m) equals x / d for every x < limit (d >= 2); 0 for d = 1
// (the kernel then skips the division); false when that cannot be guaranteed.  With
// m*d = 2^32 + e (0 <= e < d) and x = q*d + r: x*m / 2^32 = q + (r + x*e / 2^32) / d, so the
// quotient is exact whenever x*e < 2^32.
bool reciprocal(uint32_t d, uint32_t limit, uint32_t* m) {
    if (d == 1) {
        *m = 0;
        return true;
    }
    const uint64_t mm = ((1ull << 32) + d - 1) / d;
    const uint64_t e = mm * d - (1ull << 32);
    if (mm > 0xffffffffull || (limit > 0 && (uint64_t)(limit - 1) * e >= (1ull << 32))) return false;
    *m = (uint32_t)mm;
    return true;
}

// 0: launched; -1: launch error.
int launch(hipFunction_t fn, unsigned gx, unsigned gy, unsigned gz, void* args, size_t size,
           void* stream) {
    void* config[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, args, HIP_LAUNCH_PARAM_BUFFER_SIZE, &size,
                      HIP_LAUNCH_PARAM_END};
    hipError_t e = hipModuleLaunchKernel(fn, gx, gy, gz, 256, 1, 1, 0, (hipStream_t)stream, nullptr,
                                         config);
    return e == hipSuccess ? 0 : -1;
}

// Offsets the kernels form in 32 bits: a batch's qkv rows and O / dO rows must span < 2^31
// bytes, and (b*Hq + h)*S indexes LSE and D.
bool offsets_fit(int B, int S, int Hq, int Hkv) {
    const uint64_t ldb = (uint64_t)(Hq + 2 * Hkv) * 128 * 2;
    const uint64_t ldo = (uint64_t)Hq * 128 * 2;
    if ((uint64_t)S * ldb >= (1ull << 31) || (uint64_t)S * ldo >= (1ull << 31)) return false;
    // row offsets of the last (partial) block of 256 rows stay below 2^32 without wrapping
    if ((uint64_t)(S + 256) * ldb >= (1ull << 32)) return false;
    return (uint64_t)B * S * Hq < (1ull << 31);
}

struct FwdKernArgs {  // layout of tkm_fa_fwd_d128_{f16,bf16}'s argument segment (96 bytes)
    const void* qkv;
    void* out;
    float* lse;
    const int32_t* kv_len;
    uint32_t S, Hq, Hkv;
    float sl2;
    uint32_t causal, n_qblk, ldb, ldo, group;
    uint32_t n_wg, n_items, bhq;              // workgroups, items (query blocks x B x Hq), B*Hq
    uint32_t magic_nqblk, magic_hq, magic_g;  // reciprocals of n_qblk, Hq and Hq/Hkv
    uint32_t pad;
};
static_assert(sizeof(FwdKernArgs) == 96, "forward kernel argument layout");

struct DkdvKernArgs {  // layout of tkm_fa_bwd_dkdv_d128_{f16,bf16}'s argument segment (104 bytes)
    const void* qkv;
    const void* dout;
    const float* quads;  // row values: per (batch, head), tiles of 32 rows (-LSE*log2(e), then -D)
    void* dqkv;
    const int32_t* kv_len;
    uint32_t S, Hq, Hkv;
    float sl2;
    uint32_t causal, ldb, ldo, group;
    float scale;
    uint32_t n_kblk, s_pad;
    uint32_t n_wg, n_items, bh;        // workgroups, items (key blocks x B x Hkv), B*Hkv
    uint32_t magic_nkblk, magic_hkv;   // reciprocals of n_kblk and Hkv
};
static_assert(sizeof(DkdvKernArgs) == 104, "dK/dV kernel argument layout");

struct DqKernArgs {  // layout of tkm_fa_bwd_dq_d128_{f16,bf16}'s argument segment (136 bytes)
    const void* qkv;
    const void* o;
    const void* dout;
    const float* lse;
    float* delta;
    float* quads;
    void* dqkv;
    const int32_t* kv_len;
    uint32_t S, Hq, Hkv;
    float sl2;
    uint32_t causal, ldb, ldo, group;
    float scale;
    uint32_t n_qblk, s_pad, n_wg, n_items, bhq, magic_nqblk, magic_hq, magic_g;
    uint32_t compute_d;  // 1: D = <O, dO> here, written to delta and the row values; 0: read delta
};
static_assert(sizeof(DqKernArgs) == 136, "dQ kernel argument layout");

// Workgroups of a persistent launch of n_items items: with n compute units the items take R = ceil(items / n)
// rounds whatever the number of workgroups from items / R to n, so it is items / R, rounded up.  In
// snake order workgroup w then walks items w and 2W - 1 - w (R = 2) of W = items / 2, whose causal
// blocks are complementary; with W = n the last few workgroups would walk two heavy blocks and the
// others one (288 items, B 3 S 1531 Hq 16 D 128 fp16: forward 70 us with 256 workgroups, 49 with 144; dQ 94, 66).
uint32_t persistent_wgs(uint64_t n_items) {
    const uint64_t n = (uint64_t)n_cu_current_device(), rounds = (n_items + n - 1) / n;
    return (uint32_t)((n_items + rounds - 1) / rounds);
}

}  // namespace

// Each launcher returns 1: not handled here (the caller uses the HIP kernel); 0: launched;
// -1: launch error; -2: the code objects failed to load on this gfx950 device.
// Persistent: one workgroup per compute unit walks items (batch, q-head, block of 256 query
// rows), block fastest, in snake order over rounds; the blocks of a head run on one XCD.
int launch_fwd_asm(const FwdArgs& a) {
    constexpr int kRowsPerBlock = 256;
    if (a.D != 128 || (a.dtype != 0 && a.dtype != 1)) return 1;  // fp16 (0) or bf16 (1)
    if (!offsets_fit(a.B, a.S, a.Hq, a.Hkv)) return 1;
    const uint64_t n_qblk = (uint64_t)((a.S + kRowsPerBlock - 1) / kRowsPerBlock);
    const uint64_t bhq = (uint64_t)a.B * a.Hq, n_items = n_qblk * bhq;
    if (n_items >= (1ull << 31)) return 1;
    const uint32_t group = (uint32_t)(a.Hq / a.Hkv);
    uint32_t magic_nqblk = 0, magic_hq = 0, magic_g = 0;
    if (!reciprocal((uint32_t)n_qblk, (uint32_t)n_items, &magic_nqblk) ||
        !reciprocal((uint32_t)a.Hq, (uint32_t)bhq, &magic_hq) ||
        !reciprocal(group, (uint32_t)a.Hq, &magic_g))
        return 1;
    int st = 0;
    hipFunction_t fn = function_for_current_device(a.dtype == 1 ? kFwdBf16 : kFwd, a.stream, &st);
    if (!fn) return st;
    const uint32_t n_wg = persistent_wgs(n_items);
    FwdKernArgs k{a.qkv, a.o, a.lse, a.kv_len, (uint32_t)a.S, (uint32_t)a.Hq, (uint32_t)a.Hkv,
                  a.scale * 1.4426950408889634f, (uint32_t)a.causal, (uint32_t)n_qblk,
                  (uint32_t)((a.Hq + 2 * a.Hkv) * 256), (uint32_t)(a.Hq * 256), group, n_wg,
                  (uint32_t)n_items, (uint32_t)bhq, magic_nqblk, magic_hq, magic_g, 0u};
    return launch(fn, n_wg, 1, 1, &k, sizeof(k), a.stream);
}

// Persistent: one workgroup per compute unit walks items (batch, kv head, key block), key
// block fastest, in snake order over rounds; the key blocks of a head run on one XCD.
int launch_bwd_dkdv_asm(const BwdArgs& a) {
    constexpr int kKeysPerBlock = 128;
    if (a.D != 128 || (a.dtype != 0 && a.dtype != 1)) return 1;  // fp16 (0) or bf16 (1)
    if (!offsets_fit(a.B, a.S, a.Hq, a.Hkv)) return 1;
    const uint64_t n_kblk = (uint64_t)((a.S + kKeysPerBlock - 1) / kKeysPerBlock);
    const uint64_t bh = (uint64_t)a.B * a.Hkv, n_items = n_kblk * bh;
    if (n_items >= (1ull << 31)) return 1;
    uint32_t magic_nkblk = 0, magic_hkv = 0;
    if (!reciprocal((uint32_t)n_kblk, (uint32_t)n_items, &magic_nkblk) ||
        !reciprocal((uint32_t)a.Hkv, (uint32_t)bh, &magic_hkv))
        return 1;
    int st = 0;
    hipFunction_t fn = function_for_current_device(a.dtype == 1 ? kBwdDkdvBf16 : kBwdDkdv, a.stream, &st);
    if (!fn) return st;
    const uint32_t n_wg = persistent_wgs(n_items);
    DkdvKernArgs k{a.qkv, a.dout, a.ld, a.dqkv, a.kv_len, (uint32_t)a.S, (uint32_t)a.Hq,
                   (uint32_t)a.Hkv, a.scale * 1.4426950408889634f, (uint32_t)a.causal,
                   (uint32_t)((a.Hq + 2 * a.Hkv) * 256), (uint32_t)(a.Hq * 256),
                   (uint32_t)(a.Hq / a.Hkv), a.scale, (uint32_t)n_kblk,
                   (uint32_t)((a.S + 31) & ~31), n_wg, (uint32_t)n_items, (uint32_t)bh,
                   magic_nkblk, magic_hkv};
    return launch(fn, n_wg, 1, 1, &k, sizeof(k), a.stream);
}

// Persistent: one workgroup per compute unit walks items (batch, q-head, block of 256 query
// rows), block fastest, in snake order over rounds; the blocks of a head run on one XCD.
int launch_bwd_dq_asm(const BwdArgs& a, bool compute_d) {
    constexpr int kRowsPerBlock = 256;
    if (a.D != 128 || (a.dtype != 0 && a.dtype != 1)) return 1;  // fp16 (0) or bf16 (1)
    if (!offsets_fit(a.B, a.S, a.Hq, a.Hkv)) return 1;
    const uint64_t n_qblk = (uint64_t)((a.S + kRowsPerBlock - 1) / kRowsPerBlock);
    const uint64_t bhq = (uint64_t)a.B * a.Hq, n_items = n_qblk * bhq;
    if (n_items >= (1ull << 31)) return 1;
    const uint32_t group = (uint32_t)(a.Hq / a.Hkv);
    uint32_t magic_nqblk = 0, magic_hq = 0, magic_g = 0;
    if (!reciprocal((uint32_t)n_qblk, (uint32_t)n_items, &magic_nqblk) ||
        !reciprocal((uint32_t)a.Hq, (uint32_t)bhq, &magic_hq) ||
        !reciprocal(group, (uint32_t)a.Hq, &magic_g))
        return 1;
    int st = 0;
    hipFunction_t fn = function_for_current_device(a.dtype == 1 ? kBwdDqBf16 : kBwdDq, a.stream, &st);
    if (!fn) return st;
    const uint32_t n_wg = persistent_wgs(n_items);
    DqKernArgs k{a.qkv, a.o, a.dout, a.lse, a.delta, a.ld, a.dqkv, a.kv_len, (uint32_t)a.S,
                 (uint32_t)a.Hq, (uint32_t)a.Hkv, a.scale * 1.4426950408889634f, (uint32_t)a.causal,
                 (uint32_t)((a.Hq + 2 * a.Hkv) * 256), (uint32_t)(a.Hq * 256), group, a.scale,
                 (uint32_t)n_qblk, (uint32_t)((a.S + 31) & ~31), n_wg, (uint32_t)n_items,
                 (uint32_t)bhq, magic_nqblk, magic_hq, magic_g, compute_d ? 1u : 0u};
    return launch(fn, n_wg, 1, 1, &k, sizeof(k), a.stream);
}

// Loads the code objects on the current device: 0 (loaded, or not gfx950: no assembly
// path there), -2 (load failed; asm_load_error() says why).
int asm_init_current_device() {
    int dev = -1;
    if (current_device(&dev)) return -2;
    std::lock_guard<std::mutex> lock(g_mu);
    const int st = load_device_locked(dev);
    return st == -1 ? -2 : 0;
}

bool asm_available_current_device() {
    int dev = -1;
    if (current_device(&dev)) return false;
    std::lock_guard<std::mutex> lock(g_mu);
    return load_device_locked(dev) == 1;
}

const char* asm_load_error() {
    int dev = -1;
    if (current_device(&dev)) return "no current HIP device";
    std::lock_guard<std::mutex> lock(g_mu);
    return g_load_err[dev];
}

}  // namespace tkm
