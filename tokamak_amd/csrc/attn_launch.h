// attn_launch.h -- internal launch records passed from the C ABI layer to the kernels.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace tkm {

struct FwdArgs {
    const void* qkv;
    void* o;
    float* lse;
    const int32_t* kv_len;
    int B, S, Hq, Hkv, D;
    float scale;
    int causal, dtype;
    void* stream;
};

struct BwdArgs {
    const void* qkv;
    const void* o;
    const void* dout;
    const float* lse;
    void* dqkv;
    const int32_t* kv_len;
    float* delta;  // workspace: D per row, B*Hq*S floats
    float* ld;     // workspace: per (b, h) and row pair m, m+1 (rows padded to 32):
                   // -LSE*log2(e) of m, m+1, then -D of m, m+1
    int B, S, Hq, Hkv, D;
    float scale;
    int causal, dtype;
    void* stream;
};

// Kernels a call launched (tkm_attn_last_kernels); values of the TKM_ATTN_K_* bits of
// include/tkm_attn.h.
enum KernelBit : unsigned {
    kFwdAsm = 1u, kFwdHip = 2u, kDqAsm = 4u, kDqHip = 8u, kDkdvAsm = 16u, kDkdvHip = 32u,
    kDeltaHip = 64u
};
void note_kernels(unsigned bits);  // ORs bits into the calling thread's record

// Assembly code objects: load on the current device (0, or -2 with asm_load_error()),
// and whether the assembly path exists there (gfx950, loaded).
int asm_init_current_device();
bool asm_available_current_device();
const char* asm_load_error();

// Compute units of the current device (cached per device; 0 if it cannot be read).
int compute_units();

// Forms of the HIP kernels: groups of waves that split a block's tiles (merged through LDS at the end) x
// waves of 32 rows (keys) each.  Fewer rows a block give a small grid more workgroups, more
// groups give each less to walk; both read the tiles more often.
enum HipForm { kForm1x4, kForm2x4, kForm2x2, kForm4x2, kForm8x1, kForm4x1, kFormAsm };

// The forward's and dQ's form.  q: 128-row query blocks of the launch (B * Hq * blocks), n: compute units.
// Measured with 256 compute units, causal, fp16, us of the forms 1x4, 2x4, 2x2, 4x2, 4x1:
//   D 64 forward   q 64,  S 1000: 16.5 14.7 11.0 10.8  9.0     dQ: 19.6 17.7 12.8 13.1 10.7
//                  q 128, S 2048: 28.4 23.8 18.6 16.5 15.8         34.7 29.9 22.4 20.1 19.1
//                   not causal  : 28.7 23.7 19.0 17.8 19.5         35.7 31.5 23.4 23.1 24.9
//                  q 256, S 1024: 17.9 16.1 13.3 19.3 16.7         21.1 19.7 16.2 23.0 22.1
//                   not causal  : 17.4 16.1 17.5 21.5 23.1         22.5 21.0 22.5 27.1 28.9
//                  q 576, S 1531: 28.1 36.0 33.3 46.0 40.2         37.3 44.1 41.4 56.7 53.7
//                  q 1024,S 2048: 53.6 65.0 67.7 89.9 87.7         70.1 84.9 85.6  111  110
// that is, the finest form whose workgroups the chip holds at once (with one key tile there is nothing to
// split: S 64 4.2 4.7 4.7 5.4 4.3).
// D 128 (assembly; 1x4, 2x4, 4x2, 4x1):
//          forward q 64,  S 1000: 26.2; 24.6 21.9 17.1 16.6    dQ: 34.4; 36.9 29.3 21.2 18.5
//                  q 128, S 2048: 46.3; 44.4 37.2 27.9 34.3        58.7; 67.9 50.1 33.6 37.7
//                  q 256, S 1024: 27.9; 27.3 24.9 30.9 45.7        36.0; 39.5 32.7 37.9 51.9
//                  q 512, S 2048: 51.8; 54.4 52.8 75.2             68.6; 80.2 70.4 96.0
//                  q 64,  S 512 : 16.9; 15.6 15.2 12.5 11.7        22.6; 21.8 20.0 15.9 13.3
// The smallest D 128 calls (S < 768, forward q <= 64, dQ q <= 48) stay on the assembly kernels although the
// split forms are the faster ones there: that is the path that tests/test_attn_gpu.py,
// tests/test_graph_gpu.py and tests/test_trained_attention_gpu.py hold the library to (q 12 and 32 in the
// first two, forward q 64 at most in the third).  The two bounds come from those shapes and not from a
// measurement; a call between them (q 64, S 512) runs its forward on the assembly and its dQ split, which
// costs the forward 16.8 us for 11.7.
// The figures above are of before the tile loop's scalar work fell; the forward's split forms and 1x4 have
// since gained 2 to 6% (D 64 q 256, S 1024: 2x2 11.6, bf16 13.6; D 128 q 256, S 1024: 2x4 21.9).
inline HipForm pick_rows_form(int D, bool dq, long long q, int S, bool causal, int n) {
    if (D == 128) {
        if ((q <= (dq ? 48 : 64) && S < 768) || q > n) return kFormAsm;
        if (S <= 256) return kForm2x4;
        return 4 * q <= n ? kForm4x1 : 2 * q <= n ? kForm4x2 : kForm2x4;
    }
    if (S <= 64 || q > n) return kForm1x4;
    if (2 * q <= n) return causal || 4 * q <= n ? kForm4x1 : S > 256 ? kForm4x2 : kForm2x2;
    return causal ? kForm2x2 : kForm2x4;
}

// dK/dV's form.  k: 128-key blocks of the launch (B * Hkv * blocks), g: query heads per kv head.
// Measured as above, 1x4, 2x2, 4x1, 8x1:
//   D 64  k 32,  S 512,  g 2: 33.2 19.3 12.4 11.3      k 256, S 512,  g 1: 20.4 14.0 17.2 27.5
//         k 64,  S 1024, g 4:  120 65.6 38.5 30.2      k 256, S 1024, g 1: 34.6 22.5 23.5 33.6
//         k 128, S 2048, g 4:  235  129 78.0 63.5      k 256, S 4096, g 4:  474  257  201  219
//          not causal       :  238  131  100  110        not causal      :  476  347  373  428
//         k 8,   S 128,  g 1:  8.0  6.0  5.1  6.4      k 1024,S 2048, g 1:  106  112  123  188
// Short lists (k 256, S 512) do not pay for the finer forms' further reads of K and V; long ones do.
//   D 128 (assembly; 4x1): k 12, S 700, g 8: 102; 79.3       k 32, S 512, g 2: 23.9; 21.0
//         k 64, S 1024, g 4: 76.9; 61.6                      k 256, S 512, g 1: 18.0; 46.0
//         k 128, S 2048, g 4: 148; 128, not causal 160; 241  k 144, S 1531, g 4: 113; 126
// and the smallest calls (k <= 24, lists under 2048 rows) stay on the assembly kernel for the reason above: the
// bounds are those tests' shapes (k 6 and 16), and k 32, S 512, g 2 shows what they cost.
inline HipForm pick_keys_form(int D, long long k, int S, int g, bool causal, int n) {
    const long long list = (long long)g * S;   // query rows a key block meets (not causal)
    if (D == 128) {
        if ((k <= 24 && list < 2048) || S <= 256) return kFormAsm;
        return 4 * k <= n || (causal && 2 * k <= n && S >= 1024) ? kForm4x1 : kFormAsm;
    }
    if (S <= 64) return kForm2x2;
    if (4 * k <= n) return S > 256 ? kForm8x1 : kForm4x1;
    if (2 * k <= n && S > 256) return causal ? kForm8x1 : kForm4x1;
    if (k <= n) return causal && list >= 4096 ? kForm4x1 : kForm2x2;
    return kForm1x4;
}

// Launchers return 0 (launched), -1 (HIP launch error) or -2 (the assembly code objects
// failed to load on a gfx950 device).
int launch_fwd(const FwdArgs& a);
int launch_fwd_asm(const FwdArgs& a);  // also 1 = configuration not handled there
int launch_bwd_delta(const BwdArgs& a);
int launch_bwd_dkdv(const BwdArgs& a);
int launch_bwd_dkdv_asm(const BwdArgs& a);  // 1 = configuration not handled there
int launch_bwd_dq_asm(const BwdArgs& a, bool compute_d);  // 1 = not handled there
int launch_bwd_dq(const BwdArgs& a);
int launch_bwd_dq_delta(const BwdArgs& a);  // dQ, and D written for launch_bwd_dkdv

}  // namespace tkm
