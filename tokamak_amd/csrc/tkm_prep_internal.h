/* Internal declarations shared by the host sources of libtkm_attn.so (not installed). */
#ifndef TKM_PREP_INTERNAL_H
#define TKM_PREP_INTERNAL_H

#include <stdarg.h>

#include "tkm_prep.h"

#ifdef __cplusplus
extern "C" {
#endif

#define TKM_HIDDEN __attribute__((visibility("hidden")))

/* Records a formatted message as the calling thread's last error and returns status. */
TKM_HIDDEN int tkm_set_error(int status, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
TKM_HIDDEN int tkm_vset_error(int status, const char *fmt, va_list ap);

/* Launch geometry of the generated qkv-prep kernels. */
enum {
    TKM_PREP_FWD_RPW = 4,          /* forward: rows per wave per block */
    TKM_PREP_BWD_BATCH = 4,        /* backward: rows per wave loaded before the arithmetic */
    TKM_BWD_TARGET_BLOCKS = 2048,  /* backward with parameter partials: at most about this many blocks */
    TKM_BWD_FREE_BLOCKS = 16384,   /* backward without: a band costs nothing but its block */
    TKM_REDUCE_WAVES = 16          /* partial-row reduction: waves per block (1024 threads) */
};

typedef struct {
    int D, C, QK, CH, QKCH, NH, G, part_width;
} tkm_prep_geom;

TKM_HIDDEN int tkm_prep_check_desc(const tkm_prep_desc *d);
TKM_HIDDEN void tkm_prep_geometry(const tkm_prep_desc *d, tkm_prep_geom *g);
/* Rows of a band (a block row of a backward) for `rows` rows and `xblocks` blocks across a row; `side` is the
 * rows that a block takes side by side, `partials` whether each band leaves a row of parameter
 * partials.  A band is a multiple of `side`, so that no part of a block idles in its last pass (but the last
 * band's, which may be short), and no more than one pass where the target blocks allow it: the rows a wave
 * walks one after the other cost more than the larger partials' reduction (4096 x 512: 446 us for 49
 * backwards against 528 at four passes).  Before, 4096 rows of three blocks gave bands of 6 rows, two passes
 * of which half of the second was idle, and rows of 256 channels filled half of each block.
 * 4096 rows: qkv-prep of 1536 channels 13.3 -> 12.4 us and its reduction 5.8 -> 4.0, gated pair of 1376
 * 13.5 -> 12.0; the epilogues of one decoder layer 85.7 -> 80.6 us. */
TKM_HIDDEN int tkm_bwd_band(int rows, int xblocks, int side, int partials);
/* Bands of `rows` rows, at least one. */
TKM_HIDDEN int tkm_bwd_bands(int rows, int band);
TKM_HIDDEN float tkm_rope_inv_freq(const tkm_prep_desc *d, int i);

/* Checks that the current device is gfx950, compiles src with hipRTC and loads it; *module
 * receives the hipModule_t. */
TKM_HIDDEN int tkm_rtc_load(const char *src, const char *name, void **module);
TKM_HIDDEN int tkm_rtc_function(void *module, const char *name, void **fn);
TKM_HIDDEN void tkm_rtc_unload(void *module);
TKM_HIDDEN int tkm_rtc_launch(void *fn, unsigned gx, unsigned gy, unsigned block, void **args, void *stream,
                              const char *what);

#ifdef __cplusplus
}
#endif

#endif
