/*
 * hfx_rows.h -- theoretical rows of 2-bit codes and their contraction
 * (hfx_rows.hip), for the sparse and the batched forms.
 */
#pragma once

#include "hfx_common.h"

#define RW_ROWS 16     /* peptides a tile */
#define RW_MAXK 2176   /* bins of a row */
#define RW_G 9         /* groups of 256 bins of a row */

/* precision forms: planes of a spectrum, spectra a block */
#define RW_I8X3 0
#define RW_I8X6 1
#define RW_BF16 2
#define RW_PLANES(mode) ((mode) == RW_I8X3 ? 3 : (mode) == RW_I8X6 ? 6 : 4)
#define RW_NS(mode) ((mode) == RW_I8X3 ? 16u : 8u)

/* rows[l - 1]: charge level l's tiles of G KiB each, or null; slots: tile t of
 * level l at place slots[(l - 1) ntiles + t] of rows[l - 1] (null: place t);
 * ng[t]: groups tile t's peaks reach (only those are written), the array padded to
 * whole words */
struct hfx_rows {
    uint8_t *rows[HFX_MAX_CHARGE];
    const uint64_t *slots;
    uint8_t *ng;
    uint32_t ntiles, G;
};

uint32_t hfx_rows_tiles(uint32_t num_pep);
uint32_t hfx_rows_groups(uint32_t x_stride);
uint32_t hfx_rows_chunk(uint64_t rows, uint32_t cus);
uint32_t hfx_rows_item_tiles(uint32_t CH);
/* spectra that are scored without rows (hfx_xcorr_rest), in any order */
struct hfx_rest {
    uint32_t *list, *count; /* [S]; cleared before hfx_rows_split (hfx_cut_bufs) */
};
/* planes [S][RW_PLANES][RW_MAXK] and quanta of the spectra, and the charge level of
 * each, 0 for those put on the list `rest`: charges above `have`, the highest level
 * there are rows for; windows past num_pep, the peptides there are rows of; in RW_I8X6
 * spectra with a value that six digits do not hold.  norms
 * [S], if any: sum and max of |x|.  The num[s] scores of spectra whose charge is not
 * generated are set to 0, and nothing between one spectrum's scores and the next's */
int hfx_rows_split(int mode, const hfx_spectra *sp, uint8_t *planes, float *qs, uint32_t *lvl,
                   const hfx_rest *rest, uint32_t have, float2 *norms, float *scores,
                   const uint64_t *off, const uint32_t *begin, const uint32_t *num, uint32_t num_pep,
                   void *stream);
/* writes the rows of the wanted levels (non-null) and tiles (flags
 * [HFX_MAX_CHARGE][ntiles], null: all) */
int hfx_rows_build(uint32_t cus, const hfx_db *db, const hfx_rows *r, const uint32_t *flags,
                   void *stream);
/* work items of the blocks bstart (num_spec + 1 entries, empty blocks at the
 * end) of hfx_rows_item_tiles(CH) tiles each, in scratch of
 * hfx_rows_items_bytes(num_spec) */
size_t hfx_rows_items_bytes(uint32_t S);
int hfx_rows_blocks(hfx_ctx *ctx, void *scratch, const uint32_t *order, const uint32_t *bstart,
                    const uint32_t *begin, const uint32_t *num, const hfx_spectra *sp, uint32_t CH,
                    void *stream);
/* flags [HFX_MAX_CHARGE][ntiles]: the tiles those items read */
int hfx_rows_mark(void *scratch, uint32_t S, uint32_t *flags, uint32_t ntiles, void *stream);
/* the scores of every item (sp's d_zmax may hide spectra from them) */
int hfx_rows_scores(hfx_ctx *ctx, int mode, void *scratch, float *d_scores, const uint64_t *d_off,
                    const uint32_t *begin, const uint32_t *num, const uint32_t *order,
                    const uint32_t *bstart, const hfx_rows *r, const uint8_t *planes,
                    const float *qs, const hfx_spectra *sp, uint32_t CH, void *stream, void **ev);

/* spectrum order and block cut (hfx_batch.hip) */
struct hfx_order_bufs {
    uint32_t sh, nbz, nb; /* buckets, from hfx_order_shape */
    uint32_t *cnt, *tmp;  /* [nb], [S] */
    uint64_t *off;        /* [nb + 1] */
};
void hfx_order_shape(uint32_t S, uint32_t num_pep, hfx_order_bufs *o);
/* order: (fragment charge level, precursor mass, or window begin where mass is
 * null, index); a permutation whatever begin and mass hold */
int hfx_order_spectra(hfx_ctx *ctx, uint32_t *order, const hfx_order_bufs *o,
                      const uint32_t *begin, const uint32_t *zmax, const float *mass, uint32_t S,
                      void *stream);
struct hfx_cut_bufs {
    uint32_t *seg, *n; /* [hfx_cut_segs(S) * 32], [hfx_cut_segs(S)] */
    uint64_t *off;     /* [hfx_cut_segs(S) + 1] */
    uint32_t *bstart;  /* [S + 1] */
    uint32_t *clear;   /* a word cleared on the way, if any */
};
uint32_t hfx_cut_segs(uint32_t S);
/* blocks of at most ns (8 or 16) consecutive ordered spectra */
int hfx_cut_blocks(hfx_ctx *ctx, uint32_t ns, const hfx_cut_bufs *c, const uint32_t *order,
                   const uint32_t *begin, const uint32_t *num, const uint32_t *zmax, uint32_t S,
                   void *stream);
