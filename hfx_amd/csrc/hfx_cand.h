/*
 * hfx_cand.h -- candidate sets scored by the sparse XCorr and top-N kernels.
 *
 * A candidate set maps (spectrum s, k-th candidate of s) to the residues,
 * residual and residue masses of one theoretical spectrum:
 *   HfxPlainCands  unmodified peptides of the precursor window, in residual-
 *                  sorted order (Search.hs:151-165, prepare_scoring.cu:47-67);
 *   HfxModCands    modified peptides enumerated for the spectrum
 *                  (Search.hs:358-394: rows of the spectrum expanded to their
 *                  modified peptides, in enumeration order).
 */
#pragma once

#include "hfx_common.h"

#include <type_traits>

#define HFX_MTAB (32 + HFX_MAX_MA) /* residue masses, then the modable acids' additions */

/* Stage spectrum s of sp in LDS (xs) and the mass table (mtab); returns the
 * effective length, never above HFX_MAX_LEN or the stride. */
__device__ __forceinline__ uint32_t hfx_stage_spectrum(float *xs, float *mtab, const hfx_db &db,
                                                       const hfx_spectra &sp, uint32_t s)
{
    const uint32_t len = min(sp.d_len[s], min(sp.x_stride, (uint32_t)HFX_MAX_LEN));
    const float *xg = sp.d_x + (size_t)s * sp.x_stride;
    /* eight loads in flight per thread (clamped into the row) before the stores */
    constexpr uint32_t U = 8;
    for (uint32_t base = 0; base < len; base += U * blockDim.x) {
        float v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) v[u] = xg[min(base + u * blockDim.x + threadIdx.x, len - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = base + u * blockDim.x + threadIdx.x;
            if (i < len) xs[i] = v[u];
        }
    }
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? db.d_mass[threadIdx.x] : 0.0f;
    return len;
}

__device__ __forceinline__ uint32_t hfx_take(uint32_t v, uint32_t l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ float hfx_take(float v, uint32_t l)
{
    return __uint_as_float(hfx_take(__float_as_uint(v), l));
}

/* Max fragment charge actually generated: the reference launches nothing for
 * max_charge > 4 (ion_series.cu:334-342), leaving zero rows. */
__device__ __forceinline__ uint32_t hfx_zeff(uint32_t zmax)
{
    return zmax <= HFX_MAX_CHARGE ? zmax : 0u;
}

struct HfxPlainCands {
    hfx_db db;
    const uint32_t *begin; /* [S] first residual-sorted position of the window */
    const uint32_t *num;   /* [S] window size */
    const uint64_t *off;   /* [S+1] score offsets */

    __device__ __forceinline__ uint32_t count(uint32_t s) const { return num[s]; }
    __device__ __forceinline__ uint64_t base(uint32_t s) const { return off[s]; }
    __device__ __forceinline__ uint32_t zeff(uint32_t zmax) const { return hfx_zeff(zmax); }

    /* what the peaks of candidate k of spectrum s need from global memory
     * (prep: one lane's fetch; take: lane l's, to the whole wave) */
    struct Prep {
        uint32_t tc, n;
        float r;
    };
    __device__ __forceinline__ Prep prep(uint32_t s, uint32_t k) const
    {
        const uint32_t pep = db.d_idx_sorted[begin[s] + k];
        const uint32_t tc = db.d_tc[pep], tn = db.d_tn[pep];
        return Prep{tc, tn > tc ? tn - tc : 0u, db.d_r[pep]};
    }
    __device__ __forceinline__ static Prep take(const Prep &p, uint32_t l)
    {
        return Prep{hfx_take(p.tc, l), hfx_take(p.n, l), hfx_take(p.r, l)};
    }
    __device__ __forceinline__ void peaks_prep(uint32_t *map, const float *mtab, const Prep &p,
                                               uint32_t len, uint32_t zeff) const
    {
        hfx_wave_peaks(map, p.n, p.r, zeff, len, HfxPlainMass{db.d_ions + p.tc, mtab});
    }
    __device__ __forceinline__ void stage(float *) const {}
    /* one lane: the candidate's b ladder (sequential FP32 prefix of its
     * first nl residue masses) into dst, eight residues loaded ahead (the
     * last one re-read past the end) */
    __device__ __forceinline__ void ladder(const Prep &p, const float *mtab, float *dst,
                                           uint32_t nl) const
    {
        const uint8_t *res = db.d_ions + p.tc;
        float bl = 0.0f;
        for (uint32_t k = 0; k < nl; k += 8) {
            uint32_t a[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) a[j] = res[min(k + j, nl - 1u)];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                if (k + j < nl) {
                    bl = bl + mtab[HFX_ACID_IDX(a[j])];
                    dst[k + j] = bl;
                }
            }
        }
    }
};

struct HfxModCands {
    hfx_db db;
    hfx_modset ms;
    const uint64_t *off; /* [S+1] first modified peptide of each spectrum */

    __device__ __forceinline__ uint32_t count(uint32_t s) const
    {
        return (uint32_t)(off[s + 1] - off[s]);
    }
    __device__ __forceinline__ uint64_t base(uint32_t s) const { return off[s]; }
    /* addModIons dispatches max charges 1..10 (mion_series.cu:335-556) */
    __device__ __forceinline__ uint32_t zeff(uint32_t zmax) const { return zmax <= 10 ? zmax : 0u; }

    struct Prep {
        uint32_t tc, n, mod, uoff;
        float r;
    };
    __device__ __forceinline__ Prep prep(uint32_t s, uint32_t k) const
    {
        const uint64_t i = off[s] + k;
        const uint32_t pep = ms.d_mpep_pep_idx[i], mod = ms.d_mpep_mod_idx[i];
        const uint32_t tc = db.d_tc[pep], tn = db.d_tn[pep];
        return Prep{tc, tn > tc ? tn - tc : 0u, mod, ms.d_mpep_unrank_off[i],
                    db.d_r[pep] + ms.d_mod_delta[mod]};
    }
    __device__ __forceinline__ static Prep take(const Prep &p, uint32_t l)
    {
        return Prep{hfx_take(p.tc, l), hfx_take(p.n, l), hfx_take(p.mod, l), hfx_take(p.uoff, l),
                    hfx_take(p.r, l)};
    }
    __device__ __forceinline__ void peaks_prep(uint32_t *map, const float *mtab, const Prep &p,
                                               uint32_t len, uint32_t zeff) const
    {
        const uint32_t na = min(ms.num_ma, (uint32_t)HFX_MAX_MA);
        HfxModMass mm{db.d_ions + p.tc, mtab, ms.d_mod_ma_count + (size_t)p.mod * ms.num_ma,
                      ms.d_unrank + p.uoff, ms.d_ma_mass, na, {0, 0, 0, 0, 0, 0, 0}};
        hfx_wave_peaks(map, p.n, p.r, zeff, len, mm);
    }
    /* the acids' modification masses behind the residue masses */
    __device__ __forceinline__ void stage(float *mtab) const
    {
        if (threadIdx.x < HFX_MAX_MA)
            mtab[32 + threadIdx.x] = threadIdx.x < ms.num_ma ? ms.d_ma_mass[threadIdx.x] : 0.0f;
    }
    /* one lane: the modified candidate's b ladder over its first nl (<= 64)
     * positions.  A residue of modable acid a (code field a + 1) that is the
     * i-th of its acid in the peptide weighs table + ma_mass[a] when i is in
     * the acid's part of the unrank slice (HfxModMass's rule, per lane).
     * One word holds the acids' occurrence masks (64 / num_ma bits each) and one
     * their counters; four entries of the slice and eight residues are on their way at
     * a time.  A mask and a test for each acid took 940 of 3,206 us of 10.2 million
     * candidates; they take 2,800 now.  Occurrences that the masks do not hold (the
     * sixteenth of an acid, with four acids) are looked up in the slice. */
    __device__ __forceinline__ void ladder(const Prep &p, const float *mtab, float *dst,
                                           uint32_t nl) const
    {
        const uint32_t na = min(ms.num_ma, (uint32_t)HFX_MAX_MA);
        const uint32_t w = min(64u / max(na, 1u), 16u); /* bits of a mask */
        const uint32_t *row = ms.d_mod_ma_count + (size_t)p.mod * ms.num_ma;
        const uint32_t *u = ms.d_unrank + p.uoff;
        /* the acids' shares of the slice end here; then its entries, four reads at
         * a time */
        uint32_t ends[HFX_MAX_MA], tot = 0;
#pragma unroll
        for (uint32_t a = 0; a < HFX_MAX_MA; ++a) ends[a] = a < na ? row[a] : 0u;
#pragma unroll
        for (uint32_t a = 0; a < HFX_MAX_MA; ++a) ends[a] = tot += ends[a];
        uint64_t mask = 0;
        bool fits = true;
        for (uint32_t q = 0; q < tot; q += 4) {
            uint32_t e[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) e[j] = u[min(q + j, tot - 1u)];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (q + j < tot) {
                    uint32_t a = 0;
#pragma unroll
                    for (uint32_t i = 0; i + 1 < HFX_MAX_MA; ++i) a += q + j >= ends[i] ? 1u : 0u;
                    /* the last bit stays clear: it stands for every later occurrence */
                    if (e[j] + 1u < w) mask |= 1ull << (w * a + e[j]);
                    else fits = false;
                }
        }
        const uint8_t *res = db.d_ions + p.tc;
        uint32_t occ = 0; /* four bits an acid, staying at fifteen */
        float bl = 0.0f;
        for (uint32_t k = 0; k < nl; k += 8) {
            uint32_t x[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) x[j] = res[min(k + j, nl - 1u)];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
                if (k + j < nl) {
                    const uint32_t a = HFX_ACID_MOD(x[j]) - 1u;
                    float m = mtab[HFX_ACID_IDX(x[j])];
                    if (a < na) {
                        const uint32_t o = (occ >> (4 * a)) & 15u;
                        if ((mask >> (w * a + min(o, w - 1u))) & 1ull) m = m + mtab[32 + a];
                        occ += o < 15u ? 1u << (4 * a) : 0u;
                    }
                    bl = bl + m;
                    dst[k + j] = bl;
                }
        }
        if (!fits) far_ladder(p, mtab, dst, nl);
    }
    /* the same from the slice itself, for any occurrence */
    __device__ __forceinline__ void far_ladder(const Prep &p, const float *mtab, float *dst,
                                               uint32_t nl) const
    {
        const uint32_t na = min(ms.num_ma, (uint32_t)HFX_MAX_MA);
        const uint32_t *row = ms.d_mod_ma_count + (size_t)p.mod * ms.num_ma;
        const uint8_t *res = db.d_ions + p.tc;
        float bl = 0.0f;
        for (uint32_t k = 0; k < nl; ++k) {
            const uint32_t a = HFX_ACID_MOD(res[k]) - 1u;
            float m = mtab[HFX_ACID_IDX(res[k])];
            if (a < na) {
                uint32_t o = 0, off = 0;
                for (uint32_t j = 0; j < k; ++j) o += HFX_ACID_MOD(res[j]) - 1u == a ? 1u : 0u;
                for (uint32_t i = 0; i < a; ++i) off += row[i];
                bool hit = false;
                for (uint32_t q = 0; q < row[a]; ++q) hit = hit || ms.d_unrank[p.uoff + off + q] == o;
                if (hit) m = m + mtab[32 + a];
            }
            bl = bl + m;
            dst[k] = bl;
        }
    }
};
