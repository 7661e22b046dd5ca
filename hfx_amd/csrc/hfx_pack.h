/*
 * hfx_pack.h -- several short candidates in one wave: the layout and the peak
 * writes that the sparse XCorr (FP32 sums) and the top-N (exact sums) share.
 *
 * A pack is up to XP_SLOTS consecutive candidates of at most 64 ladder
 * positions in all, one lane per (candidate, position).  Lanes OR the unary
 * weight codes of their peaks into their candidate's nibble map and claim them
 * back with atomic ANDs: the first claimant of a bin gets its final code.
 */
#pragma once

#include "hfx_cand.h"

#define XP_SLOTS 4
/* b-ladder positions a wave's buffer holds (a chunk of its candidates at a
 * time; any one packable candidate has at most 64): the more, the more lanes walk
 * ladders at once; past 288 a CU holds four workgroups instead of five (10.2
 * million modified candidates: 2,945 us with 256, 2,897 with 288, 3,131 with 320) */
#define XP_LB 288
/* Peaks outside [0, len) are clamped onto margin bins whose spectrum values
 * are zero (so they add 0 when claimed): singles onto bin -1 - 8 (lane & 7)
 * or len + 8 (lane & 7), triple centres onto -2 - 8 (lane & 7) or
 * len + 1 + 8 (lane & 7) (none of a clamped triple's nibbles is inside
 * [0, len)), spread over eight words a side so that they do not queue on
 * one address.  Clamped nibbles lie in [-59, len + 58]; the staged spectrum
 * is zero from bin -XP_PAD to len + XP_PAD and the map words cover bins
 * -XP_PAD .. xstr + XP_PAD. */
#define XP_SPREAD 8
#define XP_PAD (8 * XP_SPREAD)
static_assert(XP_PAD % 8 == 0 && XP_PAD >= 8 * (XP_SPREAD - 1) + 3, "clamped peaks inside the margins");

#define XP_MAGIC 12582912.0f /* 1.5 * 2^23: x + XP_MAGIC rounds x to an integer, ties to even */
#define XP_MAGIC_BITS 0x4B400000u

/* map words per candidate for spectra of at most xstr bins: bin x in word
 * (x + XP_PAD) / 8, x in [-XP_PAD, xstr + XP_PAD) */
static uint32_t xp_map_words(uint32_t xstr) { return (xstr + 2 * XP_PAD + 7) / 8 + 1; }
/* rint(mz / 1.0005079) as the bits of the integer-valued float q + 1.5 2^23
 * (q the correctly rounded quotient): u - XP_MAGIC_BITS is the bin for
 * |bin| < 2^22 */
__device__ __forceinline__ uint32_t xp_binu(float mz)
{
    const float R = 1.0f / HFX_BIN_WIDTH_MONO;
    return __float_as_uint(hfx_div(mz, HFX_BIN_WIDTH_MONO, R) + XP_MAGIC);
}

/* division by the fragment charge, correctly rounded (exact products for
 * 1, 2, 4) */
template <int Z>
__device__ __forceinline__ float xp_zdiv(float x)
{
    if constexpr (Z == 3) return hfx_div(x, 3.0f, 1.0f / 3.0f);
    else return x * (1.0f / (float)Z);
}

/* weight of a nibble holding the OR of unary codes: 0, 1, 3, 7 -> 0, 10,
 * 25, 50, one byte lookup (v_perm: selector c picks byte c of the pool
 * 0x32000000:19000A00) */
__device__ __forceinline__ float xp_weight(uint32_t nib)
{
    return (float)(__builtin_amdgcn_perm(0x32000000u, 0x19000A00u, nib) & 0xffu);
}

/* median of three unsigned (one v_med3_u32; the compiler does not fold a
 * min of a max with non-constant bounds) */
__device__ __forceinline__ uint32_t xp_med3(uint32_t v, uint32_t lo, uint32_t hi)
{
    uint32_t r;
    asm("v_med3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(lo), "v"(hi));
    return r;
}

/* the six bins of one ladder position at charge Z, in the FP32 operation
 * order of ion_series.cu:111-156 (addIonsAB, addIonsY), as xp_binu bits
 * (XP_MAGIC_BITS + bin) clamped into [lo, hi] (singles: a, b - H2O,
 * b - NH3, y - NH3) and [lo3, hi3] (triple centres b, y) */
struct XpClamp {
    uint32_t lo, hi, lo3, hi3;
};
template <int Z>
__device__ __forceinline__ void xp_bins(float b, float y, const XpClamp &c, uint32_t (&u)[6])
{
    constexpr float zh = HFX_DEV_H * (float)Z;
    constexpr float h2o = HFX_DEV_H2O / (float)Z, nh3 = HFX_DEV_NH3 / (float)Z;
    const float ma = xp_zdiv<Z>((b - HFX_DEV_CO) + zh);
    const float mb = xp_zdiv<Z>(b + zh);
    const float my = xp_zdiv<Z>((y + HFX_DEV_H2O) + zh);
    u[0] = xp_med3(xp_binu(ma), c.lo, c.hi);
    u[1] = xp_med3(xp_binu(mb), c.lo3, c.hi3);
    u[2] = xp_med3(xp_binu(mb - h2o), c.lo, c.hi);
    u[3] = xp_med3(xp_binu(mb - nh3), c.lo, c.hi);
    u[4] = xp_med3(xp_binu(my), c.lo3, c.hi3);
    u[5] = xp_med3(xp_binu(my - nh3), c.lo, c.hi);
}

/* the words and nibble shifts of one position's peaks: singles at word
 * w[i], triples over words w[i], w[i] + 1 from nibble shift sh[i]; u[i] the
 * bits of the single's bin or of the bin before the triple's centre.  rowm
 * and xsm are the map row and the staged spectrum shifted back by
 * XP_MAGIC_BITS bins (never dereferenced themselves): the magic constant's
 * low three bits are zero, so u >> 3 and u & 7 give the word and nibble */
struct XpPeaks {
    uint32_t *w[6];
    uint32_t sh[6];
    uint32_t u[6];
};

__device__ __forceinline__ void xp_locate(uint32_t *rowm, const uint32_t (&u)[6], XpPeaks &pk)
{
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const uint32_t ui = (i == 1 || i == 4) ? u[i] - 1u : u[i];
        pk.u[i] = ui;
        pk.w[i] = rowm + (ui >> 3);
        pk.sh[i] = (ui & 7u) * 4u;
    }
}

/* ORs the peaks of one position into the candidate's map: the four
 * weight-10 peaks alone, each 25/50/25 triple as one 12-bit field over two
 * words */
__device__ __forceinline__ void xp_put(const XpPeaks &pk)
{
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        if (i == 1 || i == 4) {
            const uint64_t t = (uint64_t)(HFX_CODE25 | HFX_CODE50 << 4 | HFX_CODE25 << 8)
                               << pk.sh[i];
            atomicOr(pk.w[i], (uint32_t)t);
            atomicOr(pk.w[i] + 1, (uint32_t)(t >> 32));
        } else {
            atomicOr(pk.w[i], HFX_CODE10 << pk.sh[i]);
        }
    }
}

/* a pack: K candidates, candidate g on lanes [st_g, st_{g+1}), first
 * residue tc_g, residual r_g; wave-uniform values (no arrays: a lane picks
 * its candidate's by comparisons) */
struct XpPack {
    uint32_t K;
    uint32_t st1, st2, st3, tot;
    uint32_t lb0, lb1, lb2, lb3; /* first ladder position of each in the wave's buffer */
    float r0, r1, r2, r3;
};

/* the pack that starts at candidate p of the chunk [base's candidate, q):
 * pr_n, pofs and pr_r are a lane's candidate's positions, first position in
 * the chunk's buffer (less base) and residual */
__device__ __forceinline__ XpPack xp_form(uint32_t p, uint32_t q, uint32_t pr_n, float pr_r,
                                          uint32_t pofs, uint32_t base)
{
    /* lanes past q are not taken */
    const uint32_t p1 = min(p + 1u, (uint32_t)HFX_WAVE - 1u);
    const uint32_t p2 = min(p + 2u, (uint32_t)HFX_WAVE - 1u);
    const uint32_t p3 = min(p + 3u, (uint32_t)HFX_WAVE - 1u);
    const uint32_t n0 = hfx_take(pr_n, p), n1 = hfx_take(pr_n, p1), n2 = hfx_take(pr_n, p2),
                   n3 = hfx_take(pr_n, p3);
    const bool t1 = p + 1 < q && n0 + n1 <= HFX_WAVE;
    const bool t2 = t1 && p + 2 < q && n0 + n1 + n2 <= HFX_WAVE;
    const bool t3 = t2 && p + 3 < q && n0 + n1 + n2 + n3 <= HFX_WAVE;
    XpPack pk;
    pk.K = 1u + (uint32_t)t1 + (uint32_t)t2 + (uint32_t)t3;
    pk.st1 = t1 ? n0 : 0xffffffffu;
    pk.st2 = t2 ? n0 + n1 : 0xffffffffu;
    pk.st3 = t3 ? n0 + n1 + n2 : 0xffffffffu;
    pk.tot = n0 + (t1 ? n1 : 0u) + (t2 ? n2 : 0u) + (t3 ? n3 : 0u);
    pk.lb0 = hfx_take(pofs, p) - base;
    pk.lb1 = hfx_take(pofs, p1) - base;
    pk.lb2 = hfx_take(pofs, p2) - base;
    pk.lb3 = hfx_take(pofs, p3) - base;
    pk.r0 = hfx_take(pr_r, p);
    pk.r1 = hfx_take(pr_r, p1);
    pk.r2 = hfx_take(pr_r, p2);
    pk.r3 = hfx_take(pr_r, p3);
    return pk;
}

/* this lane's place in a pack */
struct XpLane {
    uint32_t slot, kpos; /* candidate of the pack, ladder position */
    uint32_t k1;         /* one past the candidate's last lane */
    uint32_t lad;        /* first position of the candidate in the buffer */
    float r;
    bool act;
};
__device__ __forceinline__ XpLane xp_lane(const XpPack pk, uint32_t lane)
{
    const bool g1 = lane >= pk.st1, g2 = lane >= pk.st2, g3 = lane >= pk.st3;
    XpLane l;
    l.slot = (uint32_t)g1 + (uint32_t)g2 + (uint32_t)g3;
    l.act = lane < pk.tot;
    const uint32_t k0 = g3 ? pk.st3 : g2 ? pk.st2 : g1 ? pk.st1 : 0u;
    l.k1 = g3 ? pk.tot : g2 ? min(pk.st3, pk.tot) : g1 ? min(pk.st2, pk.tot) : min(pk.st1, pk.tot);
    l.lad = g3 ? pk.lb3 : g2 ? pk.lb2 : g1 ? pk.lb1 : pk.lb0;
    l.r = g3 ? pk.r3 : g2 ? pk.r2 : g1 ? pk.r1 : pk.r0;
    l.kpos = lane - k0;
    return l;
}

/* inclusive prefix of a wave's positions: pofs + n */
__device__ __forceinline__ uint32_t xp_prefix(uint32_t n, uint32_t lane)
{
    uint32_t incl = n;
#pragma unroll
    for (int o = 1; o < HFX_WAVE; o <<= 1) {
        const uint32_t v = __shfl_up(incl, o, 64);
        if (lane >= (uint32_t)o) incl += v;
    }
    return incl;
}
