/*
 * hfx_xcorr.hip -- plain FP32 sparse XCorr, dense drop-in rows, row MVM.
 *
 * The reference scores a spectrum by materialising a dense theoretical row
 * per candidate (addIons, ion_series.cu:150-232: memset + global atomicMax +
 * int->float rewrite) and multiplying with cuBLAS sgemv (Search.hs:242-245).
 * Here the theoretical peaks of one candidate live in a 1 KiB-per-wave LDS
 * nibble map (one nibble per bin, max per bin through a unary weight code)
 * and are dotted straight against the spectrum held in LDS: no dense row ever
 * reaches HBM.
 *
 * Work decomposition: one workgroup (4 waves) per (spectrum, chunk of up to
 * XP_CHUNK candidates) tile; the spectrum is staged in LDS once per tile; each
 * wave scores several short candidates at a time (ladders -> maps -> claims).
 * Large calls write each theoretical row once instead (hfx_rows.hip).
 */
#include "hfx_pack.h"
#include "hfx_rows.h"

#include <stdlib.h>

#include <mutex>

#define XC_THREADS 256
#define XC_WAVES (XC_THREADS / HFX_WAVE)

/* largest s with off[s] <= t, off has n+1 entries, off[0] = 0 */
__device__ __forceinline__ uint32_t find_segment(const uint64_t *off, uint32_t n, uint64_t t)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= t) lo = mid; else hi = mid;
    }
    return lo;
}

/* ------------------------------------------------------------------ */
/* Plain candidates, packed: several candidates per wave                 */
/* ------------------------------------------------------------------ */

/* One workgroup (four waves) per tile of up to XP_CHUNK candidates of one
 * spectrum; each wave takes a quarter of the tile and packs up to XP_SLOTS
 * consecutive candidates of at most 64 ladder positions in all into its 64
 * lanes, one lane per (candidate, ladder position):
 *   - the b ladder is the sequential FP32 prefix of each candidate's residue
 *     masses: at step j every lane at position j adds its residue mass to its
 *     left neighbour's finished sum (a DPP shift by one lane), so lane k
 *     holds ((m_0 + m_1) + ...) + m_k, the association of a sequential loop;
 *   - each lane ORs the unary weight codes of its peaks into its candidate's
 *     nibble map (OR of codes = code of the maximum weight), then claims
 *     them back with an atomic AND that clears them: the first claimant of a
 *     bin receives its final code and every bin counts once, so no lane
 *     scans the whole map, and the map is clean for the next pack;
 *   - the lanes' partial sums are reduced per candidate.
 * A candidate of more than 64 positions takes a wave of its own through the
 * general path (hfx_wave_peaks, hfx_wave_dot).
 * 10.2 million modified candidates take 2,800 us, by vector instructions (1.02 a
 * SIMD every four cycles) and LDS atomics (bank conflicts in a third of the cycles). */
#define XP_THREADS 256
#define XP_WAVES (XP_THREADS / HFX_WAVE)
#define XP_CHUNK 128
static_assert(XP_CHUNK / XP_WAVES <= HFX_WAVE, "a wave's candidates fit its lanes");
static size_t xp_lds_bytes(uint32_t xstr)
{
    const size_t xf = ((size_t)xstr + 2 * XP_PAD + 3) & ~(size_t)3;
    return xf * 4 + (size_t)XP_WAVES * XP_SLOTS * xp_map_words(xstr) * 4 +
           (size_t)XP_WAVES * XP_LB * 4;
}

/* claims the peaks of one position (clearing them) and adds weight * x of
 * every nibble it receives (clamped peaks sit on zero spectrum values), those of
 * the b ion's side and of the y ion's to sums of their own: shorter sums round
 * less */
template <class A>
__device__ __forceinline__ void xp_claim(const XpPeaks &pk, const float *xsm, A (&acc)[2])
{
    auto add = [](uint32_t nib, float x, A &sum) {
        if constexpr (sizeof(A) == 8) sum = __builtin_fma((double)xp_weight(nib), (double)x, sum);
        else sum = __builtin_fmaf(xp_weight(nib), x, sum);
    };
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const uint32_t sh = pk.sh[i];
        A &s = acc[i >= 4];
        if (i == 1 || i == 4) {
            const uint64_t t = (uint64_t)0xfffu << sh;
            const uint32_t o0 = atomicAnd(pk.w[i], ~(uint32_t)t);
            const uint32_t o1 = atomicAnd(pk.w[i] + 1, ~(uint32_t)(t >> 32));
            const uint32_t f = (uint32_t)(((uint64_t)o1 << 32 | o0) >> sh);
            const float *xv = xsm + pk.u[i];
            add(f & 15u, xv[0], s);
            add((f >> 4) & 15u, xv[1], s);
            add((f >> 8) & 15u, xv[2], s);
        } else {
            const uint32_t old = atomicAnd(pk.w[i], ~(0xfu << sh));
            add((old >> sh) & 15u, xsm[pk.u[i]], s);
        }
    }
}

/* the value of the lane before (0 in lane 0) */
__device__ __forceinline__ float xp_prev(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v),
                                                                 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}

__device__ __forceinline__ double xp_prev(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x138, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
/* lane l's value, l a lane's own (any, where l is not one) */
__device__ __forceinline__ float xp_from(float v, uint32_t l)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute((int)(l << 2), (int)__float_as_uint(v)));
}
__device__ __forceinline__ double xp_from(double v, uint32_t l)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(l << 2), (int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(l << 2), (int)(uint32_t)(u >> 32));
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

/* Inclusive segmented sum over the wave: lane l ends with the sum of the lanes of
 * its segment from the segment's first lane (kpos = 0) to l, by doubling steps
 * taken where kpos reaches back that far: the order of the additions is that of the
 * candidate's positions alone, so that a score has the same bits wherever its
 * candidate lies in a pack. */
template <class A>
__device__ __forceinline__ A xp_segsum(A v, uint32_t kpos, uint32_t lane)
{
#pragma unroll
    for (uint32_t o = 1; o < HFX_WAVE; o <<= 1) {
        A t = v;
        if (o <= 4) {
#pragma unroll
            for (uint32_t i = 0; i < o; ++i) t = xp_prev(t);
        } else {
            t = xp_from(v, lane - o);
        }
        v = kpos >= o ? v + t : v;
    }
    return v;
}

/* one pack at fragment charges 1..Z; the candidates' b ladders are in lb; sums in
 * A (float, or double rounded once) */
template <int Z, class A>
__device__ __forceinline__ void xp_pack(uint32_t *maps, uint32_t mstr, const float *xs,
                                        const float *lb, uint32_t len, const XpPack pk,
                                        float *out)
{
    const uint32_t lane = hfx_lane();
    const XpLane ln = xp_lane(pk, lane);
    const uint32_t slot = ln.slot, kpos = ln.kpos, k1 = ln.k1;
    const bool act = ln.act;
    const float b = act ? lb[ln.lad + kpos] : 0.0f;
    const float y = ln.r - b;
    /* bin x of this lane's candidate map is in word rowp[x >> 3]; rowm and
     * xsm index by the xp_binu bits instead */
    uint32_t *rowm = maps + slot * mstr + XP_PAD / 8 - (XP_MAGIC_BITS >> 3);
    const float *xsm = xs - XP_MAGIC_BITS;
    const uint32_t sp = (lane & (XP_SPREAD - 1)) * 8u;
    const XpClamp cl{XP_MAGIC_BITS - 1u - sp, XP_MAGIC_BITS + len + sp, XP_MAGIC_BITS - 2u - sp,
                     XP_MAGIC_BITS + len + 1u + sp};
    /* charges 1..Z: the bins of each (and, for Z <= 2, their words and
     * shifts) kept in registers from the OR pass to the claim pass */
    uint32_t xz[Z][6];
    A acc[2] = {0, 0};
    if constexpr (Z <= 2) {
        XpPeaks pks[Z];
        if (act) {
            xp_bins<1>(b, y, cl, xz[0]);
            xp_locate(rowm, xz[0], pks[0]);
            if constexpr (Z >= 2) { xp_bins<2>(b, y, cl, xz[1]); xp_locate(rowm, xz[1], pks[1]); }
#pragma unroll
            for (int z = 0; z < Z; ++z) xp_put(pks[z]);
        }
        hfx_wave_sync();
        if (act) {
#pragma unroll
            for (int z = 0; z < Z; ++z) xp_claim(pks[z], xsm, acc);
        }
    } else {
        if (act) {
            xp_bins<1>(b, y, cl, xz[0]);
            xp_bins<2>(b, y, cl, xz[1]);
            xp_bins<3>(b, y, cl, xz[2]);
            if constexpr (Z >= 4) xp_bins<4>(b, y, cl, xz[3]);
#pragma unroll
            for (int z = 0; z < Z; ++z) {
                XpPeaks pk;
                xp_locate(rowm, xz[z], pk);
                xp_put(pk);
            }
        }
        hfx_wave_sync();
        if (act) {
#pragma unroll
            for (int z = 0; z < Z; ++z) {
                XpPeaks pk;
                xp_locate(rowm, xz[z], pk);
                xp_claim(pk, xsm, acc);
            }
        }
    }
    const float sc = (float)xp_segsum(acc[0] + acc[1], kpos, lane);
    hfx_wave_sync();
    /* the last lane of each candidate holds its score; a candidate without
     * positions scores 0 */
    if (act && lane + 1 == k1) out[slot] = sc;
    if (lane < pk.K) {
        const uint32_t a = lane == 0 ? 0u : lane == 1 ? pk.st1 : lane == 2 ? pk.st2 : pk.st3;
        const uint32_t e = lane == 0 ? min(pk.st1, pk.tot) : lane == 1 ? min(pk.st2, pk.tot)
                         : lane == 2 ? min(pk.st3, pk.tot) : pk.tot;
        if (a == e) out[lane] = 0.0f;
    }
}

/* the tile of spectrum s from its candidate `first` on; every thread of the
 * workgroup calls it */
template <class A, class Cands>
__device__ __forceinline__ void xp_tile(float *xp_lds, float *mtab, float *scores, const Cands &c,
                                        const hfx_spectra &sp, uint32_t mstr, uint32_t s,
                                        uint32_t first, uint32_t chunk)
{
    const uint32_t cnt = min(chunk, c.count(s) - first);
    const uint32_t xstr = sp.x_stride;
    const uint32_t xf = (xstr + 2 * XP_PAD + 3) & ~3u;
    float *xs = xp_lds + XP_PAD;
    uint32_t *maps_all = (uint32_t *)(xp_lds + xf);
    const uint32_t lane = hfx_lane(), wave = threadIdx.x / HFX_WAVE;
    uint32_t *maps = maps_all + wave * XP_SLOTS * mstr;
    float *lb = (float *)(maps_all + XP_WAVES * XP_SLOTS * mstr) + wave * XP_LB;
    const uint32_t len = hfx_stage_spectrum(xs, mtab, c.db, sp, s);
    c.stage(mtab);
    /* zeros around the spectrum: clamped peaks read them */
    for (uint32_t i = len + threadIdx.x; i < xf - XP_PAD; i += XP_THREADS) xs[i] = 0.0f;
    for (uint32_t i = threadIdx.x; i < XP_PAD; i += XP_THREADS) xp_lds[i] = 0.0f;
    for (uint32_t i = lane; i < XP_SLOTS * mstr; i += HFX_WAVE) maps[i] = 0u;
    __syncthreads();
    const uint32_t zeff = c.zeff(sp.d_zmax[s]);
    /* this wave's candidates [c0, c0 + rn) of the tile */
    const uint32_t range = chunk / XP_WAVES, c0 = wave * range;
    const uint32_t rn = __builtin_amdgcn_readfirstlane(
        c0 < cnt ? min(range, cnt - c0) : 0u);
    float *out = scores + c.base(s) + first + c0;
    if (rn == 0) return;
    if (zeff == 0) {
        /* no fragment charge generated (ion_series.cu:334-342): score 0 */
        if (lane < rn) out[lane] = 0.0f;
        return;
    }
    /* lane i < rn: candidate c0 + i's first residue, positions, residual */
    typename Cands::Prep pr{};
    if (lane < rn) pr = c.prep(s, first + c0 + lane);
    /* the packed peaks serve fragment charges 1..4; above (modified
     * candidates only: addModIons goes to 10) every candidate takes the
     * general path */
    const bool general = zeff > 4;
    /* ladder positions of the packable candidates (long ones take none):
     * exclusive prefix over the wave's candidates */
    const uint32_t nl = lane < rn && pr.n <= HFX_WAVE && !general ? pr.n : 0u;
    const uint32_t incl = xp_prefix(nl, lane);
    const uint32_t pofs = incl - nl;
    for (uint32_t p = 0; p < rn;) {
        /* a chunk [p, q) of candidates whose ladders fit the wave's buffer,
         * computed one candidate a lane: the sequential FP32 prefix of its
         * residue masses */
        const uint32_t base = hfx_take(pofs, p);
        const uint64_t fit = __ballot(lane >= p && lane < rn && incl - base <= XP_LB);
        const uint32_t q = p + (uint32_t)__builtin_popcountll(fit);
        if (lane >= p && lane < q && nl) c.ladder(pr, mtab, lb + (pofs - base), nl);
        hfx_wave_sync();
        while (p < q) {
            const uint32_t n0 = hfx_take(pr.n, p);
            if (n0 > HFX_WAVE || general) {
                /* a long candidate: the general path over chunks of 64 */
                const typename Cands::Prep qq = Cands::take(pr, p);
                c.peaks_prep(maps + XP_PAD / 8, mtab, qq, len, zeff);
                hfx_wave_sync();
                const float sc = (float)hfx_wave_dot<A>(maps + XP_PAD / 8, xs, len);
                hfx_wave_sync();
                if (lane == 0) out[p] = sc;
                ++p;
                continue;
            }
            const XpPack pk = xp_form(p, q, pr.n, pr.r, pofs, base);
            switch (zeff) {
            case 1: xp_pack<1, A>(maps, mstr, xs, lb, len, pk, out + p); break;
            case 2: xp_pack<2, A>(maps, mstr, xs, lb, len, pk, out + p); break;
            case 3: xp_pack<3, A>(maps, mstr, xs, lb, len, pk, out + p); break;
            default: xp_pack<4, A>(maps, mstr, xs, lb, len, pk, out + p); break;
            }
            p += pk.K;
        }
        hfx_wave_sync(); /* the buffer is rewritten by the next chunk */
    }
}

template <class Cands>
__global__ void __launch_bounds__(XP_THREADS)
    k_xcorr_pack(float *scores, const uint64_t *tile_off, Cands c, hfx_spectra sp, uint32_t mstr,
                 uint32_t chunk)
{
    extern __shared__ __align__(16) float xp_lds[];
    __shared__ float mtab[HFX_MTAB];
    const uint32_t S = sp.num_spec;
    const uint64_t t = blockIdx.x;
    if (t >= tile_off[S]) return;
    const uint32_t s = find_segment(tile_off, S, t);
    xp_tile<float>(xp_lds, mtab, scores, c, sp, mstr, s, (uint32_t)(t - tile_off[s]) * chunk, chunk);
}

/* The spectra that have no rows, or not in their form (seldom any: then a launch that
 * reads one word): persistent workgroups take every G-th of their tiles, of XR_CHUNK
 * candidates, so that one spectrum's window is spread over the chip. */
#define XR_CHUNK 32
template <class A>
__global__ void __launch_bounds__(XP_THREADS)
    k_xcorr_rest(float *scores, HfxPlainCands c, hfx_spectra sp, hfx_rest rest, uint32_t mstr)
{
    extern __shared__ __align__(16) float xp_lds[];
    __shared__ float mtab[HFX_MTAB];
    const uint32_t F = *rest.count;
    uint64_t at = blockIdx.x; /* of the tiles from the j-th spectrum on */
    for (uint32_t j = 0; j < F; ++j) {
        const uint32_t s = rest.list[j];
        const uint32_t nt = c.count(s) / XR_CHUNK + (c.count(s) % XR_CHUNK ? 1u : 0u);
        for (; at < nt; at += gridDim.x) {
            xp_tile<A>(xp_lds, mtab, scores, c, sp, mstr, s, (uint32_t)at * XR_CHUNK, XR_CHUNK);
            __syncthreads(); /* its LDS is staged anew */
        }
        at -= nt;
    }
}

/* Candidates a tile takes, a multiple of XP_WAVES up to XP_CHUNK.  A wave's share
 * is a chain of packs, and few tiles leave CUs idle; many small ones stage the
 * spectrum too often.  Scores of 100 spectra (33,460 pairs of short peptides):
 * 25 us with 16, 21 with 32, 31 with 64, 48 with 128; 16,183 pairs 17.4, 17.8,
 * 26, 41; 131,032 pairs 69, 51, 49, 56; 457,000 pairs 207, 140, 121, 124; long
 * peptides move the lines up (48,347 pairs 33, 37, 55, 87; 365,831 pairs 186, 146,
 * 151, 157); 10.2 million modified ones take 9 % more with 64 than with 128. */
static uint32_t xp_chunk(uint64_t total)
{
    return total <= 24000 ? 16u : total <= 160000 ? 32u : total <= 1000000 ? 64u : XP_CHUNK;
}

template <class Cands>
__global__ void k_tile_count(uint32_t *tiles, Cands c, uint32_t num_spec, uint32_t chunk)
{
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < num_spec) tiles[s] = (c.count(s) + chunk - 1) / chunk;
}

/* device scratch of the sparse XCorr for S spectra: per-spectrum tile counts
 * and their offsets */
static size_t xc_scratch_bytes(uint32_t S) { return (size_t)S * 4 + ((size_t)S + 1) * 8 + 64; }

template <class Cands>
static int launch_xcorr(void *scratch, float *d_scores, const Cands &c, uint64_t total,
                        const hfx_spectra *sp, void *stream)
{
    const uint32_t S = sp->num_spec;
    if (S == 0 || total == 0) return HFX_OK;
    HFX_REQUIRE(sp->x_stride <= HFX_MAX_LEN, HFX_ERR_ARG,
                "sparse XCorr: spectra of up to %d bins (x_stride %u)", HFX_MAX_LEN, sp->x_stride);
    const uint32_t chunk = xp_chunk(total);
    hipStream_t st = hfx_stream(stream);
    int rc;
    uint32_t *tiles = (uint32_t *)scratch;
    uint64_t *tile_off = (uint64_t *)(((uintptr_t)(tiles + S) + 15) & ~(uintptr_t)15);
    hipLaunchKernelGGL(k_tile_count<Cands>, dim3((S + 255) / 256), dim3(256), 0, st, tiles, c, S,
                       chunk);
    if ((rc = hfx_scan_offsets(nullptr, tile_off, tiles, S, stream)) != HFX_OK) return rc;
    /* sum_s ceil(n_s / chunk) <= total / chunk + S */
    const uint64_t grid = (total + chunk - 1) / chunk + S;
    HFX_REQUIRE(grid < (1ull << 31), HFX_ERR_ARG, "xcorr: %llu tiles", (unsigned long long)grid);
    hipLaunchKernelGGL(k_xcorr_pack<Cands>, dim3((uint32_t)grid), dim3(XP_THREADS),
                       xp_lds_bytes(sp->x_stride), st, d_scores, tile_off, c, *sp,
                       xp_map_words(sp->x_stride), chunk);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

int hfx_xcorr_rest(hfx_ctx *ctx, float *d_scores, const uint64_t *d_off, const uint32_t *d_begin,
                   const uint32_t *d_num, const hfx_db *db, const hfx_spectra *sp,
                   const hfx_rest *rest, int fp64, void *stream)
{
    if (sp->num_spec == 0) return HFX_OK;
    HfxPlainCands c{*db, d_begin, d_num, d_off};
    hipLaunchKernelGGL(fp64 ? k_xcorr_rest<double> : k_xcorr_rest<float>,
                       dim3((uint32_t)hfx_ctx_num_cus(ctx) * 4u), dim3(XP_THREADS),
                       xp_lds_bytes(sp->x_stride), hfx_stream(stream), d_scores, c, *sp, *rest,
                       xp_map_words(sp->x_stride));
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* ------------------------------------------------------------------ */
/* Rows route                                                            */
/* ------------------------------------------------------------------ */

/* hfx_xcorr_sparse writes each candidate's theoretical row once and contracts the
 * rows with blocks of eight spectra (hfx_rows.hip, fixed point that holds them) instead
 * of building a row per pair, where that is quicker.  In ns: a pair costs 0.2
 * more to score by itself than through its row; the rows' dozen launches 80,000 more
 * than the packed kernel's three; a tile of the database 1/3 to look at and, if a
 * window holds it, 2.7 at each charge level to write and read (as many as the
 * pairs fill, at most two levels of all).  Measured, packed and rows, us: 2,000
 * proteins, short peptides (7,293 tiles) 520,778 pairs 135 and 152, 1,043,828
 * pairs 236 and 170; longer ones (17,089 tiles) 365,831 pairs 155 and 168, 733,473
 * pairs 229 and 205; 20,000 proteins (72,760 and 170,538 tiles) 1,240,720 pairs
 * 262 and 328, 2,546,519 475 and 462; 1,839,460 446 and 534, 3,771,758 812 and 772,
 * 5,577,139 1,170 and 959, 45,788,296 9,120 and 1,790. */
static bool xr_pays(uint64_t total, uint32_t tiles)
{
    const uint64_t read = min(total / RW_ROWS, 2ull * tiles);
    return total / 5 > 80000ull + tiles / 3 + read * 27 / 10;
}

/* *taken = 0: nothing done (too few pairs, rows longer than the form's, no
 * memory to spare, a captured stream) */
static int xcorr_rows(hfx_ctx *ctx, float *d_scores, const uint64_t *d_off,
                      const uint32_t *d_begin, const uint32_t *d_num, uint64_t total,
                      const hfx_db *db, const hfx_spectra *sp, void *stream, int *taken)
{
    *taken = 0;
    /* the buffers are this call's until its work is launched */
    struct Spare {
        hfx_ctx *c;
        explicit Spare(hfx_ctx *ctx) : c(ctx) { hfx_ctx_spare_begin(c); }
        ~Spare() { hfx_ctx_spare_end(c); }
    } spare(ctx);
    const uint32_t S = sp->num_spec;
    const uint32_t nt = hfx_rows_tiles(db->num_pep), G = hfx_rows_groups(sp->x_stride);
    if (!xr_pays(total, nt) || sp->x_stride > RW_MAXK || db->num_pep == 0) return HFX_OK;
    /* a captured call keeps the packed kernel: a graph would hold these buffers, which
     * a larger call replaces and a shortage of memory takes back */
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(hfx_stream(stream), &cs) != hipSuccess ||
        cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return HFX_OK;
    }
    const uint64_t nf = (uint64_t)HFX_MAX_CHARGE * nt;
    if (nf >= 0xffffffffull) return HFX_OK;
    /* the block cut never takes more rows than the windows one by one */
    const uint64_t slots = min(nf, total / RW_ROWS + 2ull * S);
    hfx_order_bufs ob;
    hfx_order_shape(S, db->num_pep, &ob);
    const uint32_t nseg = hfx_cut_segs(S);
    auto al = [](uint64_t n) { return (n + 255) & ~(uint64_t)255; };
    const uint64_t sizes[] = {
        al((uint64_t)S * RW_PLANES(RW_I8X6) * RW_MAXK), al(4ull * S), al(4ull * S), al(4ull * S + 4),
        al(4ull * S), al(4ull * ob.nb), al(4ull * S), al(8ull * ob.nb + 8), al(4ull * nseg * 32),
        al(4ull * nseg), al(8ull * nseg + 8), al(4ull * S + 4), al(hfx_rows_items_bytes(S)),
        al(4 * nf), al(8 * nf + 8), al(nt + 4ull)};
    uint64_t bytes = 0;
    for (uint64_t z : sizes) bytes += z;
    uint8_t *p = (uint8_t *)hfx_ctx_scratch_spare(ctx, HFX_SLOT_ROWS, bytes);
    if (!p) return HFX_OK;
    uint8_t *rows = (uint8_t *)hfx_ctx_scratch_spare(ctx, HFX_SLOT_ROWS2, slots * G * 1024ull);
    if (!rows) return HFX_OK;
    uint8_t *part[sizeof sizes / sizeof *sizes];
    for (size_t i = 0; i < sizeof sizes / sizeof *sizes; ++i) {
        part[i] = p;
        p += sizes[i];
    }
    uint8_t *planes = part[0];
    float *qs = (float *)part[1];
    uint32_t *lvl = (uint32_t *)part[2], *order = (uint32_t *)part[4];
    const hfx_rest rest{(uint32_t *)part[3], (uint32_t *)part[3] + S};
    ob.cnt = (uint32_t *)part[5];
    ob.tmp = (uint32_t *)part[6];
    ob.off = (uint64_t *)part[7];
    const hfx_cut_bufs cb{(uint32_t *)part[8], (uint32_t *)part[9], (uint64_t *)part[10],
                          (uint32_t *)part[11], rest.count};
    void *items = part[12];
    uint32_t *flags = (uint32_t *)part[13];
    hfx_rows r{};
    r.slots = (uint64_t *)part[14];
    r.ng = part[15];
    r.ntiles = nt;
    r.G = G;
    for (int l = 0; l < HFX_MAX_CHARGE; ++l) r.rows[l] = rows;
    hfx_spectra sq = *sp;
    sq.d_zmax = lvl; /* the rest hidden from the items */
    const uint64_t est = max(total / 12, min(total, 2ull * db->num_pep));
    const uint32_t CH = hfx_rows_chunk(est, (uint32_t)hfx_ctx_num_cus(ctx));
    int rc;
    if ((rc = hfx_order_spectra(ctx, order, &ob, d_begin, sp->d_zmax, nullptr, S, stream)) ||
        (rc = hfx_cut_blocks(ctx, RW_NS(RW_I8X6), &cb, order, d_begin, d_num, sp->d_zmax, S, stream)) ||
        (rc = hfx_rows_split(RW_I8X6, sp, planes, qs, lvl, &rest, HFX_MAX_CHARGE, nullptr, d_scores,
                             d_off, d_begin, d_num, db->num_pep, stream)) ||
        (rc = hfx_rows_blocks(ctx, items, order, cb.bstart, d_begin, d_num, &sq, CH, stream)) ||
        (rc = hfx_rows_mark(items, S, flags, nt, stream)) ||
        (rc = hfx_scan_offsets(ctx, (uint64_t *)r.slots, flags, (uint32_t)nf, stream)) ||
        (rc = hfx_rows_build((uint32_t)hfx_ctx_num_cus(ctx), db, &r, flags, stream)) ||
        (rc = hfx_rows_scores(ctx, RW_I8X6, items, d_scores, d_off, d_begin, d_num, order,
                              cb.bstart, &r, planes, qs, &sq, CH, stream, nullptr)) ||
        (rc = hfx_xcorr_rest(ctx, d_scores, d_off, d_begin, d_num, db, sp, &rest, 0, stream)))
        return rc;
    *taken = 1;
    return HFX_OK;
}

extern "C" int hfx_xcorr_sparse(hfx_ctx *ctx, float *d_scores, const uint64_t *d_off,
                                const uint32_t *d_begin, const uint32_t *d_num, uint64_t total,
                                const hfx_db *db, const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(ctx && d_scores && d_off && d_begin && d_num && db && sp, HFX_ERR_ARG,
                "hfx_xcorr_sparse: null argument");
    HfxPlainCands c{*db, d_begin, d_num, d_off};
    void *p = nullptr;
    int rc, taken = 0;
    /* whichever kernel scores: a captured call after this one finds the table there */
    if (sp->num_spec &&
        (rc = hfx_ctx_scratch(ctx, HFX_SLOT_TILES, xc_scratch_bytes(sp->num_spec), &p)) != HFX_OK)
        return rc;
    if ((rc = xcorr_rows(ctx, d_scores, d_off, d_begin, d_num, total, db, sp, stream, &taken)) ||
        taken)
        return rc;
    return launch_xcorr(p, d_scores, c, total, sp, stream);
}

extern "C" int hfx_xcorr_sparse_mod(hfx_ctx *ctx, float *d_scores, const uint64_t *d_mp_off,
                                    uint64_t total, const hfx_modset *ms, const hfx_db *db,
                                    const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(ctx && d_scores && d_mp_off && ms && db && sp, HFX_ERR_ARG,
                "hfx_xcorr_sparse_mod: null argument");
    HFX_REQUIRE(ms->num_ma <= HFX_MAX_MA, HFX_ERR_ARG, "hfx_xcorr_sparse_mod: num_ma %u > %d",
                ms->num_ma, HFX_MAX_MA);
    HfxModCands c{*db, *ms, d_mp_off};
    void *p = nullptr;
    int rc;
    if (sp->num_spec &&
        (rc = hfx_ctx_scratch(ctx, HFX_SLOT_TILES, xc_scratch_bytes(sp->num_spec), &p)) != HFX_OK)
        return rc;
    return launch_xcorr(p, d_scores, c, total, sp, stream);
}

/* ------------------------------------------------------------------ */
/* hfx_xcorr_sparse for callers that cannot allocate                     */
/* ------------------------------------------------------------------ */

/* The tile table of up to HFX_NOALLOC_MAX_SPECTRA spectra lives in this
 * file-scope device array (12 MiB, held by every GPU the library runs on
 * until the process ends).  In host code `scratch` names a host-side stand-in,
 * never the device memory: the device address comes from
 * hipGetSymbolAddress, once per device, and only that address is passed on. */
#define NA_BYTES (((size_t)HFX_NOALLOC_MAX_SPECTRA * 4 + ((size_t)HFX_NOALLOC_MAX_SPECTRA + 1) * 8 + \
                   64 + 255) & ~(size_t)255)
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

#define NA_MAX_DEVICES 64
static std::mutex g_na_mu;
static void *g_na_ptr[NA_MAX_DEVICES];

/* the current device's address of `scratch`, looked up on the first call on
 * that device */
static int na_scratch(void **out)
{
    int dev = 0;
    HFX_CHECK_HIP(hipGetDevice(&dev));
    HFX_REQUIRE(dev >= 0 && dev < NA_MAX_DEVICES, HFX_ERR_ARG, "no-alloc scratch: device %d", dev);
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
        void *p = nullptr;
        HFX_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        HFX_REQUIRE(p != nullptr, HFX_ERR_HIP, "no-alloc scratch: no device address");
        g_na_ptr[dev] = p;
    }
    *out = g_na_ptr[dev];
    return HFX_OK;
}

extern "C" int hfx_xcorr_sparse_noalloc(float *d_scores, const uint64_t *d_off,
                                        const uint32_t *d_begin, const uint32_t *d_num,
                                        uint64_t total, const hfx_db *db, const hfx_spectra *sp,
                                        void *stream)
{
    HFX_REQUIRE(d_scores && d_off && d_begin && d_num && db && sp, HFX_ERR_ARG,
                "hfx_xcorr_sparse_noalloc: null argument");
    HFX_REQUIRE(sp->num_spec <= HFX_NOALLOC_MAX_SPECTRA, HFX_ERR_ARG,
                "hfx_xcorr_sparse_noalloc: %u spectra, at most %u in one call", sp->num_spec,
                (unsigned)HFX_NOALLOC_MAX_SPECTRA);
    static_assert(NA_BYTES >= ((size_t)HFX_NOALLOC_MAX_SPECTRA * 4 +
                               ((size_t)HFX_NOALLOC_MAX_SPECTRA + 1) * 8 + 64),
                  "no-alloc scratch holds the tile table of the largest call");
    if (sp->num_spec == 0 || total == 0) return HFX_OK;
    void *p = nullptr;
    int rc;
    if ((rc = na_scratch(&p))) return rc;
    HfxPlainCands c{*db, d_begin, d_num, d_off};
    return launch_xcorr(p, d_scores, c, total, sp, stream);
}

/* ------------------------------------------------------------------ */
/* Dense rows for the reference ABI (addIons, ion_series.cu:319-343)     */
/* ------------------------------------------------------------------ */

/* One wave per row: map -> dense row of floats 0/10/25/50, every element
 * written (no memset needed, no cross-block race).  Lanes take consecutive
 * bins, eight of them reading one map word, so that a store is 256 contiguous
 * bytes (a map word a lane made eight stores of 64 separate sectors). */
__device__ __forceinline__ void wave_map_to_row(uint32_t *map, float *row, uint32_t len)
{
    const uint32_t lane = hfx_lane(), nw = (len + 7) >> 3;
    constexpr uint32_t U = 8; /* map words read ahead of the stores */
    for (uint32_t b0 = lane; b0 < len; b0 += U * HFX_WAVE) {
        uint32_t w[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) w[u] = map[min(b0 + u * HFX_WAVE, len - 1u) >> 3];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t b = b0 + u * HFX_WAVE;
            if (b < len) row[b] = hfx_code_weight((w[u] >> (4 * (b & 7u))) & 0xFu);
        }
    }
    hfx_wave_sync();
    for (uint32_t w = lane; w < nw; w += HFX_WAVE) map[w] = 0;
}

__global__ void __launch_bounds__(XC_THREADS)
    k_add_ions(float *spec, const float *residual, const float *mass, const uint8_t *ions_all,
               const uint32_t *tc_a, const uint32_t *tn_a, const uint32_t *idx, uint32_t num_idx,
               uint32_t zmax, uint32_t len)
{
    __shared__ uint32_t maps[XC_WAVES][HFX_MAP_WORDS];
    __shared__ float mtab[32];
    const uint32_t wave = threadIdx.x / HFX_WAVE;
    uint32_t *map = maps[wave];
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? mass[threadIdx.x] : 0.0f;
    for (uint32_t w = hfx_lane(); w < HFX_MAP_WORDS; w += HFX_WAVE) map[w] = 0;
    __syncthreads();
    for (uint32_t row = blockIdx.x * XC_WAVES + wave; row < num_idx; row += gridDim.x * XC_WAVES) {
        const uint32_t pep = idx[row];
        const uint32_t tc = tc_a[pep], tn = tn_a[pep];
        const uint32_t n = tn > tc ? tn - tc : 0;
        hfx_wave_peaks(map, n, residual[pep], zmax, len, HfxPlainMass{ions_all + tc, mtab});
        hfx_wave_sync();
        wave_map_to_row(map, spec + (size_t)row * len, len);
        hfx_wave_sync();
    }
}

extern "C" void addIons(float *d_spec, const float *d_residual, const float *d_mass,
                        const uint8_t *d_ions, const uint32_t *d_tc, const uint32_t *d_tn,
                        const uint32_t *d_idx, const uint32_t num_idx, const uint32_t max_charge,
                        const uint32_t len_spec)
{
    if (num_idx == 0) return;
    if (max_charge < 1 || max_charge > HFX_MAX_CHARGE) {
        hfx_set_error("addIons: max_charge %u outside 1..4 (no kernel launched)", max_charge);
        return;
    }
    if (len_spec > HFX_MAX_LEN) {
        hfx_set_error("addIons: len_spec %u > %d", len_spec, HFX_MAX_LEN);
        return;
    }
    uint32_t blocks = min((num_idx + XC_WAVES - 1) / XC_WAVES, 65535u);
    hipLaunchKernelGGL(k_add_ions, dim3(blocks), dim3(XC_THREADS), 0, 0, d_spec, d_residual, d_mass,
                       d_ions, d_tc, d_tn, d_idx, num_idx, max_charge, len_spec);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("addIons: %s", hipGetErrorString(e));
}

/* ------------------------------------------------------------------ */
/* Row MVM replacing cuBLAS sgemv(T)                                    */
/* ------------------------------------------------------------------ */

/* A wave a row; a lane's products j = lane, lane + 64, ... are added in that
 * order, eight of its loads in flight at a time (one after the other, 366 rows
 * of 1,400 took 10.7 us: too few waves to hide the loads' latency). */
__global__ void __launch_bounds__(256) k_mvm_rows(float *y, const float *A, uint32_t lda,
                                                  const float *x, uint32_t m, uint32_t n)
{
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / HFX_WAVE;
    if (row >= m) return;
    const float *a = A + (size_t)row * lda;
    float acc = 0.0f;
    constexpr uint32_t U = 8;
    uint32_t j = hfx_lane();
    for (; j + (U - 1) * HFX_WAVE < n; j += U * HFX_WAVE) {
        float av[U], xv[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            av[u] = a[j + u * HFX_WAVE];
            xv[u] = x[j + u * HFX_WAVE];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) acc = acc + av[u] * xv[u];
    }
    /* the rest, clamped into the row; products past its end not added */
    if (j < n) {
        float av[U], xv[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t q = min(j + u * HFX_WAVE, n - 1u);
            av[u] = a[q];
            xv[u] = x[q];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (j + u * HFX_WAVE < n) acc = acc + av[u] * xv[u];
    }
    acc = hfx_wave_sum_f32(acc);
    if (hfx_lane() == 0) y[row] = acc;
}

/* mvm_ff (mvm.cu:21-56): y = A x for row-major A of m rows and n columns,
 * on the handle's stream (cublasSgemv(CUBLAS_OP_T) over the transposed
 * view, Level2.chs:65-77).  The handle replaces the cuBLAS one of
 * Execution.hs:49-53: it only carries the stream set by hfx_blas_set_stream
 * (cublasSetStream_v2). */
struct hfx_blas {
    hipStream_t stream;
};

extern "C" int hfx_blas_create(void **handle)
{
    HFX_REQUIRE(handle, HFX_ERR_ARG, "hfx_blas_create: null out");
    hfx_blas *b = (hfx_blas *)calloc(1, sizeof(hfx_blas));
    HFX_REQUIRE(b, HFX_ERR_NOMEM, "hfx_blas_create: out of host memory");
    *handle = b;
    return HFX_OK;
}

extern "C" int hfx_blas_destroy(void *handle)
{
    free(handle);
    return HFX_OK;
}

extern "C" int hfx_blas_set_stream(void *handle, void *stream)
{
    HFX_REQUIRE(handle, HFX_ERR_ARG, "hfx_blas_set_stream: null handle");
    ((hfx_blas *)handle)->stream = hfx_stream(stream);
    return HFX_OK;
}

extern "C" void mvm_ff(void *handle, float *d_y, const float *d_A, const float *d_x,
                       const uint32_t m, const uint32_t n)
{
    if (m == 0) return;
    const hipStream_t st = handle ? ((hfx_blas *)handle)->stream : nullptr;
    hipLaunchKernelGGL(k_mvm_rows, dim3((m + 3) / 4), dim3(256), 0, st, d_y, d_A, n, d_x, m, n);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("mvm_ff: %s", hipGetErrorString(e));
}

extern "C" int hfx_mvm_rows(hfx_ctx *ctx, float *d_y, const float *d_A, uint32_t lda,
                            const float *d_x, uint32_t m, uint32_t n, void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_y && d_A && d_x, HFX_ERR_ARG, "hfx_mvm_rows: null argument");
    HFX_REQUIRE(n <= lda, HFX_ERR_ARG, "hfx_mvm_rows: n %u > lda %u", n, lda);
    if (m == 0) return HFX_OK;
    hipLaunchKernelGGL(k_mvm_rows, dim3((m + 3) / 4), dim3(256), 0, hfx_stream(stream), d_y, d_A,
                       lda, d_x, m, n);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}
