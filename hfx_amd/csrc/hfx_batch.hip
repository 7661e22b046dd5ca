/*
 * hfx_batch.hip -- batched search: peptide ion index + persistent
 * work-stealing multi-spectrum XCorr, hipGraph capture, autotuner.
 *
 * The reference scores each spectrum on its own: every (spectrum, candidate)
 * pair rebuilds the candidate's theoretical spectrum (Search.hs:177-245).  A
 * candidate's peaks depend only on the peptide and the fragment charges, and
 * neighbouring precursors share most of their window, so a batch of thousands
 * of spectra here
 *   1. writes, once per database, the theoretical spectrum of every peptide
 *      for fragment charge levels 1..L (level l = charges 1..l, max per bin) as
 *      rows of 2-bit codes (hfx_rows.hip), which every form scores with where
 *      memory holds them; without them the FP32 form reads the same peaks as
 *      sorted uint16 entries bin | code << 14 (k_ix_build, one wave per peptide,
 *      from the same ladder/bin code as the plain path) and the dense forms the
 *      b ladders;
 *   2. sorts the spectra by fragment charge and precursor mass, cuts the order
 *      into blocks of up to sixteen spectra (integer form; eight in the others)
 *      and contracts each block with the rows of its windows' hull.  Without
 *      rows, FP32 form: G consecutive spectra are a block; a tile is (block, C
 *      consecutive candidates of the block's union window); a persistent kernel
 *      pulls tiles from an atomic counter (work stealing: heavy-tailed windows
 *      are cut into equal tiles), keeps the block's G spectra in LDS, streams
 *      each candidate's entries once (coalesced) and gathers every spectrum of
 *      the block that holds the candidate in its window, reducing the G partial
 *      sums with one reduce-scatter butterfly;
 *   3. selects the top N with the exact re-score of hfx_topn (flagged spectra
 *      completed in the same launch sequence, no host round trip).
 * Scores land in the same layout as hfx_xcorr_sparse, so every result is
 * checked against the same oracle.  Once planned, a batch runs without host
 * synchronisation or allocation and can be captured in a hipGraph.
 */
#include "hfx_cand.h"
#include "hfx_rows.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <numeric>
#include <tuple>
#include <vector>

#define IX_THREADS 256
#define IX_WAVES (IX_THREADS / HFX_WAVE)
#define BT_GMAX 8

/* ------------------------------------------------------------------ */
/* Ion index                                                             */
/* ------------------------------------------------------------------ */

/* capacity of position q at level l: every emitted peak fills at most one
 * bin, 10 peaks per ladder position and charge, and no more than lcap bins */
__global__ void k_ix_caps(uint32_t *caps, hfx_db db, uint32_t p0, uint32_t P, uint32_t L,
                          uint32_t lcap)
{
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= P) return;
    const uint32_t pep = db.d_idx_sorted[p0 + q];
    const uint32_t tc = db.d_tc[pep], tn = db.d_tn[pep];
    const uint32_t n = tn > tc ? tn - tc : 0;
    for (uint32_t l = 1; l <= L; ++l) caps[(size_t)q * L + l - 1] = min(10u * n * l, lcap);
}

/* compact the map (bins ascending) into entries; returns the count */
__device__ __forceinline__ uint32_t wave_compact(const uint32_t *map, uint32_t nw, uint16_t *out)
{
    const uint32_t lane = hfx_lane();
    uint32_t base = 0;
    for (uint32_t w0 = 0; w0 < nw; w0 += HFX_WAVE) {
        const uint32_t w = w0 + lane;
        const uint32_t word = w < nw ? map[w] : 0u;
        const uint32_t nz = (word | (word >> 1) | (word >> 2) | (word >> 3)) & 0x11111111u;
        const uint32_t c = (uint32_t)__builtin_popcount(nz);
        uint32_t incl = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, 64);
            if (lane >= (uint32_t)o) incl += y;
        }
        uint32_t pos = base + incl - c;
        uint32_t wd = word;
        while (wd) {
            const uint32_t sh = __builtin_ctz(wd) & ~3u;
            const uint32_t nib = (wd >> sh) & 0xFu;
            wd &= ~(0xFu << sh);
            out[pos++] = (uint16_t)(((w << 3) + (sh >> 2)) | ((uint32_t)__builtin_popcount(nib) << 14));
        }
        base += (uint32_t)__shfl(incl, 63, 64);
    }
    return base;
}

__global__ void __launch_bounds__(IX_THREADS)
    k_ix_build(uint16_t *ent, uint32_t *cnt, const uint64_t *off, hfx_db db, uint32_t p0, uint32_t P,
               uint32_t L, uint32_t lcap)
{
    __shared__ uint32_t maps[IX_WAVES][HFX_MAP_WORDS];
    __shared__ float mtab[32];
    const uint32_t wave = threadIdx.x / HFX_WAVE, lane = hfx_lane();
    uint32_t *map = maps[wave];
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? db.d_mass[threadIdx.x] : 0.0f;
    for (uint32_t w = lane; w < HFX_MAP_WORDS; w += HFX_WAVE) map[w] = 0;
    __syncthreads();
    const uint32_t nw = (lcap + 7) >> 3;
    for (uint32_t q = blockIdx.x * IX_WAVES + wave; q < P; q += gridDim.x * IX_WAVES) {
        const uint32_t pep = db.d_idx_sorted[p0 + q];
        const uint32_t tc = db.d_tc[pep], tn = db.d_tn[pep];
        const uint32_t n = tn > tc ? tn - tc : 0;
        const float r = db.d_r[pep];
        for (uint32_t l = 1; l <= L; ++l) {
            /* level l = charges 1..l: add charge l to the map of level l-1 */
            hfx_wave_peaks_z(map, n, r, l, l, lcap, HfxPlainMass{db.d_ions + tc, mtab});
            hfx_wave_sync();
            const size_t k = (size_t)q * L + l - 1;
            const uint32_t c = wave_compact(map, nw, ent + off[k]);
            if (lane == 0) cnt[k] = c;
            hfx_wave_sync();
        }
        for (uint32_t w = lane; w < nw; w += HFX_WAVE) map[w] = 0;
        hfx_wave_sync();
    }
}

/* ------------------------------------------------------------------ */
/* Blocks, tiles                                                          */
/* ------------------------------------------------------------------ */

__global__ void k_bt_blocks(uint32_t *ubeg, uint32_t *uend, uint32_t *ntiles, const uint32_t *order,
                            const uint32_t *begin, const uint32_t *num, uint32_t S, uint32_t G,
                            uint32_t B, uint32_t C)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    uint32_t lo = 0xffffffffu, hi = 0;
    for (uint32_t g = 0; g < G; ++g) {
        const uint32_t i = b * G + g;
        if (i >= S) break;
        const uint32_t s = order[i];
        if (num[s] == 0) continue;
        lo = min(lo, begin[s]);
        hi = max(hi, begin[s] + num[s]);
    }
    if (hi <= lo) { lo = 0; hi = 0; }
    ubeg[b] = lo;
    uend[b] = hi;
    ntiles[b] = (hi - lo + C - 1) / C;
}

__global__ void k_bt_reset(uint32_t *counter) { *counter = 0; }

/* zmax > 4: the reference launches nothing and the zero rows score 0 */
__global__ void k_bt_zero_unscored(float *scores, const uint64_t *off, const uint32_t *zmax,
                                   uint32_t S)
{
    const uint32_t s = blockIdx.x;
    if (s >= S || hfx_zeff(zmax[s]) != 0) return;
    for (uint64_t i = off[s] + threadIdx.x; i < off[s + 1]; i += blockDim.x) scores[i] = 0.0f;
}

struct BtArgs {
    float *scores;
    const uint64_t *score_off;
    const uint32_t *begin, *num, *order;
    uint32_t S, G, B, C;
    const uint32_t *ubeg, *uend;
    const uint64_t *tile_off;
    const uint16_t *ent;
    const uint32_t *cnt;
    const uint64_t *ent_off;
    uint32_t p0, P, L, lstr;
    uint32_t *counter;
    hfx_spectra sp;
};

__device__ __forceinline__ float code_w(uint32_t c)
{
    return c == 3 ? 50.0f : (c == 2 ? 25.0f : (c == 1 ? 10.0f : 0.0f));
}

/* Sum each of the G accumulators over the wave: a reduce-scatter butterfly
 * (halving the accumulators per lane at each of the first log2 G steps) then
 * a plain butterfly.  Lane l ends with the sum of accumulator
 * g = bit-reverse-free index ((l >> 5) & 1) * 4 + ((l >> 4) & 1) * 2 + ((l >> 3) & 1)
 * for G = 8 (first bits only for smaller G). */
template <int G>
__device__ __forceinline__ float reduce_scatter(float (&acc)[G], uint32_t lane)
{
    static_assert(G == 4 || G == 8, "G must be 4 or 8");
    float v[G];
#pragma unroll
    for (int k = 0; k < G; ++k) v[k] = acc[k];
    /* each step pairs lanes across `mask`: the lower lane keeps the lower half
     * of its live accumulators, the upper lane the upper half, each adding
     * the partner's copy of the accumulators it keeps */
    int mask = 32;
#pragma unroll
    for (int n = G; n > 1; n >>= 1, mask >>= 1) {
        const bool up = lane & (uint32_t)mask;
#pragma unroll
        for (int k = 0; k < n / 2; ++k) {
            const float send = up ? v[k] : v[k + n / 2];
            const float keep = up ? v[k + n / 2] : v[k];
            v[k] = keep + __shfl_xor(send, mask, 64);
        }
    }
    float s = v[0];
#pragma unroll
    for (; mask > 0; mask >>= 1) s += __shfl_xor(s, mask, 64);
    return s;
}

template <int G>
__device__ __forceinline__ uint32_t owner_of(uint32_t lane)
{
    if constexpr (G == 8) return ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
    else return ((lane >> 5) & 1) * 2 + ((lane >> 4) & 1);
}

template <int G>
__global__ void __launch_bounds__(512) k_batch(BtArgs a)
{
    extern __shared__ float bx[]; /* G spectra, stride lstr */
    __shared__ uint32_t m_s[BT_GMAX], m_beg[BT_GMAX], m_end[BT_GMAX], m_z[BT_GMAX], m_len[BT_GMAX];
    __shared__ uint64_t m_off[BT_GMAX];
    __shared__ uint32_t sh_t, sh_lblk;
    const uint32_t tid = threadIdx.x, lane = hfx_lane();
    const uint32_t nwaves = blockDim.x / HFX_WAVE, wave = tid / HFX_WAVE;
    const uint64_t ntiles = a.tile_off[a.B];
    uint32_t cur = 0xffffffffu;
    for (;;) {
        if (tid == 0) sh_t = atomicAdd(a.counter, 1u);
        __syncthreads();
        const uint64_t t0 = sh_t;
        if (t0 >= ntiles) break;
        /* tiles from the last to the first: blocks follow the plan's order by
         * charge level, then precursor mass, so the heaviest come first and
         * the lightest finish the launch */
        const uint64_t t = ntiles - 1u - t0;
        /* block of the tile: largest b with tile_off[b] <= t */
        uint32_t lo = 0, hi = a.B;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (a.tile_off[mid] <= t) lo = mid; else hi = mid;
        }
        const uint32_t b = lo;
        if (b != cur) {
            /* stage the block's spectra (the previous tile's readers are done:
             * the barrier above follows every wave's last read) */
            if (tid < BT_GMAX) {
                const uint32_t i = b * a.G + tid;
                uint32_t s = 0xffffffffu, be = 0, en = 0, z = 0, ln = 0;
                uint64_t of = 0;
                if (tid < a.G && i < a.S) {
                    s = a.order[i];
                    be = a.begin[s];
                    en = be + a.num[s];
                    z = hfx_zeff(a.sp.d_zmax[s]);
                    ln = min(a.sp.d_len[s], min(a.lstr, a.sp.x_stride));
                    of = a.score_off[s];
                }
                m_s[tid] = s; m_beg[tid] = be; m_end[tid] = en; m_z[tid] = z; m_len[tid] = ln;
                m_off[tid] = of;
            }
            __syncthreads();
            if (tid == 0) {
                uint32_t lb = 0;
                for (int g = 0; g < G; ++g) lb = max(lb, m_z[g]);
                sh_lblk = min(lb, a.L);
            }
            for (int g = 0; g < G; ++g) {
                const uint32_t s = m_s[g];
                if (s == 0xffffffffu) continue;
                const float *xg = a.sp.d_x + (size_t)s * a.sp.x_stride;
                for (uint32_t i = tid; i < m_len[g]; i += blockDim.x) bx[g * a.lstr + i] = xg[i];
            }
            cur = b;
            __syncthreads();
        }
        const uint32_t lblk = sh_lblk;
        const uint32_t chunk = (uint32_t)(t - a.tile_off[b]);
        const uint32_t pa = a.ubeg[b] + chunk * a.C;
        const uint32_t pb = min(pa + a.C, a.uend[b]);
        for (uint32_t p = pa + wave; p < pb; p += nwaves) {
            const uint32_t q = p - a.p0;
            for (uint32_t l = 1; l <= lblk; ++l) {
                bool act[G];
                bool any = false;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    act[g] = m_z[g] == l && m_beg[g] <= p && p < m_end[g];
                    any |= act[g];
                }
                if (!any) continue;
                const size_t k = (size_t)q * a.L + l - 1;
                const uint16_t *e = a.ent + a.ent_off[k];
                const uint32_t ne = a.cnt[k];
                float acc[G];
#pragma unroll
                for (int g = 0; g < G; ++g) acc[g] = 0.0f;
                for (uint32_t j = lane; j < ne; j += HFX_WAVE) {
                    const uint32_t v = e[j];
                    const uint32_t bin = v & 0x3fffu;
                    const float w = code_w(v >> 14);
#pragma unroll
                    for (int g = 0; g < G; ++g)
                        if (act[g] && bin < m_len[g]) acc[g] = acc[g] + w * bx[g * a.lstr + bin];
                }
                const float sum = reduce_scatter<G>(acc, lane);
                const uint32_t g = owner_of<G>(lane);
                if ((lane & 7) == 0 && act[g])
                    a.scores[m_off[g] + (p - m_beg[g])] = sum;
            }
        }
        __syncthreads();
    }
}

/* ------------------------------------------------------------------ */
/* Per-database peptide index                                            */
/* ------------------------------------------------------------------ */

/* Everything the batched forms precompute per peptide: it depends on the
 * database only, so it is built once and shared by every batch. */
struct hfx_pepix {
    hfx_ctx *ctx;
    hfx_db db;
    uint32_t forms, L, lcap;
    /* HFX_PEPIX_LADDER: b ladders of every peptide, residual-sorted order */
    void *lad_mem[2];
    hfx_dn_ladder lad;
    /* HFX_PEPIX_IONS: peptide q (residual-sorted position), level l <= L:
     * cnt[q L + l - 1] entries at ent + ent_off[q L + l - 1] */
    uint32_t *caps, *cnt;
    uint64_t *ent_off;
    uint16_t *ent;
    uint64_t n_ent, n_pos, bytes;
    uint64_t key[2]; /* of the database's contents */
    struct RowSet *rs; /* its theoretical rows, once a batch has needed them */
};

/* The theoretical rows of a database (hfx_rows.hip), one copy for all indexes over
 * the same contents: 1.57 GB a charge level for 2.7 M peptides.  A level is written
 * when a batch first needs it and not moved while a batch uses the set; a set
 * that no batch uses gives its rows back where memory is short (they are written
 * again when next needed), one that no index holds either is freed.  Two databases are the
 * same by a 128-bit key of what rows are made from, never by their addresses. */
struct RowSet {
    int device;
    uint32_t num_pep;
    uint64_t key[2];
    hfx_rows rows;
    uint64_t bytes;
    uint32_t keepers, users; /* indexes, batches */
    RowSet *next;
};
static std::mutex g_rows_mu; /* the sets and what they hold */
static RowSet *g_rowsets;

/* frees a set's rows; called with g_rows_mu held and no batch using it */
static void rowset_clear(RowSet *rs)
{
    (void)hipDeviceSynchronize(); /* work of batches that used it */
    for (uint8_t *&p : rs->rows.rows) {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
    if (rs->rows.ng) (void)hipFree(rs->rows.ng);
    rs->rows.ng = nullptr;
    rs->bytes = 0;
}

/* one keeper or user less, g_rows_mu held */
static void rowset_leave(RowSet *rs, uint32_t RowSet::*count)
{
    if (--(rs->*count) || rs->keepers || rs->users) return;
    rowset_clear(rs);
    RowSet **at = &g_rowsets;
    while (*at != rs) at = &(*at)->next;
    *at = rs->next;
    free(rs);
}

bool hfx_rowsets_release(int device)
{
    std::lock_guard<std::mutex> lk(g_rows_mu);
    bool any = false;
    for (RowSet *rs = g_rowsets; rs; rs = rs->next)
        if (rs->device == device && rs->users == 0 && rs->bytes) {
            rowset_clear(rs);
            any = true;
        }
    return any;
}

__global__ void k_ord_fill(uint32_t *a, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}

/* A 128-bit key of what rows are made from: residuals, ladder bounds and residual
 * order of the peptides, the residues up to the last ladder's end (mod bits aside) and
 * the residue masses, each value mixed with its place (D. Stafford's variant 13 of the
 * 64-bit finaliser) and added up.  key[2]: the last ladder's end, which the residues
 * are read up to by the second kernel.  The 52 MB of 2.7 M peptides, read in order, take
 * 70 us; an atomic a wave, not one a workgroup, 500. */
__device__ __forceinline__ uint64_t key_mix(uint64_t x)
{
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}
struct KeySum {
    uint64_t a = 0, b = 0;
    __device__ __forceinline__ void add(uint32_t array, uint64_t i, uint32_t v)
    {
        const uint64_t at = (i << 32 | v) + (uint64_t)(array + 1u) * 0x9e3779b97f4a7c15ull;
        a += key_mix(at);
        b += key_mix(at ^ 0xd1b54a32d192ed03ull);
    }
    /* by every thread of a workgroup, which adds once: atomics on one word queue */
    __device__ __forceinline__ void to(unsigned long long *key)
    {
        __shared__ unsigned long long sum[2];
        if (threadIdx.x < 2) sum[threadIdx.x] = 0;
        for (int o = 32; o > 0; o >>= 1) {
            a += __shfl_xor(a, o, 64);
            b += __shfl_xor(b, o, 64);
        }
        __syncthreads();
        if (hfx_lane() == 0) {
            atomicAdd(&sum[0], (unsigned long long)a);
            atomicAdd(&sum[1], (unsigned long long)b);
        }
        __syncthreads();
        if (threadIdx.x < 2) atomicAdd(key + threadIdx.x, sum[threadIdx.x]);
    }
};
__global__ void __launch_bounds__(256) k_db_key_peptides(unsigned long long *key, hfx_db db)
{
    KeySum k;
    uint32_t end = 0;
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t < 26) k.add(0, t, __float_as_uint(db.d_mass[t]));
    for (uint64_t p = t; p < db.num_pep; p += gridDim.x * 256ull) {
        const uint32_t tn = db.d_tn[p];
        k.add(1, p, __float_as_uint(db.d_r[p]));
        k.add(2, p, db.d_tc[p]);
        k.add(3, p, tn);
        k.add(4, p, db.d_idx_sorted[p]);
        end = max(end, tn);
    }
    for (int o = 32; o > 0; o >>= 1) end = max(end, (uint32_t)__shfl_xor((int)end, o, 64));
    if (hfx_lane() == 0 && end) atomicMax(key + 2, (unsigned long long)end);
    k.to(key);
}
__global__ void __launch_bounds__(256) k_db_key_residues(unsigned long long *key, hfx_db db)
{
    KeySum k;
    const uint64_t n = key[2];
    /* four residues a step, those before the first multiple of four on their own */
    const uint64_t head = min(n, (uint64_t)(-(uintptr_t)db.d_ions & 3u)), words = (n - head) / 4;
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    /* (a residue's own place and code: the same sum wherever the words lie) */
    auto one = [&](uint64_t i, uint32_t c) { k.add(5, i, HFX_ACID_IDX(c)); };
    for (uint64_t w = t; w < words; w += gridDim.x * 256ull) {
        const uint32_t v = *(const uint32_t *)(db.d_ions + head + 4 * w);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) one(head + 4 * w + j, v >> (8 * j));
    }
    const uint64_t tail = head + 4 * words;
    if (t < head) one(t, db.d_ions[t]);
    if (t < n - tail) one(tail + t, db.d_ions[tail + t]);
    k.to(key);
}

template <class T>
static int dalloc(T **p, size_t n)
{
    hipError_t e = hfx_device_malloc((void **)p, (n ? n : 1) * sizeof(T));
    if (e != hipSuccess) {
        *p = nullptr;
        hfx_set_error("device allocation of %zu bytes failed: %s", n * sizeof(T),
                      hipGetErrorString(e));
        return HFX_ERR_NOMEM;
    }
    return HFX_OK;
}

extern "C" int hfx_pepix_destroy(hfx_pepix *ix)
{
    if (!ix) return HFX_OK;
    (void)hipDeviceSynchronize();
    if (ix->rs) {
        std::lock_guard<std::mutex> lk(g_rows_mu);
        rowset_leave(ix->rs, &RowSet::keepers);
    }
    void *ps[] = {ix->lad_mem[0], ix->lad_mem[1], ix->caps, ix->cnt, ix->ent_off, ix->ent};
    for (void *p : ps)
        if (p) (void)hipFree(p);
    free(ix);
    return HFX_OK;
}

extern "C" int hfx_pepix_build(hfx_ctx *ctx, const hfx_db *db, uint32_t forms, uint32_t levels,
                               uint32_t max_len, void *stream, hfx_pepix **out)
{
    HFX_REQUIRE(ctx && db && out, HFX_ERR_ARG, "hfx_pepix_build: null argument");
    HFX_REQUIRE(forms && !(forms & ~(HFX_PEPIX_LADDER | HFX_PEPIX_IONS)), HFX_ERR_ARG,
                "hfx_pepix_build: forms 0x%x", forms);
    HFX_REQUIRE(!(forms & HFX_PEPIX_IONS) || (levels >= 1 && levels <= HFX_MAX_CHARGE &&
                                                max_len >= 8 && max_len <= HFX_MAX_LEN),
                HFX_ERR_ARG, "hfx_pepix_build: levels 1..%d and max_len 8..%d", HFX_MAX_CHARGE,
                HFX_MAX_LEN);
    *out = nullptr;
    hfx_pepix *ix = (hfx_pepix *)calloc(1, sizeof(hfx_pepix));
    HFX_REQUIRE(ix, HFX_ERR_NOMEM, "hfx_pepix_build: out of host memory");
    ix->ctx = ctx;
    ix->db = *db;
    ix->forms = forms;
    hipStream_t st = hfx_stream(stream);
    const uint32_t P = db->num_pep;
    int rc = HFX_OK;
    unsigned long long *key = nullptr;
    rc = dalloc(&key, 3);
    if (!rc && P) {
        hipLaunchKernelGGL(k_ord_fill, dim3(1), dim3(64), 0, st, (uint32_t *)key, 6u);
        const dim3 g(std::min((P + 255) / 256, 512u));
        hipLaunchKernelGGL(k_db_key_peptides, g, dim3(256), 0, st, key, *db);
        hipLaunchKernelGGL(k_db_key_residues, g, dim3(256), 0, st, key, *db);
    }
    if (!rc && (forms & HFX_PEPIX_LADDER)) {
        rc = hfx_dense_ladder_build(ctx, db, 0, P, 1, &ix->lad, ix->lad_mem, stream);
        if (!rc) {
            ix->n_pos = 0;
            rc = hipMemcpyAsync(&ix->n_pos, ix->lad.off + P, 8, hipMemcpyDeviceToHost, st) ||
                         hipStreamSynchronize(st)
                     ? HFX_ERR_HIP
                     : HFX_OK;
            ix->bytes += ((uint64_t)P + 1) * 8 + (uint64_t)P * 8 +
                         std::max<uint64_t>(ix->n_pos, 1) * sizeof(hfx_dn_pos);
        }
    }
    if (!rc && (forms & HFX_PEPIX_IONS)) {
        ix->L = levels;
        ix->lcap = max_len;
        const uint64_t PL = (uint64_t)P * levels;
        if (PL >= 0xffffffffull) {
            hfx_set_error("hfx_pepix_build: %u peptides x %u levels", P, levels);
            rc = HFX_ERR_ARG;
        }
        if (!rc) rc = dalloc(&ix->caps, PL);
        if (!rc) rc = dalloc(&ix->ent_off, PL + 1);
        if (!rc) rc = dalloc(&ix->cnt, PL);
        if (!rc && P) {
            hipLaunchKernelGGL(k_ix_caps, dim3((P + 255) / 256), dim3(256), 0, st, ix->caps, *db,
                               0u, P, levels, max_len);
            rc = hfx_scan_offsets(ctx, ix->ent_off, ix->caps, (uint32_t)PL, stream);
            if (!rc && (hipMemcpyAsync(&ix->n_ent, ix->ent_off + PL, 8, hipMemcpyDeviceToHost,
                                       st) != hipSuccess ||
                        hipStreamSynchronize(st) != hipSuccess)) {
                hfx_set_error("hfx_pepix_build: reading the index size failed");
                rc = HFX_ERR_HIP;
            }
        }
        if (!rc) rc = dalloc(&ix->ent, ix->n_ent);
        if (!rc && P) {
            const uint32_t grid = (uint32_t)std::min<uint64_t>(
                (P + IX_WAVES - 1) / IX_WAVES, (uint64_t)hfx_ctx_num_cus(ctx) * 16);
            hipLaunchKernelGGL(k_ix_build, dim3(grid), dim3(IX_THREADS), 0, st, ix->ent, ix->cnt,
                               ix->ent_off, *db, 0u, P, levels, max_len);
        }
        ix->bytes += PL * 4 * 2 + (PL + 1) * 8 + ix->n_ent * 2;
    }
    if (!rc && hipGetLastError() != hipSuccess) {
        hfx_set_error("hfx_pepix_build: kernel launch failed");
        rc = HFX_ERR_HIP;
    }
    if (!rc && P && hipMemcpyAsync(ix->key, key, 16, hipMemcpyDeviceToHost, st) != hipSuccess) {
        hfx_set_error("hfx_pepix_build: reading the key failed");
        rc = HFX_ERR_HIP;
    }
    if (hipStreamSynchronize(st) != hipSuccess && !rc) {
        hfx_set_error("hfx_pepix_build: synchronize failed");
        rc = HFX_ERR_HIP;
    }
    if (key) (void)hipFree(key);
    if (rc) {
        hfx_pepix_destroy(ix);
        return rc;
    }
    *out = ix;
    return HFX_OK;
}

/* The rows of charge levels 1..L of the index's database, for one more batch
 * (rowset_leave(.., &RowSet::users) when it is done): written now where they are
 * missing (waits for the stream then).  Null when a quarter of the free memory does
 * not hold them: the batch keeps the ladder or ion-list kernels. */
static RowSet *pepix_use_rows(hfx_pepix *ix, uint32_t L, uint32_t cus, hipStream_t st, hfx_rows *out)
{
    std::lock_guard<std::mutex> lk(g_rows_mu);
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    if (!ix->rs) {
        for (RowSet *rs = g_rowsets; rs; rs = rs->next)
            if (rs->device == dev && rs->num_pep == ix->db.num_pep && rs->key[0] == ix->key[0] &&
                rs->key[1] == ix->key[1])
                ix->rs = rs;
        if (!ix->rs) {
            ix->rs = (RowSet *)calloc(1, sizeof(RowSet));
            if (!ix->rs) return nullptr;
            ix->rs->device = dev;
            ix->rs->num_pep = ix->db.num_pep;
            ix->rs->key[0] = ix->key[0];
            ix->rs->key[1] = ix->key[1];
            ix->rs->next = g_rowsets;
            g_rowsets = ix->rs;
        }
        ++ix->rs->keepers;
    }
    RowSet *rs = ix->rs;
    const uint32_t nt = hfx_rows_tiles(ix->db.num_pep);
    const uint64_t level = std::max<uint64_t>((uint64_t)nt * RW_G * 1024, 256);
    hfx_rows want{};
    want.ntiles = nt;
    want.G = RW_G;
    uint64_t need = 0;
    for (uint32_t l = 0; l < L; ++l) need += rs->rows.rows[l] ? 0 : level;
    if (need) {
        size_t fr = 0, tot = 0;
        bool ok = hipMemGetInfo(&fr, &tot) == hipSuccess && need <= fr / 4;
        if (ok && !rs->rows.ng) ok = hipMalloc((void **)&rs->rows.ng, nt + 4ull) == hipSuccess;
        for (uint32_t l = 0; l < L && ok; ++l)
            if (!rs->rows.rows[l]) ok = hipMalloc((void **)&want.rows[l], level) == hipSuccess;
        want.ng = rs->rows.ng;
        ok = ok && hfx_rows_build(cus, &ix->db, &want, nullptr, (void *)st) == HFX_OK &&
             hipStreamSynchronize(st) == hipSuccess;
        for (uint32_t l = 0; l < HFX_MAX_CHARGE; ++l) {
            if (!want.rows[l]) continue;
            if (!ok) {
                (void)hipFree(want.rows[l]);
                continue;
            }
            rs->rows.rows[l] = want.rows[l];
            rs->bytes += level;
        }
        (void)hipGetLastError();
        if (!ok) return nullptr;
        rs->rows.ntiles = nt;
        rs->rows.G = RW_G;
    }
    ++rs->users;
    *out = rs->rows;
    return rs;
}

extern "C" int hfx_pepix_info(const hfx_pepix *ix, uint64_t *info /*[6]*/)
{
    HFX_REQUIRE(ix && info, HFX_ERR_ARG, "hfx_pepix_info: null argument");
    info[0] = ix->forms; info[1] = ix->L; info[2] = ix->lcap; info[3] = ix->n_pos;
    std::lock_guard<std::mutex> lk(g_rows_mu);
    info[4] = ix->n_ent; info[5] = ix->bytes + (ix->rs ? ix->rs->bytes : 0);
    return HFX_OK;
}

/* ------------------------------------------------------------------ */
/* Spectrum order and dense blocks, on the device                        */
/* ------------------------------------------------------------------ */

/* Spectra are ordered by (fragment charge level, precursor mass, index):
 * bucket = level * nbz + (window begin >> sh) -- the window's first
 * residual-sorted position is a monotone function of the precursor mass --
 * counted, scattered, then ranked inside each bucket by (mass, index).  Without
 * masses the window's begin takes their place.  Any input gives a permutation: the
 * begin of an empty window, which nothing else reads, may be anything, and masses
 * that are NaN come last. */
__device__ __forceinline__ uint32_t ord_bucket(uint32_t s, const uint32_t *begin,
                                               const uint32_t *zmax, uint32_t sh, uint32_t nbz)
{
    return hfx_zeff(zmax[s]) * nbz + min(begin[s] >> sh, nbz - 1u);
}

__global__ void k_ord_count(uint32_t *cnt, const uint32_t *begin, const uint32_t *zmax, uint32_t S,
                            uint32_t sh, uint32_t nbz)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < S) atomicAdd(&cnt[ord_bucket(s, begin, zmax, sh, nbz)], 1u);
}

/* counts down to zero, leaving cnt cleared */
__global__ void k_ord_scatter(uint32_t *tmp, uint32_t *cnt, const uint64_t *boff,
                              const uint32_t *begin, const uint32_t *zmax, uint32_t S, uint32_t sh,
                              uint32_t nbz)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    const uint32_t k = ord_bucket(s, begin, zmax, sh, nbz);
    tmp[boff[k] + atomicSub(&cnt[k], 1u) - 1u] = s;
}

__global__ void k_ord_rank(uint32_t *order, const uint32_t *tmp, const uint64_t *boff,
                           const uint32_t *begin, const uint32_t *zmax, const float *mass,
                           uint32_t S, uint32_t sh, uint32_t nbz)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S) return;
    const uint32_t s = tmp[i];
    const uint32_t k = ord_bucket(s, begin, zmax, sh, nbz);
    const uint32_t a = (uint32_t)boff[k], e = (uint32_t)boff[k + 1];
    auto key = [&](uint32_t t) {
        if (!mass) return begin[t];
        const float m = mass[t] + 0.0f; /* -0 as 0 */
        return m == m ? hfx_f2key(m) : 0xffffffffu;
    };
    const uint32_t ks = key(s);
    uint32_t rank = 0;
    for (uint32_t j = a; j < e; ++j) {
        const uint32_t t = tmp[j], kt = key(t);
        rank += (kt < ks || (kt == ks && t < s)) ? 1u : 0u;
    }
    order[a + rank] = s;
}

/* Dense blocks: the order cut into runs of at most DN_NS spectra that
 * minimise the sum over blocks of (charge levels x rows of the hull of the
 * windows) -- a block spanning a gap in precursor mass would score every
 * candidate in the gap.  A dynamic programme per segment of CUT_SEG order
 * positions (segments are cut independently, which costs about 1% more
 * rows than one programme over the whole order), a wave a segment.  First the
 * costs of every block, which depend on nothing: sixteen lanes take the newest
 * 1 .. 16 of j positions, their hulls by inclusive row scans (min of starts, max
 * of ends, OR of charge levels).  Then the chain of 32 steps, cut to what hangs on
 * the step before: an addition, a row minimum, a shift by a lane (DPP row_shr:1).
 * Costs are whole and below 2^43, so exact in FP64, with length / 16 below the
 * point: the shortest block among equal costs, the one a serial scan of lengths
 * 1, 2, ... with strict improvement keeps.  11 us, 14.2 with the hulls in the
 * chain and 64-bit integers. */
#define CUT_SEG 32
#define CUT_ROW 16
#define CUT_WG 256
#define CUT_SPW (CUT_WG / HFX_WAVE) /* segments a workgroup */

template <int CTRL>
__device__ __forceinline__ uint32_t cut_dpp(uint32_t old, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ double cut_dpp64(double old, double v)
{
    return __hiloint2double(
        (int)cut_dpp<CTRL>((uint32_t)__double2hiint(old), (uint32_t)__double2hiint(v)),
        (int)cut_dpp<CTRL>((uint32_t)__double2loint(old), (uint32_t)__double2loint(v)));
}

template <int CUT_NS>
__global__ void __launch_bounds__(CUT_WG) k_cut_seg(uint32_t *seg_cuts, uint32_t *seg_n,
                                                   const uint32_t *order, const uint32_t *begin,
                                                   const uint32_t *num, const uint32_t *zmax,
                                                   uint32_t S)
{
    static_assert(CUT_NS <= CUT_ROW, "every block length has its lane");
    __shared__ uint32_t lo_s[CUT_SPW * CUT_SEG], hi_s[CUT_SPW * CUT_SEG], lv_s[CUT_SPW * CUT_SEG];
    __shared__ double cost_s[CUT_SPW][CUT_SEG][CUT_ROW];
    __shared__ uint8_t from_s[CUT_SPW][CUT_SEG + 1];
    const uint32_t base = blockIdx.x * CUT_SPW * CUT_SEG;
    for (uint32_t i = threadIdx.x; i < CUT_SPW * CUT_SEG; i += CUT_WG) {
        const uint32_t p = base + i;
        uint32_t lo = 0xffffffffu, hi = 0, lv = 0;
        if (p < S) {
            const uint32_t s = order[p], z = hfx_zeff(zmax[s]), n = num[s];
            if (z && n) {
                lo = begin[s];
                hi = lo + n;
                lv = 1u << z;
            }
        }
        lo_s[i] = lo;
        hi_s[i] = hi;
        lv_s[i] = lv;
    }
    __syncthreads();
    const uint32_t r = threadIdx.x / HFX_WAVE, lane = hfx_lane(), i = lane % CUT_ROW;
    const uint32_t seg = blockIdx.x * CUT_SPW + r;
    const uint32_t p0 = seg * CUT_SEG;
    if (p0 >= S) return; /* the whole wave leaves together */
    const uint32_t len = min((uint32_t)CUT_SEG, S - p0);
    const uint32_t *lo = lo_s + r * CUT_SEG, *hi = hi_s + r * CUT_SEG, *lv = lv_s + r * CUT_SEG;
    uint8_t *from = from_s[r];
    /* lane i of a row: the block of the newest i + 1 of j positions, four j a turn */
#pragma unroll
    for (uint32_t q = 0; q < CUT_SEG * CUT_ROW / HFX_WAVE; ++q) {
        const uint32_t j = q * (HFX_WAVE / CUT_ROW) + lane / CUT_ROW + 1;
        const bool in = i < j;
        const uint32_t at = in ? j - 1u - i : 0u;
        uint32_t l = in ? lo[at] : 0xffffffffu, h = in ? hi[at] : 0u, v = in ? lv[at] : 0u;
        l = min(l, cut_dpp<0x111>(0xffffffffu, l));
        h = max(h, cut_dpp<0x111>(0u, h));
        v |= cut_dpp<0x111>(0u, v);
        l = min(l, cut_dpp<0x112>(0xffffffffu, l));
        h = max(h, cut_dpp<0x112>(0u, h));
        v |= cut_dpp<0x112>(0u, v);
        l = min(l, cut_dpp<0x114>(0xffffffffu, l));
        h = max(h, cut_dpp<0x114>(0u, h));
        v |= cut_dpp<0x114>(0u, v);
        l = min(l, cut_dpp<0x118>(0xffffffffu, l));
        h = max(h, cut_dpp<0x118>(0u, h));
        v |= cut_dpp<0x118>(0u, v);
        const uint64_t rows = h > l ? (uint64_t)(h - l) : 0ull;
        cost_s[r][j - 1][i] = i < (uint32_t)CUT_NS && in
                                  ? (double)(rows * (uint64_t)__builtin_popcount(v)) + 0.0625 * (double)i
                                  : (double)INFINITY;
    }
    hfx_wave_sync();
    /* lane i: the best cost of the positions before that block (finite for i < j) */
    double bst = i == 0 ? 0.0 : (double)INFINITY;
#pragma unroll 8
    for (uint32_t j = 1; j <= len; ++j) {
        double key = bst + cost_s[r][j - 1][i], t;
        t = cut_dpp64<0xB1>(0.0, key);  /* quad_perm [1,0,3,2] */
        key = t < key ? t : key;
        t = cut_dpp64<0x4E>(0.0, key);  /* quad_perm [2,3,0,1] */
        key = t < key ? t : key;
        t = cut_dpp64<0x141>(0.0, key); /* row_half_mirror */
        key = t < key ? t : key;
        t = cut_dpp64<0x140>(0.0, key); /* row_mirror */
        key = t < key ? t : key;
        const double whole = floor(key);
        bst = cut_dpp64<0x111>(whole, bst);
        if (lane == 0) from[j] = (uint8_t)(j - 1u - (uint32_t)((key - whole) * 16.0));
    }
    if (lane != 0) return;
    /* block starts, back from the segment's end, then written in order */
    uint32_t cnt = 0;
    for (uint32_t j = len; j > 0; j = from[j]) ++cnt;
    uint32_t w = cnt;
    for (uint32_t j = len; j > 0; j = from[j]) seg_cuts[(size_t)seg * CUT_SEG + --w] = p0 + from[j];
    seg_n[seg] = cnt;
}

/* bstart[0 .. nb) = the segments' block starts in order, bstart[nb .. cap]
 * = S (empty blocks), nb = seg_off[nseg] */
/* also clears a word for what follows, if asked to */
__global__ void k_cut_place(uint32_t *clear, uint32_t *bstart, const uint32_t *seg_cuts, const uint32_t *seg_n,
                            const uint64_t *seg_off, uint32_t nseg, uint32_t cap, uint32_t S)
{
    if (clear && blockIdx.x == 0 && threadIdx.x == 0) *clear = 0;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t seg = t / CUT_SEG, i = t % CUT_SEG;
    if (seg < nseg && i < seg_n[seg]) bstart[seg_off[seg] + i] = seg_cuts[t];
    const uint32_t nb = (uint32_t)seg_off[nseg];
    if (t <= cap && t >= nb) bstart[t] = S;
}

/* buckets of the spectrum order: about two spectra a bucket on average */
void hfx_order_shape(uint32_t S, uint32_t num_pep, hfx_order_bufs *o)
{
    o->sh = 0;
    while (((uint64_t)num_pep >> o->sh) > std::max<uint64_t>(S / 2, 64)) ++o->sh;
    o->nbz = (num_pep >> o->sh) + 1;
    o->nb = (HFX_MAX_CHARGE + 1) * o->nbz;
}

int hfx_order_spectra(hfx_ctx *ctx, uint32_t *order, const hfx_order_bufs *o,
                      const uint32_t *begin, const uint32_t *zmax, const float *mass, uint32_t S,
                      void *stream)
{
    hipStream_t st = hfx_stream(stream);
    const uint32_t g = (S + 255) / 256;
    hipLaunchKernelGGL(k_ord_fill, dim3((o->nb + 255) / 256), dim3(256), 0, st, o->cnt, o->nb);
    hipLaunchKernelGGL(k_ord_count, dim3(g), dim3(256), 0, st, o->cnt, begin, zmax, S, o->sh,
                       o->nbz);
    int rc;
    if ((rc = hfx_scan_offsets(ctx, o->off, o->cnt, o->nb, stream))) return rc;
    hipLaunchKernelGGL(k_ord_scatter, dim3(g), dim3(256), 0, st, o->tmp, o->cnt, o->off, begin,
                       zmax, S, o->sh, o->nbz);
    hipLaunchKernelGGL(k_ord_rank, dim3(g), dim3(256), 0, st, order, o->tmp, o->off, begin, zmax,
                       mass, S, o->sh, o->nbz);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

uint32_t hfx_cut_segs(uint32_t S) { return (S + CUT_SEG - 1) / CUT_SEG; }

int hfx_cut_blocks(hfx_ctx *ctx, uint32_t ns, const hfx_cut_bufs *c, const uint32_t *order,
                   const uint32_t *begin, const uint32_t *num, const uint32_t *zmax, uint32_t S,
                   void *stream)
{
    hipStream_t st = hfx_stream(stream);
    const uint32_t nseg = hfx_cut_segs(S);
    const dim3 g((nseg + CUT_SPW - 1) / CUT_SPW);
    if (ns == 16)
        hipLaunchKernelGGL(k_cut_seg<16>, g, dim3(CUT_WG), 0, st, c->seg, c->n, order, begin, num,
                           zmax, S);
    else
        hipLaunchKernelGGL(k_cut_seg<8>, g, dim3(CUT_WG), 0, st, c->seg, c->n, order, begin, num,
                           zmax, S);
    int rc;
    if ((rc = hfx_scan_offsets(ctx, c->off, c->n, nseg, stream))) return rc;
    const uint32_t nt = std::max(nseg * CUT_SEG, S + 1);
    hipLaunchKernelGGL(k_cut_place, dim3((nt + 255) / 256), dim3(256), 0, st, c->clear, c->bstart, c->seg,
                       c->n, c->off, nseg, S, S);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* ------------------------------------------------------------------ */
/* The batch object                                                       */
/* ------------------------------------------------------------------ */

struct hfx_batch {
    hfx_ctx *ctx;
    hfx_db db;
    hfx_spectra sp;
    float eps;
    uint32_t N, margin;
    uint32_t S, G, C, threads, B, L, lstr;
    uint64_t total;
    bool planned;
    const hfx_pepix *ix; /* the caller's index, or own */
    hfx_pepix *own;      /* built on first need when the caller gave none */
    /* device buffers (owned) */
    uint32_t *begin, *num, *order, *ubeg, *uend, *ntiles, *counter;
    uint64_t *score_off, *tile_off;
    float *scores;
    uint32_t *top_pos, *top_cnt, *flag;
    double *top_exact;
    float *top_f32;
    uint8_t *tx_scratch; /* top-N exact route */
    /* spectrum order: buckets */
    uint32_t ord_sh, ord_nbz, ord_nb;
    uint32_t *ord_cnt, *ord_tmp;
    uint64_t *ord_off;
    uint32_t precision; /* HFX_BATCH_FP32_SPARSE, _BF16X2_DENSE or _I8X3_DENSE */
    uint32_t CH;        /* rows, dense: candidates per work item */
    uint8_t *dn_scratch; /* dense: hi/lo spectra, blocks (allocated with the dense form) */
    uint32_t *dn_bstart; /* dense: [S + 1] block starts in order (S past the last block) */
    uint32_t *cut_seg, *cut_n;
    uint64_t *cut_off;
    uint32_t nseg;
    bool dense_set;      /* a dense form was chosen since the plan */
    bool chunk_set;      /* CH is the caller's or the tuner's */
    bool rows_tried, use_rows; /* scores come from the database's rows */
    RowSet *rs;                /* the set they are in, and what this batch reads of it */
    hfx_rows rows;
    uint32_t have;             /* the highest charge level of those rows */
    uint8_t *rw_planes;  /* rows, FP32 form: six digits of every spectrum | item bookkeeping */
    uint32_t *rw_small;  /* rows: [S] sum and max of |x|, [S] quanta, [S] levels, the rest's list */
    hipGraph_t graph;
    hipGraphExec_t exec;
};

/* the rows are decided anew at the next run */
static void bt_rows_drop(hfx_batch *b)
{
    if (b->rs) {
        std::lock_guard<std::mutex> lk(g_rows_mu);
        rowset_leave(b->rs, &RowSet::users);
    }
    b->rs = nullptr;
    b->rows_tried = b->use_rows = false;
}

static void bt_free(hfx_batch *b)
{
    bt_rows_drop(b);
    void *ps[] = {b->begin,    b->num,       b->order,     b->ubeg,      b->uend,
                  b->ntiles,   b->counter,   b->score_off, b->tile_off,  b->scores,
                  b->top_pos,  b->top_cnt,   b->flag,      b->top_exact, b->top_f32,
                  b->tx_scratch, b->ord_cnt, b->ord_tmp,   b->ord_off,   b->dn_scratch,
                  b->dn_bstart, b->cut_seg,  b->cut_n,     b->cut_off,   b->rw_small,
                  b->rw_planes};
    for (void *p : ps)
        if (p) (void)hipFree(p);
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    hfx_ctx *ctx = b->ctx;
    const hfx_pepix *ix = b->ix;
    hfx_pepix *own = b->own;
    memset(b, 0, sizeof *b);
    b->ctx = ctx;
    b->own = own;
    b->ix = ix == own ? nullptr : ix; /* the caller's index stays attached */
}

extern "C" int hfx_batch_create(hfx_ctx *ctx, hfx_batch **out)
{
    HFX_REQUIRE(ctx && out, HFX_ERR_ARG, "hfx_batch_create: null argument");
    hfx_batch *b = (hfx_batch *)calloc(1, sizeof(hfx_batch));
    HFX_REQUIRE(b, HFX_ERR_NOMEM, "hfx_batch_create: out of host memory");
    b->ctx = ctx;
    *out = b;
    return HFX_OK;
}

extern "C" int hfx_batch_destroy(hfx_batch *b)
{
    if (!b) return HFX_OK;
    (void)hipDeviceSynchronize();
    bt_free(b);
    if (b->own) hfx_pepix_destroy(b->own);
    free(b);
    return HFX_OK;
}

static int bt_ready_attached(hfx_batch *b, hipStream_t st);

extern "C" int hfx_batch_use_index(hfx_batch *b, const hfx_pepix *ix)
{
    HFX_REQUIRE(b, HFX_ERR_ARG, "hfx_batch_use_index: null batch");
    HFX_REQUIRE(!b->planned || !ix ||
                    (ix->db.d_idx_sorted == b->db.d_idx_sorted && ix->db.num_pep == b->db.num_pep),
                HFX_ERR_ARG, "hfx_batch_use_index: the index belongs to another database");
    b->ix = ix;
    bt_rows_drop(b);
    if (b->exec) {
        (void)hipGraphExecDestroy(b->exec);
        b->exec = nullptr;
        (void)hipGraphDestroy(b->graph);
        b->graph = nullptr;
    }
    /* its rows now, so that no run waits or allocates for them */
    return b->planned ? bt_ready_attached(b, nullptr) : HFX_OK;
}

/* Shape-bucketed autotuner results of this process: (S bucket, P bucket, L)
 * -> (G, C, threads) of the ion-list kernel; the chunk of each precision form over
 * rows, and of the dense forms' ladder kernels. */
typedef std::tuple<int, int, uint32_t> tune_shape;
static std::mutex g_tune_mu;
static std::map<tune_shape, std::tuple<uint32_t, uint32_t, uint32_t>> g_tune;
struct TuneChunks {
    const char *name; /* in the cache file */
    uint32_t precision;
    bool rows;
    std::map<tune_shape, uint32_t> chunk;
};
static TuneChunks g_tune_chunks[] = {{"fp32", HFX_BATCH_FP32_SPARSE, true, {}},
                                     {"bf16", HFX_BATCH_BF16X2_DENSE, true, {}},
                                     {"int8", HFX_BATCH_I8X3_DENSE, true, {}},
                                     {"bf16-ladder", HFX_BATCH_BF16X2_DENSE, false, {}},
                                     {"int8-ladder", HFX_BATCH_I8X3_DENSE, false, {}}};
/* null: the form without rows has no chunk */
static std::map<tune_shape, uint32_t> *tune_chunks(uint32_t precision, bool rows)
{
    for (TuneChunks &t : g_tune_chunks)
        if (t.precision == precision && t.rows == rows) return &t.chunk;
    return nullptr;
}

/* the two dense forms share the ladders, block cut and work items */
static inline bool bt_is_dense(uint32_t precision)
{
    return precision == HFX_BATCH_BF16X2_DENSE || precision == HFX_BATCH_I8X3_DENSE;
}
/* the dense forms' per-batch scratch: the larger of the two */
static size_t bt_dense_scratch(uint32_t S)
{
    return std::max(hfx_dense_scratch_bytes(S), hfx_dense8_scratch_bytes(S));
}

/* the launch shapes the kernels support: sparse G in {4, 8}, C in 1..4096,
 * threads in {256, 512}; a dense chunk a multiple of its tile (16 candidates
 * for BF16, 64 for int8) up to 8192 */
static bool tune_sparse_ok(uint32_t G, uint32_t C, uint32_t threads)
{
    return (G == 4 || G == 8) && C >= 1 && C <= 4096 && (threads == 256 || threads == 512);
}
static uint32_t tune_dense_step(uint32_t precision)
{
    return precision == HFX_BATCH_I8X3_DENSE ? 64u : 16u;
}
static bool tune_dense_ok(uint32_t precision, uint32_t CH)
{
    const uint32_t step = tune_dense_step(precision);
    return CH >= step && CH % step == 0 && CH <= 8192;
}

/* candidates a work item takes over rows, untuned: by the rows the blocks read --
 * about a twelfth of the pairs, but every row of the database's two usual
 * levels once the batch covers it */
static uint32_t bt_chunk(const hfx_batch *b)
{
    const uint64_t rows = std::max<uint64_t>(b->total / 12, std::min<uint64_t>(b->total, 2ull * b->db.num_pep));
    return hfx_rows_chunk(rows, (uint32_t)hfx_ctx_num_cus(b->ctx));
}

static tune_shape tune_key(const hfx_batch *b)
{
    auto lg = [](uint64_t v) { int k = 0; while (v > 1) { v >>= 1; ++k; } return k; };
    return std::make_tuple(lg(b->S), lg(b->total), b->L);
}

/* The tuned shapes persist across processes when HFX_TUNE_CACHE names a
 * file: one line a shape, "sparse <S bucket> <pairs bucket> <levels> <G> <C>
 * <threads>", or "fp32 ... <chunk>", "bf16", "int8" over rows, "bf16-ladder",
 * "int8-ladder" without (other lines are ignored).  It is read when a lookup first sees the path (its entries
 * replace this process's for the same shapes) and rewritten whole, through a
 * temporary file and a rename, after each tuning.  Callers hold g_tune_mu. */
static std::string g_tune_path;
static void tune_load_locked()
{
    const char *p = getenv("HFX_TUNE_CACHE");
    const std::string path = p ? p : "";
    if (path == g_tune_path) return;
    g_tune_path = path;
    if (path.empty()) return;
    FILE *f = fopen(path.c_str(), "r");
    if (!f) return;
    char kind[16];
    int sb, pb;
    unsigned L, a, c, t;
    char line[256];
    while (fgets(line, sizeof line, f)) {
        const int n = sscanf(line, "%15s %d %d %u %u %u %u", kind, &sb, &pb, &L, &a, &c, &t);
        const auto key = std::make_tuple(sb, pb, (uint32_t)L);
        /* entries outside the supported shapes (a damaged or hand-edited
         * file) are skipped, never launched */
        if (n == 7 && !strcmp(kind, "sparse") && tune_sparse_ok(a, c, t))
            g_tune[key] = std::make_tuple((uint32_t)a, (uint32_t)c, (uint32_t)t);
        else if (n == 5)
            for (TuneChunks &k : g_tune_chunks)
                if (!strcmp(kind, k.name) && tune_dense_ok(k.precision, a)) k.chunk[key] = a;
    }
    fclose(f);
}
static void tune_save_locked()
{
    if (g_tune_path.empty()) return;
    /* a temporary name of this process's own, so that processes tuning at
     * once never write one file together (the last rename wins) */
    const std::string tmp = g_tune_path + ".tmp." + std::to_string((long)getpid());
    FILE *f = fopen(tmp.c_str(), "w");
    if (!f) return;
    for (const auto &e : g_tune)
        fprintf(f, "sparse %d %d %u %u %u %u\n", std::get<0>(e.first), std::get<1>(e.first),
                std::get<2>(e.first), std::get<0>(e.second), std::get<1>(e.second),
                std::get<2>(e.second));
    for (const TuneChunks &k : g_tune_chunks)
        for (const auto &e : k.chunk)
            fprintf(f, "%s %d %d %u %u\n", k.name, std::get<0>(e.first), std::get<1>(e.first),
                    std::get<2>(e.first), e.second);
    if (fclose(f) == 0) rename(tmp.c_str(), g_tune_path.c_str());
}

/* The chunk of the current form, unless the caller or the tuner set one: tuned for
 * batches of this shape, or by the rows it reads; 256 for the ladder kernels.  Until
 * the rows are decided on they are taken to be there. */
static void bt_pick_chunk(hfx_batch *b)
{
    if (b->chunk_set) return;
    const bool rows = b->rows_tried ? b->use_rows : b->sp.x_stride <= RW_MAXK;
    b->CH = rows ? bt_chunk(b) : 256u;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    tune_load_locked();
    if (auto *m = tune_chunks(b->precision, rows)) {
        auto it = m->find(tune_key(b));
        if (it != m->end()) b->CH = it->second;
    }
}

/* the form of the peptide index the current precision reads */
static uint32_t bt_form(const hfx_batch *b)
{
    return bt_is_dense(b->precision) ? HFX_PEPIX_LADDER : HFX_PEPIX_IONS;
}

/* makes sure the index holds the current precision's form: the caller's,
 * or one the batch builds (never while a stream is being captured) */
static int bt_need_index(hfx_batch *b, hipStream_t st)
{
    const uint32_t f = bt_form(b);
    if (b->ix && (b->ix->forms & f) && (f != HFX_PEPIX_IONS || b->ix->L >= b->L)) return HFX_OK;
    HFX_REQUIRE(!b->ix || b->ix == b->own, HFX_ERR_ARG,
                "batch: the attached peptide index lacks the %s form this precision reads",
                f == HFX_PEPIX_LADDER ? "ladder" : "ion list");
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HFX_CHECK_HIP(hipStreamIsCapturing(st, &cs));
    HFX_REQUIRE(cs == hipStreamCaptureStatusNone, HFX_ERR_ARG,
                "batch: the peptide index is built on first use, not under capture "
                "(run or set the precision once before capturing)");
    uint32_t forms = f;
    if (b->own) forms |= b->own->forms;
    hfx_pepix *nx = nullptr;
    int rc = hfx_pepix_build(b->ctx, &b->db, forms, HFX_MAX_CHARGE, HFX_MAX_LEN, (void *)st, &nx);
    if (rc) return rc;
    if (b->own) hfx_pepix_destroy(b->own);
    b->own = nx;
    b->ix = nx;
    bt_rows_drop(b);
    return HFX_OK;
}

static int bt_cut_alloc(hfx_batch *b);
static int bt_dense_alloc(hfx_batch *b);
/* the FP32 form's planes and work items */
static size_t bt_planes_bytes(uint32_t S)
{
    return (size_t)S * RW_PLANES(RW_I8X6) * RW_MAXK + hfx_rows_items_bytes(S);
}

/* the current form's own buffers of the rows route are there */
static bool bt_rows_bufs(const hfx_batch *b)
{
    return b->rw_small && (bt_is_dense(b->precision) ? b->dn_scratch : b->rw_planes);
}
/* the next scores come from rows */
static bool bt_rows(const hfx_batch *b) { return b->use_rows && bt_rows_bufs(b); }

/* the index, and its rows where they fit (decided once a plan, index and form, never
 * under capture: a batch captured by its caller without a run before it keeps
 * the other kernels) */
static int bt_ready_rows(hfx_batch *b, hipStream_t st);
static int bt_ready(hfx_batch *b, hipStream_t st)
{
    int rc = bt_need_index(b, st);
    if (rc || b->S == 0 || (b->rows_tried && (!b->use_rows || bt_rows_bufs(b)))) return rc;
    /* (the null stream cannot be asked while another one is captured) */
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return HFX_OK;
    }
    rc = bt_ready_rows(b, st);
    bt_pick_chunk(b);
    return rc;
}
static int bt_ready_rows(hfx_batch *b, hipStream_t st)
{
    b->rows_tried = true;
    if (b->sp.x_stride > RW_MAXK || b->db.num_pep == 0) return HFX_OK;
    size_t fr = 0, tot = 0;
    HFX_CHECK_HIP(hipMemGetInfo(&fr, &tot));
    if (!bt_rows_bufs(b) && (uint64_t)b->S * 16384 > fr / 4) {
        bt_rows_drop(b);
        b->rows_tried = true;
        return HFX_OK;
    }
    if (!b->rs) b->rs = pepix_use_rows(const_cast<hfx_pepix *>(b->ix), b->L, (uint32_t)hfx_ctx_num_cus(b->ctx),
                           st, &b->rows);
    if (!b->rs) return HFX_OK;
    if (bt_cut_alloc(b) || (!b->rw_small && dalloc(&b->rw_small, 5 * (size_t)b->S + 1)) ||
        (bt_is_dense(b->precision) ? bt_dense_alloc(b)
                                   : !b->rw_planes && dalloc(&b->rw_planes, bt_planes_bytes(b->S)))) {
        (void)hipGetLastError();
        bt_rows_drop(b);
        b->rows_tried = true;
        return HFX_OK;
    }
    for (b->have = 0; b->have < HFX_MAX_CHARGE && b->rows.rows[b->have];) ++b->have;
    b->use_rows = true;
    return HFX_OK;
}

/* bt_ready as far as it goes without building an index of the batch's own */
static int bt_ready_attached(hfx_batch *b, hipStream_t st)
{
    const uint32_t f = bt_form(b);
    if (!b->ix || !(b->ix->forms & f) || (f == HFX_PEPIX_IONS && b->ix->L < b->L)) return HFX_OK;
    return bt_ready(b, st);
}

/* Device bytes a batch allocates for S spectra with `total` scored pairs (the
 * precision form's own buffers included, the per-database index and rows not):
 * the same sums as the allocations.  rows: with what it takes to score through
 * rows, which it does without where memory is short; the FP32 form's is counted
 * for the others too, as a plan starts in that form. */
static uint64_t bt_bytes(uint32_t S, uint64_t total, uint32_t N, uint32_t num_pep,
                         uint32_t precision, bool rows = true)
{
    auto al = [](uint64_t n, uint64_t sz) { return (std::max<uint64_t>(n, 1) * sz + 255) & ~255ull; };
    uint32_t sh = 0;
    while (((uint64_t)num_pep >> sh) > std::max<uint64_t>(S / 2, 64)) ++sh;
    const uint64_t nb = (uint64_t)(HFX_MAX_CHARGE + 1) * ((num_pep >> sh) + 1);
    const uint64_t bmax = (S + 3) / 4;
    uint64_t b = al(S, 4) * 3 + al((uint64_t)S + 1, 8)                  /* begin, num, order, off */
                 + al(nb, 4) + al(nb + 1, 8) + al(S, 4)                   /* order buckets */
                 + al(total, 4) + al(1, 4)                               /* scores, counter */
                 + al((uint64_t)S * N, 4) + al((uint64_t)S * N, 8) + al((uint64_t)S * N, 4) +
                 al(S, 4) * 2                                            /* top-N */
                 + al(hfx_topn_scratch_bytes(S, total), 1)               /* exact route */
                 + al(bmax, 4) * 3 + al(bmax + 1, 8);                    /* sparse blocks */
    const uint64_t nseg = (S + CUT_SEG - 1) / CUT_SEG;
    if (rows || bt_is_dense(precision))
        b += al((uint64_t)S + 1, 4) + al(nseg * CUT_SEG, 4) + al(nseg, 4) + al(nseg + 1, 8);
    if (rows) b += al(5ull * S + 1, 4) + al(bt_planes_bytes(S), 1);
    if (bt_is_dense(precision)) b += al(bt_dense_scratch(S), 1);
    return b;
}

extern "C" int hfx_batch_required_bytes(uint32_t S, uint64_t total, uint32_t N, uint32_t num_pep,
                                        uint32_t precision, uint64_t *bytes)
{
    HFX_REQUIRE(bytes, HFX_ERR_ARG, "hfx_batch_required_bytes: null out");
    HFX_REQUIRE(precision <= HFX_BATCH_I8X3_DENSE, HFX_ERR_ARG,
                "hfx_batch_required_bytes: unknown precision %u", precision);
    *bytes = bt_bytes(S, total, N, num_pep, precision);
    return HFX_OK;
}

/* Search.hs:427-433 / Execution.hs:77-93 (groupScorePlan): consecutive runs
 * of spectra whose batch fits `budget` device bytes, each as long as it can
 * be (h_off: the S + 1 score offsets, window sizes summed).  A spectrum that
 * alone needs more than the budget is an error (the reference splits such a
 * spectrum's candidates instead; a batch here scores whole windows). */
extern "C" int hfx_batch_split(const uint64_t *h_off, uint32_t S, uint32_t N, uint32_t num_pep,
                               uint32_t precision, uint64_t budget, uint32_t *h_first,
                               uint32_t cap, uint32_t *num_batches)
{
    HFX_REQUIRE(h_off && num_batches, HFX_ERR_ARG, "hfx_batch_split: null argument");
    HFX_REQUIRE(precision <= HFX_BATCH_I8X3_DENSE, HFX_ERR_ARG,
                "hfx_batch_split: unknown precision %u", precision);
    for (uint32_t s = 0; s < S; ++s)
        HFX_REQUIRE(h_off[s + 1] >= h_off[s], HFX_ERR_ARG,
                    "hfx_batch_split: score offsets decrease at spectrum %u", s);
    uint32_t nb = 0, a = 0;
    while (a < S) {
        /* the longest run [a, e) that fits: the requirement grows with the
         * run, so a binary search over its end */
        uint32_t lo = a, hi = S;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo + 1) / 2;
            if (bt_bytes(mid - a, h_off[mid] - h_off[a], N, num_pep, precision) <= budget) lo = mid;
            else hi = mid - 1;
        }
        HFX_REQUIRE(lo > a, HFX_ERR_NOMEM,
                    "hfx_batch_split: spectrum %u alone needs %llu bytes, budget %llu", a,
                    (unsigned long long)bt_bytes(1, h_off[a + 1] - h_off[a], N, num_pep, precision),
                    (unsigned long long)budget);
        if (h_first && nb < cap) h_first[nb] = a;
        ++nb;
        a = lo;
    }
    if (h_first && nb < cap) h_first[nb] = S;
    *num_batches = nb;
    return HFX_OK;
}

extern "C" int hfx_batch_plan(hfx_batch *b, const hfx_db *db, const hfx_spectra *sp, float eps,
                              uint32_t N, uint32_t margin, void *stream)
{
    HFX_REQUIRE(b && db && sp, HFX_ERR_ARG, "hfx_batch_plan: null argument");
    HFX_REQUIRE(N >= 1 && N + margin <= 128 && N <= 64, HFX_ERR_ARG,
                "hfx_batch_plan: N + margin must be <= 128 and N <= 64");
    hipStream_t st = hfx_stream(stream);
    bt_free(b);
    if (b->own && (b->own->db.d_idx_sorted != db->d_idx_sorted ||
                   b->own->db.num_pep != db->num_pep || b->own->db.d_ions != db->d_ions)) {
        hfx_pepix_destroy(b->own);
        b->own = nullptr;
    }
    if (b->ix && (b->ix->db.d_idx_sorted != db->d_idx_sorted || b->ix->db.num_pep != db->num_pep))
        HFX_REQUIRE(false, HFX_ERR_ARG, "hfx_batch_plan: the attached index belongs to another "
                                        "database");
    if (!b->ix) b->ix = b->own;
    b->db = *db;
    b->sp = *sp;
    b->eps = eps;
    b->N = N;
    b->margin = margin;
    const uint32_t S = b->S = sp->num_spec;
    int rc;
    if ((rc = dalloc(&b->begin, S)) || (rc = dalloc(&b->num, S)) ||
        (rc = dalloc(&b->score_off, (size_t)S + 1)) || (rc = dalloc(&b->order, S)))
        return rc;
    /* the windows once, to size the score arrays (the run computes them again) */
    if ((rc = hfx_window(b->ctx, b->begin, b->num, db, sp->d_mass, S, eps, stream))) return rc;
    if ((rc = hfx_scan_offsets(b->ctx, b->score_off, b->num, S, stream))) return rc;
    std::vector<uint32_t> hz(S), hl(S);
    if (S) {
        HFX_CHECK_HIP(hipMemcpyAsync(hz.data(), sp->d_zmax, 4ull * S, hipMemcpyDeviceToHost, st));
        HFX_CHECK_HIP(hipMemcpyAsync(hl.data(), sp->d_len, 4ull * S, hipMemcpyDeviceToHost, st));
    }
    HFX_CHECK_HIP(hipMemcpyAsync(&b->total, b->score_off + S, 8, hipMemcpyDeviceToHost, st));
    HFX_CHECK_HIP(hipStreamSynchronize(st));
    {
        /* fail with a clear message, before allocating, when the batch
         * cannot fit (hfx_batch_split cuts a larger set into batches that do) */
        size_t fr = 0, tot = 0;
        HFX_CHECK_HIP(hipMemGetInfo(&fr, &tot));
        const uint64_t need = bt_bytes(S, b->total, N, db->num_pep, HFX_BATCH_FP32_SPARSE, false);
        if (need > fr && hfx_spare_release()) HFX_CHECK_HIP(hipMemGetInfo(&fr, &tot));
        HFX_REQUIRE(need <= fr, HFX_ERR_NOMEM,
                    "hfx_batch_plan: %u spectra with %llu scores need %llu device bytes, %zu free "
                    "(split them with hfx_batch_split)",
                    S, (unsigned long long)b->total, (unsigned long long)need, fr);
    }
    uint32_t L = 0, lmax = 0;
    for (uint32_t s = 0; s < S; ++s) {
        lmax = std::max(lmax, std::min(hl[s], std::min(sp->x_stride, (uint32_t)HFX_MAX_LEN)));
        L = std::max(L, hz[s] <= HFX_MAX_CHARGE ? hz[s] : 0u);
    }
    b->L = std::max(L, 1u);
    b->lstr = (std::max(lmax, 8u) + 15) & ~15u;
    hfx_order_bufs o{};
    hfx_order_shape(S, db->num_pep, &o);
    b->ord_sh = o.sh;
    b->ord_nbz = o.nbz;
    b->ord_nb = o.nb;
    if ((rc = dalloc(&b->ord_cnt, b->ord_nb)) || (rc = dalloc(&b->ord_off, (size_t)b->ord_nb + 1)) ||
        (rc = dalloc(&b->ord_tmp, S)))
        return rc;
    /* defaults, replaced by the autotuner's choice for this shape */
    b->G = 8;
    b->C = 64;
    b->threads = 512;
    b->precision = HFX_BATCH_FP32_SPARSE;
    bt_pick_chunk(b);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        tune_load_locked();
        auto it = g_tune.find(tune_key(b));
        if (it != g_tune.end()) std::tie(b->G, b->C, b->threads) = it->second;
    }
    if ((rc = dalloc(&b->scores, b->total)) || (rc = dalloc(&b->counter, 1)) ||
        (rc = dalloc(&b->top_pos, (size_t)S * N)) || (rc = dalloc(&b->top_exact, (size_t)S * N)) ||
        (rc = dalloc(&b->top_f32, (size_t)S * N)) || (rc = dalloc(&b->top_cnt, S)) ||
        (rc = dalloc(&b->flag, S)))
        return rc;
    /* the top-N exact route's scratch is owned by the batch, so that a
     * captured graph never allocates and never sees it move */
    if ((rc = dalloc(&b->tx_scratch, hfx_topn_scratch_bytes(S, b->total)))) return rc;
    /* blocks are sized for the smallest G the tuner may pick (4) */
    const uint32_t bmax = (S + 3) / 4;
    if ((rc = dalloc(&b->ubeg, bmax)) || (rc = dalloc(&b->uend, bmax)) ||
        (rc = dalloc(&b->ntiles, bmax)) || (rc = dalloc(&b->tile_off, (size_t)bmax + 1)))
        return rc;
    b->planned = true;
    HFX_CHECK_LAUNCH();
    return bt_ready_attached(b, st);
}

extern "C" int hfx_batch_plan_ix(hfx_batch *b, const hfx_pepix *ix, const hfx_spectra *sp,
                                 float eps, uint32_t N, uint32_t margin, void *stream)
{
    HFX_REQUIRE(b && ix, HFX_ERR_ARG, "hfx_batch_plan_ix: null argument");
    b->ix = ix;
    return hfx_batch_plan(b, &ix->db, sp, eps, N, margin, stream);
}

/* the block cut's buffers */
static int bt_cut_alloc(hfx_batch *b)
{
    int rc;
    b->nseg = (b->S + CUT_SEG - 1) / CUT_SEG;
    if ((!b->dn_bstart && (rc = dalloc(&b->dn_bstart, (size_t)b->S + 1))) ||
        (!b->cut_seg && (rc = dalloc(&b->cut_seg, (size_t)b->nseg * CUT_SEG))) ||
        (!b->cut_n && (rc = dalloc(&b->cut_n, b->nseg))) ||
        (!b->cut_off && (rc = dalloc(&b->cut_off, (size_t)b->nseg + 1))))
        return rc;
    return HFX_OK;
}

/* the dense form's per-batch buffers (hi/lo rows of every spectrum, block
 * bookkeeping), allocated when the form is first chosen */
static int bt_dense_alloc(hfx_batch *b)
{
    const int rc = bt_cut_alloc(b);
    if (rc || b->dn_scratch) return rc;
    return dalloc(&b->dn_scratch, bt_dense_scratch(b->S));
}

/* ---- the phases of one batched search ---- */

/* windows and score offsets */
static int bt_windows(hfx_batch *b, hipStream_t st)
{
    int rc;
    if ((rc = hfx_window(b->ctx, b->begin, b->num, &b->db, b->sp.d_mass, b->S, b->eps, (void *)st)))
        return rc;
    return hfx_scan_offsets(b->ctx, b->score_off, b->num, b->S, (void *)st);
}

/* spectrum order (fragment charge level, precursor mass, index) */
static int bt_order(hfx_batch *b, hipStream_t st)
{
    const hfx_order_bufs o{b->ord_sh, b->ord_nbz, b->ord_nb, b->ord_cnt, b->ord_tmp, b->ord_off};
    return hfx_order_spectra(b->ctx, b->order, &o, b->begin, b->sp.d_zmax, b->sp.d_mass, b->S,
                             (void *)st);
}

/* the rows form of the current precision */
static int bt_mode(const hfx_batch *b)
{
    return b->precision == HFX_BATCH_I8X3_DENSE     ? RW_I8X3
           : b->precision == HFX_BATCH_BF16X2_DENSE ? RW_BF16
                                                    : RW_I8X6;
}
/* dn_scratch (dense forms) or rw_planes as the rows route carves them: planes | item
 * bookkeeping; norms, quanta, levels and the list of the rest in rw_small */
static float2 *bt_norms(const hfx_batch *b) { return (float2 *)b->rw_small; }
static float *bt_quanta(const hfx_batch *b) { return (float *)(b->rw_small + 2 * (size_t)b->S); }
static uint32_t *bt_levels(const hfx_batch *b) { return b->rw_small + 3 * (size_t)b->S; }
static hfx_rest bt_rest(const hfx_batch *b)
{
    return {b->rw_small + 4 * (size_t)b->S, b->rw_small + 5 * (size_t)b->S};
}
static uint8_t *bt_planes(const hfx_batch *b)
{
    return bt_is_dense(b->precision) ? b->dn_scratch : b->rw_planes;
}
static void *bt_items(const hfx_batch *b)
{
    return bt_planes(b) + (size_t)b->S * (bt_is_dense(b->precision) ? 4 : RW_PLANES(RW_I8X6)) * RW_MAXK;
}

/* blocks (segment DP; sixteen spectra a block in the integer form, eight in the
 * others) and the spectra's hi/lo rows or digits */
static int bt_dense_prep(hfx_batch *b, hipStream_t st)
{
    const bool i8 = b->precision == HFX_BATCH_I8X3_DENSE;
    const hfx_rest rest = bt_rest(b);
    const hfx_cut_bufs c{b->cut_seg, b->cut_n, b->cut_off, b->dn_bstart, bt_rows(b) ? rest.count : nullptr};
    int rc;
    if ((rc = hfx_cut_blocks(b->ctx, i8 ? 16u : 8u, &c, b->order, b->begin, b->num, b->sp.d_zmax,
                             b->S, (void *)st)))
        return rc;
    if (bt_rows(b)) {
        return hfx_rows_split(bt_mode(b), &b->sp, bt_planes(b), bt_quanta(b), bt_levels(b), &rest,
                              b->have, bt_norms(b), b->scores, b->score_off, b->begin, b->num,
                              b->db.num_pep, (void *)st);
    }
    return i8 ? hfx_dense8_split(&b->sp, b->dn_scratch, (void *)st)
              : hfx_dense_split(&b->sp, b->dn_scratch, (void *)st);
}

/* blocks of G spectra in order + tiles for the current (G, C) */
static int bt_tiles(hfx_batch *b, hipStream_t st)
{
    b->B = (b->S + b->G - 1) / b->G;
    if (b->B == 0) return HFX_OK;
    hipLaunchKernelGGL(k_bt_blocks, dim3((b->B + 255) / 256), dim3(256), 0, st, b->ubeg, b->uend,
                       b->ntiles, b->order, b->begin, b->num, b->S, b->G, b->B, b->C);
    return hfx_scan_offsets(b->ctx, b->tile_off, b->ntiles, b->B, (void *)st);
}

static int bt_prep(hfx_batch *b, hipStream_t st)
{
    int rc;
    if ((rc = bt_order(b, st))) return rc;
    if (bt_rows(b) || bt_is_dense(b->precision)) return bt_dense_prep(b, st);
    return bt_tiles(b, st);
}

static int bt_score(hfx_batch *b, hipStream_t st, void **ev)
{
    if (b->B == 0 || b->total == 0) return HFX_OK;
    const hfx_pepix *ix = b->ix;
    hipLaunchKernelGGL(k_bt_reset, dim3(1), dim3(1), 0, st, b->counter);
    BtArgs a{b->scores, b->score_off, b->begin,   b->num,     b->order,   b->S,
             b->G,      b->B,         b->C,       b->ubeg,    b->uend,    b->tile_off,
             ix->ent,   ix->cnt,      ix->ent_off, 0u,        b->db.num_pep, ix->L,
             b->lstr,   b->counter,   b->sp};
    const size_t smem = (size_t)b->G * b->lstr * 4;
    const uint32_t grid = (uint32_t)hfx_ctx_num_cus(b->ctx) * (b->G == 8 ? 2u : 4u) *
                          (b->threads == 256 ? 2u : 1u);
    /* gfx950 gives a workgroup up to 160 KiB of LDS; ask for what this
     * configuration stages (G spectra of lstr floats) */
    if (b->G == 8) {
        HFX_CHECK_HIP(hipFuncSetAttribute((const void *)k_batch<8>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        if (ev) HFX_CHECK_HIP(hipEventRecord((hipEvent_t)ev[0], st));
        hipLaunchKernelGGL(k_batch<8>, dim3(grid), dim3(b->threads), smem, st, a);
    } else {
        HFX_CHECK_HIP(hipFuncSetAttribute((const void *)k_batch<4>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        if (ev) HFX_CHECK_HIP(hipEventRecord((hipEvent_t)ev[0], st));
        hipLaunchKernelGGL(k_batch<4>, dim3(grid), dim3(b->threads), smem, st, a);
    }
    if (ev) HFX_CHECK_HIP(hipEventRecord((hipEvent_t)ev[1], st));
    hipLaunchKernelGGL(k_bt_zero_unscored, dim3(b->S), dim3(256), 0, st, b->scores, b->score_off,
                       b->sp.d_zmax, b->S);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* scores from the database's rows, in the current precision; the spectra that these do
 * not serve -- a charge above those the plan's spectra had, or, in the FP32 form, values
 * that the digits do not hold -- by sums within the form's bound */
static int bt_row_scores(hfx_batch *b, hipStream_t st, void **ev)
{
    if (b->total == 0) return HFX_OK;
    const int mode = bt_mode(b);
    const float *qs = bt_quanta(b);
    hfx_spectra sq = b->sp;
    sq.d_zmax = bt_levels(b); /* the rest hidden */
    const hfx_rest rest = bt_rest(b);
    int rc;
    if ((rc = hfx_rows_blocks(b->ctx, bt_items(b), b->order, b->dn_bstart, b->begin, b->num, &sq,
                              b->CH, (void *)st)) ||
        (rc = hfx_rows_scores(b->ctx, mode, bt_items(b), b->scores, b->score_off, b->begin, b->num,
                              b->order, b->dn_bstart, &b->rows, bt_planes(b), qs, &sq, b->CH,
                              (void *)st, ev)))
        return rc;
    return hfx_xcorr_rest(b->ctx, b->scores, b->score_off, b->begin, b->num, &b->db, &b->sp, &rest,
                          mode != RW_I8X6, (void *)st);
}

/* ev (optional): events recorded around the scoring kernel itself */
static int bt_scores(hfx_batch *b, hipStream_t st, void **ev = nullptr)
{
    if (bt_rows(b)) return bt_row_scores(b, st, ev);
    if (b->precision == HFX_BATCH_I8X3_DENSE) {
        if (b->total == 0) return HFX_OK;
        return hfx_dense8_scores(b->ctx, b->scores, b->score_off, b->begin, b->num, b->order,
                                 b->dn_bstart, b->S, &b->ix->lad, &b->sp, b->CH, b->dn_scratch, 1,
                                 (void *)st, ev);
    }
    if (b->precision == HFX_BATCH_BF16X2_DENSE) {
        if (b->total == 0) return HFX_OK;
        return hfx_dense_scores(b->ctx, b->scores, b->score_off, b->begin, b->num, b->order,
                                b->dn_bstart, b->S, &b->ix->lad, &b->sp, b->CH, b->dn_scratch, 1,
                                (void *)st, ev);
    }
    return bt_score(b, st, ev);
}

/* |dense - exact| <= (2^-16 + 210 * 2^-24) * 50 * sum|x|: the hi/lo split
 * (2^-16 per bin) plus at most 100 FP32 additions on any term's path (32 in
 * one MFMA, one per k-step after it) and the hi + lo sum, each allowed 2 ulp */
#define BT_REL_DENSE (1.52587890625e-05f + 210.0f * 5.9604644775390625e-08f)
#define BT_REL_F32 (80.0f * 5.9604644775390625e-08f)
/* integer form: |score - exact| <= max|x| / 8355711 * 50 len (the rounding of
 * x 2^k to integers) + 2^-24 * 50 sum|x| (the one FP32 rounding) */
#define BT_REL_I8 5.9604644775390625e-08f
#define BT_RELQ_I8 (1.0f / 8355711.0f)

static int bt_topn(hfx_batch *b, hipStream_t st)
{
    const bool i8 = b->precision == HFX_BATCH_I8X3_DENSE;
    const float rel0 = i8 ? BT_REL_I8 : b->precision == HFX_BATCH_BF16X2_DENSE ? BT_REL_DENSE
                                                                             : BT_REL_F32;
    return hfx_topn_device(b->ctx, b->top_pos, b->top_exact, b->top_f32, b->top_cnt, b->flag,
                           b->N, b->margin, b->scores, b->score_off, b->total, b->begin, b->num,
                           &b->db, &b->sp, rel0, 0.0f, i8 ? BT_RELQ_I8 : 0.0f,
                           bt_rows(b) ? bt_norms(b) : nullptr, b->tx_scratch, (void *)st);
}

extern "C" int hfx_batch_run(hfx_batch *b, void *stream)
{
    HFX_REQUIRE(b && b->planned, HFX_ERR_ARG, "hfx_batch_run: batch not planned");
    hipStream_t st = hfx_stream(stream);
    int rc;
    if (b->S == 0) return HFX_OK;
    if ((rc = bt_ready(b, st))) return rc;
    if ((rc = bt_windows(b, st)) || (rc = bt_prep(b, st)) || (rc = bt_scores(b, st))) return rc;
    return bt_topn(b, st);
}

extern "C" int hfx_batch_set_precision(hfx_batch *b, uint32_t precision)
{
    HFX_REQUIRE(b && b->planned, HFX_ERR_ARG, "hfx_batch_set_precision: batch not planned");
    HFX_REQUIRE(precision == HFX_BATCH_FP32_SPARSE || bt_is_dense(precision), HFX_ERR_ARG,
                "hfx_batch_set_precision: unknown precision %u", precision);
    HFX_REQUIRE(!bt_is_dense(precision) || b->sp.x_stride <= hfx_dense_max_len(),
                HFX_ERR_ARG,
                "hfx_batch_set_precision: the dense form takes spectra of up to %u bins "
                "(x_stride %u)", hfx_dense_max_len(), b->sp.x_stride);
    int rc;
    if (bt_is_dense(precision) && (rc = bt_dense_alloc(b))) return rc;
    if (bt_is_dense(precision)) b->dense_set = true;
    const bool other = precision != b->precision;
    if (other && b->exec) {
        (void)hipGraphExecDestroy(b->exec);
        b->exec = nullptr;
        (void)hipGraphDestroy(b->graph);
        b->graph = nullptr;
    }
    b->precision = precision;
    if (other) {
        b->chunk_set = false;
        bt_pick_chunk(b);
    }
    return bt_ready_attached(b, nullptr);
}

extern "C" int hfx_batch_capture(hfx_batch *b, void *stream)
{
    HFX_REQUIRE(b && b->planned, HFX_ERR_ARG, "hfx_batch_capture: batch not planned");
    HFX_REQUIRE(stream != nullptr, HFX_ERR_ARG, "hfx_batch_capture: needs a non-null stream");
    hipStream_t st = hfx_stream(stream);
    int rc;
    if ((rc = bt_ready(b, st))) return rc;
    if (b->exec) { (void)hipGraphExecDestroy(b->exec); b->exec = nullptr; }
    if (b->graph) { (void)hipGraphDestroy(b->graph); b->graph = nullptr; }
    /* kernel attributes are set outside the capture */
    HFX_CHECK_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    rc = hfx_batch_run(b, stream);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(st, &g);
    HFX_REQUIRE(rc == HFX_OK, rc, "hfx_batch_capture: run failed during capture: %s",
                hfx_last_error());
    HFX_CHECK_HIP(e);
    b->graph = g;
    HFX_CHECK_HIP(hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
    return HFX_OK;
}

extern "C" int hfx_batch_replay(hfx_batch *b, void *stream)
{
    HFX_REQUIRE(b && b->exec, HFX_ERR_ARG, "hfx_batch_replay: no captured graph");
    HFX_CHECK_HIP(hipGraphLaunch(b->exec, hfx_stream(stream)));
    return HFX_OK;
}

/* Times the scoring kernel of the planned batch for each configuration in a
 * small grid and keeps the fastest; the choice is remembered for batches of
 * the same shape bucket in this process.  Over rows, any form, and in the dense
 * ones: the chunk of candidates per work item; the FP32 form over ion lists: (G, C,
 * threads). */
extern "C" int hfx_batch_autotune(hfx_batch *b, void *stream, uint32_t *out_cfg)
{
    HFX_REQUIRE(b && b->planned, HFX_ERR_ARG, "hfx_batch_autotune: batch not planned");
    hipStream_t st = hfx_stream(stream);
    int rc;
    /* index, windows and order once */
    if ((rc = hfx_batch_run(b, stream))) return rc;
    hipEvent_t e0, e1;
    HFX_CHECK_HIP(hipEventCreate(&e0));
    HFX_CHECK_HIP(hipEventCreate(&e1));
    /* a warm run, then the fastest of three timed runs (the minimum is the
     * least disturbed by clocks and other work) */
    auto time2 = [&](float *ms) -> int {
        int r;
        if ((r = bt_prep(b, st)) || (r = bt_scores(b, st))) return r; /* warm */
        *ms = 1e30f;
        for (int k = 0; k < 3; ++k) {
            float t = 0.0f;
            HFX_CHECK_HIP(hipEventRecord(e0, st));
            if ((r = bt_scores(b, st))) return r;
            HFX_CHECK_HIP(hipEventRecord(e1, st));
            HFX_CHECK_HIP(hipEventSynchronize(e1));
            HFX_CHECK_HIP(hipEventElapsedTime(&t, e0, e1));
            *ms = t < *ms ? t : *ms;
        }
        return HFX_OK;
    };
    float best = 1e30f;
    uint32_t bG = b->G, bC = b->C, bT = b->threads, bCH = b->CH;
    const bool rows = bt_rows(b), chunks = rows || bt_is_dense(b->precision);
    if (chunks) {
        /* the untuned one is among them */
        const uint32_t own = rows ? bt_chunk(b) : 256u;
        const uint32_t CHs[6] = {512, 1024, 2048, 4096, 8192, own};
        for (uint32_t i = 0; i < 6; ++i) {
            const uint32_t CH = CHs[i];
            bool seen = false;
            for (uint32_t j = 0; j < i; ++j)
                seen |= rows ? hfx_rows_item_tiles(CHs[j]) == hfx_rows_item_tiles(CH) : CHs[j] == CH;
            if (seen) continue;
            b->CH = CH;
            float ms = 0;
            if ((rc = time2(&ms))) return rc;
            if (ms < best) { best = ms; bCH = CH; }
        }
    } else {
        const uint32_t Gs[2] = {4, 8}, Cs[4] = {32, 64, 128, 256}, Ts[2] = {256, 512};
        for (uint32_t G : Gs)
            for (uint32_t C : Cs)
                for (uint32_t T : Ts) {
                    b->G = G;
                    b->C = C;
                    b->threads = T;
                    float ms = 0;
                    if ((rc = time2(&ms))) return rc;
                    if (ms < best) { best = ms; bG = G; bC = C; bT = T; }
                }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    b->G = bG;
    b->C = bC;
    b->threads = bT;
    b->CH = bCH;
    b->chunk_set = chunks;
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        tune_load_locked();
        if (chunks) (*tune_chunks(b->precision, rows))[tune_key(b)] = bCH;
        else g_tune[tune_key(b)] = std::make_tuple(bG, bC, bT);
        tune_save_locked();
    }
    if (b->exec) {
        /* the captured graph holds the old launch shapes */
        (void)hipGraphExecDestroy(b->exec);
        b->exec = nullptr;
        (void)hipGraphDestroy(b->graph);
        b->graph = nullptr;
    }
    /* leave the batch's outputs those of the chosen configuration */
    if ((rc = hfx_batch_run(b, stream))) return rc;
    if (out_cfg) {
        out_cfg[0] = bG; out_cfg[1] = bC; out_cfg[2] = bT;
        if (bt_is_dense(b->precision)) {
            out_cfg[0] = 0;
            out_cfg[1] = bCH;
            out_cfg[2] = 1024u; /* workgroup threads of both ladder kernels */
        }
    }
    return HFX_OK;
}

/* Runs the planned batch phase by phase with events between the phases:
 * ms[0] windows + offsets, ms[1] per-batch preparation (spectrum order;
 * dense form: block cut and hi/lo rows; sparse form: tiles), ms[2] scoring,
 * ms[3] top-N (+ exact route). */
extern "C" int hfx_batch_time(hfx_batch *b, void *stream, float *ms)
{
    HFX_REQUIRE(b && b->planned && ms, HFX_ERR_ARG, "hfx_batch_time: batch not planned");
    hipStream_t st = hfx_stream(stream);
    int rc = HFX_OK;
    for (int i = 0; i < 5; ++i) ms[i] = 0.0f;
    if (b->S == 0) return HFX_OK;
    if ((rc = bt_ready(b, st))) return rc;
    hipEvent_t ev[7];
    for (auto &e : ev) HFX_CHECK_HIP(hipEventCreate(&e));
    void *kev[2] = {ev[5], ev[6]};
    HFX_CHECK_HIP(hipEventRecord(ev[0], st));
    if (!rc) rc = bt_windows(b, st);
    HFX_CHECK_HIP(hipEventRecord(ev[1], st));
    if (!rc) rc = bt_prep(b, st);
    HFX_CHECK_HIP(hipEventRecord(ev[2], st));
    const bool scored = b->total != 0 && (bt_rows(b) || bt_is_dense(b->precision) || b->B != 0);
    if (!rc) rc = bt_scores(b, st, kev);
    HFX_CHECK_HIP(hipEventRecord(ev[3], st));
    if (!rc) rc = bt_topn(b, st);
    HFX_CHECK_HIP(hipEventRecord(ev[4], st));
    HFX_CHECK_HIP(hipEventSynchronize(ev[4]));
    for (int i = 0; i < 4; ++i) HFX_CHECK_HIP(hipEventElapsedTime(&ms[i], ev[i], ev[i + 1]));
    if (scored && !rc) HFX_CHECK_HIP(hipEventElapsedTime(&ms[4], ev[5], ev[6]));
    for (auto &e : ev) (void)hipEventDestroy(e);
    return rc;
}

extern "C" int hfx_batch_set_config(hfx_batch *b, uint32_t G, uint32_t C, uint32_t threads)
{
    HFX_REQUIRE(b && b->planned, HFX_ERR_ARG, "hfx_batch_set_config: batch not planned");
    if (bt_is_dense(b->precision)) {
        /* dense forms: C = candidates per work item (G, threads fixed) */
        const uint32_t step = tune_dense_step(b->precision);
        HFX_REQUIRE(tune_dense_ok(b->precision, C), HFX_ERR_ARG,
                    "hfx_batch_set_config: dense chunk must be a multiple of %u in %u..8192",
                    step, step);
        b->CH = C;
        b->chunk_set = true;
        return HFX_OK;
    }
    HFX_REQUIRE(tune_sparse_ok(G, C, threads), HFX_ERR_ARG,
                "hfx_batch_set_config: G in {4,8}, C in 1..4096, threads in {256,512}");
    b->G = G;
    b->C = C;
    b->threads = threads;
    return HFX_OK;
}

extern "C" int hfx_batch_dense_blocks(const hfx_batch *b, uint32_t *h_bstart, uint32_t cap,
                                      uint32_t *num_blocks)
{
    HFX_REQUIRE(b && num_blocks, HFX_ERR_ARG, "hfx_batch_dense_blocks: null argument");
    HFX_REQUIRE(b->planned && b->dense_set, HFX_ERR_ARG,
                "hfx_batch_dense_blocks: no dense run of this batch");
    uint64_t nb = 0;
    HFX_CHECK_HIP(hipDeviceSynchronize());
    HFX_CHECK_HIP(hipMemcpy(&nb, b->cut_off + b->nseg, 8, hipMemcpyDeviceToHost));
    *num_blocks = (uint32_t)nb;
    if (h_bstart && cap) {
        const size_t n = std::min<size_t>(cap, (size_t)nb + 1);
        HFX_CHECK_HIP(hipMemcpy(h_bstart, b->dn_bstart, 4 * n, hipMemcpyDeviceToHost));
    }
    return HFX_OK;
}

extern "C" int hfx_batch_order(const hfx_batch *b, uint32_t *h_order)
{
    HFX_REQUIRE(b && b->planned && h_order, HFX_ERR_ARG, "hfx_batch_order: batch not planned");
    HFX_CHECK_HIP(hipDeviceSynchronize());
    if (b->S) HFX_CHECK_HIP(hipMemcpy(h_order, b->order, 4ull * b->S, hipMemcpyDeviceToHost));
    return HFX_OK;
}

extern "C" int hfx_batch_info(const hfx_batch *b, uint64_t *info /*[12]*/)
{
    HFX_REQUIRE(b && info, HFX_ERR_ARG, "hfx_batch_info: null argument");
    const hfx_pepix *ix = b->ix;
    info[0] = b->S; info[1] = b->total; info[2] = b->db.num_pep; info[3] = b->L;
    info[4] = ix ? ix->n_ent : 0; info[5] = b->G; info[6] = b->C; info[7] = b->threads;
    info[8] = b->lstr; info[9] = 0; info[10] = b->precision; info[11] = b->CH;
    return HFX_OK;
}

extern "C" int hfx_batch_outputs(const hfx_batch *b, void **ptrs /*[10]*/)
{
    HFX_REQUIRE(b && ptrs, HFX_ERR_ARG, "hfx_batch_outputs: null argument");
    ptrs[0] = b->top_pos; ptrs[1] = b->top_exact; ptrs[2] = b->top_f32; ptrs[3] = b->top_cnt;
    ptrs[4] = b->flag; ptrs[5] = b->scores; ptrs[6] = b->score_off; ptrs[7] = b->begin;
    ptrs[8] = b->num; ptrs[9] = b->ix ? (void *)b->ix->ent : nullptr;
    return HFX_OK;
}
