/*
 * hfx_mods.hip -- modified-peptide enumeration and modified theoretical rows.
 *
 *   findModablePeptides  filter_by_mod.cu:150-378
 *   calcTotalModCands    calc_mod_cands.cu:27-119
 *   prepareGenMod        prepare_gen_mod.cu:23-129
 *   genModCands          gen_mod_pep.cu:127-312, combinatorics.h:13-134
 *   addModIons           mion_series.cu:174-556 (dense rows, drop-in)
 *   hfx_mpep_offsets     Search.hs:381-386 on the device
 *
 * Integer work throughout; outputs are bit-identical to the reference's
 * (including unrankComb's reflection trick, which repeats some subsets and
 * misses others for e.g. n=5, k=2 -- reproduced, not fixed).  The one
 * deliberate difference: a modified residue's occurrence index counts its own
 * acid (check_series.cu:61-99, filter_by_mod.cu:216-230) where
 * mion_series.cu:252-269 counts every modable acid.
 */
#include "hfx_cand.h"

/* ------------------------------------------------------------------ */
/* Combinatorics                                                         */
/* ------------------------------------------------------------------ */

struct ChooseTab {
    uint32_t t[43][12];
};
static constexpr ChooseTab make_choose()
{
    ChooseTab c{};
    for (int a = 0; a <= 42; ++a)
        for (int b = 0; b <= 11; ++b)
            c.t[a][b] = (b == 0) ? 1u : (a == 0 ? 0u : c.t[a - 1][b - 1] + c.t[a - 1][b]);
    return c;
}
/* C(n, k) for n <= 42, k <= 11: the table of combinatorics.h:13-57 */
__constant__ ChooseTab k_choose = make_choose();

/* a workgroup's copy of the table in LDS: lanes look up different entries, which
 * constant memory serves one at a time */
typedef uint32_t ChooseLds[43 * 12];
__device__ __forceinline__ void choose_load(uint32_t *t)
{
    for (uint32_t i = threadIdx.x; i < 43 * 12; i += blockDim.x) t[i] = (&k_choose.t[0][0])[i];
    __syncthreads();
}

/* combinatorics.h:59-88 */
__device__ __forceinline__ uint32_t d_choose(const uint32_t *tab, uint32_t n, uint32_t k)
{
    if (n > 42 || k > 11) {
        if (k == 0 || n == k) return 1;
        if (n < k) return 0;
        uint32_t t = 1;
        if (k < n - k) {
            for (uint32_t i = n; i >= n - k + 1; --i) t = t * i / (n - i + 1);
        } else {
            for (uint32_t i = n; i >= k + 1; --i) t = t * i / (n - i + 1);
        }
        return t;
    }
    return tab[n * 12 + k];
}

/* combinatorics.h:90-134 largestV + unrankComb */
__device__ __forceinline__ void d_unrank_comb(const uint32_t *tab, uint32_t *ans, uint32_t n, uint32_t k,
                                              uint32_t rank)
{
    uint32_t a = n, b = k;
    const uint32_t total = d_choose(tab, n, k);
    uint32_t x;
    bool dual = false;
    if ((total / 2) >= rank) x = rank;
    else { x = total - 1 - rank; dual = true; }
    for (uint32_t i = 0; i < k; ++i) {
        uint32_t v = a - 1, c;
        while ((c = d_choose(tab, v, b)) > x) --v;
        ans[i] = dual ? (n - 1) - v : v;
        x = x - c;
        a = v;
        b = b - 1;
    }
}

/* A kernel's instance for na modable acids: every number that prepare_ions packs (1
 * to 7) has its own, whose loops over the acids keep their values in registers; up to
 * 10, which these steps take, share one.  Finding the rows and unranking for 1,500
 * spectra, us: one acid 93 and 17 by the shared instance, 90 and 16 by its own; three
 * 124 and 36, 116 and 33; seven 337 and 173, 292 and 130. */
#define MOD_NA(k, na) \
    ((na) == 1 ? k<1> : (na) == 2 ? k<2> : (na) == 3 ? k<3> : (na) == 4 ? k<4> : (na) == 5 ? k<5> \
     : (na) == 6 ? k<6> : (na) == 7 ? k<7> : k<0>)
static_assert(HFX_MAX_MA == 7, "an instance for each packed number of acids");

/* ------------------------------------------------------------------ */
/* findModablePeptides                                                   */
/* ------------------------------------------------------------------ */

/* counts of each modable acid over [tc, tn) (fillPepMACount :193-231) of
 * the peptide at every residual-sorted position below npos, and for each
 * modification a bit per position: the peptide holds the acids it needs
 * (checkModable :234-262).  One wave per 64 positions, a word of bits each. */
__global__ void __launch_bounds__(256)
    k_mod_bits(uint32_t *pcnt, uint64_t *bits, uint32_t W, const uint32_t *idx_sorted, uint32_t npos,
               const uint8_t *ions, const uint32_t *tc, const uint32_t *tn, const uint8_t *ma,
               uint32_t num_ma, const uint32_t *mod_ma_count, uint32_t num_mod)
{
    const uint32_t w = blockIdx.x * 4 + threadIdx.x / HFX_WAVE, k = w * HFX_WAVE + hfx_lane();
    if (w >= W) return;
    uint32_t c[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (k < npos) {
        const uint32_t pep = idx_sorted[k];
        uint8_t mac[10];
#pragma unroll
        for (uint32_t a = 0; a < 10; ++a) mac[a] = a < num_ma ? ma[a] : 0;
        const uint32_t j1 = tn[pep];
        for (uint32_t j = tc[pep]; j < j1; ++j) {
            const uint8_t ch = (uint8_t)(HFX_ACID_IDX(ions[j]) + 'A');
#pragma unroll
            for (uint32_t a = 0; a < 10; ++a) c[a] += (ch == mac[a]) ? 1u : 0u;
        }
#pragma unroll
        for (uint32_t a = 0; a < 10; ++a)
            if (a < num_ma) pcnt[(size_t)k * num_ma + a] = c[a];
    }
    for (uint32_t m = 0; m < num_mod; ++m) {
        const uint32_t *need = mod_ma_count + (size_t)m * num_ma;
        bool ok = k < npos;
#pragma unroll
        for (uint32_t a = 0; a < 10; ++a)
            if (a < num_ma) ok = ok && c[a] >= need[a];
        const uint64_t v = __ballot(ok);
        if (hfx_lane() == 0) bits[(size_t)m * W + w] = v;
    }
}

/* rank[m][w]: the bits of modification m before word w.  A workgroup each. */
__global__ void __launch_bounds__(1024) k_mod_rank(uint32_t *rank, const uint64_t *bits, uint32_t W)
{
    __shared__ uint32_t wt[16];
    const uint64_t *b = bits + (size_t)blockIdx.x * W;
    uint32_t *r = rank + (size_t)blockIdx.x * W;
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (uint32_t w0 = 0; w0 < W; w0 += 1024) {
        const uint32_t w = w0 + threadIdx.x;
        const uint32_t v = w < W ? (uint32_t)__popcll(b[w]) : 0u;
        uint32_t x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) wt[wid] = x;
        __syncthreads();
        uint32_t pre = carry;
        for (uint32_t i = 0; i < 16; ++i) {
            pre += i < wid ? wt[i] : 0u;
            carry += wt[i];
        }
        if (w < W) r[w] = pre + x - v;
        __syncthreads();
    }
}

struct ModBits {
    const uint64_t *bits; /* [num_mod][W], W words past the last position */
    const uint32_t *rank;
    uint32_t W;
    /* modable peptides of m at positions below k */
    __device__ __forceinline__ uint32_t below(uint32_t m, uint32_t k) const
    {
        const size_t w = (size_t)m * W + k / 64;
        return rank[w] + (uint32_t)__popcll(bits[w] & ((1ull << (k % 64)) - 1ull));
    }
};

/* the windows of a part of the modifications, [m0, m0 + M) of num_mod: the i-th of
 * them, spectrum by spectrum */
struct ModPart {
    uint32_t m0, M, num_mod;
    uint64_t pairs; /* spectra x M */
    __device__ __forceinline__ uint64_t window(uint64_t i) const { return i / M * num_mod + m0 + i % M; }
};

/* modable peptides of every (spectrum, modification) window */
__global__ void k_mod_counts(uint32_t *cnt, const uint32_t *begin, const uint32_t *end, ModPart p,
                             ModBits mb)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.pairs) return;
    const uint64_t pr = p.window(i);
    const uint32_t m = (uint32_t)(i % p.M), b = begin[pr], e = end[pr];
    cnt[pr] = b < e ? mb.below(m, e) - mb.below(m, b) : 0u;
}

/* The modable rows (pep, mod): spectrum-major, mod-minor, residual-sorted
 * within a window (fillPepAndModIdx :151-190, remove_if :345-358), with each
 * row's acid counts; one wave per (spectrum, mod), a word of bits a step.
 * Only the rows that stay are written -- 5.8 of 50.9 million for 5,000 spectra
 * and 34 modifications; writing, scanning and compacting all of them took 1,300
 * us; the bits, their ranks, the counts and their scan take 60, this 78 (190
 * with a read of the bits, and of each acid's count, after every store). */
template <uint32_t NA> /* num_ma, or 0: any up to 10 */
__global__ void __launch_bounds__(256)
    k_mod_rows(uint32_t *__restrict__ out_pep, uint32_t *__restrict__ out_mod,
               uint32_t *__restrict__ out_cnt, const uint64_t *off,
               const uint32_t *__restrict__ idx_sorted, const uint32_t *begin, const uint32_t *end,
               ModPart part, const uint32_t *__restrict__ pcnt, uint32_t num_ma, ModBits mb)
{
    const uint64_t i = (uint64_t)blockIdx.x * 4 + threadIdx.x / HFX_WAVE;
    if (i >= part.pairs) return;
    const uint64_t pr = part.window(i);
    const uint32_t m = (uint32_t)(i % part.M), lane = hfx_lane();
    const uint32_t na = NA ? NA : num_ma;
    const uint32_t b = begin[pr], e = end[pr];
    const uint64_t *bits = mb.bits + (size_t)m * mb.W;
    uint64_t o = off[pr];
    if (b >= e) return;
    const uint32_t w1 = (e - 1) / 64;
    for (uint32_t w0 = b / 64; w0 <= w1; w0 += HFX_WAVE) {
        /* lane l: word w0 + l of the window */
        const uint32_t wl = w0 + lane;
        uint64_t mine = wl <= w1 ? bits[wl] : 0ull;
        if (wl == b / 64) mine &= ~0ull << (b % 64);
        if (wl == e / 64) mine &= (1ull << (e % 64)) - 1ull;
        const uint32_t nw = min(w1 - w0 + 1u, (uint32_t)HFX_WAVE);
        for (uint32_t j = 0; j < nw; ++j) {
            const uint64_t v = (uint64_t)hfx_take((uint32_t)(mine >> 32), j) << 32 |
                               hfx_take((uint32_t)mine, j);
            if ((v >> lane) & 1ull) {
                const uint64_t p = o + (uint32_t)__popcll(v & ((1ull << lane) - 1ull));
                const uint32_t k = (w0 + j) * 64 + lane;
                const uint32_t *from = pcnt + (size_t)k * na;
                uint32_t c[NA ? NA : 10];
#pragma unroll
                for (uint32_t a = 0; a < (NA ? NA : 10u); ++a)
                    if (a < na) c[a] = from[a];
                out_pep[p] = idx_sorted[k];
                out_mod[p] = part.m0 + m;
#pragma unroll
                for (uint32_t a = 0; a < (NA ? NA : 10u); ++a)
                    if (a < na) out_cnt[p * na + a] = c[a];
            }
            o += (uint32_t)__popcll(v);
        }
    }
}

/* largest window end (every window position lies below it), by workgroup */
#define ME_BLOCKS 64u
__global__ void __launch_bounds__(1024) k_max_end(const uint32_t *end, uint64_t n, uint32_t *out)
{
    __shared__ uint32_t w[16];
    uint32_t v = 0;
    for (uint64_t i = blockIdx.x * 1024ull + threadIdx.x; i < n; i += gridDim.x * 1024ull)
        v = max(v, end[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int i = 0; i < 16; ++i) t = max(t, w[i]);
        out[blockIdx.x] = t;
    }
}

/* lower_bound(kept row ids, spec_num_cand_scan[s]) == number of kept rows of
 * the spectra before s (:364-366) */
__global__ void k_mod_valid_scan(uint32_t *out, const uint64_t *off, uint32_t num_mod,
                                 uint32_t num_spec)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < num_spec) out[s] = off ? (uint32_t)off[(uint64_t)s * num_mod] : 0u;
}

static int read_u64(const uint64_t *d, uint64_t *out)
{
    HFX_CHECK_HIP(hipMemcpy(out, d, 8, hipMemcpyDeviceToHost));
    return HFX_OK;
}

extern "C" uint32_t findModablePeptides(
    uint32_t *d_out_pep_idx_raw, uint32_t *d_out_pep_mod_idx_raw, uint32_t *d_out_pep_ma_count_raw,
    uint32_t *d_out_spec_num_valid_scan, const uint32_t *d_spec_num_cand_scan,
    const uint32_t num_spec, uint32_t num_cand_total, const uint8_t *d_ions, const uint32_t *d_tc,
    const uint32_t *d_tn, const uint32_t *d_pep_idx_r_sorted_raw, const uint32_t *d_begin_raw,
    const uint32_t *d_end_raw, const uint32_t *d_num_pep_scan_raw, const uint32_t *d_mod_ma_count,
    const uint32_t num_mod, const uint8_t *d_ma, const uint32_t num_ma)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return 0;
    if (num_ma > 10) {
        hfx_set_error("findModablePeptides: num_ma %u > 10", num_ma);
        return 0;
    }
    (void)d_spec_num_cand_scan;
    (void)d_num_pep_scan_raw;
    if (num_spec == 0 || num_mod == 0) return 0;
    const uint64_t pairs = (uint64_t)num_spec * num_mod;
    const dim3 gs((num_spec + 255) / 256), t(256);
    if (num_cand_total == 0) {
        hipLaunchKernelGGL(k_mod_valid_scan, gs, t, 0, 0, d_out_spec_num_valid_scan,
                           (const uint64_t *)nullptr, num_mod, num_spec);
        if (hipStreamSynchronize(0) != hipSuccess) hfx_set_error("findModablePeptides: sync failed");
        return 0;
    }
    if (pairs >= 0xffffffffull) {
        hfx_set_error("findModablePeptides: %llu windows", (unsigned long long)pairs);
        return 0;
    }
    /* the positions the windows reach (one small read back) */
    uint32_t npos = 0;
    {
        void *q, *h;
        const uint32_t g = (uint32_t)min((pairs + 1023) / 1024, (uint64_t)ME_BLOCKS);
        if (hfx_ctx_scratch(ctx, HFX_SLOT_MODS2, 4 * ME_BLOCKS, &q) != HFX_OK) return 0;
        if (hfx_ctx_pinned(ctx, 4 * ME_BLOCKS, &h) != HFX_OK) return 0;
        hipLaunchKernelGGL(k_max_end, dim3(g), dim3(1024), 0, 0, d_end_raw, pairs, (uint32_t *)q);
        if (hipMemcpy(h, q, 4 * g, hipMemcpyDeviceToHost) != hipSuccess) {
            hfx_set_error("findModablePeptides: read back failed");
            return 0;
        }
        for (uint32_t i = 0; i < g; ++i) npos = max(npos, ((uint32_t *)h)[i]);
    }
    /* The bits and ranks take 12 bytes for 64 positions and a modification, however
     * few of them a window holds: so many modifications at a time that they take no
     * more than 64 MiB, or than the rows of all candidates would. */
    const uint32_t W = npos / 64 + 1;
    const uint64_t room = max((uint64_t)num_cand_total * (20 + 4 * num_ma), 64ull << 20);
    const uint32_t M = (uint32_t)min((uint64_t)num_mod, max(room / (12ull * W), 1ull));
    void *p;
    const size_t words = (size_t)W * M;
    const size_t bytes = words * 12 + (pairs + 1) * 8 + pairs * 4 + (size_t)npos * 4 * num_ma + 64;
    if (hfx_ctx_scratch(ctx, HFX_SLOT_MODS, bytes, &p) != HFX_OK) return 0;
    uint64_t *off = (uint64_t *)p, *bits = off + pairs + 1;
    uint32_t *rank = (uint32_t *)(bits + words), *cnt = rank + words, *pcnt = cnt + pairs;
    const ModBits mb{bits, rank, W};
    auto part = [&](uint32_t m0) {
        const uint32_t m = min(M, num_mod - m0);
        return ModPart{m0, m, num_mod, (uint64_t)num_spec * m};
    };
    auto find = [&](const ModPart &q) {
        hipLaunchKernelGGL(k_mod_bits, dim3((W + 3) / 4), t, 0, 0, pcnt, bits, W, d_pep_idx_r_sorted_raw,
                           npos, d_ions, d_tc, d_tn, d_ma, num_ma,
                           d_mod_ma_count + (size_t)q.m0 * num_ma, q.M);
        hipLaunchKernelGGL(k_mod_rank, dim3(q.M), dim3(1024), 0, 0, rank, bits, W);
    };
    for (uint64_t m0 = 0; m0 < num_mod; m0 += M) {
        const ModPart q = part((uint32_t)m0);
        find(q);
        hipLaunchKernelGGL(k_mod_counts, dim3((uint32_t)((q.pairs + 255) / 256)), t, 0, 0, cnt,
                           d_begin_raw, d_end_raw, q, mb);
    }
    if (hfx_scan_offsets(ctx, off, cnt, (uint32_t)pairs, nullptr) != HFX_OK) return 0;
    const auto rows = MOD_NA(k_mod_rows, num_ma);
    for (uint64_t m0 = 0; m0 < num_mod; m0 += M) {
        const ModPart q = part((uint32_t)m0);
        if (M < num_mod) find(q);
        hipLaunchKernelGGL(rows, dim3((uint32_t)((q.pairs + 3) / 4)), t, 0, 0, d_out_pep_idx_raw,
                           d_out_pep_mod_idx_raw, d_out_pep_ma_count_raw, off, d_pep_idx_r_sorted_raw,
                           d_begin_raw, d_end_raw, q, pcnt, num_ma, mb);
    }
    hipLaunchKernelGGL(k_mod_valid_scan, gs, t, 0, 0, d_out_spec_num_valid_scan, off, num_mod,
                       num_spec);
    uint64_t total = 0;
    if (read_u64(off + pairs, &total) != HFX_OK) return 0;
    return (uint32_t)total;
}

/* ------------------------------------------------------------------ */
/* calcTotalModCands                                                      */
/* ------------------------------------------------------------------ */

__global__ void k_calc_mod_cands(uint32_t *num_mpep, uint32_t *comb_scan, const uint32_t *mod_ma_count,
                                 const uint32_t *pep_mod_idx, const uint32_t *pep_ma_count,
                                 uint32_t n, uint32_t num_ma)
{
    __shared__ ChooseLds tab;
    choose_load(tab);
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t m = pep_mod_idx[p];
    uint32_t have[10], need[10], num = 1;
    if (num_ma > 10) {
        for (int32_t i = (int32_t)num_ma - 1; i >= 0; --i) {
            num *= d_choose(tab, pep_ma_count[(size_t)num_ma * p + i],
                            mod_ma_count[(size_t)num_ma * m + i]);
            comb_scan[(size_t)num_ma * p + i] = num;
        }
        num_mpep[p] = num;
        return;
    }
#pragma unroll
    for (uint32_t i = 0; i < 10; ++i)
        if (i < num_ma) {
            have[i] = pep_ma_count[(size_t)num_ma * p + i];
            need[i] = mod_ma_count[(size_t)num_ma * m + i];
        }
#pragma unroll
    for (int32_t i = 9; i >= 0; --i)
        if (i < (int32_t)num_ma) {
            num *= d_choose(tab, have[i], need[i]);
            comb_scan[(size_t)num_ma * p + i] = num;
        }
    num_mpep[p] = num;
}

extern "C" uint32_t calcTotalModCands(uint32_t *d_out_pep_num_mpep_raw,
                                      uint32_t *d_out_pep_ma_num_comb_scan_raw,
                                      const uint32_t *d_mod_ma_count_raw, const uint32_t *d_pep_idx_raw,
                                      const uint32_t *d_pep_mod_idx_raw,
                                      const uint32_t *d_pep_ma_count_raw, const uint32_t nPep,
                                      const uint32_t num_mod, const uint32_t num_ma)
{
    (void)d_pep_idx_raw;
    (void)num_mod;
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx || nPep == 0) return 0;
    hipLaunchKernelGGL(k_calc_mod_cands, dim3((nPep + 255) / 256), dim3(256), 0, 0,
                       d_out_pep_num_mpep_raw, d_out_pep_ma_num_comb_scan_raw, d_mod_ma_count_raw,
                       d_pep_mod_idx_raw, d_pep_ma_count_raw, nPep, num_ma);
    return hfx_sum_u32_to_host(ctx, d_out_pep_num_mpep_raw, nPep);
}

/* ------------------------------------------------------------------ */
/* prepareGenMod                                                          */
/* ------------------------------------------------------------------ */

/* GE_ITEMS modified peptides a workgroup: a 64-way search finds the row of the
 * first, the rows that start among them are marked in LDS, and the largest mark
 * so far gives each its row.  A search of 23 steps for every one took 210 us for
 * 10.2 million, 87 now (204 MB written). */
#define GE_THREADS 256
#define GE_PER 8
#define GE_ITEMS (GE_THREADS * GE_PER)
__global__ void __launch_bounds__(GE_THREADS)
    k_gen_expand(uint32_t *o_pep, uint32_t *o_mod, uint32_t *o_rank, uint32_t *o_ith, uint32_t *o_sum,
                 const uint32_t *mod_ma_count_sum, const uint32_t *pep_idx, const uint32_t *pep_mod_idx,
                 const uint64_t *row_off, uint32_t num_rows, uint32_t num_mpep)
{
    __shared__ uint32_t mark[GE_ITEMS], wmax[GE_THREADS / HFX_WAVE];
    const uint32_t tid = threadIdx.x, lane = hfx_lane(), wave = tid / HFX_WAVE;
    const uint64_t i0 = (uint64_t)blockIdx.x * GE_ITEMS;
    const uint32_t cnt = (uint32_t)min((uint64_t)num_mpep - i0, (uint64_t)GE_ITEMS);
    for (uint32_t i = tid; i < GE_ITEMS; i += GE_THREADS) mark[i] = 0;
    /* the last row that starts at or before i0: in [lo, lo + n) */
    uint32_t lo = 0, n = num_rows;
    while (n > 1) {
        const uint32_t step = (n + HFX_WAVE - 1) / HFX_WAVE;
        const uint64_t at = (uint64_t)lane * step;
        const uint64_t in = __ballot(at < n && row_off[lo + min(at, (uint64_t)n - 1)] <= i0);
        const uint32_t c = (uint32_t)__popcll(in) - 1u; /* lane 0 is always in */
        lo += c * step;
        n = min(step, n - c * step);
    }
    __syncthreads();
    for (uint32_t r = lo + 1 + tid;; r += GE_THREADS) {
        const uint64_t o = r < num_rows ? row_off[r] : ~0ull;
        if (o < i0 + cnt) atomicMax(&mark[o - i0], r - lo);
        /* rows start in order: past the last of them when any lies beyond */
        if (__ballot(o < i0 + cnt) != ~0ull) break;
    }
    __syncthreads();
    uint32_t m[GE_PER], x = 0;
#pragma unroll
    for (uint32_t q = 0; q < GE_PER; ++q) {
        x = max(x, mark[tid * GE_PER + q]);
        m[q] = x;
    }
#pragma unroll
    for (uint32_t o = 1; o < HFX_WAVE; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x = max(x, y);
    }
    if (lane == HFX_WAVE - 1) wmax[wave] = x;
    uint32_t pre = __shfl_up(x, 1, 64);
    if (lane == 0) pre = 0;
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) pre = max(pre, wmax[w]);
#pragma unroll
    for (uint32_t q = 0; q < GE_PER; ++q) mark[tid * GE_PER + q] = lo + max(m[q], pre);
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < GE_PER; ++q) {
        const uint32_t j = q * GE_THREADS + tid;
        if (j >= cnt) break;
        const uint64_t i = i0 + j;
        const uint32_t row = mark[j], md = pep_mod_idx[row];
        o_pep[i] = pep_idx[row];
        o_mod[i] = md;
        o_rank[i] = (uint32_t)(i - row_off[row]);
        o_ith[i] = row;
        o_sum[i] = mod_ma_count_sum[md];
    }
}

extern "C" uint32_t prepareGenMod(uint32_t *d_out_mpep_pep_idx, uint32_t *d_out_mpep_pep_mod_idx,
                                  uint32_t *d_out_mpep_rank, uint32_t *d_out_mpep_ith_valid,
                                  uint32_t *d_out_mpep_mod_ma_count_sum_scan,
                                  const uint32_t *d_mod_ma_count_sum, const uint32_t *d_pep_idx,
                                  const uint32_t *d_pep_mod_idx, const uint32_t *d_pep_num_mpep,
                                  const uint32_t num_pep, const uint32_t num_mpep)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx || num_pep == 0 || num_mpep == 0) return 0;
    void *p;
    if (hfx_ctx_scratch(ctx, HFX_SLOT_MODS2, ((size_t)num_pep + 1) * 8, &p) != HFX_OK) return 0;
    uint64_t *row_off = (uint64_t *)p;
    if (hfx_scan_offsets(ctx, row_off, d_pep_num_mpep, num_pep, nullptr) != HFX_OK) return 0;
    uint64_t avail = 0;
    if (read_u64(row_off + num_pep, &avail) != HFX_OK) return 0;
    const uint32_t m = (uint32_t)min((uint64_t)num_mpep, avail);
    hipLaunchKernelGGL(k_gen_expand, dim3((uint32_t)(((uint64_t)m + GE_ITEMS - 1) / GE_ITEMS)),
                       dim3(GE_THREADS), 0, 0, d_out_mpep_pep_idx,
                       d_out_mpep_pep_mod_idx, d_out_mpep_rank, d_out_mpep_ith_valid,
                       d_out_mpep_mod_ma_count_sum_scan, d_mod_ma_count_sum, d_pep_idx,
                       d_pep_mod_idx, row_off, num_pep, m);
    const uint32_t total = hfx_sum_u32_to_host(ctx, d_out_mpep_mod_ma_count_sum_scan, m);
    hfx_scan_u32_inplace(d_out_mpep_mod_ma_count_sum_scan, m, nullptr);
    if (hipStreamSynchronize(0) != hipSuccess) hfx_set_error("prepareGenMod: sync failed");
    return total;
}

/* ------------------------------------------------------------------ */
/* genModCands                                                            */
/* ------------------------------------------------------------------ */

/* 10.2 million: 273 us with the table in constant memory and a read of the next
 * acid's counts behind every store; 117 now, 0.5 GB. */
template <uint32_t NA> /* num_ma, or 0: any up to 10 */
__global__ void k_gen_mod_cands(uint32_t *__restrict__ out_unrank,
                                const uint32_t *__restrict__ mod_ma_count,
                                const uint32_t *__restrict__ mpep_ith,
                                const uint32_t *__restrict__ mpep_rank,
                                const uint32_t *__restrict__ mpep_scan,
                                const uint32_t *__restrict__ pep_mod_idx,
                                const uint32_t *__restrict__ pep_ma_count,
                                const uint32_t *__restrict__ comb_scan, uint32_t num_mpep,
                                uint32_t num_ma)
{
    __shared__ ChooseLds tab;
    choose_load(tab);
    const uint32_t mp = blockIdx.x * blockDim.x + threadIdx.x;
    if (mp >= num_mpep) return;
    constexpr uint32_t MA = NA ? NA : 10;
    const uint32_t na = NA ? NA : num_ma;
    const uint32_t ith = mpep_ith[mp];
    uint32_t x = mpep_rank[mp], pos = mpep_scan[mp];
    const uint32_t pm = pep_mod_idx[ith];
    uint32_t have[MA], need[MA], comb[MA];
#pragma unroll
    for (uint32_t i = 0; i < MA; ++i)
        if (i < na) {
            have[i] = pep_ma_count[(size_t)ith * na + i];
            comb[i] = comb_scan[(size_t)ith * na + i];
            need[i] = mod_ma_count[(size_t)pm * na + i];
        }
    /* add_ma_ranks, gen_mod_pep.cu:127-157 */
#pragma unroll
    for (uint32_t i = 0; i < MA; ++i)
        if (i < na) {
            uint32_t rank = x;
            if (i + 1 < MA && i + 1 < na) {
                const uint32_t nxt = comb[i + 1 < MA ? i + 1 : i];
                rank = 0;
                if (x >= nxt) {
                    rank = x / nxt;
                    x = x % nxt;
                }
            }
            if (need[i] != 0) {
                d_unrank_comb(tab, out_unrank + pos, have[i], need[i], rank);
                pos += need[i];
            }
        }
}

extern "C" void genModCands(uint32_t *d_out_mpep_unrank, const uint32_t *d_mod_ma_count,
                            const uint32_t *d_mpep_ith_valid, const uint32_t *d_mpep_rank,
                            const uint32_t *d_mpep_mod_ma_count_sum_scan,
                            const uint32_t *d_pep_mod_idx, const uint32_t *d_pep_ma_count,
                            const uint32_t *d_pep_ma_num_comb_scan, const uint32_t total,
                            const uint32_t mod_num_ma)
{
    if (total == 0) return;
    if (mod_num_ma < 1 || mod_num_ma > 10) {
        hfx_set_error("genModCands: num_ma %u outside 1..10", mod_num_ma);
        return;
    }
    hipLaunchKernelGGL(MOD_NA(k_gen_mod_cands, mod_num_ma), dim3((total + 255) / 256), dim3(256), 0, 0,
                       d_out_mpep_unrank, d_mod_ma_count, d_mpep_ith_valid, d_mpep_rank,
                       d_mpep_mod_ma_count_sum_scan, d_pep_mod_idx, d_pep_ma_count,
                       d_pep_ma_num_comb_scan, total, mod_num_ma);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("genModCands: %s", hipGetErrorString(e));
}

/* ------------------------------------------------------------------ */
/* addModIons: dense rows of modified peptides                           */
/* ------------------------------------------------------------------ */

#define AM_THREADS 256
#define AM_WAVES (AM_THREADS / HFX_WAVE)

__global__ void __launch_bounds__(AM_THREADS)
    k_add_mod_ions(float *spec, const float *residual, const float *mass, const uint8_t *ions_all,
                   const uint32_t *tc_a, const uint32_t *tn_a, const uint32_t *mp_pep,
                   const uint32_t *mp_mod, const uint32_t *unrank, const uint32_t *mp_scan,
                   uint32_t num_mpep, const uint32_t *mod_ma_count, const float *mod_delta,
                   const float *ma_mass, uint32_t num_ma, uint32_t len, uint32_t zmax)
{
    __shared__ uint32_t maps[AM_WAVES][HFX_MAP_WORDS];
    __shared__ float mtab[32];
    const uint32_t wave = threadIdx.x / HFX_WAVE;
    uint32_t *map = maps[wave];
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? mass[threadIdx.x] : 0.0f;
    for (uint32_t w = hfx_lane(); w < HFX_MAP_WORDS; w += HFX_WAVE) map[w] = 0;
    __syncthreads();
    for (uint32_t row = blockIdx.x * AM_WAVES + wave; row < num_mpep; row += gridDim.x * AM_WAVES) {
        const uint32_t pep = mp_pep[row], mod = mp_mod[row];
        const uint32_t tc = tc_a[pep], tn = tn_a[pep];
        const uint32_t n = tn > tc ? tn - tc : 0;
        HfxModMass mm{ions_all + tc, mtab, mod_ma_count + (size_t)mod * num_ma,
                      unrank + mp_scan[row], ma_mass, num_ma, {0, 0, 0, 0, 0, 0, 0}};
        hfx_wave_peaks(map, n, residual[pep] + mod_delta[mod], zmax, len, mm);
        hfx_wave_sync();
        const uint32_t nw = (len + 7) >> 3;
        float *out = spec + (size_t)row * len;
        for (uint32_t w = hfx_lane(); w < nw; w += HFX_WAVE) {
            const uint32_t word = map[w];
            map[w] = 0;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t b = (w << 3) + k;
                if (b < len) out[b] = hfx_code_weight((word >> (4 * k)) & 0xFu);
            }
        }
        hfx_wave_sync();
    }
}

extern "C" void addModIons(float *d_out_mspec, const float *d_residual, const float *d_mass,
                           const uint8_t *d_ions, const uint32_t *d_tc, const uint32_t *d_tn,
                           const uint32_t *d_mpep_pep_idx, const uint32_t *d_mpep_pep_mod_idx,
                           const uint32_t *d_mpep_unrank,
                           const uint32_t *d_mpep_mod_ma_count_sum_scan, const uint32_t len_unrank,
                           const uint32_t num_mpep, const uint32_t *d_mod_ma_count,
                           const float *d_mod_delta, const uint8_t *d_ma, const float *d_ma_mass,
                           const uint32_t num_ma, const uint32_t len_spec,
                           const uint32_t max_charge, void *stream)
{
    (void)len_unrank;
    (void)d_ma;
    if (num_mpep == 0) return;
    /* mion_series.cu:443-556 dispatches MaxCharge 1..10 and NumMA 1..10; the
     * 3-bit packing of prepare_ions limits modable acids to 7 */
    if (max_charge < 1 || max_charge > 10 || num_ma < 1 || num_ma > HFX_MAX_MA ||
        len_spec > HFX_MAX_LEN) {
        hfx_set_error("addModIons: unsupported max_charge %u / num_ma %u / len %u", max_charge,
                      num_ma, len_spec);
        return;
    }
    const uint32_t blocks = min((num_mpep + AM_WAVES - 1) / AM_WAVES, 65535u);
    hipLaunchKernelGGL(k_add_mod_ions, dim3(blocks), dim3(AM_THREADS), 0, hfx_stream(stream),
                       d_out_mspec, d_residual, d_mass, d_ions, d_tc, d_tn, d_mpep_pep_idx,
                       d_mpep_pep_mod_idx, d_mpep_unrank, d_mpep_mod_ma_count_sum_scan, num_mpep,
                       d_mod_ma_count, d_mod_delta, d_ma_mass, num_ma, len_spec, max_charge);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("addModIons: %s", hipGetErrorString(e));
}

/* ------------------------------------------------------------------ */
/* Per-spectrum offsets of the modified peptides                          */
/* ------------------------------------------------------------------ */

__global__ void k_mpep_offsets(uint64_t *mp_off, const uint64_t *row_off, uint32_t num_rows,
                               const uint32_t *valid_scan, uint32_t num_spec)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < num_spec) mp_off[s] = row_off[min(valid_scan[s], num_rows)];
    else if (s == num_spec) mp_off[s] = row_off[num_rows];
}

extern "C" int hfx_mpep_offsets(hfx_ctx *ctx, uint64_t *d_mp_off, const uint32_t *d_pep_num_mpep,
                                uint32_t num_rows, const uint32_t *d_spec_num_valid_scan,
                                uint32_t num_spec, void *stream)
{
    HFX_REQUIRE(ctx && d_mp_off && d_spec_num_valid_scan, HFX_ERR_ARG,
                "hfx_mpep_offsets: null argument");
    void *p;
    int rc;
    if ((rc = hfx_ctx_scratch(ctx, HFX_SLOT_MODS2, ((size_t)num_rows + 1) * 8, &p)) != HFX_OK)
        return rc;
    uint64_t *row_off = (uint64_t *)p;
    if ((rc = hfx_scan_offsets(ctx, row_off, d_pep_num_mpep, num_rows, stream)) != HFX_OK) return rc;
    hipLaunchKernelGGL(k_mpep_offsets, dim3((num_spec + 256) / 256), dim3(256), 0,
                       hfx_stream(stream), d_mp_off, row_off, num_rows, d_spec_num_valid_scan,
                       num_spec);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}
