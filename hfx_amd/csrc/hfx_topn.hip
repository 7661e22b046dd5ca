/*
 * hfx_topn.hip -- per-spectrum top-N with an exact re-score.
 *
 * The reference sorts every score of a spectrum with a b40c radix sort and
 * copies them all to the host (Search.hs:250-276, sort_b40c.cu:34-41); the
 * final order is descending score, ties by ascending candidate position
 * (stable ascending sort, then reverse twice: Search.hs:119-123, :276).
 *
 * Here, in three launches:
 *   1. k_topn_select, one workgroup per spectrum: the T = min(N + margin, n)
 *      best FP32 scores (key desc, position asc), and every other candidate
 *      whose FP32 score is >= fN - 2B, fN being the N-th best FP32 score (B
 *      bounds |FP32 - exact|): the N-th best exact score exN is >= fN - B, so no
 *      candidate left out can reach the top N;
 *   2. k_topn_exact, one wave per spectrum (long lists shared out among all
 *      waves): the exact scores of those candidates, several a wave: int64
 *      fixed point, sum of round(w*x*2^36), independent of summation order, so
 *      the GPU and the CPU oracle agree bit for bit;
 *   3. k_topn_rank, one wave per spectrum: the re-scored candidates by (exact
 *      desc, position asc), the best N written.
 * If the band holds more than TN_EXT candidates, the spectrum is flagged and
 * the exact route scores every candidate at or above exN - B exactly.
 * Bound: |score - exact| <= (rel0 + rel1 * z) * 50 * sum_b |x_b|
 *                           + relq * max_b |x_b| * 50 * len + 1e-6, with
 * z the spectrum's fragment charge count and sum|w*x| <= 50 * sum_b |x_b|
 * (each bin counts once, weights <= 50).  The sparse FP32 scores use
 * rel0 = 80 * 2^-24 (<= 71 roundings per score), rel1 = 0; the dense BF16
 * scores pass their own (split error + one rounding per non-zero bin).
 *
 * One workgroup per spectrum for all three, a wave per candidate, spends half of
 * its time on exact scores with a quarter of the lanes busy, and a spectrum
 * with 200 tied candidates holds up a small batch by itself.
 * Select + exact + rank: 10,000 spectra, 1120 candidates each, top 10: 128 + 125 +
 * 15 us, 445 in one kernel; 20,000 spectra, top 5: 159 + 135 + 15 us and 430 (179
 * where the selection reads the spectra for their norms); 250 spectra: 13 + 21 + 7
 * us and 171.  The selection is a chain of short steps (63 % of the waves' cycles
 * are waits, 55 % of the vector issue is used); the exact scores are bound by their
 * FP64 terms and the maps' LDS atomics.
 */
#define HFX_TOPN_REL_F32 (80.0f * 5.9604644775390625e-08f)
#include "hfx_pack.h"

#define TN_THREADS 256
#define TN_WAVES (TN_THREADS / HFX_WAVE)
#define TN_MAXT 128
#define TN_EXT 256
#define TN_MAXC (TN_MAXT + TN_EXT)

/* T at most this: a threshold from the lanes' largest scores, then one
 * collection; above, a radix select.  Whole top-N by the first and by radix: 250
 * spectra, N = 5: 46 and 56 us, 32: 124 and 146, 48: 152 and 162, 64: 169 and
 * 165; 2,000 spectra, 5: 168 and 184, 32: 325 and 333, 48: 381 and 378, 64: 433
 * and 423. */
#define TN_LT 32
/* scores a thread keeps in registers between its two looks at them: windows of
 * up to 6144 candidates are read once */
#define TN_HOLD 24

/* the first select pass histograms the key's 11 high bits */
#define TN_HBITS 11
#define TN_HBINS (1u << TN_HBITS)

/* candidates of a spectrum that its own wave re-scores; the rest of a longer
 * list goes out in tasks of as many, first to the waves without a spectrum (4
 * workgroups a CU at least).  Up to TN_FEW spectra half as many.  With eight and
 * with sixteen, whole top-N: 250 spectra, N = 16: 58 and 79 us; 2,000, N = 16:
 * 234 and 250, N = 64: 359 and 397, N = 5: 168 and 167; a plain search of 10,000,
 * N = 10: 2170 and 2088; a BF16 batch of 6,000: 1150 and 1105. */
#define TN_TASK 16
#define TN_TASK_FEW 8
#define TN_FEW 4096
#define TN_SPILL ((TN_MAXC - 1) / TN_TASK_FEW)

__device__ __forceinline__ bool before_fx(int64_t fa, uint32_t pa, int64_t fb, uint32_t pb)
{
    return fa > fb || (fa == fb && pa < pb);
}

/* One radix-select step on an nb-bucket histogram: the digit holding the
 * rem-th largest element (counting from bucket nb - 1 down) and the rank
 * left inside it.  Wave 0 does it: lane l sums its run of nb / 64 buckets
 * (one at least), an inclusive scan over the lanes finds the run that holds
 * rank rem, and that lane walks it.  Every thread must call it (it ends with
 * a barrier); all get the same (digit, rem). */
__device__ __forceinline__ void tn_select_digit(const uint32_t *hist, uint32_t nb,
                                                uint32_t *sh_digit, uint32_t *sh_rem)
{
    const uint32_t tid = threadIdx.x, lane = hfx_lane();
    if (tid < HFX_WAVE) {
        const uint32_t rem = *sh_rem;
        const uint32_t per = (nb + HFX_WAVE - 1) / HFX_WAVE;
        const int top = (int)nb - 1 - (int)(lane * per);
        uint32_t sum = 0;
        for (uint32_t k = 0; k < per; ++k)
            if (top - (int)k >= 0) sum += hist[top - (int)k];
        uint32_t incl = sum;
#pragma unroll
        for (uint32_t o = 1; o < HFX_WAVE; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        const uint32_t excl = incl - sum;
        if (excl < rem && rem <= incl) {
            uint32_t cum = excl;
            for (uint32_t k = 0; k < per && top - (int)k >= 0; ++k) {
                const uint32_t h = hist[top - (int)k];
                if (cum + h >= rem) {
                    *sh_digit = (uint32_t)(top - (int)k);
                    *sh_rem = rem - cum;
                    break;
                }
                cum += h;
            }
        }
    }
    __syncthreads();
}

/* The `want` first of a wave's candidates in order of (key desc, position asc):
 * R a lane, key 0 for none.  want rounds of a wave-wide best; emit(r, key, pos)
 * in every lane.  A few rounds where counting every candidate's place compares
 * them all: 25 us for 261 of them. */
template <int R, class Emit>
__device__ __forceinline__ void tn_wave_top(uint64_t (&k)[R], uint32_t (&p)[R], uint32_t want,
                                            Emit &&emit)
{
    for (uint32_t r = 0; r < want; ++r) {
        uint64_t bk = k[0];
        uint32_t bp = p[0];
#pragma unroll
        for (int i = 1; i < R; ++i) {
            const bool c = k[i] > bk || (k[i] == bk && p[i] < bp);
            bk = c ? k[i] : bk;
            bp = c ? p[i] : bp;
        }
#pragma unroll
        for (uint32_t o = 1; o < HFX_WAVE; o <<= 1) {
            const uint64_t ok = (uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(bk >> 32), o, 64) << 32 |
                                (uint32_t)__shfl_xor((int)(uint32_t)bk, o, 64);
            const uint32_t op = (uint32_t)__shfl_xor((int)bp, o, 64);
            const bool c = ok > bk || (ok == bk && op < bp);
            bk = c ? ok : bk;
            bp = c ? op : bp;
        }
        emit(r, bk, bp);
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (k[i] == bk && p[i] == bp) {
                k[i] = 0;
                p[i] = 0xffffffffu;
            }
    }
}

/* Histogram increment of digit d for the active lanes of a wave: lanes that
 * share the first pending lane's digit add their count with one atomic (a
 * few rounds: score keys crowd into few high-byte buckets), the rest add one
 * each. */
__device__ __forceinline__ void tn_hist_add(uint32_t *hist, uint32_t d, bool act)
{
    const uint32_t lane = hfx_lane();
    uint64_t m = __ballot(act);
    for (int it = 0; it < 4 && m; ++it) {
        const uint32_t leader = (uint32_t)__builtin_ctzll(m);
        const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)d, (int)leader);
        const uint64_t same = __ballot(((m >> lane) & 1ull) && d == v);
        if (lane == leader) atomicAdd(&hist[v], (uint32_t)__builtin_popcountll(same));
        m &= ~same;
    }
    if ((m >> lane) & 1ull) atomicAdd(&hist[d], 1u);
}

#define TN_BIG 0x80000000u /* in mcnt: terms may pass 2^50 */
/* sixteen bytes at any multiple of four */
typedef float tn_f4 __attribute__((ext_vector_type(4), aligned(4)));

/* exact-route and candidate scratch of a call, see tx_carve */
struct TnLists {
    uint32_t *cand;  /* [S][TN_MAXC] positions: the T selected, then the band */
    uint32_t *mcnt;  /* [S] their number, and TN_BIG */
    uint2 *spill;    /* [S * TN_SPILL] (spectrum, first candidate) */
    uint32_t *nspill;
    double *tau;     /* [S] the bound, then the exact route's threshold */
    uint32_t *band;  /* [S] band size of flagged spectra */
    uint32_t task;   /* candidates a task */
};

template <class Cands>
__global__ void __launch_bounds__(TN_THREADS)
    k_topn_select(TnLists o, uint32_t *flag, uint32_t N, uint32_t margin, const float *scores,
                  Cands c, hfx_spectra sp, float rel0, float rel1, float relq, const float2 *norms)
{
    __shared__ uint32_t hist[TN_HBINS];
    __shared__ uint64_t kv[TN_MAXC]; /* (key, ~position) */
    __shared__ uint32_t cp[TN_MAXC];
    __shared__ uint32_t wcnt[TN_WAVES], sh_low[TN_WAVES];
    __shared__ float sh_x1[TN_WAVES], sh_xm[TN_WAVES];
    __shared__ uint32_t sh_digit, sh_rem, sh_gt, sh_last, sh_ext, sh_cnt, sh_task;
    __shared__ float sh_fN;

    const uint32_t s = blockIdx.x, tid = threadIdx.x, wave = tid / HFX_WAVE;
    const uint32_t lane = hfx_lane();
    const uint32_t n = c.count(s);
    const float *sc = scores + c.base(s);
    if (n == 0) {
        if (tid == 0) {
            o.mcnt[s] = 0;
            flag[s] = 0;
        }
        return;
    }
    const uint32_t T = min(N + margin, n);

    /* every sweep over memory visits this thread's keys through for_keys(f),
     * f(i, key), eight loads in flight at a time (clamped into the window, so
     * that none is conditional); i >= n past the window, where all lanes of a
     * wave still take part (for the ballots) */
    auto for_keys = [&](auto &&f) {
        constexpr uint32_t U = 8;
        for (uint32_t base = 0; base < n; base += U * TN_THREADS) {
            uint32_t kk[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u)
                kk[u] = hfx_f2key(sc[min(base + u * TN_THREADS + tid, n - 1u)]);
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) f(base + u * TN_THREADS + tid, kk[u]);
        }
    };
    if (tid == 0) {
        sh_rem = T;
        sh_gt = 0;
        sh_ext = 0;
        sh_last = 0;
        sh_cnt = 0;
    }

    /* 1. the scores, once, four at a time, and the largest of each thread;
     * sum|x| and max|x|, where the caller does not have them (norms) */
    const bool held = n <= TN_HOLD * TN_THREADS;
    const uint32_t len = min(sp.d_len[s], min(sp.x_stride, (uint32_t)HFX_MAX_LEN));
    const float *xg = sp.d_x + (size_t)s * sp.x_stride;
    tn_f4 v4[TN_HOLD / 4];
    uint32_t km = 0;
    if (held) {
        /* thread t's scores are 1024 u + 4 t + e; absent ones are NaN, which
         * the largest skips */
#pragma unroll
        for (uint32_t u = 0; u < TN_HOLD / 4; ++u) {
            v4[u] = tn_f4{NAN, NAN, NAN, NAN};
            const uint32_t i = u * 4 * TN_THREADS + 4 * tid;
            if (i + 4 <= n) v4[u] = *(const tn_f4 *)(sc + i);
            else if (i < n)
#pragma unroll
                for (uint32_t e = 0; e < 3; ++e)
                    if (i + e < n) v4[u][e] = sc[i + e];
        }
    }
    float x1 = 0.0f, xm = 0.0f;
    for (uint32_t base = 0; !norms && base < len; base += 8 * TN_THREADS) {
        float v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) v[u] = xg[min(base + u * TN_THREADS + tid, len - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            if (base + u * TN_THREADS + tid < len) {
                x1 += fabsf(v[u]);
                xm = fmaxf(xm, fabsf(v[u]));
            }
    }
    /* a score that is NaN orders by its bits, as the radix select has it */
    bool nan = false;
    if (held) {
        float m = -INFINITY;
        uint32_t cnt = 0;
#pragma unroll
        for (uint32_t u = 0; u < TN_HOLD / 4; ++u)
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                m = fmaxf(m, v4[u][e]);
                cnt += v4[u][e] == v4[u][e] ? 1u : 0u;
            }
        /* this thread's scores: 4 for every whole step, the rest in the last */
        const uint32_t step = 4 * TN_THREADS, whole = n / step, rest = n % step;
        const uint32_t mine = whole * 4 + min(4u, rest > 4 * tid ? rest - 4 * tid : 0u);
        nan = cnt != mine;
        km = mine ? hfx_f2key(m) : 0u;
    } else {
        for_keys([&](uint32_t i, uint32_t k) { km = max(km, i < n ? k : 0u); });
    }
    x1 = hfx_wave_sum_f32(x1);
    for (uint32_t q = 32; q > 0; q >>= 1) xm = fmaxf(xm, __shfl_xor(xm, q, 64));
    /* a key that at least T of the wave's keys reach: the T-th largest of the
     * lanes' largest, bit by bit (0 if fewer lanes have any); the low twelve
     * bits left out, which takes a few more scores into the list */
    uint32_t low = 0;
    if (T <= TN_LT)
        for (int b = 31; b >= 12; --b) {
            const uint32_t t = low | 1u << b;
            if ((uint32_t)__builtin_popcountll(__ballot(km >= t)) >= T) low = t;
        }
    const uint64_t anynan = __ballot(nan);
    if (lane == 0) {
        sh_x1[wave] = x1;
        sh_xm[wave] = xm;
        sh_low[wave] = low;
        wcnt[wave] = anynan != 0;
    }
    __syncthreads();
    const bool direct = T <= TN_LT && !(wcnt[0] | wcnt[1] | wcnt[2] | wcnt[3]);
    static_assert(TN_WAVES == 4, "every wave's mark");
    const uint32_t zeff = c.zeff(sp.d_zmax[s]);
    float xa = 0.0f, xmax = 0.0f;
    for (uint32_t w = 0; w < TN_WAVES; ++w) {
        xa += sh_x1[w];
        xmax = fmaxf(xmax, sh_xm[w]);
        low = max(low, sh_low[w]);
    }
    if (norms) {
        xa = norms[s].x;
        xmax = norms[s].y;
    }
    const double rel = (double)rel0 + (double)rel1 * (double)zeff;
    const double bound = rel * 50.0 * (double)xa * 1.001 +
                         (double)relq * (double)xmax * 50.0 * (double)len * 1.001 + 1e-6;
    /* scores below it can be neither selected nor in the band when the N-th
     * best is f or more (a relative 1e-12 margin covers the double roundings) */
    auto reach = [&](float f) {
        const double d = (double)f;
        return d - 2.0 * bound - 1e-12 * (fabs(d) + 2.0 * bound);
    };

    /* 2. T <= TN_LT: fN >= low, so every key at or above reach(low) holds the
     * selection and the band.  They are ranked exactly; the band is taken from
     * them once fN is known.  Should they pass TN_MAXC (long runs of
     * near-equal scores), the radix select below takes over. */
    uint32_t ne = 0, fl = 0;
    bool done = false;
    if (direct) {
        uint32_t kthr = low;
        if (low) {
            const double thr = reach(hfx_key2f(low));
            if (thr == thr) {
                /* the smallest key whose value is >= thr (-0 and +0 are equal
                 * values, but not keys) */
                const float tf = (float)thr;
                uint32_t kt = hfx_f2key(tf) + ((double)tf < thr ? 1u : 0u);
                if (tf == 0.0f && !((double)tf < thr)) kt = 0x7fffffffu;
                kthr = min(kt, low);
            }
        }
        auto collect = [&](uint32_t i, uint32_t k, bool f) {
            const uint64_t bal = __ballot(f);
            if (bal) {
                const uint32_t lead = (uint32_t)__builtin_ctzll(bal);
                uint32_t at = 0;
                if (lane == lead) at = atomicAdd(&sh_cnt, (uint32_t)__builtin_popcountll(bal));
                at = hfx_take(at, lead) +
                     (uint32_t)__builtin_popcountll(bal & ((1ull << lane) - 1ull));
                if (f && at < TN_MAXC) kv[at] = (uint64_t)k << 32 | (0xffffffffu - i);
            }
        };
        if (held) {
            /* the threshold as a value: no NaN here, and -0 is taken with +0 */
            const float fthr = kthr <= hfx_f2key(-INFINITY) ? -INFINITY : hfx_key2f(kthr);
#pragma unroll
            for (uint32_t u = 0; u < TN_HOLD / 4; ++u)
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e)
                    if (__ballot(v4[u][e] >= fthr))
                        collect(u * 4 * TN_THREADS + 4 * tid + e,
                                v4[u][e] >= fthr ? hfx_f2key(v4[u][e]) : 0u, v4[u][e] >= fthr);
        } else {
            for_keys([&](uint32_t i, uint32_t k) { collect(i, k, i < n && k >= kthr); });
        }
        __syncthreads();
        const uint32_t M0 = sh_cnt;
        done = M0 <= TN_MAXC;
        if (done) {
            uint32_t rk[(TN_MAXC + TN_THREADS - 1) / TN_THREADS];
#pragma unroll
            for (uint32_t q = 0; q < (TN_MAXC + TN_THREADS - 1) / TN_THREADS; ++q) {
                const uint32_t a = q * TN_THREADS + tid;
                rk[q] = 0xffffffffu;
                if (a < M0) {
                    const uint64_t v = kv[a];
                    uint32_t r = 0;
#pragma unroll 8
                    for (uint32_t b = 0; b < M0; ++b) r += kv[b] > v ? 1u : 0u;
                    rk[q] = r;
                    if (r < T) cp[r] = 0xffffffffu - (uint32_t)v;
                    if (r == N - 1u) sh_fN = hfx_key2f((uint32_t)(v >> 32));
                }
            }
            __syncthreads();
            if (n > T) {
                const double tau2 = reach(sh_fN);
#pragma unroll
                for (uint32_t q = 0; q < (TN_MAXC + TN_THREADS - 1) / TN_THREADS; ++q) {
                    const uint32_t a = q * TN_THREADS + tid;
                    if (a < M0 && rk[q] >= T &&
                        (double)hfx_key2f((uint32_t)(kv[a] >> 32)) >= tau2) {
                        const uint32_t slot = atomicAdd(&sh_ext, 1u);
                        if (slot < TN_EXT) cp[T + slot] = 0xffffffffu - (uint32_t)kv[a];
                    }
                }
                __syncthreads();
                ne = sh_ext;
            }
        }
    }
    if (!done) {
        /* Radix select, first over the key's 11 high bits (sign, exponent, two
         * mantissa bits: a quarter octave a bucket), then 8, 8 and 5 bits; after
         * each pass, once the keys at or above the prefix found so far -- M of
         * them, known from the histograms -- number at most TN_MAXC, they are
         * collected and ranked exactly.  Otherwise (long runs of near-equal
         * scores) the full threshold key K is found and the keys above it, then
         * the smallest positions equal to it, are collected. */
        uint32_t prefix = 0, pmask = 0;
        bool ranked = false;
        for (int pass = 0; pass < 4; ++pass) {
            const uint32_t shift = pass == 0 ? 32u - TN_HBITS : pass == 1 ? 13u : pass == 2 ? 5u : 0u;
            const uint32_t nb = pass == 0 ? TN_HBINS : pass == 3 ? 32u : 256u;
            for (uint32_t b = tid; b < nb; b += TN_THREADS) hist[b] = 0;
            __syncthreads();
            for_keys([&](uint32_t i, uint32_t k) {
                tn_hist_add(hist, (k >> shift) & (nb - 1u), i < n && (k & pmask) == prefix);
            });
            __syncthreads();
            tn_select_digit(hist, nb, &sh_digit, &sh_rem);
            prefix |= sh_digit << shift;
            pmask |= (nb - 1u) << shift;
            const uint32_t M = T - sh_rem + hist[sh_digit];
            __syncthreads(); /* every thread has read hist before it is cleared */
            if (M <= TN_MAXC) {
                for_keys([&](uint32_t i, uint32_t k) {
                    if (i < n && (k & pmask) >= prefix)
                        kv[atomicAdd(&sh_gt, 1u)] = (uint64_t)k << 32 | (0xffffffffu - i);
                });
                __syncthreads();
                for (uint32_t a = tid; a < M; a += TN_THREADS) {
                    const uint64_t va = kv[a];
                    uint32_t rk = 0;
                    for (uint32_t b = 0; b < M; ++b) rk += kv[b] > va ? 1u : 0u;
                    const uint32_t pa = 0xffffffffu - (uint32_t)va;
                    if (rk < T) cp[rk] = pa;
                    if (rk == T - 1u) {
                        sh_digit = (uint32_t)(va >> 32);
                        sh_last = pa;
                    }
                }
                __syncthreads();
                ranked = true;
                break;
            }
        }
        const uint32_t K = ranked ? sh_digit : prefix;
        if (!ranked) {
            const uint32_t need_eq = sh_rem; /* >= 1 */
            const uint32_t n_gt = T - need_eq;
            for_keys([&](uint32_t i, uint32_t k) {
                if (i < n && k > K) {
                    const uint32_t slot = atomicAdd(&sh_gt, 1u);
                    if (slot < n_gt) cp[slot] = i;
                }
            });
            /* keys equal to the threshold: the need_eq smallest positions */
            uint32_t eq_base = 0;
            for (uint32_t base = 0; base < n && eq_base < need_eq; base += TN_THREADS) {
                const uint32_t i = base + tid;
                const bool f = i < n && hfx_f2key(sc[i]) == K;
                const uint64_t bal = __ballot(f);
                const uint32_t wr = (uint32_t)__builtin_popcountll(bal & ((1ull << lane) - 1ull));
                if (lane == 0) wcnt[wave] = (uint32_t)__builtin_popcountll(bal);
                __syncthreads();
                uint32_t wpre = 0, tot = 0;
                for (uint32_t w = 0; w < TN_WAVES; ++w) {
                    if (w < wave) wpre += wcnt[w];
                    tot += wcnt[w];
                }
                const uint32_t r = eq_base + wpre + wr;
                if (f && r < need_eq) {
                    cp[n_gt + r] = i;
                    if (r == need_eq - 1) sh_last = i;
                }
                eq_base += tot;
                __syncthreads();
            }
        }
        __syncthreads();
        if (n > T) {
            /* the N-th best of the selection, then the band */
            for (uint32_t i = tid; i < T; i += TN_THREADS) {
                const uint32_t pi = cp[i], ki = hfx_f2key(sc[pi]);
                kv[i] = (uint64_t)ki << 32 | (0xffffffffu - pi);
            }
            __syncthreads();
            for (uint32_t i = tid; i < T; i += TN_THREADS) {
                uint32_t rk = 0;
                for (uint32_t j = 0; j < T; ++j) rk += kv[j] > kv[i] ? 1u : 0u;
                if (rk == N - 1) sh_fN = hfx_key2f((uint32_t)(kv[i] >> 32));
            }
            __syncthreads();
            const double tau2 = reach(sh_fN);
            const uint32_t last = sh_last;
            for_keys([&](uint32_t i, uint32_t k) {
                const bool selected = k > K || (k == K && i <= last);
                if (i < n && !selected && (double)hfx_key2f(k) >= tau2) {
                    const uint32_t slot = atomicAdd(&sh_ext, 1u);
                    if (slot < TN_EXT) cp[T + slot] = i;
                }
            });
            __syncthreads();
            ne = sh_ext;
        }
    }

    /* 3. the list.  More than TN_EXT in the band: the spectrum is flagged, the
     * selection alone is re-scored, and the exact route takes every candidate at
     * or above exN - B. */
    if (ne > TN_EXT) {
        fl = 1;
        if (tid == 0) o.band[s] = ne; /* sizes the exact route's tiles */
        ne = 0;
    }
    const uint32_t M = T + ne;
    /* spectra whose terms 50 |x| 2^36 stay below 2^50 take the short rounding
     * (fmaxf skips a NaN, the sum keeps it) */
    const uint32_t big = xmax < 300.0f && xa == xa ? 0u : TN_BIG;
    for (uint32_t i = tid; i < M; i += TN_THREADS) o.cand[(size_t)s * TN_MAXC + i] = cp[i];
    const uint32_t ntask = M > o.task ? (M - 1u) / o.task : 0u;
    if (tid == 0) {
        o.mcnt[s] = M | big;
        flag[s] = fl;
        o.tau[s] = bound;
        sh_task = ntask ? atomicAdd(o.nspill, ntask) : 0u;
    }
    if (ntask) {
        __syncthreads();
        if (tid < ntask) o.spill[sh_task + tid] = make_uint2(s, (tid + 1u) * o.task);
    }
}

/* ------------------------------------------------------------------ */
/* Exact scores, several candidates a wave                               */
/* ------------------------------------------------------------------ */

/* LDS of a wave: XP_SLOTS maps (cleared), the ladder buffer, the pack's sums */
struct FxWave {
    uint32_t *maps;
    float *lb;
    unsigned long long *acc;
};
static size_t fx_lds_bytes(uint32_t xstr)
{
    return (size_t)TN_WAVES * (XP_SLOTS * xp_map_words(xstr) + XP_LB) * 4 + TN_WAVES * XP_SLOTS * 8;
}
__device__ __forceinline__ FxWave fx_wave(unsigned char *lds, uint32_t mstr, uint32_t wave)
{
    unsigned long long *acc = (unsigned long long *)lds;
    uint32_t *maps = (uint32_t *)(acc + TN_WAVES * XP_SLOTS);
    float *lb = (float *)(maps + TN_WAVES * XP_SLOTS * mstr);
    const FxWave f{maps + wave * XP_SLOTS * mstr, lb + wave * XP_LB, acc + wave * XP_SLOTS};
    for (uint32_t i = hfx_lane(); i < XP_SLOTS * mstr; i += HFX_WAVE) f.maps[i] = 0u;
    return f;
}

/* one pack at fragment charges 1..Z: the exact sum of each candidate into its
 * accumulator.  The spectrum is read where it lies (a row is a few KiB, in L2
 * after the first pack); its values come before the claims, whose codes decide
 * what is added; bins outside [0, len) add nothing. */
template <int Z, bool BIG>
__device__ __forceinline__ void fx_pack(const FxWave &f, uint32_t mstr, const float *x, uint32_t len,
                                        const XpPack pk)
{
    const uint32_t lane = hfx_lane();
    const XpLane ln = xp_lane(pk, lane);
    if (lane < XP_SLOTS) f.acc[lane] = 0ull;
    const float b = ln.act ? f.lb[ln.lad + ln.kpos] : 0.0f;
    const float y = ln.r - b;
    uint32_t *rowm = f.maps + ln.slot * mstr + XP_PAD / 8 - (XP_MAGIC_BITS >> 3);
    const uint32_t spr = (lane & (XP_SPREAD - 1)) * 8u;
    const XpClamp cl{XP_MAGIC_BITS - 1u - spr, XP_MAGIC_BITS + len + spr,
                     XP_MAGIC_BITS - 2u - spr, XP_MAGIC_BITS + len + 1u + spr};
    auto put = [&](auto zc) {
        uint32_t u[6];
        XpPeaks p;
        xp_bins<decltype(zc)::value>(b, y, cl, u);
        xp_locate(rowm, u, p);
        xp_put(p);
    };
    if (ln.act) {
        put(std::integral_constant<int, 1>{});
        if constexpr (Z >= 2) put(std::integral_constant<int, 2>{});
        if constexpr (Z >= 3) put(std::integral_constant<int, 3>{});
        if constexpr (Z >= 4) put(std::integral_constant<int, 4>{});
    }
    hfx_wave_sync();
    if (ln.act) {
        uint64_t sum = 0; /* modulo 2^64 */
        /* rint(w x 2^36): adding 1.5 * 2^16 rounds w x, below 2^15, to a multiple
         * of 2^-36, ties to even, and leaves the integer in the low bits, the
         * constant's bits taken off the sum once for all terms.  Fused, so
         * rounded once: three instructions fewer a term, 137.7 -> 135.6 us for 20,000
         * spectra (the LDS atomics bound it). */
        constexpr double MAGIC = 98304.0;
        auto term = [&](uint32_t nib, uint32_t bin, float xv) {
            /* selector bytes 1..3 are zero and pick zeros */
            const uint32_t w = bin < len ? __builtin_amdgcn_perm(0x32000000u, 0x19000A00u, nib & 15u)
                                         : 0u;
            if constexpr (BIG) {
                sum += (uint64_t)hfx_fx_term((float)w, xv);
            } else {
                const double t = __builtin_fma((double)w, (double)xv, MAGIC);
                sum += (uint64_t)__double_as_longlong(t);
            }
        };
        /* the bins again, not kept from the first pass: eight waves a SIMD
         * would not hold them for four charges */
        auto claim = [&](auto zc) {
            float b2 = b;
            asm volatile("" : "+v"(b2));
            uint32_t u[6];
            XpPeaks p;
            xp_bins<decltype(zc)::value>(b2, y, cl, u);
            xp_locate(rowm, u, p);
            float xv[6][3];
#pragma unroll
            for (int i = 0; i < 6; ++i)
#pragma unroll
                for (int q = 0; q < (i == 1 || i == 4 ? 3 : 1); ++q)
                    xv[i][q] = x[min(p.u[i] - XP_MAGIC_BITS + q, len - 1u)];
#pragma unroll
            for (int i = 0; i < 6; ++i) {
                const uint32_t bin = p.u[i] - XP_MAGIC_BITS, sh = p.sh[i];
                if (i == 1 || i == 4) {
                    const uint64_t t = (uint64_t)0xfffu << sh;
                    const uint32_t o0 = atomicAnd(p.w[i], ~(uint32_t)t);
                    const uint32_t o1 = atomicAnd(p.w[i] + 1, ~(uint32_t)(t >> 32));
                    const uint32_t g = (uint32_t)(((uint64_t)o1 << 32 | o0) >> sh);
                    term(g, bin, xv[i][0]);
                    term(g >> 4, bin + 1u, xv[i][1]);
                    term(g >> 8, bin + 2u, xv[i][2]);
                } else {
                    term(atomicAnd(p.w[i], ~(0xfu << sh)) >> sh, bin, xv[i][0]);
                }
            }
        };
        claim(std::integral_constant<int, 1>{});
        if constexpr (Z >= 2) claim(std::integral_constant<int, 2>{});
        if constexpr (Z >= 3) claim(std::integral_constant<int, 3>{});
        if constexpr (Z >= 4) claim(std::integral_constant<int, 4>{});
        if constexpr (!BIG) sum -= 10ull * Z * (uint64_t)__double_as_longlong(MAGIC);
        atomicAdd(&f.acc[ln.slot], (unsigned long long)sum);
    }
    hfx_wave_sync();
}

/* the exact scores of rn <= 64 candidates of one spectrum, candidate i's
 * metadata in lane i: emit(i, score) once each, by one lane.  BIG: terms may
 * pass 2^50. */
template <bool BIG, class Cands, class Emit>
__device__ __forceinline__ void fx_scores(const FxWave &f, uint32_t mstr, const float *mtab,
                                          const float *x, uint32_t len, uint32_t zeff,
                                          const Cands &c, const typename Cands::Prep &pr,
                                          uint32_t rn, Emit &&emit)
{
    const uint32_t lane = hfx_lane();
    if (zeff == 0 || len == 0) {
        /* no fragment charge generated, or no bins */
        if (lane < rn) emit(lane, (int64_t)0);
        return;
    }
    const bool general = zeff > 4;
    const uint32_t nl = lane < rn && pr.n <= HFX_WAVE && !general ? pr.n : 0u;
    const uint32_t incl = xp_prefix(nl, lane), pofs = incl - nl;
    for (uint32_t p = 0; p < rn;) {
        const uint32_t base = hfx_take(pofs, p);
        const uint64_t fit = __ballot(lane >= p && lane < rn && incl - base <= XP_LB);
        const uint32_t q = p + (uint32_t)__builtin_popcountll(fit);
        if (lane >= p && lane < q && nl) c.ladder(pr, mtab, f.lb + (pofs - base), nl);
        hfx_wave_sync();
        while (p < q) {
            if (hfx_take(pr.n, p) > HFX_WAVE || general) {
                c.peaks_prep(f.maps + XP_PAD / 8, mtab, Cands::take(pr, p), len, zeff);
                hfx_wave_sync();
                const int64_t v = hfx_wave_dot_fx(f.maps + XP_PAD / 8, x, len);
                hfx_wave_sync();
                if (lane == 0) emit(p, v);
                ++p;
                continue;
            }
            const XpPack pk = xp_form(p, q, pr.n, pr.r, pofs, base);
            switch (zeff) {
            case 1: fx_pack<1, BIG>(f, mstr, x, len, pk); break;
            case 2: fx_pack<2, BIG>(f, mstr, x, len, pk); break;
            case 3: fx_pack<3, BIG>(f, mstr, x, len, pk); break;
            default: fx_pack<4, BIG>(f, mstr, x, len, pk); break;
            }
            if (lane < pk.K) emit(p + lane, (int64_t)f.acc[lane]);
            hfx_wave_sync(); /* the accumulators are cleared by the next pack */
            p += pk.K;
        }
        hfx_wave_sync(); /* the buffer is rewritten by the next chunk */
    }
}

/* exact scores of the listed candidates: wave w takes the first o.task of
 * spectrum w, then all waves share the spilled tasks.  fx: [s][TN_MAXC]. */
template <class Cands>
__global__ void __launch_bounds__(TN_THREADS)
    k_topn_exact(int64_t *fx, TnLists o, Cands c, hfx_spectra sp, uint32_t mstr)
{
    extern __shared__ __align__(16) unsigned char tn_dyn[];
    __shared__ float mtab[HFX_MTAB];
    const uint32_t wave = threadIdx.x / HFX_WAVE, lane = hfx_lane(), S = sp.num_spec;
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? c.db.d_mass[threadIdx.x] : 0.0f;
    c.stage(mtab);
    const FxWave f = fx_wave(tn_dyn, mstr, wave);
    __syncthreads();
    auto task = [&](uint32_t s, uint32_t k0) {
        const uint32_t mc = __builtin_amdgcn_readfirstlane(o.mcnt[s]), M = mc & ~TN_BIG;
        const uint32_t rn = M > k0 ? min(M - k0, o.task) : 0u;
        if (rn == 0) return;
        typename Cands::Prep pr{};
        if (lane < rn) pr = c.prep(s, o.cand[(size_t)s * TN_MAXC + k0 + lane]);
        const uint32_t len = min(sp.d_len[s], min(sp.x_stride, (uint32_t)HFX_MAX_LEN));
        int64_t *out = fx + (size_t)s * TN_MAXC + k0;
        const float *x = sp.d_x + (size_t)s * sp.x_stride;
        const uint32_t zeff = c.zeff(sp.d_zmax[s]);
        auto emit = [&](uint32_t i, int64_t v) { out[i] = v; };
        if (mc & TN_BIG) fx_scores<true>(f, mstr, mtab, x, len, zeff, c, pr, rn, emit);
        else fx_scores<false>(f, mstr, mtab, x, len, zeff, c, pr, rn, emit);
    };
    const uint32_t w = __builtin_amdgcn_readfirstlane(blockIdx.x * TN_WAVES + wave);
    if (w < S) task(w, 0);
    /* the waves without a spectrum first */
    const uint32_t ns = *o.nspill, W = gridDim.x * TN_WAVES;
    for (uint32_t i = w < S ? w + (W - S) : w - S; i < ns; i += W) {
        const uint2 t = o.spill[i];
        task(__builtin_amdgcn_readfirstlane(t.x), __builtin_amdgcn_readfirstlane(t.y));
    }
}

#define TX_CHUNK 256
/* a flagged spectrum's tiles also number at least its band count / TX_LIVE,
 * so that the candidates the exact route re-scores spread over the tiles */
#define TX_LIVE 32

/* the exact route's work: the flagged spectra (in any order), their number, the
 * first tile of each (off[number] = all tiles), and the place of each one's exact
 * scores (a sum of window sizes, wherever the spectra's own scores lie) */
struct TxPlan {
    uint64_t *off, *at;
    uint32_t *list, *count;
};

/* by one workgroup: few spectra are flagged, so the tiles need no table per
 * spectrum */
template <class Cands>
__device__ void tx_plan(TxPlan p, const uint32_t *flag, const uint32_t *band, const Cands &c,
                        uint32_t S)
{
    __shared__ uint32_t nl;
    __shared__ uint64_t wt[TN_THREADS / HFX_WAVE], wa[TN_THREADS / HFX_WAVE];
    const uint32_t lane = hfx_lane(), wave = threadIdx.x / HFX_WAVE;
    if (threadIdx.x == 0) nl = 0;
    __syncthreads();
    for (uint32_t s0 = threadIdx.x; s0 < S; s0 += 8 * TN_THREADS) {
        uint32_t fv[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) fv[u] = flag[min(s0 + u * TN_THREADS, S - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            if (s0 + u * TN_THREADS < S && fv[u] != 0u)
                p.list[atomicAdd(&nl, 1u)] = s0 + u * TN_THREADS;
    }
    __syncthreads(); /* the list is this workgroup's own: visible to it from here */
    const uint32_t F = nl;
    uint64_t nt = 0, na = 0;
    for (uint32_t q0 = 0; q0 < F; q0 += TN_THREADS) {
        const uint32_t q = q0 + threadIdx.x;
        uint64_t t = 0, n = 0;
        if (q < F) {
            const uint32_t s = p.list[q], b = min(band[s], c.count(s));
            n = c.count(s);
            t = max((n + TX_CHUNK - 1) / TX_CHUNK, ((uint64_t)b + TX_LIVE - 1) / TX_LIVE);
        }
        uint64_t x = t, y = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint64_t v = __shfl_up(x, o, 64), u = __shfl_up(y, o, 64);
            if (lane >= (uint32_t)o) {
                x += v;
                y += u;
            }
        }
        if (lane == HFX_WAVE - 1) {
            wt[wave] = x;
            wa[wave] = y;
        }
        __syncthreads();
        uint64_t to = nt + x - t, at = na + y - n;
        for (uint32_t w = 0; w < TN_THREADS / HFX_WAVE; ++w) {
            if (w < wave) {
                to += wt[w];
                at += wa[w];
            }
            nt += wt[w];
            na += wa[w];
        }
        if (q < F) {
            p.off[q] = to;
            p.at[q] = at;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        p.off[F] = nt;
        *p.count = F;
    }
}

/* the lists in order of (exact desc, position asc): the best N, and for
 * flagged spectra exN - B as the exact route's threshold.  A wave a spectrum; the
 * first workgroup plans the exact route meanwhile, from what the selection left
 * (its own launch took 2 to 6 us, and the gap). */
template <class Cands>
__global__ void __launch_bounds__(TN_THREADS)
    k_topn_rank(uint32_t *top_pos, double *top_exact, float *top_f32, uint32_t *top_cnt,
                const uint32_t *flag, uint32_t N, const int64_t *fx, TnLists o, const float *scores,
                Cands c, uint32_t S, TxPlan plan)
{
    const uint32_t wave = threadIdx.x / HFX_WAVE, lane = hfx_lane();
    if (blockIdx.x == 0) {
        tx_plan(plan, flag, o.band, c, S);
        return;
    }
    const uint32_t s = (blockIdx.x - 1u) * TN_WAVES + wave;
    if (s >= S) return;
    const uint32_t M = o.mcnt[s] & ~TN_BIG, n = c.count(s), outn = min(N, n);
    const float *sc = scores + c.base(s);
    const bool fl = M && flag[s] != 0u;
    const int64_t *f = fx + (size_t)s * TN_MAXC;
    const uint32_t *p = o.cand + (size_t)s * TN_MAXC;
    auto put = [&](uint32_t rk, uint64_t k, uint32_t pos) {
        const double v = (double)(int64_t)(k ^ 0x8000000000000000ull) * (1.0 / HFX_FX_SCALE);
        top_pos[(size_t)s * N + rk] = pos;
        top_exact[(size_t)s * N + rk] = v;
        top_f32[(size_t)s * N + rk] = sc[pos];
        if (fl && rk == N - 1u) o.tau[s] = v - o.tau[s];
    };
    if (M <= HFX_WAVE) {
        /* each lane counts its candidate's place */
        uint64_t k = 0;
        uint32_t pos = 0xffffffffu;
        if (lane < M) {
            k = (uint64_t)f[lane] ^ 0x8000000000000000ull;
            pos = p[lane];
        }
        uint32_t rk = 0;
        for (uint32_t j = 0; j < M; ++j) {
            const uint64_t kj = (uint64_t)hfx_take((uint32_t)(k >> 32), j) << 32 |
                                hfx_take((uint32_t)k, j);
            const uint32_t pj = hfx_take(pos, j);
            rk += kj > k || (kj == k && pj < pos) ? 1u : 0u;
        }
        if (lane < M && rk < outn) put(rk, k, pos);
    } else {
        constexpr int R = TN_MAXC / HFX_WAVE;
        uint64_t k[R];
        uint32_t pos[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const uint32_t j = (uint32_t)i * HFX_WAVE + lane;
            k[i] = 0;
            pos[i] = 0xffffffffu;
            if (j < M) {
                k[i] = (uint64_t)f[j] ^ 0x8000000000000000ull;
                pos[i] = p[j];
            }
        }
        tn_wave_top<R>(k, pos, outn, [&](uint32_t rk, uint64_t kb, uint32_t pb) {
            if (lane == 0) put(rk, kb, pb);
        });
    }
    if (lane == 0) top_cnt[s] = outn;
}

/* ------------------------------------------------------------------ */
/* Exact route: every candidate of a flagged spectrum scored exactly     */
/* (tile-parallel, persistent), then a 64-bit radix select of the top N. */
/* Runs on the device after the re-score without a host round trip.      */
/* ------------------------------------------------------------------ */

#define TX_MAXN 64
/* a wave fetches the metadata of its share of a tile one lane per candidate */
static_assert(TX_CHUNK / TN_WAVES <= HFX_WAVE && TN_TASK <= HFX_WAVE,
              "one lane per candidate of a wave's share");

/* the list of the flagged spectra as a launch of its own, where the caller names
 * them */
template <class Cands>
__global__ void __launch_bounds__(TN_THREADS)
    k_tx_plan(TxPlan p, const uint32_t *flag, const uint32_t *band, Cands c, uint32_t S)
{
    tx_plan(p, flag, band, c, S);
}

__global__ void k_tx_reset(uint32_t *counter)
{
    counter[0] = 0;
    counter[1] = 0;
}

__global__ void k_zero_flags(uint32_t *flag, uint32_t S)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < S) flag[i] = 0;
}
__global__ void k_mark_list(uint32_t *flag, double *tau, uint32_t *band, const uint32_t *list,
                            uint32_t num_list, uint32_t S)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < num_list && list[i] < S) {
        flag[list[i]] = 1;
        tau[list[i]] = -INFINITY; /* every candidate scored exactly */
        band[list[i]] = 0xffffffffu;
    }
}

/* persistent: workgroup g takes tiles g, g + grid, ... of the flagged
 * spectra (about one each: no shared counter to queue on).  A spectrum's nt
 * tiles interleave its candidates (tile k takes k, k + nt, k + 2 nt, ...):
 * candidates near tau sit together in the window's order, and so are
 * spread over the tiles. */
template <class Cands>
__global__ void __launch_bounds__(TN_THREADS)
    k_exact_tiles(int64_t *fxbuf, const uint64_t *tile_off, const uint64_t *fx_at,
                  const uint32_t *list, const uint32_t *count, Cands c, hfx_spectra sp, const float *scores,
                  const double *tau, uint32_t mstr)
{
    extern __shared__ __align__(16) unsigned char tn_dyn[];
    __shared__ float mtab[HFX_MTAB];
    __shared__ uint32_t lpos[TN_WAVES][HFX_WAVE];
    const uint32_t wave = threadIdx.x / HFX_WAVE, lane = hfx_lane();
    const uint32_t F = *count;
    const uint64_t ntiles = tile_off[F];
    if (blockIdx.x >= ntiles) return;
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? c.db.d_mass[threadIdx.x] : 0.0f;
    c.stage(mtab);
    const FxWave f = fx_wave(tn_dyn, mstr, wave);
    __syncthreads();
    for (uint64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t lo = 0, hi = F;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (tile_off[mid] <= t) lo = mid; else hi = mid;
        }
        const uint32_t s = list[lo];
        const uint32_t k = (uint32_t)(t - tile_off[lo]);
        const uint32_t nt = (uint32_t)(tile_off[lo + 1] - tile_off[lo]);
        const uint32_t n = c.count(s);
        const double ts = tau[s];
        const uint32_t len = min(sp.d_len[s], min(sp.x_stride, (uint32_t)HFX_MAX_LEN));
        /* the wave's candidates: tile slots m = wave + 4 j (j < 64), lane j
         * reading candidate i = k + nt m's score.  A candidate below tau
         * cannot reach the top N (its exact score is below the N-th exact
         * score): it keeps the smallest key, stored by its own lane.  The
         * others are moved to the first lanes and re-scored. */
        const float *sc = scores + c.base(s);
        int64_t *fx = fxbuf + fx_at[lo];
        const uint64_t mi64 = k + (uint64_t)nt * (wave + TN_WAVES * lane);
        const uint32_t mi = (uint32_t)mi64;
        bool live = false;
        if (wave + TN_WAVES * lane < TX_CHUNK && mi64 < n) {
            live = !((double)sc[mi] < ts);
            if (!live) fx[mi] = INT64_MIN;
        }
        const uint64_t lm = __ballot(live);
        const uint32_t rn = (uint32_t)__builtin_popcountll(lm);
        if (live) lpos[wave][__builtin_popcountll(lm & ((1ull << lane) - 1ull))] = mi;
        hfx_wave_sync();
        uint32_t pos = 0;
        typename Cands::Prep pr{};
        if (lane < rn) {
            pos = lpos[wave][lane];
            pr = c.prep(s, pos);
        }
        fx_scores<true>(f, mstr, mtab, sp.d_x + (size_t)s * sp.x_stride, len,
                        c.zeff(sp.d_zmax[s]), c, pr, rn,
                        [&](uint32_t i, int64_t v) { fx[lpos[wave][i]] = v; });
        hfx_wave_sync();
    }
}

/* top N of a flagged spectrum by (exact desc, position asc).
 *
 * Only the live candidates count: the exact route leaves INT64_MIN for every
 * candidate below tau, and more than N are live.  They are gathered into LDS
 * in one sweep (up to FX_CAP of them) and selected there, a few by rounds of the
 * best (46 -> 15 us for 110 spectra of 10,000 candidates, top 5), more by radix over the
 * bits in which their 64-bit keys differ, 11 bits a pass, then, for keys
 * tied in full, over the complemented position.  Windows with more live
 * candidates (or fewer than N) take the 8-bit radix select over global
 * memory.  A persistent grid walks the list of flagged spectra. */
#define FX_CAP 4096
/* a workgroup per flagged spectrum, of few: sixteen waves each, so that a
 * sweep over the window has 8192 loads in flight */
#define FX_THREADS 1024
#define FX_WAVES (FX_THREADS / HFX_WAVE)
#define FX_DBITS 11
/* up to this many wanted: rounds of the best (two shuffles' depth each) instead of
 * digits (six passes with four barriers each where keys tie in full) */
#define FX_ROUNDS 16
static_assert(3 * FX_WAVES * FX_ROUNDS <= 1u << FX_DBITS && FX_WAVES * FX_ROUNDS % HFX_WAVE == 0 &&
                  FX_CAP % FX_THREADS == 0,
              "the waves' best fit the histogram's words");

template <class Cands>
__global__ void __launch_bounds__(FX_THREADS)
    k_topn_fx(uint32_t *top_pos, double *top_exact, float *top_f32, uint32_t *top_cnt,
              uint32_t *flag, uint32_t N, const uint32_t *list, const uint32_t *list_cnt,
              const int64_t *fxbuf, const uint64_t *fx_at, const float *scores, Cands c)
{
    __shared__ uint64_t lk[FX_CAP];
    __shared__ uint32_t lp[FX_CAP];
    __shared__ __align__(8) uint32_t hist[1u << FX_DBITS];
    __shared__ uint32_t sel_p[TX_MAXN];
    __shared__ int64_t sel_f[TX_MAXN];
    __shared__ uint32_t wcnt[FX_WAVES];
    __shared__ uint32_t sh_digit, sh_rem, sh_gt, sh_cnt;
    __shared__ uint64_t sh_diff;
    const uint32_t tid = threadIdx.x, wave = tid / HFX_WAVE, lane = hfx_lane();
    const uint32_t F = *list_cnt;

    for (uint32_t q = blockIdx.x; q < F; q += gridDim.x) {
        const uint32_t s = list[q];
        const uint32_t n = c.count(s);
        const int64_t *fx = fxbuf + fx_at[q];
        const float *sc = scores + c.base(s);
        uint32_t want = min(N, n);
        if (want == 0) {
            if (tid == 0) top_cnt[s] = 0;
            continue;
        }
        auto key = [&](uint32_t i) { return (uint64_t)fx[i] ^ 0x8000000000000000ull; };
        /* f(i, key) over this thread's keys, eight loads in flight
         * (clamped into the window); i >= n past it, where all lanes
         * still take part */
        auto for_keys = [&](auto &&f) {
            constexpr uint32_t U = 8;
            for (uint32_t base = 0; base < n; base += U * FX_THREADS) {
                uint64_t kk[U];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    kk[u] = key(min(base + u * FX_THREADS + tid, n - 1u));
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) f(base + u * FX_THREADS + tid, kk[u]);
            }
        };

        /* 1. the live keys (key 0 is INT64_MIN) into LDS, one LDS atomic
         * per wave and batch */
        if (tid == 0) {
            sh_cnt = 0;
            sh_gt = 0;
            sh_diff = 0;
            sh_rem = want;
        }
        __syncthreads();
        for_keys([&](uint32_t i, uint64_t k) {
            const bool live = i < n && k != 0ull;
            const uint64_t b = __ballot(live);
            if (b) {
                const uint32_t leader = (uint32_t)__builtin_ctzll(b);
                uint32_t wb = 0;
                if (lane == leader) wb = atomicAdd(&sh_cnt, (uint32_t)__builtin_popcountll(b));
                wb = (uint32_t)__builtin_amdgcn_readlane((int)wb, (int)leader);
                const uint32_t slot =
                    wb + (uint32_t)__builtin_popcountll(b & ((1ull << lane) - 1ull));
                if (live && slot < FX_CAP) {
                    lk[slot] = k;
                    lp[slot] = i;
                }
            }
        });
        __syncthreads();
        const uint32_t M = sh_cnt;
        if (M < want) {
            /* Fewer live candidates than N: the N-th exact score of the
             * selection lies above tau + bound, so at least N candidates
             * have exact scores >= tau + bound, and each of them whose FP32
             * score fell below tau lies further below its exact score than
             * the stated bound allows.  Only the live candidates are ranked
             * and the spectrum is marked for the host. */
            want = M;
            if (tid == 0) {
                flag[s] |= HFX_FLAG_SHORT;
                sh_rem = want;
                if (want == 0) top_cnt[s] = 0;
            }
            __syncthreads();
            if (want == 0) continue;
        }
        if (M <= FX_CAP && want <= FX_ROUNDS) {
            /* 2. few wanted: each wave's best of its share, then the best of
             * those */
            uint64_t *wk = (uint64_t *)hist;
            uint32_t *wp = hist + 2 * FX_WAVES * FX_ROUNDS;
            uint64_t k[FX_CAP / FX_THREADS];
            uint32_t pos[FX_CAP / FX_THREADS];
#pragma unroll
            for (uint32_t u = 0; u < FX_CAP / FX_THREADS; ++u) {
                const uint32_t i = u * FX_THREADS + tid;
                k[u] = i < M ? lk[i] : 0ull;
                pos[u] = i < M ? lp[i] : 0xffffffffu;
            }
            tn_wave_top(k, pos, want, [&](uint32_t r, uint64_t kb, uint32_t pb) {
                if (lane == 0) {
                    wk[wave * FX_ROUNDS + r] = kb;
                    wp[wave * FX_ROUNDS + r] = pb;
                }
            });
            __syncthreads();
            if (wave == 0) {
                constexpr uint32_t E = FX_WAVES * FX_ROUNDS / HFX_WAVE;
                uint64_t k2[E];
                uint32_t p2[E];
#pragma unroll
                for (uint32_t u = 0; u < E; ++u) {
                    const uint32_t i = u * HFX_WAVE + lane;
                    const bool in = i % FX_ROUNDS < want;
                    k2[u] = in ? wk[i] : 0ull;
                    p2[u] = in ? wp[i] : 0xffffffffu;
                }
                tn_wave_top(k2, p2, want, [&](uint32_t r, uint64_t kb, uint32_t pb) {
                    if (lane == 0) {
                        sel_p[r] = pb;
                        sel_f[r] = (int64_t)(kb ^ 0x8000000000000000ull);
                    }
                });
            }
            __syncthreads();
        } else if (M <= FX_CAP) {
            /* 2. the bits in which the live keys differ */
            const uint64_t k0 = lk[0];
            uint64_t d = 0;
            for (uint32_t i = tid; i < M; i += FX_THREADS) d |= lk[i] ^ k0;
            if (d) atomicOr((unsigned long long *)&sh_diff, (unsigned long long)d);
            __syncthreads();
            const uint64_t diff = sh_diff;
            /* 3. radix select over the key: prefix/pmask fix the bits
             * found so far; done once the bucket is taken whole */
            const int top = diff ? 63 - __builtin_clzll(diff) : -1;
            /* bits above the top differing one (none when it is bit 63:
             * 2 << 63 wraps to 0) */
            uint64_t pmask = diff ? ~((2ull << top) - 1ull) : ~0ull;
            uint64_t prefix = k0 & pmask;
            int hi = top;
            bool whole = false;
            while (hi >= 0 && !whole) {
                const int lo = hi - (FX_DBITS - 1) > 0 ? hi - (FX_DBITS - 1) : 0;
                const uint32_t width = (uint32_t)(hi - lo + 1), nb = 1u << width;
                for (uint32_t b = tid; b < nb; b += FX_THREADS) hist[b] = 0;
                __syncthreads();
                for (uint32_t i = tid; i < M; i += FX_THREADS) {
                    const uint64_t k = lk[i];
                    if ((k & pmask) == prefix)
                        atomicAdd(&hist[(uint32_t)(k >> lo) & (nb - 1u)], 1u);
                }
                __syncthreads();
                tn_select_digit(hist, nb, &sh_digit, &sh_rem);
                prefix |= (uint64_t)sh_digit << lo;
                pmask |= (uint64_t)(nb - 1u) << lo;
                whole = hist[sh_digit] == sh_rem;
                hi = lo - 1;
                __syncthreads();
            }
            /* 4. keys tied in full (pmask all ones): the rem smallest
             * positions among them, by radix over ~position */
            uint32_t qprefix = 0, qmask = 0;
            if (!whole) {
                for (int qh = 31; qh >= 0 && !whole;) {
                    const int lo = qh - (FX_DBITS - 1) > 0 ? qh - (FX_DBITS - 1) : 0;
                    const uint32_t width = (uint32_t)(qh - lo + 1), nb = 1u << width;
                    for (uint32_t b = tid; b < nb; b += FX_THREADS) hist[b] = 0;
                    __syncthreads();
                    for (uint32_t i = tid; i < M; i += FX_THREADS) {
                        const uint32_t q = ~lp[i];
                        if (lk[i] == prefix && (q & qmask) == qprefix)
                            atomicAdd(&hist[(q >> lo) & (nb - 1u)], 1u);
                    }
                    __syncthreads();
                    tn_select_digit(hist, nb, &sh_digit, &sh_rem);
                    qprefix |= sh_digit << lo;
                    qmask |= (nb - 1u) << lo;
                    whole = hist[sh_digit] == sh_rem;
                    qh = lo - 1;
                    __syncthreads();
                }
            }
            /* 5. the selection: keys above the prefix, and the bucket
             * (or the tied key's chosen positions) -- want of them */
            for (uint32_t i = tid; i < M; i += FX_THREADS) {
                const uint64_t k = lk[i];
                const uint32_t q = ~lp[i];
                const bool take = qmask == 0u
                                      ? (k & pmask) >= prefix
                                      : (k > prefix || (k == prefix && (q & qmask) >= qprefix));
                if (take) {
                    const uint32_t slot = atomicAdd(&sh_gt, 1u);
                    if (slot < want) {
                        sel_p[slot] = lp[i];
                        sel_f[slot] = (int64_t)(k ^ 0x8000000000000000ull);
                    }
                }
            }
            __syncthreads();
        } else {
            /* the 8-bit radix select over global memory */
            uint64_t prefix = 0, pmask = 0;
            for (int shift = 56; shift >= 0; shift -= 8) {
                if (tid < 256u) hist[tid] = 0;
                __syncthreads();
                for_keys([&](uint32_t i, uint64_t k) {
                    tn_hist_add(hist, (uint32_t)(k >> shift) & 255u,
                                i < n && (k & pmask) == prefix);
                });
                __syncthreads();
                tn_select_digit(hist, 256u, &sh_digit, &sh_rem);
                prefix |= (uint64_t)sh_digit << shift;
                pmask |= 255ull << shift;
            }
            const uint64_t K = prefix;
            const uint32_t need_eq = sh_rem, n_gt = want - need_eq;
            for_keys([&](uint32_t i, uint64_t k) {
                if (i < n && k > K) {
                    const uint32_t slot = atomicAdd(&sh_gt, 1u);
                    if (slot < n_gt) {
                        sel_p[slot] = i;
                        sel_f[slot] = (int64_t)(k ^ 0x8000000000000000ull);
                    }
                }
            });
            uint32_t eq_base = 0;
            for (uint32_t base = 0; base < n && eq_base < need_eq; base += FX_THREADS) {
                const uint32_t i = base + tid;
                const bool f = i < n && key(i) == K;
                const uint64_t bal = __ballot(f);
                const uint32_t wr = (uint32_t)__builtin_popcountll(bal & ((1ull << lane) - 1ull));
                if (lane == 0) wcnt[wave] = (uint32_t)__builtin_popcountll(bal);
                __syncthreads();
                uint32_t wpre = 0, tot = 0;
                for (uint32_t w = 0; w < FX_WAVES; ++w) {
                    if (w < wave) wpre += wcnt[w];
                    tot += wcnt[w];
                }
                const uint32_t r = eq_base + wpre + wr;
                if (f && r < need_eq) {
                    sel_p[n_gt + r] = i;
                    sel_f[n_gt + r] = fx[i];
                }
                eq_base += tot;
                __syncthreads();
            }
            __syncthreads();
        }
        for (uint32_t i = tid; i < want; i += FX_THREADS) {
            uint32_t rk = 0;
            for (uint32_t j = 0; j < want; ++j)
                rk += before_fx(sel_f[j], sel_p[j], sel_f[i], sel_p[i]) ? 1u : 0u;
            top_pos[(size_t)s * N + rk] = sel_p[i];
            top_exact[(size_t)s * N + rk] = (double)sel_f[i] * (1.0 / HFX_FX_SCALE);
            top_f32[(size_t)s * N + rk] = sc[sel_p[i]];
        }
        if (tid == 0) top_cnt[s] = want;
        __syncthreads();
    }
}

/* ------------------------------------------------------------------ */
/* Launch helpers                                                        */
/* ------------------------------------------------------------------ */

/* scratch of a call:
 * fxbuf[total] | tile_off[S+1] | fx_at[S] | tau[S] | lfx[S][TN_MAXC] |
 * spill[S * TN_SPILL] | counters (256 B) | list[S] | band[S] | mcnt[S] |
 * cand[S][TN_MAXC].  No place follows the caller's score offsets, which may start
 * anywhere and leave room between the spectra. */
size_t hfx_topn_scratch_bytes(uint32_t S, uint64_t total)
{
    return total * 8 + ((size_t)S + 1) * 8 + (size_t)S * (16 + 8 * TN_MAXC + 8 * TN_SPILL) + 256 +
           (size_t)S * 4 * (3 + TN_MAXC);
}

/* the bins of a row that are read, whatever its stride */
static uint32_t tn_bins(const hfx_spectra *sp) { return min(sp->x_stride, (uint32_t)HFX_MAX_LEN); }

struct TxScratch {
    int64_t *fxbuf, *lfx;
    uint64_t *tile_off, *fx_at;
    uint32_t *counter, *list; /* counter: spilled tasks, flagged spectra */
    TnLists l;
};
static TxScratch tx_carve(void *p, uint32_t S, uint64_t total)
{
    TxScratch x;
    x.fxbuf = (int64_t *)p;
    x.tile_off = (uint64_t *)(x.fxbuf + total);
    x.fx_at = x.tile_off + S + 1;
    x.l.tau = (double *)(x.fx_at + S);
    x.lfx = (int64_t *)(x.l.tau + S);
    x.l.spill = (uint2 *)(x.lfx + (size_t)S * TN_MAXC);
    x.counter = (uint32_t *)(x.l.spill + (size_t)S * TN_SPILL);
    x.l.nspill = x.counter;
    x.list = x.counter + 64;
    x.l.band = x.list + S;
    x.l.mcnt = x.l.band + S;
    x.l.cand = x.l.mcnt + S;
    x.l.task = S <= TN_FEW ? TN_TASK_FEW : TN_TASK;
    return x;
}
static TxPlan tx_plan_of(const TxScratch &x) { return {x.tile_off, x.fx_at, x.list, x.counter + 1}; }
static int tx_scratch(hfx_ctx *ctx, void *given, uint32_t S, uint64_t total, void **out)
{
    *out = given;
    if (given) return HFX_OK;
    return hfx_ctx_scratch(ctx, HFX_SLOT_TOPN, hfx_topn_scratch_bytes(S, total), out);
}

template <class Cands>
static int exact_route(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact, float *d_top_f32,
                       uint32_t *d_top_cnt, uint32_t N, uint32_t *d_flag,
                       const float *d_scores, const Cands &c, uint64_t total,
                       const hfx_spectra *sp, void *scratch, bool planned, hipStream_t st)
{
    const uint32_t S = sp->num_spec;
    if (S == 0) return HFX_OK;
    HFX_REQUIRE(N >= 1 && N <= TX_MAXN, HFX_ERR_ARG, "top-N: N must be in 1..%d", TX_MAXN);
    void *p;
    int rc;
    if ((rc = tx_scratch(ctx, scratch, S, total, &p))) return rc;
    const TxScratch x = tx_carve(p, S, total);
    if (!planned)
        hipLaunchKernelGGL(k_tx_plan<Cands>, dim3(1), dim3(TN_THREADS), 0, st, tx_plan_of(x), d_flag,
                           x.l.band, c, S);
    hipLaunchKernelGGL(k_exact_tiles<Cands>, dim3((uint32_t)hfx_ctx_num_cus(ctx) * 4),
                       dim3(TN_THREADS), fx_lds_bytes(tn_bins(sp)), st, x.fxbuf, x.tile_off, x.fx_at,
                       x.list, x.counter + 1, c, *sp, d_scores, x.l.tau, xp_map_words(tn_bins(sp)));
    hipLaunchKernelGGL(k_topn_fx<Cands>, dim3(min(S, (uint32_t)hfx_ctx_num_cus(ctx))),
                       dim3(FX_THREADS), 0, st, d_top_pos, d_top_exact, d_top_f32, d_top_cnt,
                       d_flag, N, x.list, x.counter + 1, x.fxbuf, x.fx_at, d_scores, c);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

template <class Cands>
static int launch_topn(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact, float *d_top_f32,
                       uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N, uint32_t margin,
                       const float *d_scores, const Cands &c, uint64_t total,
                       const hfx_spectra *sp, float rel0, float rel1, float relq,
                       const float2 *norms, void *scratch, void *stream)
{
    HFX_REQUIRE(ctx && d_top_pos && d_top_exact && d_top_f32 && d_top_cnt && d_flag && d_scores &&
                    sp,
                HFX_ERR_ARG, "hfx_topn: null argument");
    HFX_REQUIRE(N >= 1 && N <= TX_MAXN && N + margin <= TN_MAXT, HFX_ERR_ARG,
                "hfx_topn: need 1 <= N <= %d and N + margin <= %d (N=%u margin=%u)", TX_MAXN,
                TN_MAXT, N, margin);
    const uint32_t S = sp->num_spec;
    if (S == 0) return HFX_OK;
    hipStream_t st = hfx_stream(stream);
    void *p;
    int rc;
    if ((rc = tx_scratch(ctx, scratch, S, total, &p))) return rc;
    const TxScratch x = tx_carve(p, S, total);
    const uint32_t gw = (S + TN_WAVES - 1) / TN_WAVES;
    hipLaunchKernelGGL(k_tx_reset, dim3(1), dim3(1), 0, st, x.counter);
    hipLaunchKernelGGL(k_topn_select<Cands>, dim3(S), dim3(TN_THREADS), 0, st, x.l, d_flag, N,
                       margin, d_scores, c, *sp, rel0, rel1, relq, norms);
    /* at least four workgroups a CU: the spilled tasks spread over them */
    hipLaunchKernelGGL(k_topn_exact<Cands>, dim3(max(gw, 4u * (uint32_t)hfx_ctx_num_cus(ctx))),
                       dim3(TN_THREADS), fx_lds_bytes(tn_bins(sp)), st, x.lfx, x.l, c, *sp,
                       xp_map_words(tn_bins(sp)));
    hipLaunchKernelGGL(k_topn_rank<Cands>, dim3(gw + 1), dim3(TN_THREADS), 0, st, d_top_pos,
                       d_top_exact, d_top_f32, d_top_cnt, d_flag, N, x.lfx, x.l, d_scores, c, S,
                       tx_plan_of(x));
    HFX_CHECK_LAUNCH();
    return exact_route(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, N, d_flag, d_scores, c,
                       total, sp, p, true, st);
}

template <class Cands>
static int launch_topn_exact(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                             float *d_top_f32, uint32_t *d_top_cnt, uint32_t N,
                             const uint32_t *d_list, uint32_t num_list, const float *d_scores,
                             const Cands &c, uint64_t total, const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(ctx && d_top_pos && d_top_exact && d_top_f32 && d_top_cnt && d_list && sp,
                HFX_ERR_ARG, "hfx_topn_exact: null argument");
    const uint32_t S = sp->num_spec;
    if (S == 0 || num_list == 0) return HFX_OK;
    hipStream_t st = hfx_stream(stream);
    void *p, *q;
    int rc;
    if ((rc = hfx_ctx_scratch(ctx, HFX_SLOT_FLAGS, 4ull * S + 64, &p)) != HFX_OK) return rc;
    if ((rc = tx_scratch(ctx, nullptr, S, total, &q))) return rc;
    uint32_t *flag = (uint32_t *)p;
    const TxScratch x = tx_carve(q, S, total);
    hipLaunchKernelGGL(k_zero_flags, dim3((S + 255) / 256), dim3(256), 0, st, flag, S);
    hipLaunchKernelGGL(k_mark_list, dim3((num_list + 255) / 256), dim3(256), 0, st, flag, x.l.tau,
                       x.l.band, d_list, num_list, S);
    return exact_route(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, N, flag, d_scores, c,
                       total, sp, q, false, st);
}

/* used by the batched path: the whole top-N on the device */
int hfx_topn_device(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact, float *d_top_f32,
                    uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N, uint32_t margin,
                    const float *d_scores, const uint64_t *d_off, uint64_t total,
                    const uint32_t *d_begin, const uint32_t *d_num, const hfx_db *db,
                    const hfx_spectra *sp, float rel0, float rel1, float relq, const float2 *norms,
                    void *scratch, void *stream)
{
    HFX_REQUIRE(rel0 >= 0.0f && rel1 >= 0.0f && relq >= 0.0f && rel0 < 1.0f && rel1 < 1.0f &&
                    relq < 1.0f,
                HFX_ERR_ARG,
                "top-N: error bound factors must lie in [0, 1) (rel0=%g rel1=%g relq=%g)", rel0,
                rel1, relq);
    HfxPlainCands c{*db, d_begin, d_num, d_off};
    return launch_topn(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, d_flag, N, margin,
                       d_scores, c, total, sp, rel0, rel1, relq, norms, scratch, stream);
}

extern "C" int hfx_topn(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact, float *d_top_f32,
                        uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N, uint32_t margin,
                        const float *d_scores, const uint64_t *d_off, uint64_t total,
                        const uint32_t *d_begin, const uint32_t *d_num, const hfx_db *db,
                        const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(d_off && d_begin && d_num && db, HFX_ERR_ARG, "hfx_topn: null argument");
    return hfx_topn_device(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, d_flag, N, margin,
                           d_scores, d_off, total, d_begin, d_num, db, sp, HFX_TOPN_REL_F32, 0.0f,
                           0.0f, nullptr, nullptr, stream);
}

extern "C" int hfx_topn_rel(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                            float *d_top_f32, uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N,
                            uint32_t margin, float rel0, float rel1, const float *d_scores,
                            const uint64_t *d_off, uint64_t total, const uint32_t *d_begin,
                            const uint32_t *d_num, const hfx_db *db, const hfx_spectra *sp,
                            void *stream)
{
    HFX_REQUIRE(d_off && d_begin && d_num && db, HFX_ERR_ARG, "hfx_topn_rel: null argument");
    return hfx_topn_device(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, d_flag, N, margin,
                           d_scores, d_off, total, d_begin, d_num, db, sp, rel0, rel1, 0.0f,
                           nullptr, nullptr, stream);
}

extern "C" int hfx_topn_rel_q(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                              float *d_top_f32, uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N,
                              uint32_t margin, float rel0, float rel1, float relq,
                              const float *d_scores, const uint64_t *d_off, uint64_t total,
                              const uint32_t *d_begin, const uint32_t *d_num, const hfx_db *db,
                              const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(d_off && d_begin && d_num && db, HFX_ERR_ARG, "hfx_topn_rel_q: null argument");
    return hfx_topn_device(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, d_flag, N, margin,
                           d_scores, d_off, total, d_begin, d_num, db, sp, rel0, rel1, relq,
                           nullptr, nullptr, stream);
}

extern "C" int hfx_topn_exact(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                              float *d_top_f32, uint32_t *d_top_cnt, uint32_t N,
                              const uint32_t *d_spec_list, uint32_t num_list,
                              const float *d_scores, const uint64_t *d_off, uint64_t total,
                              const uint32_t *d_begin, const uint32_t *d_num, const hfx_db *db,
                              const hfx_spectra *sp, void *stream)
{
    HFX_REQUIRE(d_off && d_begin && d_num && db && d_scores, HFX_ERR_ARG,
                "hfx_topn_exact: null argument");
    HfxPlainCands c{*db, d_begin, d_num, d_off};
    return launch_topn_exact(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, N, d_spec_list,
                             num_list, d_scores, c, total, sp, stream);
}

extern "C" int hfx_topn_mod(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                            float *d_top_f32, uint32_t *d_top_cnt, uint32_t *d_flag, uint32_t N,
                            uint32_t margin, const float *d_scores, const uint64_t *d_mp_off,
                            const hfx_modset *ms, const hfx_db *db, const hfx_spectra *sp,
                            void *stream)
{
    HFX_REQUIRE(d_mp_off && ms && db, HFX_ERR_ARG, "hfx_topn_mod: null argument");
    HFX_REQUIRE(ms->num_ma <= HFX_MAX_MA, HFX_ERR_ARG, "hfx_topn_mod: num_ma %u", ms->num_ma);
    HfxModCands c{*db, *ms, d_mp_off};
    return launch_topn(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, d_flag, N, margin,
                       d_scores, c, ms->num_mpep, sp, HFX_TOPN_REL_F32, 0.0f, 0.0f, nullptr,
                       nullptr, stream);
}

extern "C" int hfx_topn_exact_mod(hfx_ctx *ctx, uint32_t *d_top_pos, double *d_top_exact,
                                  float *d_top_f32, uint32_t *d_top_cnt, uint32_t N,
                                  const uint32_t *d_spec_list, uint32_t num_list,
                                  const float *d_scores, const uint64_t *d_mp_off,
                                  const hfx_modset *ms, const hfx_db *db, const hfx_spectra *sp,
                                  void *stream)
{
    HFX_REQUIRE(d_mp_off && ms && db && d_scores, HFX_ERR_ARG, "hfx_topn_exact_mod: null argument");
    HFX_REQUIRE(ms->num_ma <= HFX_MAX_MA, HFX_ERR_ARG, "hfx_topn_exact_mod: num_ma %u", ms->num_ma);
    HfxModCands c{*db, *ms, d_mp_off};
    return launch_topn_exact(ctx, d_top_pos, d_top_exact, d_top_f32, d_top_cnt, N, d_spec_list,
                             num_list, d_scores, c, ms->num_mpep, sp, stream);
}
