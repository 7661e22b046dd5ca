/*
 * hfx_stats.hip -- E-values and SP ion matches of a search, on the device.
 *
 * E-values (Util/Statistics.hs:37-100, applied per spectrum by
 * Search.hs:118-123 to every match of the spectrum, unmodified and modified):
 * the reference sorts all scores ascending, keeps sorted positions
 * [round(0.3 n), round((1 - p/100) n)), shifts them by 1 - min, drops those at
 * or below 4000, histograms the rest in bins of width w and fits log10 of the
 * heights against the bin centres by least squares (statistics-linreg).
 *
 * No sort is needed here: x -> bin is monotone, so the sorted positions of the
 * scores of one bin form the range [C(k-1), C(k)) of the cumulative bin counts
 * C, and the kept count of bin k is that range's overlap with the cut.  One
 * workgroup per spectrum:
 *   1. min and max of the spectrum's scores, kept in registers (the part past
 *      EV_HOLD chunks is read again);
 *   2. key(x) = 0 for (x + 1) - min <= 4000, else ceil(((x + 1) - min) / w)
 *      - kbase (>= 1), counted per key in LDS (EV_KEYS keys per pass; a wider
 *      spread takes one pass per range of keys).  FP32 decides the key unless
 *      the quotient lies within its error of an edge;
 *   3. a block scan of the counts gives every key's sorted range, hence the
 *      kept counts and the histogram points (x_k, log10(c_k / w));
 *   4. least squares in FP64: sums about the middle of the key range.
 *
 * SP ions (IonSeries.hs:99-147, Match.hs:33-40): extractPeaks keeps the 200
 * largest values of the spectrum and folds them by max into bins i div 3; a
 * b or y ion matches when its bin round(m/z / bin width / 3) holds a value
 * above zero.  sp_flags turns a spectrum into those flags (one bit per bin;
 * one wave per spectrum, the row in registers, the 200th value selected bit by
 * bit over the float bits by ballot counts; k_sp_peaks does the same with a
 * workgroup for rows longer than 3072); sp_matches matches peptides along their
 * FP32 b ladders, a position a lane.  k_sp_topn does both, a wave a spectrum.
 */
#include "hfx_common.h"

#include <math.h>
#include <type_traits>

#define ST_THREADS 256
#define ST_WAVES (ST_THREADS / HFX_WAVE)

#define EV_THREADS 256
#define EV_WAVES (EV_THREADS / HFX_WAVE)
#define EV_CHUNK (4 * EV_THREADS)    /* scores a workgroup loads at once       */
#define EV_HOLD 6                   /* chunks kept in registers               */
#define EV_KEYS 1024                /* histogram keys per pass                */
#define EV_KPT (EV_KEYS / EV_THREADS)
#define EV_COPY_SHIFT 4             /* 16 counts of a key where keys are few  */
#define EV_MAGIC 12582912.0f        /* 1.5 * 2^23: adding it rounds to an integer */
#define EV_MAGIC_BITS 0x4B400000u

#define SP_TOP 200                  /* IonSeries.hs:104                       */
#define SP_CACHE 8192               /* spectrum values kept in LDS            */
#define SP_WORDS 256                /* flag words: len / 3 + 1 <= 8192 bins   */

/* Host constants of the ion ladder (Mass.hs:19-27) */
#define SP_H 1.007276f
#define SP_H2O 18.010565f

/* ------------------------------------------------------------------ */
/* Block primitives (ST_THREADS threads)                                */
/* ------------------------------------------------------------------ */

template <typename T>
__device__ __forceinline__ T st_wave_sum(T v)
{
#pragma unroll
    for (int m = HFX_WAVE / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, HFX_WAVE);
    return v;
}

/* sum over the block, partial sums added in wave order (deterministic) */
template <typename T>
__device__ __forceinline__ T st_block_sum(T v, T *red)
{
    v = st_wave_sum(v);
    __syncthreads();
    if (threadIdx.x % HFX_WAVE == 0) red[threadIdx.x / HFX_WAVE] = v;
    __syncthreads();
    T t = red[0];
#pragma unroll
    for (int i = 1; i < ST_WAVES; ++i) t += red[i];
    return t;
}

/* exclusive prefix sum over the block in thread order */
template <typename T>
__device__ __forceinline__ T st_block_excl_scan(T v, T *red)
{
    const int lane = threadIdx.x % HFX_WAVE, w = threadIdx.x / HFX_WAVE;
    T x = v;
#pragma unroll
    for (int d = 1; d < HFX_WAVE; d <<= 1) {
        const T y = __shfl_up(x, d, HFX_WAVE);
        if (lane >= d) x += y;
    }
    __syncthreads();
    if (lane == HFX_WAVE - 1) red[w] = x;
    __syncthreads();
    T off = 0;
    for (int i = 0; i < w; ++i) off += red[i];
    return off + x - v;
}

/* ------------------------------------------------------------------ */
/* E-value fit                                                           */
/* ------------------------------------------------------------------ */

/* ------------------------------------------------------------------ */
/* Wave reductions over DPP lane moves (no LDS round trips)              */
/* ------------------------------------------------------------------ */

/* quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror:
 * every lane of a row of 16 ends with the row's total; row_bcast15 (rows 1
 * and 3) and row_bcast31 (rows 2 and 3) carry the rows into lane 63. */
#define ST_DPP32(old, v, ctrl, rm) \
    ((uint32_t)__builtin_amdgcn_update_dpp((int)(old), (int)(v), (ctrl), (rm), 0xF, false))

template <int CTRL, int RM>
__device__ __forceinline__ uint64_t st_dpp64(uint64_t v, uint64_t old)
{
    const uint32_t lo = ST_DPP32((uint32_t)old, (uint32_t)v, CTRL, RM);
    const uint32_t hi = ST_DPP32((uint32_t)(old >> 32), (uint32_t)(v >> 32), CTRL, RM);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t st_readlane63(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
    return ((uint64_t)hi << 32) | lo;
}

/* op-reduction of a 64-bit value over the wave; ident is op's identity */
template <class Op>
__device__ __forceinline__ uint64_t st_wave_reduce64(uint64_t v, uint64_t ident, Op op)
{
    v = op(v, st_dpp64<0xB1, 0xF>(v, ident));
    v = op(v, st_dpp64<0x4E, 0xF>(v, ident));
    v = op(v, st_dpp64<0x141, 0xF>(v, ident));
    v = op(v, st_dpp64<0x140, 0xF>(v, ident));
    v = op(v, st_dpp64<0x142, 0xA>(v, ident));
    v = op(v, st_dpp64<0x143, 0xC>(v, ident));
    return st_readlane63(v);
}

__device__ __forceinline__ double st_wsum_f64(double v)
{
    const uint64_t r = st_wave_reduce64(__double_as_longlong(v), 0ull, [](uint64_t a, uint64_t b) {
        return (uint64_t)__double_as_longlong(__longlong_as_double(a) + __longlong_as_double(b));
    });
    return __longlong_as_double(r);
}

/* least lo and greatest hi of the wave, in every lane */
__device__ __forceinline__ void st_wave_minmax(float &lo, float &hi)
{
    auto step = [&](auto ctrl, auto rm) {
        const uint32_t l = ST_DPP32(__float_as_uint(lo), __float_as_uint(lo), decltype(ctrl)::value,
                                    decltype(rm)::value);
        const uint32_t h = ST_DPP32(__float_as_uint(hi), __float_as_uint(hi), decltype(ctrl)::value,
                                    decltype(rm)::value);
        lo = fminf(lo, __uint_as_float(l));
        hi = fmaxf(hi, __uint_as_float(h));
    };
    using std::integral_constant;
    step(integral_constant<int, 0xB1>{}, integral_constant<int, 0xF>{});
    step(integral_constant<int, 0x4E>{}, integral_constant<int, 0xF>{});
    step(integral_constant<int, 0x141>{}, integral_constant<int, 0xF>{});
    step(integral_constant<int, 0x140>{}, integral_constant<int, 0xF>{});
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});
    lo = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(lo), 63));
    hi = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(hi), 63));
}

/* inclusive prefix sum of uint32 over the wave: row_shr 1, 2, 4, 8 within
 * rows of 16, then row_bcast15 / row_bcast31 across rows */
__device__ __forceinline__ uint32_t st_wave_incl_scan32(uint32_t x)
{
    x += ST_DPP32(0u, x, 0x111, 0xF);
    x += ST_DPP32(0u, x, 0x112, 0xF);
    x += ST_DPP32(0u, x, 0x114, 0xF);
    x += ST_DPP32(0u, x, 0x118, 0xF);
    x += ST_DPP32(0u, x, 0x142, 0xA);
    x += ST_DPP32(0u, x, 0x143, 0xC);
    return x;
}

/* ------------------------------------------------------------------ */
/* E-value fit                                                           */
/* ------------------------------------------------------------------ */

struct EvArgs {
    double *fit;        /* [S][2] alpha, beta          */
    uint32_t *npts;     /* [S] histogram points, opt.  */
    uint64_t *nused;    /* [S] scores kept, opt.       */
    const float *sa;
    const uint64_t *oa;
    const float *sb;    /* second score set, opt.      */
    const uint64_t *ob;
    double w, rw, kb;   /* bin width, RN(1 / w), kbase */
    float perc;
};

#define EV_NSUM 4   /* sum dx, sum y, sum dx^2, sum dx y */

struct EvShared {
    uint32_t hist[EV_KEYS];       /* counts per key (several of each, if few) */
    uint32_t red32[EV_KPT * EV_WAVES];
    double redd[EV_NSUM * EV_WAVES];
    uint64_t redu[2 * EV_WAVES];
    uint32_t redn[2 * EV_WAVES];
};

/* sixteen bytes at any multiple of four */
typedef float ev_f4 __attribute__((ext_vector_type(4), aligned(4)));

/* one spectrum's view: n scores in chunks of EV_CHUNK (the first ca of set a,
 * the rest of set b), the cut, the key map */
struct EvSpec {
    const float *sa, *sb;
    uint64_t na, nb, n;
    uint64_t ca, nch;
    int64_t cb, ce;
    double h0, w, kb, x0;
    double rw;          /* RN(1 / w) */
    /* the key map in FP32: q = fma(v, rwf, cf) is within eps of the quotient
     * ((v + 1) - h0) / w less a half; above qhi the score is kept for certain,
     * below qlo filtered out, and within in of an integer its ceiling holds */
    float rwf, cf, qlo, qhi, in;

    /* thread tid's four scores of chunk u; NaN past the end, which no key
     * counts */
    __device__ __forceinline__ ev_f4 load(uint64_t u) const
    {
        const bool a = u < ca;
        const float *p = a ? sa : sb;
        const uint64_t i = (a ? u : u - ca) * EV_CHUNK + 4 * threadIdx.x, m = a ? na : nb;
        ev_f4 v = {NAN, NAN, NAN, NAN};
        if (i + 4 <= m) v = *(const ev_f4 *)(p + i);
        else if (i < m)
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (i + e < m) v[e] = p[i + e];
        return v;
    }

    /* 0 for (x + 1) - min <= 4000 (filtered out, Statistics.hs:76), else
     * the bin ceiling(y / w) less kbase: monotone in x.  q = y * RN(1/w) is
     * within 2 ulp of y / w (below 2^20: 5e-10), so its ceiling is that of
     * the correctly rounded quotient unless q lies within 1e-9 of an
     * integer: only then (or for q >= 2^20) divide. */
    __device__ __forceinline__ uint64_t key(float v) const
    {
        const double y = ((double)v + 1.0) - h0;
        if (!(y > 4000.0)) return 0;
        const double q = y * rw;
        const double f = q - floor(q);
        const double c = (f > 1e-9 && f < 1.0 - 1e-9 && q < 1048576.0) ? ceil(q) : ceil(y / w);
        const double kd = c - kb;
        return kd < 4.6e18 ? (uint64_t)kd : (uint64_t)4.6e18;
    }

    /* valBin = i * w - w / 2 with i = ceiling(y / w); x = valBin / 10000
     * (here times RN(1e-4): within an ulp) */
    __device__ __forceinline__ double xof(uint64_t k) const
    {
        return (((double)k + kb) * w - w / 2.0) * 1e-4;
    }
};

/* a thread's part of the histogram points */
struct EvSums {
    double v[EV_NSUM];
    uint32_t points, kept;
};

/* f(score, its place in the group) for every score of thread tid, group(first
 * chunk) after each group of up to 8 chunks: H = EV_HOLD from the registers that hold
 * them (none if H = 0), then two at a time from memory */
template <int H, class F, class G>
__device__ __forceinline__ void ev_each(const EvSpec &e, const ev_f4 (&v)[EV_HOLD], F &&f, G &&group)
{
    if constexpr (H > 0) {
#pragma unroll
        for (int u = 0; u < H; ++u) {
            if ((uint64_t)u < e.nch) {
#pragma unroll
                for (int i = 0; i < 4; ++i) f(v[u][i], 4 * (u % 8) + i);
            }
            if (u % 8 == 7) group((uint64_t)u - 7);
        }
        if (H % 8) group((uint64_t)(H - H % 8));
    }
    for (uint64_t u = H; u < e.nch; u += 2) {
        ev_f4 t[2];
        t[0] = e.load(u);
        t[1] = e.load(u + 1); /* past the last chunk: NaN */
#pragma unroll
        for (int i = 0; i < 8; ++i) f(t[i >> 2][i & 3], i);
        group(u);
    }
}

/* Histogram of keys [base, base + EV_KEYS); the kept part of each key's
 * scores becomes a point (x, logh), added to the thread's sums (x shifted by
 * x0).  ALL: no score lies above the range.  next = the smallest key above the
 * range (~0 if none).  hist is clear, and left so if not ALL. */
template <bool ALL>
__device__ __forceinline__ void ev_window(const EvSpec &e, EvShared &sh, const ev_f4 (&v)[EV_HOLD],
                                          uint64_t base, uint64_t khi, EvSums &acc, uint64_t &next)
{
    const uint32_t tid = threadIdx.x, lane = tid % HFX_WAVE, wv = tid / HFX_WAVE;
    /* few keys: up to 16 counts of each, by lane, so that fewer lanes of an
     * atomic meet on a word */
    uint32_t shl = 0;
    if (ALL)
        while (shl < EV_COPY_SHIFT && (khi + 1) << (shl + 1) <= EV_KEYS) ++shl;
    const uint32_t cp = lane & ((1u << shl) - 1u);
    uint64_t above = 0, nxt = ~(uint64_t)0;
    auto add = [&](uint64_t k) {
        if (k < base || k == 0) return;
        if (ALL || k - base < EV_KEYS) {
            atomicAdd(&sh.hist[(uint32_t)(k - base) << shl | cp], 1u);
        } else {
            ++above;
            nxt = k < nxt ? k : nxt;
        }
    };
    uint32_t edge = 0; /* scores of the group that FP32 cannot decide */
    const uint32_t kofs = EV_MAGIC_BITS - 1u + (uint32_t)e.kb;
    /* several ranges are rare: their passes read the scores again */
    ev_each<ALL ? EV_HOLD : 0>(
        e, v,
        [&](float x, int i) {
            /* the sum with 1.5 * 2^23 rounds quotient - 1/2: its ceiling less 1 */
            const float q = __builtin_fmaf(x, e.rwf, e.cf), t = q + EV_MAGIC;
            const bool ok = fabsf(q - (t - EV_MAGIC)) < e.in && q > e.qhi;
            if (ok) {
                const uint32_t k = __float_as_uint(t) - kofs; /* the key */
                if constexpr (ALL) atomicAdd(&sh.hist[k << shl | cp], 1u); /* base 0, none above */
                else add(k);
            }
            edge |= (!ok && q >= e.qlo ? 1u : 0u) << i;
        },
        [&](uint64_t u) {
            while (edge) {
                const uint32_t i = (uint32_t)__builtin_ctz(edge);
                edge &= edge - 1u;
                const uint64_t c = u + i / 4;
                const bool a = c < e.ca;
                add(e.key((a ? e.sa : e.sb)[(a ? c : c - e.ca) * EV_CHUNK + 4 * threadIdx.x + i % 4]));
            }
        });
    if constexpr (!ALL) {
        above = st_wave_reduce64(above, 0ull, [](uint64_t a, uint64_t b) { return a + b; });
        nxt = st_wave_reduce64(nxt, ~0ull, [](uint64_t a, uint64_t b) { return a < b ? a : b; });
        if (lane == 0) {
            sh.redu[2 * wv] = above;
            sh.redu[2 * wv + 1] = nxt;
        }
    }
    __syncthreads();
    next = ~(uint64_t)0;
    uint64_t ta = 0;
    if constexpr (!ALL) {
#pragma unroll
        for (int i = 0; i < EV_WAVES; ++i) {
            ta += sh.redu[2 * i];
            next = sh.redu[2 * i + 1] < next ? sh.redu[2 * i + 1] : next;
        }
    }
    /* thread t's keys are t + 256 j: the sorted position of each from a scan of
     * the counts */
    const uint32_t nj = max((uint32_t)EV_KPT >> shl, 1u);
    auto counted = [&](uint32_t j) {
        const uint32_t k = j * EV_THREADS + tid;
        if (shl < 2) return sh.hist[k << shl] + (shl ? sh.hist[k << 1 | 1u] : 0u);
        uint32_t n = 0;
        if (k << shl < EV_KEYS)
            for (uint32_t i = 0; i < 1u << shl; i += 4) {
                const uint4 q = *(const uint4 *)&sh.hist[(k << shl) + ((i + 4 * k) & ((1u << shl) - 4u))];
                n += q.x + q.y + q.z + q.w;
            }
        return n;
    };
#pragma unroll 1
    for (uint32_t j = 0; j < nj; ++j) {
        const uint32_t incl = st_wave_incl_scan32(counted(j));
        if (lane == HFX_WAVE - 1) sh.red32[j * EV_WAVES + wv] = incl;
    }
    __syncthreads();
    /* scores of keys below the range: all but those counted or above */
    uint32_t pre = (uint32_t)(e.n - ta);
    for (uint32_t i = 0; i < nj * EV_WAVES; ++i) pre -= sh.red32[i];
#pragma unroll 1
    for (uint32_t j = 0; j < nj; ++j) {
        const uint32_t c = counted(j);
        uint32_t o = pre + st_wave_incl_scan32(c) - c;
#pragma unroll
        for (uint32_t i = 0; i < EV_WAVES; ++i) {
            o += i < wv ? sh.red32[j * EV_WAVES + i] : 0u;
            pre += sh.red32[j * EV_WAVES + i];
        }
        if (!ALL) sh.hist[j * EV_THREADS + tid] = 0;
        const int64_t kp = min((int64_t)o + c, e.ce) - max((int64_t)o, e.cb);
        if (c && kp > 0) {
            /* logh = logBase 10 (count / w) = log h / log 10 (here log10:
             * within an ulp) */
            const double dx = e.xof(base + j * EV_THREADS + tid) - e.x0;
            const double y = log10((double)kp / e.w);
            acc.v[0] += dx;
            acc.v[1] += y;
            acc.v[2] += dx * dx;
            acc.v[3] += dx * y;
            acc.points += 1;
            acc.kept += (uint32_t)kp;
        }
    }
    if constexpr (!ALL) __syncthreads(); /* the next range counts in hist again */
}

/* spectrum s's sets */
__device__ __forceinline__ EvSpec ev_sets(const EvArgs &a, uint32_t s)
{
    EvSpec e;
    const uint64_t a0 = a.oa[s];
    e.na = a.oa[s + 1] - a0;
    e.sa = a.sa + a0;
    e.nb = 0;
    e.sb = nullptr;
    if (a.sb) {
        const uint64_t b0 = a.ob[s];
        e.nb = a.ob[s + 1] - b0;
        e.sb = a.sb + b0;
    }
    e.n = e.na + e.nb;
    e.ca = (e.na + EV_CHUNK - 1) / EV_CHUNK;
    e.nch = e.ca + (e.nb + EV_CHUNK - 1) / EV_CHUNK;
    return e;
}

/* its cut and key map, the scores lying in [lo, hi]; the key of hi */
__device__ __forceinline__ uint64_t ev_map(EvSpec &e, const EvArgs &a, float lo, float hi)
{
    /* the cut (Statistics.hs:72-73): Float for cut_end, Double for cut_beg,
     * halves to even */
    const float fe = (1.0f - a.perc / 100.0f) * (float)e.n;
    e.ce = min((int64_t)e.n, max((int64_t)0, (int64_t)__builtin_rintf(fe)));
    e.cb = max((int64_t)0, (int64_t)rint((30.0 / 100.0) * (double)e.n));
    e.h0 = (double)lo;
    e.w = a.w;
    e.rw = a.rw;
    e.kb = a.kb;
    /* rwf, cf and the sum are each within 2^-24 relative, of |v| rw, |cf| and no
     * more than both together; eps is more than twice that.  Nothing is decided
     * in FP32 where it passes a quarter of a bin. */
    e.rwf = (float)e.rw;
    e.cf = (float)((1.0 - e.h0) * e.rw - 0.5);
    const float q4 = (float)(4000.0 * e.rw - 0.5);
    const float eps =
        (fmaxf(fabsf(lo), fabsf(hi)) * e.rwf + fabsf(e.cf) + fabsf(q4) + 1.0f) * 2.4e-7f * 2.0f;
    const bool use = eps < 0.25f;
    e.in = use ? 0.5f - eps : -1.0f;
    e.qhi = q4 + eps;
    e.qlo = use ? q4 - eps : -INFINITY;
    /* sums are taken about x0, the middle of the key range of the scores,
     * and centred at the end (no cancellation beyond the data's own spread) */
    const uint64_t khi = e.key(hi);
    e.x0 = khi ? 0.5 * (e.xof(1) + e.xof(khi)) : 0.0;
    return khi;
}

/* the sums' least squares: over the block in wave order (deterministic) */
__device__ __forceinline__ void ev_solve(const EvArgs &a, EvShared &sh, uint32_t s, double x0, EvSums acc)
{
    const uint32_t tid = threadIdx.x, lane = tid % HFX_WAVE, wv = tid / HFX_WAVE;
    if (__ballot(acc.points != 0)) { /* often the first wave only */
#pragma unroll
        for (int q = 0; q < EV_NSUM; ++q) acc.v[q] = st_wsum_f64(acc.v[q]);
        const uint64_t pk = st_wave_reduce64((uint64_t)acc.points << 32 | acc.kept, 0ull,
                                             [](uint64_t x, uint64_t y) { return x + y; });
        acc.points = (uint32_t)(pk >> 32);
        acc.kept = (uint32_t)pk;
    }
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < EV_NSUM; ++q) sh.redd[EV_NSUM * wv + q] = acc.v[q];
        sh.redn[2 * wv] = acc.points;
        sh.redn[2 * wv + 1] = acc.kept;
    }
    __syncthreads();
    if (tid == 0) {
        double t[EV_NSUM];
        uint32_t points = 0, kept = 0;
        for (int i = 0; i < EV_WAVES; ++i) {
            points += sh.redn[2 * i];
            kept += sh.redn[2 * i + 1];
        }
#pragma unroll
        for (int q = 0; q < EV_NSUM; ++q) {
            t[q] = sh.redd[q];
            for (int i = 1; i < EV_WAVES; ++i) t[q] += sh.redd[EV_NSUM * i + q];
        }
        const double m = (double)points;
        const double sxx = t[2] - t[0] * t[0] / m;
        const double sxy = t[3] - t[0] * t[1] / m;
        const double beta = sxy / sxx;
        const double mx = x0 + t[0] / m, my = t[1] / m;
        a.fit[2 * s] = my - beta * mx;
        a.fit[2 * s + 1] = beta;
        if (a.npts) a.npts[s] = points;
        if (a.nused) a.nused[s] = kept;
    }
}

/* a spectrum whose keys take several ranges: a function of its own (the
 * kernel's arguments through their segment), called last, so that its registers are not those of the usual case */
__device__ __attribute__((noinline)) void
ev_wide(const __attribute__((address_space(4))) void *args, EvShared &sh, uint32_t s, float lo, float hi)
{
    const EvArgs a = *(const EvArgs *)args;
    EvSpec e = ev_sets(a, s);
    const uint64_t khi = ev_map(e, a, lo, hi);
    const ev_f4 v[EV_HOLD] = {};
    EvSums acc{};
    uint64_t next = 0;
    for (uint64_t base = 0; base <= khi; base = next) /* no key passes khi */
        ev_window<false>(e, sh, v, base, khi, acc, next);
    ev_solve(a, sh, s, e.x0, acc);
}

/* A workgroup a spectrum, eight of them a CU (64 registers, 4.5 KiB of LDS):
 * each step waits on the one before it (loads, least, counts, scan, logarithms,
 * sums; half of a wave's cycles), so the CU is kept busy by the other workgroups,
 * up to 0.97 vector instructions a SIMD every four cycles: they bound it.  With the
 * scores in LDS four workgroups fit, and keys in FP64 alone take a dozen FP64
 * operations a score.  10,000 spectra of 4600 scores on average: 162 us that way, 70
 * so (185 MB, 2.6 TB/s; 128 threads and 5120 scores held: 75, one wave and 4096: 110). */
__global__ __launch_bounds__(EV_THREADS, 8) void k_evfit(EvArgs a)
{
    __shared__ __align__(16) EvShared sh;
    const uint32_t s = blockIdx.x, tid = threadIdx.x, lane = tid % HFX_WAVE;
    const uint32_t wv = tid / HFX_WAVE;
    EvSpec e = ev_sets(a, s);
    auto no_fit = [&]() {
        if (tid == 0) {
            a.fit[2 * s] = NAN;
            a.fit[2 * s + 1] = NAN;
            if (a.npts) a.npts[s] = 0;
            if (a.nused) a.nused[s] = 0;
        }
    };
    /* positions are counted in 32 bits */
    if (e.n == 0 || e.n > 0xFFFFFFFFull) {
        no_fit();
        return;
    }

    /* 1. the scores, their min and max */
    ev_f4 v[EV_HOLD];
#pragma unroll
    for (int u = 0; u < EV_HOLD; ++u) v[u] = (uint64_t)u < e.nch ? e.load(u) : ev_f4{NAN, NAN, NAN, NAN};
    for (uint32_t k = tid; k < EV_KEYS / 4; k += EV_THREADS)
        ((uint4 *)sh.hist)[k] = make_uint4(0u, 0u, 0u, 0u);
    float lo = INFINITY, hi = -INFINITY;
    ev_each<EV_HOLD>(
        e, v,
        [&](float x, int) {
            lo = fminf(lo, x);
            hi = fmaxf(hi, x);
        },
        [](uint64_t) {});
    {
        st_wave_minmax(lo, hi);
        if (lane == 0) sh.redu[wv] = (uint64_t)__float_as_uint(hi) << 32 | __float_as_uint(lo);
        __syncthreads();
        lo = INFINITY;
        hi = -INFINITY;
#pragma unroll
        for (int i = 0; i < EV_WAVES; ++i) {
            lo = fminf(lo, __uint_as_float((uint32_t)sh.redu[i]));
            hi = fmaxf(hi, __uint_as_float((uint32_t)(sh.redu[i] >> 32)));
        }
    }
    if (!(isfinite(lo) && isfinite(hi))) {
        /* no histogram over non-finite scores */
        no_fit();
        return;
    }

    const uint64_t khi = ev_map(e, a, lo, hi);

    /* 2-4. histogram points and their least squares */
    if (khi >= EV_KEYS) {
        __syncthreads(); /* redu is written again */
        ev_wide((const __attribute__((address_space(4))) void *)__builtin_amdgcn_kernarg_segment_ptr(), sh, s, lo, hi);
        return;
    }
    EvSums acc{};
    uint64_t next = 0;
    ev_window<true>(e, sh, v, 0, khi, acc, next);
    ev_solve(a, sh, s, e.x0, acc);
}

/* Statistics.hs:41: E = 10 ** (alpha + beta * (score / 10000)) */
__global__ void k_evapply(double *ev, const double *fit, const double *score,
                          const uint32_t *cnt, uint32_t N, uint32_t S)
{
    const uint64_t m = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= (uint64_t)N * S) return;
    const uint32_t s = (uint32_t)(m / N), k = (uint32_t)(m % N);
    if (cnt && k >= cnt[s]) {
        ev[m] = 0.0;
        return;
    }
    ev[m] = pow(10.0, fit[2 * s] + fit[2 * s + 1] * (score[m] / 10000.0));
}

/* ------------------------------------------------------------------ */
/* SP ions                                                               */
/* ------------------------------------------------------------------ */

struct SpShared {
    float xs[SP_CACHE];
    uint32_t flags[SP_WORDS];
    uint32_t redu[ST_WAVES];
};

/* positive values by their bits (order preserving), the rest as 0 */
__device__ __forceinline__ uint32_t sp_key(float v) { return v > 0.0f ? __float_as_uint(v) : 0u; }

/* extractPeaks (IonSeries.hs:99-107) of one spectrum per workgroup: bit t of
 * the W flag words set where bin t = i div 3 holds one of the 200 largest
 * values and that value is above zero.  Ties at the 200th value keep the
 * lowest positions. */
__global__ __launch_bounds__(ST_THREADS) void k_sp_peaks(uint32_t *on, uint32_t W, hfx_spectra sp)
{
    __shared__ SpShared sh;
    const uint32_t s = blockIdx.x, tid = threadIdx.x;
    const uint32_t L = min(sp.d_len[s], sp.x_stride);
    const float *row = sp.d_x + (size_t)s * sp.x_stride;
    const bool cached = L <= SP_CACHE;
    if (cached)
        for (uint32_t i = tid; i < L; i += ST_THREADS) sh.xs[i] = row[i];
    for (uint32_t k = tid; k < W; k += ST_THREADS) sh.flags[k] = 0;
    __syncthreads();
    const float *src = cached ? sh.xs : row;

    uint32_t P = 0;
    for (uint32_t i = tid; i < L; i += ST_THREADS) P += src[i] > 0.0f;
    P = st_block_sum(P, sh.redu);

    if (P > SP_TOP) {
        /* T = key of the 200th largest value: the largest T with
         * #{key >= T} >= 200, bit by bit from the top */
        uint32_t T = 0;
        for (int bit = 30; bit >= 0; --bit) {
            const uint32_t cand = T | (1u << bit);
            uint32_t c = 0;
            for (uint32_t i = tid; i < L; i += ST_THREADS) c += sp_key(src[i]) >= cand;
            c = st_block_sum(c, sh.redu);
            if (c >= SP_TOP) T = cand;
        }
        uint32_t gt = 0;
        for (uint32_t i = tid; i < L; i += ST_THREADS) gt += sp_key(src[i]) > T;
        gt = st_block_sum(gt, sh.redu);
        const uint32_t need = SP_TOP - gt;
        /* ties in position order: contiguous runs per thread */
        const uint32_t per = (L + ST_THREADS - 1) / ST_THREADS;
        const uint32_t i0 = min(L, tid * per), i1 = min(L, i0 + per);
        uint32_t ties = 0;
        for (uint32_t i = i0; i < i1; ++i) ties += sp_key(src[i]) == T;
        uint32_t rank = st_block_excl_scan(ties, sh.redu);
        for (uint32_t i = i0; i < i1; ++i) {
            const uint32_t k = sp_key(src[i]);
            const bool sel = k > T || (k == T && rank++ < need);
            if (sel) atomicOr(&sh.flags[(i / 3) >> 5], 1u << ((i / 3) & 31));
        }
    } else {
        for (uint32_t i = tid; i < L; i += ST_THREADS)
            if (src[i] > 0.0f) atomicOr(&sh.flags[(i / 3) >> 5], 1u << ((i / 3) & 31));
    }
    __syncthreads();
    for (uint32_t k = tid; k < W; k += ST_THREADS) on[(size_t)s * W + k] = sh.flags[k];
}

#define SPW_MAXE 48                                          /* values per lane */
#define SPW_WORDS ((SPW_MAXE * HFX_WAVE / 3 + 1 + 31) / 32)     /* 33 flag words  */

/* k_sp_peaks' flags for a row of L <= E * 64 values (E <= SPW_MAXE, a multiple
 * of 4) by one wave: the row in registers (values 4 q .. 4 q + 3 of a lane are
 * positions 256 q + 4 lane + 0 .. 3, 0 past the row, which no count sees), every
 * count a ballot.  The 200th value is found bit by bit; once 64 values or fewer
 * share its leading bits -- a dozen steps, where a spectrum's largest value and
 * its 200th differ by a few octaves -- those go one to a lane, and a step is one
 * ballot instead of E.  fw: the wave's flag words, clear; u: 64 words of LDS. */
template <int E>
__device__ __forceinline__ void sp_flags(uint32_t *fw, uint32_t *u, const float *row, uint32_t L)
{
    const uint32_t lane = hfx_lane();
    uint32_t kv[E];
#pragma unroll
    for (int q = 0; q < E / 4; ++q) {
        const uint32_t i = 4 * (HFX_WAVE * q + lane);
        ev_f4 t = {0.0f, 0.0f, 0.0f, 0.0f};
        if (i + 4 <= L) t = *(const ev_f4 *)(row + i);
        else if (i < L)
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (i + e < L) t[e] = row[i + e];
#pragma unroll
        for (int e = 0; e < 4; ++e) kv[4 * q + e] = __float_as_uint(t[e]);
    }
    uint32_t P = 0, top = 0;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        kv[j] = sp_key(__uint_as_float(kv[j]));
        P += __popcll(__builtin_amdgcn_ballot_w64(kv[j] != 0));
        top = max(top, kv[j]);
    }
    uint32_t T = 1, need = 0, eq = 0; /* all positive values */
    if (P > SP_TOP) {
#pragma unroll
        for (int m = 1; m < HFX_WAVE; m <<= 1) top = max(top, (uint32_t)__shfl_xor((int)top, m, 64));
        top = __builtin_amdgcn_readfirstlane(top);
        /* T: the largest with ge = #{key >= T} >= 200; hi = #{key >= T + 2^(bit + 1)} */
        T = 0;
        uint32_t ge = P, hi = 0;
        int bit = 31 - __builtin_clz(top);
        for (; bit >= 0 && ge - hi > HFX_WAVE; --bit) {
            const uint32_t cand = T | (1u << bit);
            uint32_t c = 0;
#pragma unroll
            for (int j = 0; j < E; ++j) c += __popcll(__builtin_amdgcn_ballot_w64(kv[j] >= cand));
            if (c >= SP_TOP) {
                T = cand;
                ge = c;
            } else {
                hi = c;
            }
        }
        if (bit >= 0) {
            /* the ge - hi <= 64 keys of [T, T + 2^(bit + 1)), one to a lane */
            const uint32_t end = T + (2u << bit), lo = max(T, 1u);
            const uint64_t below = __lanemask_lt();
            uint32_t at = 0;
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const bool in = kv[j] >= lo && kv[j] < end;
                const uint64_t m = __builtin_amdgcn_ballot_w64(in);
                if (in) u[at + (uint32_t)__popcll(m & below)] = kv[j];
                at += (uint32_t)__popcll(m);
            }
            hfx_wave_sync();
            const uint32_t w = lane < at ? u[lane] : 0u;
            for (; bit >= 0; --bit) {
                const uint32_t cand = T | (1u << bit);
                const uint32_t c = hi + (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(w >= cand));
                if (c >= SP_TOP) {
                    T = cand;
                    ge = c;
                }
            }
            eq = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(w == T));
        } else {
            eq = ge - hi; /* of [T, T + 1) */
        }
        need = SP_TOP - (ge - eq);
    }
    auto flag = [&](int q, int e) {
        const uint32_t t = (4 * (HFX_WAVE * q + lane) + e) / 3;
        atomicOr(&fw[t >> 5], 1u << (t & 31));
    };
    if (need == eq) {
#pragma unroll
        for (int j = 0; j < E; ++j)
            if (kv[j] >= T) flag(j / 4, j % 4);
    } else {
        /* ties of T past the 200: the lowest positions */
        const uint64_t below = __lanemask_lt();
        uint32_t base = 0;
#pragma unroll
        for (int q = 0; q < E / 4; ++q) {
            uint32_t before = base;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint64_t m = __builtin_amdgcn_ballot_w64(kv[4 * q + e] == T);
                before += (uint32_t)__popcll(m & below);
                base += (uint32_t)__popcll(m);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t k = kv[4 * q + e];
                if (k > T || (k == T && before < need)) flag(q, e);
                before += k == T;
            }
        }
    }
    hfx_wave_sync();
}

template <int E>
__global__ __launch_bounds__(ST_THREADS) void k_sp_peaks_w(uint32_t *on, uint32_t W,
                                                            hfx_spectra sp)
{
    __shared__ uint32_t words[ST_WAVES * SPW_WORDS], und[ST_THREADS];
    const uint32_t wv = threadIdx.x / HFX_WAVE, lane = threadIdx.x % HFX_WAVE;
    const uint32_t s = blockIdx.x * ST_WAVES + wv;
    if (s >= sp.num_spec) return;
    uint32_t *fw = words + wv * SPW_WORDS;
    for (uint32_t k = lane; k < SPW_WORDS; k += HFX_WAVE) fw[k] = 0;
    hfx_wave_sync();
    sp_flags<E>(fw, und + wv * HFX_WAVE, sp.d_x + (size_t)s * sp.x_stride,
                min(min(sp.d_len[s], sp.x_stride), (uint32_t)(E * HFX_WAVE)));
    for (uint32_t k = lane; k < W; k += HFX_WAVE) on[(size_t)s * W + k] = k < SPW_WORDS ? fw[k] : 0u;
}

struct SpArgs {
    uint32_t *nb, *ny, *tot;
    const uint32_t *on;
    uint32_t W;
    float bw;
    hfx_db db;
    const uint32_t *len, *zmax;
    uint32_t stride, num_spec;
};

/* bin = round(v / bin width / 3), halves to even; matched when in range and
 * flagged (IonSeries.hs:142-147) */
__device__ __forceinline__ uint32_t sp_on(const uint32_t *f, uint32_t npk, float v, float bw)
{
    const float q = __builtin_rintf((v / bw) / 3.0f);
    if (!(q >= 0.0f && q < (float)npk)) return 0;
    const uint32_t i = (uint32_t)q;
    return (f[i >> 5] >> (i & 31)) & 1u;
}

/* Matches of a wave, SPM_ROWS at a time: lane i < SPM_ROWS holds match i.  Its
 * lane sums the FP32 ladder (in order, as everywhere) into LDS, SPM_POS positions
 * at a time; then the wave's lanes take one position each, whatever the peptides'
 * lengths.  One thread a match took 70 us for 50,000 of them, most lanes waiting
 * on the residues, masses and flags of the longest. */
#define SPM_ROWS 16
#define SPM_POS 32

struct SpMatch {
    uint32_t tc, n;   /* first residue, residues taken (Location.hs:42-58) */
    uint32_t nz, npk; /* fragment charges, peak bins */
    uint32_t nmod, s;
    float r;
    bool live;
};

struct SpLds {
    float b[SPM_ROWS * SPM_POS];
    uint8_t row[SPM_ROWS * SPM_POS];
    uint32_t first[SPM_ROWS]; /* ladder position of b[0], were it this row's */
    uint32_t n[SPM_ROWS], nz[SPM_ROWS], npk[SPM_ROWS], s[SPM_ROWS];
    float r[SPM_ROWS];
    uint32_t nb[SPM_ROWS], ny[SPM_ROWS];
};

/* peptide p against spectrum s, s < num_spec; live: p < num_pep */
__device__ __forceinline__ SpMatch sp_get(const SpArgs &a, uint32_t p, uint32_t s, uint32_t nmod,
                                          bool live)
{
    SpMatch m{};
    m.live = live;
    if (!live) return m;
    m.tc = a.db.d_tc[p];
    const uint32_t tn = a.db.d_tn[p];
    m.n = (uint64_t)tn < a.db.num_ions ? tn - m.tc + 1 : tn - m.tc;
    m.r = (a.db.d_r[p] + SP_H) + SP_H2O;
    m.npk = min(a.len[s], a.stride) / 3 + 1;
    m.nz = max(a.zmax[s], 1u);
    m.nmod = nmod;
    m.s = s;
    return m;
}

/* lookup + matchIonSequence (IonSeries.hs:136-147) + scoreSP (Match.hs:33-40) of
 * cnt <= SPM_ROWS matches, results to out + i; flags(s) = words of spectrum s */
template <class Flags>
__device__ __forceinline__ void sp_matches(const SpArgs &a, SpLds &w, const float *mtab,
                                           const SpMatch &m, uint32_t cnt, uint64_t out,
                                           Flags &&flags)
{
    const uint32_t lane = hfx_lane();
    const uint32_t n = lane < cnt && m.live ? m.n : 0u;
    if (lane < SPM_ROWS) {
        w.n[lane] = n;
        w.nz[lane] = m.nz;
        w.npk[lane] = m.npk;
        w.s[lane] = m.s;
        w.r[lane] = m.r;
        w.nb[lane] = 0;
        w.ny[lane] = 0;
    }
    uint32_t nmax = lane < SPM_ROWS ? n : 0u;
#pragma unroll
    for (uint32_t o = 1; o < SPM_ROWS; o <<= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o, 64));
    nmax = __builtin_amdgcn_readfirstlane(nmax);
    const uint8_t *res = a.db.d_ions + m.tc;
    float pm = 0.0f;
    for (uint32_t k0 = 0; k0 < nmax; k0 += SPM_POS) {
        const uint32_t cn = n > k0 ? min(n - k0, (uint32_t)SPM_POS) : 0u;
        uint32_t incl = lane < SPM_ROWS ? cn : 0u;
#pragma unroll
        for (uint32_t o = 1; o < SPM_ROWS; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        const uint32_t np = __builtin_amdgcn_readlane(incl, SPM_ROWS - 1);
        if (cn) {
            const uint32_t at = incl - cn;
            w.first[lane] = k0 - at; /* modulo 2^32 */
            for (uint32_t k = 0; k < cn; k += 8) {
                uint32_t x[8];
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) x[j] = res[k0 + min(k + j, cn - 1u)];
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j)
                    if (k + j < cn) {
                        pm = pm + mtab[HFX_ACID_IDX(x[j])];
                        w.b[at + k + j] = pm;
                        w.row[at + k + j] = (uint8_t)lane;
                    }
            }
        }
        hfx_wave_sync();
        for (uint32_t i = lane; i < np; i += HFX_WAVE) {
            const uint32_t q = w.row[i], k = w.first[q] + i, nq = w.n[q], nz = w.nz[q];
            const uint32_t npk = w.npk[q];
            const uint32_t *f = flags(w.s[q]);
            const float b = w.b[i], r = w.r[q];
            uint32_t nb = 0, ny = 0;
            for (uint32_t c = 1; c <= nz; ++c) {
                const float cf = (float)c;
                const float mz = (b + SP_H * cf) / cf;
                if (c < nz || k + 1u < nq) nb += sp_on(f, npk, mz, a.bw);   /* init */
                if (c > 1 || k > 0) ny += sp_on(f, npk, r - mz, a.bw);      /* tail */
            }
            if (nb) atomicAdd(&w.nb[q], nb);
            if (ny) atomicAdd(&w.ny[q], ny);
        }
        hfx_wave_sync();
    }
    hfx_wave_sync();
    if (lane < cnt) {
        a.nb[out + lane] = m.live ? w.nb[lane] : 0u;
        a.ny[out + lane] = m.live ? w.ny[lane] : 0u;
        a.tot[out + lane] = m.live ? (m.n - 1 + m.nmod) * 2 : 0u;
    }
    hfx_wave_sync(); /* the rows are set again by the next matches */
}

__global__ __launch_bounds__(ST_THREADS) void k_sp_list(SpArgs a, const uint32_t *pep,
                                                        const uint32_t *spec, const uint32_t *nmod,
                                                        uint64_t M)
{
    __shared__ SpLds lds[ST_WAVES];
    __shared__ float mtab[32];
    const uint32_t wv = threadIdx.x / HFX_WAVE, lane = hfx_lane();
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? a.db.d_mass[threadIdx.x] : 0.0f;
    __syncthreads();
    const uint64_t m0 = ((uint64_t)blockIdx.x * ST_WAVES + wv) * SPM_ROWS;
    if (m0 >= M) return;
    const uint32_t cnt = (uint32_t)min(M - m0, (uint64_t)SPM_ROWS);
    SpMatch m{};
    if (lane < cnt) {
        const uint32_t p = pep[m0 + lane], s = spec[m0 + lane];
        /* 0xFFFFFFFF: no peptide */
        m = sp_get(a, p, s, nmod ? nmod[m0 + lane] : 0u, p < a.db.num_pep && s < a.num_spec);
    }
    sp_matches(a, lds[wv], mtab, m, cnt, m0, [&](uint32_t s) { return a.on + (size_t)s * a.W; });
}

/* top-N of an unmodified search: entry k of spectrum s is the window
 * position top_pos[s][k] (sorted peptide begin[s] + position) */
struct SpPlainTop {
    const uint32_t *top_pos, *top_cnt, *begin;
    uint32_t N;
    __device__ __forceinline__ SpMatch get(const SpArgs &a, uint32_t s, uint32_t k) const
    {
        const bool live = k < top_cnt[s];
        return sp_get(a, live ? a.db.d_idx_sorted[begin[s] + top_pos[(uint64_t)s * N + k]] : 0u, s, 0u,
                      live);
    }
};

/* top-N of a modified search: entry k of spectrum s is modified peptide
 * mp_off[s] + top_pos[s][k]; matched on its unmodified peptide
 * (Search.hs:296-299), the printed length grows by its modified sites */
struct SpModTop {
    const uint32_t *top_pos, *top_cnt;
    const uint64_t *mp_off;
    uint32_t N;
    hfx_modset ms;
    __device__ __forceinline__ SpMatch get(const SpArgs &a, uint32_t s, uint32_t k) const
    {
        if (k >= top_cnt[s]) return SpMatch{};
        const uint64_t i = mp_off[s] + top_pos[(uint64_t)s * N + k];
        const uint32_t md = ms.d_mpep_mod_idx[i];
        uint32_t nmod = 0;
        for (uint32_t q = 0; q < ms.num_ma; ++q) nmod += ms.d_mod_ma_count[(size_t)md * ms.num_ma + q];
        return sp_get(a, ms.d_mpep_pep_idx[i], s, nmod, true);
    }
};

/* a wave a spectrum: its N matches, the flags of its row found here (E > 0) or
 * read from a.on (E = 0).  10,000 spectra of 2176 bins, top 5: 54 us; in launches of
 * their own the flags take 53 (31 steps of 36 ballots) and the matches 70 (a thread
 * each).  The chains of reads and of select steps bound it: two thirds of the waves'
 * cycles are waits and 36 % of the vector issue is used, 24 waves a CU at most; 64
 * registers for 32 waves spill (61 us). */
template <int E, class Top>
__global__ __launch_bounds__(ST_THREADS) void k_sp_topn(SpArgs a, Top top, const float *x)
{
    __shared__ uint32_t words[ST_WAVES * SPW_WORDS], und[ST_THREADS];
    __shared__ SpLds lds[ST_WAVES];
    __shared__ float mtab[32];
    const uint32_t wv = threadIdx.x / HFX_WAVE, lane = hfx_lane();
    const uint32_t s = blockIdx.x * ST_WAVES + wv;
    uint32_t *fw = words + wv * SPW_WORDS;
    if constexpr (E > 0)
        for (uint32_t k = lane; k < SPW_WORDS; k += HFX_WAVE) fw[k] = 0;
    if (threadIdx.x < 32) mtab[threadIdx.x] = threadIdx.x < 26 ? a.db.d_mass[threadIdx.x] : 0.0f;
    __syncthreads();
    if (s >= a.num_spec) return;
    /* the first matches' chain of reads starts before the row's */
    SpMatch m{};
    if (lane < min(top.N, (uint32_t)SPM_ROWS)) m = top.get(a, s, lane);
    if constexpr (E > 0)
        sp_flags<E>(fw, und + wv * HFX_WAVE, x + (size_t)s * a.stride,
                    min(min(a.len[s], a.stride), (uint32_t)(E * HFX_WAVE)));
    for (uint32_t k = 0; k < top.N; k += SPM_ROWS) {
        const uint32_t cnt = min(top.N - k, (uint32_t)SPM_ROWS);
        if (k && lane < cnt) m = top.get(a, s, k + lane);
        sp_matches(a, lds[wv], mtab, m, cnt, (uint64_t)s * top.N + k, [&](uint32_t) {
            return E > 0 ? (const uint32_t *)fw : a.on + (size_t)s * a.W;
        });
    }
}

/* ------------------------------------------------------------------ */
/* Host                                                                  */
/* ------------------------------------------------------------------ */

extern "C" int hfx_evalue_fit(hfx_ctx *ctx, double *d_fit, uint32_t *d_npts, uint64_t *d_nused,
                              const float *d_scores_a, const uint64_t *d_off_a,
                              const float *d_scores_b, const uint64_t *d_off_b,
                              uint32_t num_spec, uint32_t bin_width, float cutoff_perc,
                              void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_fit && d_off_a && d_scores_a, HFX_ERR_ARG, "hfx_evalue_fit: null argument");
    HFX_REQUIRE(!d_scores_b == !d_off_b, HFX_ERR_ARG,
                "hfx_evalue_fit: second score set needs both scores and offsets");
    HFX_REQUIRE(bin_width >= 1, HFX_ERR_ARG, "hfx_evalue_fit: bin width 0");
    HFX_REQUIRE(cutoff_perc >= 0.0f && cutoff_perc <= 100.0f, HFX_ERR_ARG,
                "hfx_evalue_fit: cut-off percentage %g outside [0, 100]", (double)cutoff_perc);
    if (num_spec == 0) return HFX_OK;
    EvArgs a{d_fit, d_npts, d_nused, d_scores_a, d_off_a, d_scores_b, d_off_b,
             (double)bin_width, 1.0 / bin_width,
             fmax(floor(4000.0 / bin_width) - 1.0, 0.0), cutoff_perc};
    hipLaunchKernelGGL(k_evfit, dim3(num_spec), dim3(EV_THREADS), 0, hfx_stream(stream), a);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

extern "C" int hfx_evalues(hfx_ctx *ctx, double *d_ev, const double *d_fit,
                           const double *d_score, const uint32_t *d_cnt, uint32_t N,
                           uint32_t num_spec, void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_ev && d_fit && d_score, HFX_ERR_ARG, "hfx_evalues: null argument");
    const uint64_t M = (uint64_t)N * num_spec;
    if (M == 0) return HFX_OK;
    hipLaunchKernelGGL(k_evapply, dim3((unsigned)((M + 255) / 256)), dim3(256), 0,
                       hfx_stream(stream), d_ev, d_fit, d_score, d_cnt, N, num_spec);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

extern "C" uint32_t hfx_sp_peak_words(uint32_t x_stride) { return (x_stride / 3 + 1 + 31) / 32; }

/* run(values per lane) for rows that a wave holds; 0 for longer ones */
template <class F>
static int sp_rows(const hfx_spectra *sp, F &&run)
{
    const uint32_t rows = (sp->x_stride + HFX_WAVE - 1) / HFX_WAVE;
    if (rows <= 12) return run(std::integral_constant<int, 12>{});
    if (rows <= 24) return run(std::integral_constant<int, 24>{});
    if (rows <= 36) return run(std::integral_constant<int, 36>{});
    if (rows <= SPW_MAXE) return run(std::integral_constant<int, SPW_MAXE>{});
    return 0;
}

extern "C" int hfx_sp_peaks(hfx_ctx *ctx, uint32_t *d_on, uint32_t words, const hfx_spectra *sp,
                            void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_on && sp, HFX_ERR_ARG, "hfx_sp_peaks: null argument");
    HFX_REQUIRE(words >= hfx_sp_peak_words(sp->x_stride), HFX_ERR_ARG,
                "hfx_sp_peaks: %u flag words < %u for stride %u", words,
                hfx_sp_peak_words(sp->x_stride), sp->x_stride);
    HFX_REQUIRE(hfx_sp_peak_words(sp->x_stride) <= SP_WORDS, HFX_ERR_ARG,
                "hfx_sp_peaks: spectrum stride %u above %u", sp->x_stride,
                3u * (32u * SP_WORDS - 1u) + 2u);
    if (sp->num_spec == 0) return HFX_OK;
    const dim3 gw((sp->num_spec + ST_WAVES - 1) / ST_WAVES);
    const int rc = sp_rows(sp, [&](auto e) {
        hipLaunchKernelGGL(k_sp_peaks_w<decltype(e)::value>, gw, dim3(ST_THREADS), 0,
                           hfx_stream(stream), d_on, words, *sp);
        return 1;
    });
    if (!rc)
        hipLaunchKernelGGL(k_sp_peaks, dim3(sp->num_spec), dim3(ST_THREADS), 0, hfx_stream(stream),
                           d_on, words, *sp);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

static int sp_args(SpArgs &a, uint32_t *d_nb, uint32_t *d_ny, uint32_t *d_total,
                   const uint32_t *d_on, uint32_t words, const hfx_db *db, const hfx_spectra *sp,
                   int mono)
{
    HFX_REQUIRE(d_nb && d_ny && d_total && d_on && db && sp, HFX_ERR_ARG,
                "hfx_sp_ions: null argument");
    HFX_REQUIRE(words >= hfx_sp_peak_words(sp->x_stride), HFX_ERR_ARG,
                "hfx_sp_ions: %u flag words < %u", words, hfx_sp_peak_words(sp->x_stride));
    a.nb = d_nb;
    a.ny = d_ny;
    a.tot = d_total;
    a.on = d_on;
    a.W = words;
    a.bw = mono ? HFX_BIN_WIDTH_MONO : HFX_BIN_WIDTH_AVG; /* Correlation.hs:29-30 */
    a.db = *db;
    a.len = sp->d_len;
    a.zmax = sp->d_zmax;
    a.stride = sp->x_stride;
    a.num_spec = sp->num_spec;
    return HFX_OK;
}

extern "C" int hfx_sp_ions(hfx_ctx *ctx, uint32_t *d_nb, uint32_t *d_ny, uint32_t *d_total,
                           const uint32_t *d_pep, const uint32_t *d_spec, const uint32_t *d_nmod,
                           uint64_t num_match, const uint32_t *d_on, uint32_t words,
                           const hfx_db *db, const hfx_spectra *sp, int mono, void *stream)
{
    (void)ctx;
    SpArgs a;
    int rc = sp_args(a, d_nb, d_ny, d_total, d_on, words, db, sp, mono);
    if (rc) return rc;
    HFX_REQUIRE(d_pep && d_spec, HFX_ERR_ARG, "hfx_sp_ions: null match list");
    if (num_match == 0) return HFX_OK;
    const uint64_t per = (uint64_t)ST_WAVES * SPM_ROWS;
    hipLaunchKernelGGL(k_sp_list, dim3((unsigned)((num_match + per - 1) / per)), dim3(ST_THREADS), 0,
                       hfx_stream(stream), a, d_pep, d_spec, d_nmod, num_match);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* the matches of every spectrum's top N: rows that a wave holds in one launch
 * without scratch, longer ones through their flags in scratch */
template <class Top>
static int sp_topn(hfx_ctx *ctx, uint32_t *d_nb, uint32_t *d_ny, uint32_t *d_total, const Top &top,
                   const hfx_db *db, const hfx_spectra *sp, int mono, void *stream)
{
    HFX_REQUIRE(ctx, HFX_ERR_ARG, "hfx_sp_ions_topn: null argument");
    const uint32_t W = hfx_sp_peak_words(sp->x_stride);
    HFX_REQUIRE(W <= SP_WORDS, HFX_ERR_ARG, "hfx_sp_ions_topn: spectrum stride %u above %u",
                sp->x_stride, 3u * (32u * SP_WORDS - 1u) + 2u);
    const dim3 g((sp->num_spec + ST_WAVES - 1) / ST_WAVES), t(ST_THREADS);
    SpArgs a;
    /* any non-null flags: not read where the kernel finds them */
    int rc = sp_args(a, d_nb, d_ny, d_total, (const uint32_t *)sp, W, db, sp, mono);
    if (rc) return rc;
    if (top.N == 0 || sp->num_spec == 0) return HFX_OK;
    if (!sp_rows(sp, [&](auto e) {
            a.on = nullptr;
            hipLaunchKernelGGL((k_sp_topn<decltype(e)::value, Top>), g, t, 0, hfx_stream(stream), a,
                               top, sp->d_x);
            return 1;
        })) {
        void *p = nullptr;
        rc = hfx_ctx_scratch(ctx, HFX_SLOT_STATS, (size_t)4 * W * sp->num_spec, &p);
        if (rc) return rc;
        rc = hfx_sp_peaks(ctx, (uint32_t *)p, W, sp, stream);
        if (rc) return rc;
        a.on = (const uint32_t *)p;
        hipLaunchKernelGGL((k_sp_topn<0, Top>), g, t, 0, hfx_stream(stream), a, top, sp->d_x);
    }
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

extern "C" int hfx_sp_ions_topn(hfx_ctx *ctx, uint32_t *d_nb, uint32_t *d_ny, uint32_t *d_total,
                                const uint32_t *d_top_pos, const uint32_t *d_top_cnt,
                                const uint32_t *d_begin, uint32_t N, const hfx_db *db,
                                const hfx_spectra *sp, int mono, void *stream)
{
    HFX_REQUIRE(d_top_pos && d_top_cnt && d_begin && db && sp, HFX_ERR_ARG,
                "hfx_sp_ions_topn: null argument");
    return sp_topn(ctx, d_nb, d_ny, d_total, SpPlainTop{d_top_pos, d_top_cnt, d_begin, N}, db, sp, mono,
                   stream);
}

extern "C" int hfx_sp_ions_topn_mod(hfx_ctx *ctx, uint32_t *d_nb, uint32_t *d_ny,
                                    uint32_t *d_total, const uint32_t *d_top_pos,
                                    const uint32_t *d_top_cnt, const uint64_t *d_mp_off,
                                    uint32_t N, const hfx_modset *ms, const hfx_db *db,
                                    const hfx_spectra *sp, int mono, void *stream)
{
    HFX_REQUIRE(d_top_pos && d_top_cnt && d_mp_off && ms && db && sp, HFX_ERR_ARG,
                "hfx_sp_ions_topn_mod: null argument");
    return sp_topn(ctx, d_nb, d_ny, d_total, SpModTop{d_top_pos, d_top_cnt, d_mp_off, N, *ms}, db, sp,
                   mono, stream);
}
