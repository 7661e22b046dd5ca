/*
 * hfx_preprocess.hip -- fast-XCorr spectrum preprocessing on the GPU.
 *
 * Restates Correlation.hs:37-109 (sequestXCorr = crossCorrolation .
 * normaliseByRegion . observedIntensity), one workgroup per spectrum, the
 * whole spectrum resident in LDS:
 *   1. observedIntensity (:57-71): len = 75 + ceiling(min(50 + pcr*z,
 *      trunc(last_mz/10)*10)); peaks with mz <= cutoff (outside pcr +- 15 when
 *      removing the precursor) binned with rint(mz / bin width), max sqrt(I)
 *      per bin (LDS atomicMax on the bit pattern: values are >= 0).
 *   2. normaliseByRegion (:84-96): 10 regions of sel = (len-75) div 10 bins,
 *      50 * e / region max (max > 1e-6 and i < 10*sel), else 0.  A region's
 *      maximum is that of its peaks, taken while they are binned.
 *   3. crossCorrolation (:105-109): x_i = e_i - sum(a[max(0,i-75) .. +150]) / 150,
 *      the 151-bin window summed left to right in FP32 (mean_mode 0, the
 *      reference's foldl') or in FP64 (mean_mode 1).
 *
 * In FP64 the window sums are differences of the bins' prefix sums, as long as
 * every non-zero a is at least 2^-13 (its square at least 6e-12 of its region's
 * largest intensity) and all of them add up to less than 2^17 (2,621 bins at the
 * largest value, 50): those sums are exact in any order.
 * Otherwise, and in FP32, they run over the bins that hold a peak only: a is nowhere
 * negative, so the zeros between them leave a left-to-right sum unchanged to
 * the last bit, and a spectrum of a few hundred peaks over 2,000 bins has about
 * 13 of them in a window of 151.  The non-zero values are compacted in bin
 * order (one 64-bit mask a 64-bin chunk, and the chunks' running counts), so
 * that a window is a contiguous run of that list whose ends are two population
 * counts.
 * 20,000 spectra of 167 peaks: 1,075 us with 151 LDS reads and additions a bin,
 * 181 over the peaks only, 109 with the prefix sums (170 MB written, 1.6 TB/s).
 * The vector instructions of a bin (scaling, scan, FP64 division) bound it: 1.1 a
 * SIMD every four cycles, the most measured in any kernel here.
 */
#include "hfx_common.h"

#define PP_THREADS 256
#define PP_WAVES (PP_THREADS / HFX_WAVE)
#define PP_CHUNKS (HFX_MAX_LEN / HFX_WAVE)
static_assert(PP_CHUNKS <= HFX_WAVE, "one lane a chunk in the scan of counts");

/* dynamic LDS: the bins (ceil(cap / 64) * 64 words) and the list of non-zero
 * values (as many), or one FP64 prefix sum a bin and the last; cap = the longest
 * spectrum the stride allows */
static size_t pp_lds_bytes(uint32_t stride)
{
    const uint32_t cap = min(stride, (uint32_t)HFX_MAX_LEN);
    return 2 * (size_t)((cap + HFX_WAVE - 1) / HFX_WAVE) * HFX_WAVE * 4 + 8;
}

/* inclusive prefix sum over the wave by lane moves: rows of 16 by shifts of 1,
 * 2, 4 and 8, then across rows */
template <int CTRL, int ROWS>
__device__ __forceinline__ double pp_step(double x)
{
    const uint64_t v = __double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS,
                                                              0xf, false);
    return x + __longlong_as_double((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double pp_wave_incl(double x)
{
    x = pp_step<0x111, 0xf>(x);
    x = pp_step<0x112, 0xf>(x);
    x = pp_step<0x114, 0xf>(x);
    x = pp_step<0x118, 0xf>(x);
    x = pp_step<0x142, 0xa>(x);
    x = pp_step<0x143, 0xc>(x);
    return x;
}
/* lane l's value (l uniform) */
__device__ __forceinline__ double pp_take(double x, uint32_t l)
{
    const uint64_t v = __double_as_longlong(x);
    return __longlong_as_double(
        (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), (int)l) << 32 |
        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)l));
}

/* sum of list[a .. e) in order, as T */
template <class T>
__device__ __forceinline__ T pp_sum(const float *list, uint32_t a, uint32_t e)
{
    T sum = 0;
    for (uint32_t k = a; k < e; ++k) sum = sum + (T)list[k];
    return sum;
}

/* PER: chunks of a wave, for the longest spectrum the stride allows */
template <uint32_t PER>
__global__ void __launch_bounds__(PP_THREADS, PER <= 9 ? 8 : 6)
    k_preprocess(float *x, uint32_t stride, uint32_t *len_out, uint32_t *status, const float *mz,
                 const float *inten, const uint32_t *off, const float *pcr_a, const float *chg_a,
                 int remove_precursor, float bw, int mean_mode)
{
    extern __shared__ __align__(16) uint32_t sbin[];
    __shared__ uint32_t rmax[11];
    __shared__ uint64_t mask[PP_CHUNKS + 1];
    __shared__ uint32_t pre[PP_CHUNKS + 1];
    __shared__ double tot[PP_CHUNKS];
    __shared__ uint32_t sh_odd;
    const uint32_t s = blockIdx.x, t = threadIdx.x, lane = hfx_lane(), wave = t / HFX_WAVE;
    const uint32_t p0 = off[s], p1 = off[s + 1];
    float *xs = x + (size_t)s * stride;
    const float pcr = pcr_a[s], chg = chg_a[s];
    uint32_t st = 0, len = 0;
    if (p1 <= p0) {
        st = 1;
    } else {
        const float mzcut = 50.0f + pcr * chg;
        const float q = mz[p1 - 1] / 10.0f;
        const float mzlim = (float)((int64_t)__builtin_truncf(q) * 10);
        const float cutoff = (mzcut <= mzlim) ? mzcut : mzlim; /* Haskell min */
        const float lenf = 75.0f + __builtin_ceilf(cutoff);
        if (!(lenf >= 1.0f) || lenf > (float)min(stride, (uint32_t)HFX_MAX_LEN)) {
            st = 3;
        } else {
            len = (uint32_t)lenf;
            if (len < 85) st = 2; /* sel = (len-75) div 10 <= 0 */
        }
        if (st == 0) {
            const uint32_t nch = (len + HFX_WAVE - 1) / HFX_WAVE;
            float *list = (float *)(sbin + nch * HFX_WAVE);
            for (uint32_t i = t; i < nch * HFX_WAVE; i += PP_THREADS) sbin[i] = 0;
            if (t < 11) rmax[t] = 0;
            if (t == 0) sh_odd = 0;
            __syncthreads();
            const uint32_t sel = (len - 75) / 10;
            /* bin / sel: a bin and a half lies 1 / (2 sel) from the next quotient */
            const float rsel = 1.0f / (float)sel;
            auto region = [&](uint32_t b) { return min(10u, (uint32_t)(((float)b + 0.5f) * rsel)); };
            const float plo = pcr - 15.0f, phi = pcr + 15.0f;
            for (uint32_t p = p0 + t; p < p1; p += PP_THREADS) {
                const float m = mz[p];
                const bool keep = remove_precursor ? (m <= cutoff && (m <= plo || phi <= m))
                                                   : (m <= cutoff);
                if (keep) {
                    const int32_t b = (int32_t)__builtin_rintf(m / bw);
                    const uint32_t v = __float_as_uint(__builtin_sqrtf(inten[p])) & 0x7fffffffu;
                    if (b >= 0 && (uint32_t)b < len) {
                        atomicMax(&sbin[b], v);
                        atomicMax(&rmax[region((uint32_t)b)], v);
                    }
                }
            }
            __syncthreads();
            /* each bin scaled: 50 e / (the region's largest) */
            auto scaled = [&](uint32_t i) -> float {
                const uint32_t v = sbin[i];
                if (v == 0u) return 0.0f;
                const float m = __uint_as_float(rmax[region(i)]);
                return (m > 1e-6f && i < sel * 10) ? 50.0f * (__uint_as_float(v) / m) : 0.0f;
            };
            float av[PER];
            bool whole = false;
            if (mean_mode != 0) {
                /* Where every value is 0 or in [2^-13, 64), sums below 2^17 of them
                 * are exact in FP64 (multiples of 2^-36): the windows are
                 * differences of prefix sums, in any order the same bits. */
                double ex[PER];
                bool ok = true;
#pragma unroll
                for (uint32_t q = 0; q < PER; ++q) {
                    const uint32_t c = wave + q * PP_WAVES;
                    av[q] = 0.0f;
                    ex[q] = 0.0;
                    if (c < nch) {
                        const float a = scaled(c * HFX_WAVE + lane);
                        ok = ok && (a == 0.0f || (a >= 0x1p-13f && a < 64.0f));
                        const double incl = pp_wave_incl((double)a);
                        av[q] = a;
                        ex[q] = incl - (double)a;
                        if (lane == HFX_WAVE - 1) tot[c] = incl;
                    }
                }
                if (__ballot(!ok) && lane == 0) sh_odd = 1;
                __syncthreads(); /* the bins have been read: their prefix sums may take their place */
                const double mine = lane < nch ? tot[lane] : 0.0;
                const double run = pp_wave_incl(mine);
                whole = sh_odd == 0 && pp_take(run, nch - 1) < 0x1p17;
                if (whole) {
                    double *pb = (double *)sbin; /* sums of the bins below i <= nch * 64 */
#pragma unroll
                    for (uint32_t q = 0; q < PER; ++q) {
                        const uint32_t c = wave + q * PP_WAVES;
                        if (c < nch)
                            pb[c * HFX_WAVE + lane] = ex[q] + pp_take(run - mine, c);
                    }
                    if (t == 0) pb[nch * HFX_WAVE] = pp_take(run, nch - 1);
                    __syncthreads();
#pragma unroll
                    for (uint32_t q = 0; q < PER; ++q) {
                        const uint32_t i = (wave + q * PP_WAVES) * HFX_WAVE + lane;
                        if (i < len) {
                            const uint32_t w0 = i >= 75 ? i - 75 : 0;
                            xs[i] = (float)((double)av[q] - (pb[min(len, w0 + 151)] - pb[w0]) / 150.0);
                        }
                    }
                } else {
#pragma unroll
                    for (uint32_t q = 0; q < PER; ++q) {
                        const uint32_t c = wave + q * PP_WAVES;
                        if (c < nch) sbin[c * HFX_WAVE + lane] = __float_as_uint(av[q]);
                    }
                }
            }
            if (!whole) {
                for (uint32_t c = wave; c < nch; c += PP_WAVES) {
                    const uint32_t i = c * HFX_WAVE + lane;
                    const float a = mean_mode != 0 ? __uint_as_float(sbin[i]) : scaled(i);
                    sbin[i] = __float_as_uint(a);
                    const uint64_t nz = __ballot(a != 0.0f);
                    if (lane == 0) mask[c] = nz;
                }
                __syncthreads();
                /* non-zero bins before each chunk */
                if (wave == 0) {
                    const uint32_t n = lane < nch ? (uint32_t)__builtin_popcountll(mask[lane]) : 0u;
                    uint32_t incl = n;
    #pragma unroll
                    for (uint32_t o = 1; o < HFX_WAVE; o <<= 1) {
                        const uint32_t y = __shfl_up(incl, o, 64);
                        if (lane >= o) incl += y;
                    }
                    pre[lane] = incl - n;
                    if (lane == HFX_WAVE - 1) pre[HFX_WAVE] = incl;
                    if (lane == 0) mask[nch] = 0;
                }
                __syncthreads();
                /* non-zero bins below bin i (i <= nch * 64) */
                auto below = [&](uint32_t i) -> uint32_t {
                    const uint64_t m = mask[i / HFX_WAVE] & ((1ull << (i % HFX_WAVE)) - 1ull);
                    return pre[i / HFX_WAVE] + (uint32_t)__builtin_popcountll(m);
                };
                for (uint32_t c = wave; c < nch; c += PP_WAVES) {
                    const uint32_t i = c * HFX_WAVE + lane;
                    if ((mask[c] >> lane) & 1ull) list[below(i)] = __uint_as_float(sbin[i]);
                }
                __syncthreads();
                for (uint32_t i = t; i < len; i += PP_THREADS) {
                    const uint32_t w0 = i >= 75 ? i - 75 : 0;
                    const uint32_t k0 = below(w0), k1 = below(min(len, w0 + 151));
                    const float a = __uint_as_float(sbin[i]);
                    if (mean_mode == 0) xs[i] = a - pp_sum<float>(list, k0, k1) / 150.0f;
                    else xs[i] = (float)((double)a - pp_sum<double>(list, k0, k1) / 150.0);
                }
            }
        }
    }
    for (uint32_t i = len + t; i < stride; i += PP_THREADS) xs[i] = 0.0f;
    if (t == 0) {
        len_out[s] = len;
        status[s] = st;
    }
}

extern "C" int hfx_preprocess(hfx_ctx *ctx, float *d_x, uint32_t x_stride, uint32_t *d_len,
                              uint32_t *d_status, const float *d_mz, const float *d_int,
                              const uint32_t *d_peak_off, const float *d_pcr, const float *d_charge,
                              uint32_t num_spec, int remove_precursor, int mono, int mean_mode,
                              void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_x && d_len && d_status && d_peak_off && d_pcr && d_charge, HFX_ERR_ARG,
                "hfx_preprocess: null argument");
    HFX_REQUIRE(mean_mode == 0 || mean_mode == 1, HFX_ERR_ARG, "hfx_preprocess: mean_mode %d",
                mean_mode);
    if (num_spec == 0) return HFX_OK;
    const float bw = mono ? HFX_BIN_WIDTH_MONO : HFX_BIN_WIDTH_AVG;
    const uint32_t cap = min(x_stride, (uint32_t)HFX_MAX_LEN);
    constexpr uint32_t SHORT = 9, LONG = PP_CHUNKS / PP_WAVES; /* up to 2304, 4096 bins */
    hipLaunchKernelGGL(cap <= SHORT * PP_THREADS ? k_preprocess<SHORT> : k_preprocess<LONG>,
                       dim3(num_spec), dim3(PP_THREADS), pp_lds_bytes(x_stride),
                       hfx_stream(stream), d_x, x_stride, d_len, d_status, d_mz, d_int, d_peak_off,
                       d_pcr, d_charge, remove_precursor, bw, mean_mode);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}
