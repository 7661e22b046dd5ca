/*
 * hfx_rows.hip -- theoretical spectra as rows of 2-bit codes in HBM, and their
 * contraction with blocks of spectra on the MFMA units.
 *
 * A candidate's theoretical spectrum depends only on its peptide and the
 * fragment charge level, and a peptide is a candidate of every spectrum whose
 * window holds it (hundreds, in a batch of thousands).  Its row is therefore
 * written once -- per database for the batched forms (kept by the peptide
 * index), per call for hfx_xcorr_sparse -- and every block of spectra then
 * reads finished rows: the inner loop of the contraction is loads, code lookups
 * and matrix instructions, with no ladder, no bins, no LDS atomics and no
 * barrier.
 *
 * Rows.  Sixteen consecutive residual-sorted peptides form a tile, the M of a
 * 16x16 matrix instruction.  A tile is up to RW_G groups of 256 bins, 1 KiB
 * each: lane (row, kg) of a wave owns 16 bytes of a group, word i holding the
 * codes of bins 64 i + 16 kg .. + 15 of the group, so a wave reads a group of
 * a tile with one 16-byte load a lane, contiguous.  Nibble n of a word holds bin
 * n in bits 0-1 and bin n + 8 in bits 2-3.  Codes 0, 1, 3, 2 stand for the
 * weights 0, 10, 25, 50 (two bits of the unary code that orders them in the
 * LDS map).  Four v_perm turn a word into 16 int8 weights in the order
 * rw_bin_of gives; the spectra's planes are stored in the same order.
 *
 * Spectra.  Precision forms (see hfx_dense.hip for their bounds):
 *   RW_I8X3  three balanced base-256 digits of X = rint(x 2^k),
 *            max|x| 2^k <= 8355711; a block is sixteen spectra;
 *   RW_I8X6  six digits, max|x| in [2^45, 2^46) of the last one's unit, for the FP32
 *            forms: they hold every FP32 value from max|x| 2^-22 up with all of
 *            its 24 bits, so that the sums are exact and a score is rounded once.  A
 *            spectrum with a value that they do not hold (smaller, and not a
 *            multiple of the unit; or not finite) keeps the packed kernel.  A column of the
 *            matrix instructions is half a spectrum's digits, a block eight
 *            spectra;
 *   RW_BF16  hi and lo BF16 of eight spectra, FP32 accumulation.
 *
 * Scoring kernels, 20,000 proteins (2.7 M peptides), with rows written per
 * block into LDS (dense forms) or gathered per pair (FP32), and so: three digits,
 * 20,000 spectra 1,978 and 864 us; BF16, 6,000 spectra 1,937 and 773; FP32 batched,
 * 4,000 spectra 10,114 and 570.  Writing two levels' rows of the database takes
 * 0.89 ms, once.
 */
#include "hfx_cand.h"
#include "hfx_rows.h"

#include <algorithm>
#include <type_traits>

typedef __bf16 rw_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rw_f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t rw_i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t rw_u32x4 __attribute__((ext_vector_type(4)));

#define RW_NKS (RW_MAXK / 64)  /* k-steps of 64 bins */
static_assert(RW_MAXK % 64 == 0 && RW_G * 256 >= RW_MAXK, "groups cover a row");

/* bin within a k-step's 64 of byte j (0..15) of k-group kg */
__host__ __device__ inline uint32_t rw_bin_of(uint32_t kg, uint32_t j)
{
    return kg * 16u + ((j >> 2) & 1u) * 8u + 2u * (j & 3u) + (j >> 3);
}

/* wave-uniform tables nothing in the kernel writes, through scalar loads */
template <class T>
__device__ __forceinline__ T rw_sload(const T *p, uint64_t i)
{
    return ((const __attribute__((address_space(4))) T *)p)[i];
}

/* ------------------------------------------------------------------ */
/* Spectra as planes                                                     */
/* ------------------------------------------------------------------ */

__device__ __forceinline__ uint32_t rw_bf16(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

/* planes[s][plane][RW_MAXK]: byte 64 ks + 16 kg + j of a digit plane (the lowest
 * digit first) is the digit of bin 64 ks + rw_bin_of(kg, j); the BF16 planes (hi of bytes j < 8,
 * hi of j >= 8, lo, lo) hold eight BF16 in the 16 bytes of a k-group.
 * qs[s] = 2^-k.  norms (if any): sum and max of |x|.  A spectrum whose charge has no
 * rows (above `have`; a later one than those a batch was planned with), whose window
 * passes the last peptide that has any (num_pep), or, in the FP32 form, which the
 * digits do not serve, goes to the list `rest`, and its lvl[s] is 0; the others' lvl[s]
 * is their fragment charge. */
template <int MODE>
__global__ void __launch_bounds__(256)
    k_rw_split(uint8_t *planes, float *qs, uint32_t *lvl, hfx_rest rest, uint32_t have,
               float2 *norms, float *scores, const uint64_t *off, const uint32_t *begin,
               const uint32_t *num, uint32_t num_pep, hfx_spectra sp)
{
    constexpr uint32_t NP = RW_PLANES(MODE);
    __shared__ float red[2][256 / HFX_WAVE];
    __shared__ uint32_t bad;
    const uint32_t s = blockIdx.x, tid = threadIdx.x;
    const uint32_t len = min(sp.d_len[s], min(sp.x_stride, (uint32_t)RW_MAXK));
    const float *x = sp.d_x + (size_t)s * sp.x_stride;
    /* spectra whose fragment charge is not generated score 0 */
    const uint32_t z = hfx_zeff(sp.d_zmax[s]);
    if (z == 0)
        for (uint32_t i = tid; i < num[s]; i += 256) scores[off[s] + i] = 0.0f;
    /* thread t takes the four bins of words t + 256 u (bytes 4 w .. 4 w + 3) */
    constexpr uint32_t NW = RW_MAXK / 4, NU = (NW + 255) / 256;
    float v[NU][4];
    float m = 0.0f, x1 = 0.0f;
    bool odd = false;
    if (tid == 0) bad = 0;
#pragma unroll
    for (uint32_t u = 0; u < NU; ++u) {
        const uint32_t w = tid + 256 * u;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t bin = (w >> 4) * 64u + rw_bin_of((w >> 2) & 3u, (w & 3u) * 4u + i);
            v[u][i] = w < NW && bin < len ? x[bin] : 0.0f;
            const float a = fabsf(v[u][i]);
            m = fmaxf(m, a);
            x1 += a;
            odd |= !(a < INFINITY);
        }
    }
    for (uint32_t k = 32; k > 0; k >>= 1) {
        m = fmaxf(m, __shfl_xor(m, k, 64));
        x1 += __shfl_xor(x1, k, 64);
    }
    if (hfx_lane() == 0) {
        red[0][tid / HFX_WAVE] = m;
        red[1][tid / HFX_WAVE] = x1;
    }
    __syncthreads();
    if (odd) bad = 1;
    __syncthreads();
    m = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    x1 = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    if (tid == 0 && norms) norms[s] = make_float2(x1, m);
    bool out = z > have || (num[s] && (uint64_t)begin[s] + num[s] > num_pep);
    /* RW_I8X6, k: m 2^k in [2^45, 2^46), at most 126 */
    [[maybe_unused]] double sc6 = 1.0;
    if constexpr (MODE == RW_I8X6) {
        int k = 0;
        if (m > 0.0f && !bad) k = min(45 - ((int)((__float_as_uint(m) >> 23) & 255u) - 127), 126);
        sc6 = ldexp(1.0, k);
        if (tid == 0) qs[s] = ldexpf(1.0f, -k);
        bool lost = bad != 0;
#pragma unroll
        for (uint32_t u = 0; u < NU; ++u)
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const double d = (double)v[u][i] * sc6;
                lost |= !(rint(d) == d);
            }
        out |= __syncthreads_or(lost) != 0;
    }
    if (tid == 0) {
        lvl[s] = out ? 0u : z;
        if (out && z) rest.list[atomicAdd(rest.count, 1u)] = s;
    }
    if (out) return; /* its planes are read into no score */
    uint8_t *o = planes + (size_t)s * NP * RW_MAXK;
    if constexpr (MODE == RW_BF16) {
#pragma unroll
        for (uint32_t u = 0; u < NU; ++u) {
            const uint32_t w = tid + 256 * u;
            if (w >= NW) break;
            uint32_t h[4], l[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                h[i] = rw_bf16(v[u][i]);
                l[i] = rw_bf16(v[u][i] - __uint_as_float(h[i] << 16));
            }
            /* four bins are 8 bytes; word w & 3 < 2: the first eight bins */
            const uint32_t part = (w >> 1) & 1u;
            const size_t at = (size_t)(w >> 2) * 16u + (w & 1u) * 8u;
            *(uint2 *)(o + part * RW_MAXK + at) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
            *(uint2 *)(o + (2 + part) * RW_MAXK + at) =
                make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
        }
        return;
    }
    /* RW_I8X3, k: m 2^k in [2^22, 2^23) from m's exponent, one less where that passes
     * the largest value the digits reach; at most 126 */
    [[maybe_unused]] float sc = 1.0f;
    if constexpr (MODE == RW_I8X3) {
        int k = 0;
        if (m > 0.0f) {
            const int e = (int)((__float_as_uint(m) >> 23) & 255u) - 127;
            k = 22 - e;
            if (k > 126) k = 126;
            else if (ldexpf(m, k) > 8355711.0f) --k;
        }
        sc = ldexpf(1.0f, k);
        if (tid == 0) qs[s] = ldexpf(1.0f, -k);
    }
    using X_t = std::conditional_t<MODE == RW_I8X6, int64_t, int32_t>;
#pragma unroll
    for (uint32_t u = 0; u < NU; ++u) {
        const uint32_t t = tid + 256 * u;
        if (t >= NW) break;
        uint32_t w[NP];
#pragma unroll
        for (uint32_t d = 0; d < NP; ++d) w[d] = 0u;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            X_t X;
            if constexpr (MODE == RW_I8X6) X = (int64_t)((double)v[u][i] * sc6);
            else X = (int32_t)rintf(v[u][i] * sc);
#pragma unroll
            for (uint32_t d = 0; d < NP; ++d) {
                const int32_t g = d + 1 < NP ? (((int32_t)X + 128) & 255) - 128 : (int32_t)X;
                w[d] |= (uint32_t)(g & 255) << (8 * i);
                X = (X - g) >> 8;
            }
        }
#pragma unroll
        for (uint32_t d = 0; d < NP; ++d) ((uint32_t *)(o + d * RW_MAXK))[t] = w[d];
    }
}

/* ------------------------------------------------------------------ */
/* Rows                                                                  */
/* ------------------------------------------------------------------ */

/* Persistent workgroups of four waves, a tile at a time.  The nibble map of its
 * sixteen rows (bin x of a row in word 2 + x / 8, unary codes OR-ed = max per
 * bin) takes 18.7 KiB of LDS, so that seven workgroups fill a CU; a row stride of
 * 36 mod 64 words puts the 32 lanes of half an emission read on 64 different
 * banks.  A tile is a chain: order, offsets, residues, masses, sums, peaks,
 * codes.  The reads of the next three tiles are under way while one is written;
 * masses are looked up a position a lane and only their sums (one lane a
 * peptide, sequential FP32 as everywhere) go one after the other.  Ladders lie
 * in LDS one peptide after the other, sixteen peptides x RB_CHUNK positions at a
 * time, so that each thread then takes one position whatever the peptides'
 * lengths.  A peak whose bins all lie outside the row goes to one of the words
 * past it, by lane; a triple that straddles an end spills into the row's margin
 * words.  Neither is emitted.  Words are cleared as they are emitted for the last
 * time.  Rows go out past the caches: they are read again only after gigabytes
 * of others.
 * Two levels of 2.7 M peptides (2.4 GB written, 0.7 GB of scattered reads): 1,340
 * us with a workgroup of two waves a tile, no reads ahead and a lane a peptide
 * for residues, masses and sums; 890 us so (960 through the caches; 6
 * workgroups a CU 50 us more, 5 150 more).  Memory at 3.5 TB/s and vector
 * instructions (69 % of issue; two thirds of the waves' cycles are waits) share it. */
#define RB_THREADS 256
#define RB_WAVES (RB_THREADS / HFX_WAVE)
#define RB_PER_CU 7
#define RB_MSTR 292
#define RB_CHUNK 48
static_assert(RB_MSTR >= 2 + RW_MAXK / 8 + 2 && RB_MSTR % 64 == 36, "map row stride");
static_assert(RB_THREADS == 16 * RW_ROWS && RB_CHUNK % 16 == 0, "sixteen threads a peptide");
#define RB_MAGIC 12582912.0f /* 1.5 * 2^23: adding it rounds to an integer, ties to even */
#define RB_MAGIC_BITS 0x4B400000u

/* bin + RB_MAGIC_BITS: |mz| < 2^21 */
__device__ __forceinline__ uint32_t rb_binu(float mz)
{
    return __float_as_uint(hfx_div(mz, HFX_BIN_WIDTH_MONO, 1.0f / HFX_BIN_WIDTH_MONO) + RB_MAGIC);
}

/* ladder masses are cut to this, whose peaks are past the row at any charge and
 * do not pass the magic sum's 2^22 bins */
#define RB_MZMAX 1.0e6f
/* bins past the row that a lane's peaks outside it go to: words 276 .. 291 */
#define RB_OUT(lane) (RW_MAXK + 16u + ((lane) & 7u) * 16u)
static_assert(2 + RB_OUT(7u) / 8 + 1 < RB_MSTR, "the last word outside the row");

struct RbPut {
    uint32_t *row; /* word of bin -16 */
    uint32_t out;  /* RB_OUT + 16 */
    __device__ __forceinline__ void one(float mz) const
    {
        const uint32_t u = min(rb_binu(mz) - (RB_MAGIC_BITS - 16u), out);
        atomicOr(row + (u >> 3), HFX_CODE10 << ((u << 2) & 31u));
    }
    /* 25 at x - 1, 50 at x, 25 at x + 1 */
    __device__ __forceinline__ void three(float mz) const
    {
        const uint32_t u = min(rb_binu(mz) - (RB_MAGIC_BITS - 15u), out); /* x - 1 */
        const uint64_t t = (uint64_t)(HFX_CODE25 | HFX_CODE50 << 4 | HFX_CODE25 << 8)
                           << ((u << 2) & 31u);
        atomicOr(row + (u >> 3), (uint32_t)t);
        if (t >> 32) atomicOr(row + (u >> 3) + 1, (uint32_t)(t >> 32));
    }
};

template <int Z>
__device__ __forceinline__ void rb_peaks(const RbPut &p, float b, float y)
{
    constexpr float zh = HFX_DEV_H * (float)Z;
    constexpr float h2o = HFX_DEV_H2O / (float)Z, nh3 = HFX_DEV_NH3 / (float)Z;
    auto zdiv = [](float x) {
        if constexpr (Z == 3) return hfx_div(x, 3.0f, 1.0f / 3.0f);
        else return x * (1.0f / (float)Z);
    };
    const float ma = zdiv((b - HFX_DEV_CO) + zh);
    const float mb = zdiv(b + zh);
    const float my = zdiv((y + HFX_DEV_H2O) + zh);
    p.one(ma);
    p.three(mb);
    p.one(mb - h2o);
    p.one(mb - nh3);
    p.three(my);
    p.one(my - nh3);
}

struct RbArgs {
    hfx_db db;
    uint32_t ntiles;
    uint8_t *rows[HFX_MAX_CHARGE];       /* null: level not written */
    const uint32_t *flags;               /* [level - 1][ntiles]: tiles wanted, or null: all */
    const uint64_t *slots;               /* their places in rows[level - 1] */
    uint8_t *ng;                         /* [ntiles] groups a tile's peaks reach */
    uint32_t G;                          /* groups a tile holds */
};

/* two words of eight nibbles 0 / 1 / 3 / 7 -> sixteen 2-bit codes */
__device__ __forceinline__ uint32_t rb_pack(uint32_t a, uint32_t b)
{
    const uint32_t ca = (a & 0x22222222u) | ((a ^ (a >> 2)) & 0x11111111u);
    const uint32_t cb = (b & 0x22222222u) | ((b ^ (b >> 2)) & 0x11111111u);
    return ca | cb << 2;
}

__global__ void __launch_bounds__(RB_THREADS, RB_PER_CU) k_rw_build(RbArgs a)
{
    __shared__ __align__(16) uint32_t maps[RW_ROWS * RB_MSTR];
    __shared__ float lb[RW_ROWS * RB_CHUNK];
    __shared__ uint8_t lrow[RW_ROWS * RB_CHUNK];
    __shared__ float mtab[32], rr[RW_ROWS];
    __shared__ float topb;
    const uint32_t tid = threadIdx.x, lane = hfx_lane(), wave = tid / HFX_WAVE;
    for (uint32_t i = tid; i < RW_ROWS * RB_MSTR / 4; i += RB_THREADS)
        ((uint4 *)maps)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (tid < 32) mtab[tid] = tid < 26 ? a.db.d_mass[tid] : 0.0f;
    /* lane: peptide lane & 15 of a tile; thread: residues lk, lk + 16, ... of its
     * peptide lr */
    const uint32_t lr = tid >> 4, lk = tid & 15u;
    const uint32_t G = gridDim.x;
    auto order = [&](uint64_t t) {
        const uint64_t q = t * RW_ROWS + (lane & 15u);
        return t < a.ntiles && q < a.db.num_pep ? a.db.d_idx_sorted[q] : 0xffffffffu;
    };
    struct Meta {
        uint32_t tc, tn;
        float r;
    };
    auto meta = [&](uint32_t pep) {
        Meta m{0u, 0u, 0.0f};
        if (pep != 0xffffffffu) m = Meta{a.db.d_tc[pep], a.db.d_tn[pep], a.db.d_r[pep]};
        return m;
    };
    auto count = [](const Meta &m) { return m.tn > m.tc ? m.tn - m.tc : 0u; };
    auto residues = [&](const Meta &m, uint32_t (&x)[2]) {
        const uint32_t tc = (uint32_t)__shfl((int)m.tc, (int)lr, 64);
        const uint32_t n = (uint32_t)__shfl((int)count(m), (int)lr, 64);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) x[j] = lk + 16 * j < n ? a.db.d_ions[tc + lk + 16 * j] : 0u;
    };
    /* the wanted tiles among blockIdx.x, blockIdx.x + G, ...: 64 looked at at once,
     * a tile a lane; ~0 past the last */
    uint64_t look = blockIdx.x, from = 0, left = 0;
    uint32_t lane_want = 0;
    auto next = [&](uint32_t &want) -> uint64_t {
        while (!left) {
            want = 0;
            if (look >= a.ntiles) return ~0ull;
            from = look;
            const uint64_t t = from + (uint64_t)lane * G;
            lane_want = 0;
#pragma unroll
            for (uint32_t l = 0; l < HFX_MAX_CHARGE; ++l)
                if (a.rows[l] && t < a.ntiles && (!a.flags || a.flags[(size_t)l * a.ntiles + t] != 0u))
                    lane_want |= 1u << l;
            left = __ballot(lane_want != 0u);
            look += 64ull * G;
        }
        const uint32_t i = (uint32_t)__builtin_ctzll(left);
        left &= left - 1ull;
        want = (uint32_t)__builtin_amdgcn_readlane((int)lane_want, (int)i);
        return from + (uint64_t)i * G;
    };
    /* the tile written: its offsets and residues; the one after it: its offsets;
     * the one after that: its order */
    uint32_t w0, w1, w2, x[2];
    uint64_t t0 = next(w0), t1 = next(w1), t2 = next(w2);
    Meta m0 = meta(order(t0)), m1 = meta(order(t1));
    uint32_t pep = order(t2);
    residues(m0, x);
    __syncthreads();
    for (uint32_t turn = blockIdx.x; t0 != ~0ull; ++turn) {
        const uint64_t t = t0;
        const Meta m = m0;
        const uint32_t want = w0, x0 = x[0], x1 = x[1];
        t0 = t1;
        t1 = t2;
        w0 = w1;
        w1 = w2;
        m0 = m1;
        residues(m0, x);
        m1 = meta(pep);
        t2 = next(w2);
        pep = order(t2);
        const uint32_t n = count(m);
        uint32_t nmax = n;
#pragma unroll
        for (uint32_t o = 8; o > 0; o >>= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o, 64));
        nmax = __builtin_amdgcn_readfirstlane(nmax);
        const uint32_t nch = max((nmax + RB_CHUNK - 1) / RB_CHUNK, 1u);
        const uint32_t top = 31u - (uint32_t)__builtin_clz(want); /* highest level - 1 */
        const uint32_t wv = (wave + turn) % RB_WAVES; /* the sums go round the SIMDs */
        if (tid < RW_ROWS) rr[tid] = m.r;
        float bl = 0.0f;

        /* positions [c RB_CHUNK, ...) of the sixteen ladders into lb, row after
         * row; their number */
        auto ladders = [&](uint32_t c) {
            const uint32_t k0 = c * RB_CHUNK;
            const uint32_t cn = n > k0 ? min(n - k0, (uint32_t)RB_CHUNK) : 0u;
            uint32_t incl = cn;
#pragma unroll
            for (uint32_t o = 1; o < RW_ROWS; o <<= 1) {
                const uint32_t y = __shfl_up(incl, o, 16);
                if ((lane & 15u) >= o) incl += y;
            }
            const uint32_t at = incl - cn;
            const uint32_t la = (uint32_t)__shfl((int)at, (int)lr, 64);
            const uint32_t ln = (uint32_t)__shfl((int)cn, (int)lr, 64);
            const uint32_t ltc = (uint32_t)__shfl((int)m.tc, (int)lr, 64);
#pragma unroll
            for (uint32_t j = 0; j < RB_CHUNK / 16; ++j) {
                const uint32_t k = lk + 16 * j;
                if (k < ln) {
                    const uint32_t xr = c == 0 && j < 2 ? (j ? x1 : x0) : a.db.d_ions[ltc + k0 + k];
                    lb[la + k] = mtab[HFX_ACID_IDX(xr)];
                    lrow[la + k] = (uint8_t)lr;
                }
            }
            __syncthreads();
            if (wv == 0) {
                float mx = 0.0f;
                if (lane < RW_ROWS) {
                    if (c == 0) bl = 0.0f;
                    for (uint32_t k = 0; k < cn; k += 8) {
                        float v[8];
#pragma unroll
                        for (uint32_t j = 0; j < 8; ++j) v[j] = lb[at + min(k + j, cn - 1u)];
#pragma unroll
                        for (uint32_t j = 0; j < 8; ++j)
                            if (k + j < cn) {
                                bl = bl + v[j];
                                lb[at + k + j] = bl;
                                mx = fmaxf(mx, fmaxf(bl, m.r - bl));
                            }
                    }
                }
#pragma unroll
                for (uint32_t o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
                if (lane == 0) topb = c == 0 ? mx : fmaxf(topb, mx);
            }
            __syncthreads();
            return (uint32_t)__builtin_amdgcn_readlane((int)incl, RW_ROWS - 1);
        };
        uint32_t np = 0;
        for (uint32_t z = 1; z <= top + 1u; ++z) {
            for (uint32_t c = 0; c < nch; ++c) {
                if (z == 1 || nch > 1) np = ladders(c);
                for (uint32_t i = tid; i < np; i += RB_THREADS) {
                    const uint32_t row = lrow[i];
                    const float b0 = lb[i];
                    const float b = __builtin_amdgcn_fmed3f(b0, -RB_MZMAX, RB_MZMAX);
                    const float y = __builtin_amdgcn_fmed3f(rr[row] - b0, -RB_MZMAX, RB_MZMAX);
                    const RbPut p{maps + row * RB_MSTR, RB_OUT(lane) + 16u};
                    switch (z) {
                    case 1: rb_peaks<1>(p, b, y); break;
                    case 2: rb_peaks<2>(p, b, y); break;
                    case 3: rb_peaks<3>(p, b, y); break;
                    default: rb_peaks<4>(p, b, y); break;
                    }
                }
                __syncthreads();
            }
            /* groups the peaks reach: every bin lies below top / 1.0005 + 24 */
            const float tf = fminf(topb, 1.0e6f);
            const uint32_t ng = min(a.G, ((uint32_t)tf + 28u) / 256u + 1u);
            if (z == 1 && tid == 0) a.ng[t] = (uint8_t)ng;
            if ((want >> (z - 1u)) & 1u) {
                const bool last = z > top;
                const uint64_t slot = a.slots ? rw_sload(a.slots, (uint64_t)(z - 1u) * a.ntiles + t) : t;
                rw_u32x4 *out = (rw_u32x4 *)(a.rows[z - 1u] + slot * ((size_t)a.G * 1024u));
                uint32_t *mrow = maps + (lane & 15u) * RB_MSTR + 2 + 2 * (lane >> 4);
                for (uint32_t g = wv; g < ng; g += RB_WAVES) {
                    rw_u32x4 v;
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) {
                        /* the last group's words past the row hold no bins */
                        const uint32_t w = g * 32 + k * 8;
                        uint2 ab = make_uint2(0u, 0u);
                        if (w < RW_MAXK / 8) {
                            ab = *(const uint2 *)(mrow + w);
                            if (last) *(uint2 *)(mrow + w) = make_uint2(0u, 0u);
                        }
                        v[k] = rb_pack(ab.x, ab.y);
                    }
                    __builtin_nontemporal_store(v, out + g * 64 + lane);
                }
                if (!last) __syncthreads(); /* read before the next charge's peaks */
            }
        }
    }
}

/* ------------------------------------------------------------------ */
/* Work items                                                             */
/* ------------------------------------------------------------------ */

/* block b: the tiles of its windows' hull, fragment charge levels (bit z),
 * longest row in k-steps, work items (CT tiles each, per level).  Sixteen lanes a
 * block, a spectrum each (a thread a block read them one after the other: 18 us
 * for 20,000 spectra, 4.7 now); the first also clears the items' counter. */
__global__ void __launch_bounds__(256)
    k_rw_blocks(uint32_t *tbeg, uint32_t *tend, uint32_t *binfo, uint32_t *items, uint32_t *counter,
                const uint32_t *order, const uint32_t *bstart, const uint32_t *begin,
                const uint32_t *num, hfx_spectra sp, uint32_t B, uint32_t CT)
{
    const uint32_t b = (blockIdx.x * 256 + threadIdx.x) / 16, g = threadIdx.x & 15u;
    if (b == 0 && g == 0) *counter = 0;
    if (b >= B) return;
    uint32_t lo = 0xffffffffu, hi = 0, mask = 0, kmax = 0;
    const uint32_t i = bstart[b] + g;
    if (i < bstart[b + 1]) {
        const uint32_t s = order[i];
        const uint32_t z = hfx_zeff(sp.d_zmax[s]), n = num[s], bg = begin[s], ln = sp.d_len[s];
        if (z && n) {
            lo = bg;
            hi = bg + n;
            mask = 1u << z;
            kmax = min(ln, min(sp.x_stride, (uint32_t)RW_MAXK));
        }
    }
#pragma unroll
    for (uint32_t o = 8; o > 0; o >>= 1) {
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 16));
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 16));
        mask |= (uint32_t)__shfl_xor((int)mask, o, 16);
        kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o, 16));
    }
    if (g != 0) return;
    const bool any = hi > lo;
    const uint32_t t0 = any ? lo / RW_ROWS : 0u, t1 = any ? (hi + RW_ROWS - 1) / RW_ROWS : 0u;
    if (!any) mask = 0;
    tbeg[b] = t0;
    tend[b] = t1;
    binfo[b] = (kmax + 63u) / 64u | mask << 16;
    items[b] = ((t1 - t0 + CT - 1) / CT) * (uint32_t)__builtin_popcount(mask);
}

__global__ void k_rw_fill(uint32_t *a, uint64_t n, uint32_t v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = v;
}

/* the tiles the blocks read: one workgroup a block (equal stores race) */
__global__ void k_rw_mark(uint32_t *flags, const uint32_t *tbeg, const uint32_t *tend,
                          const uint32_t *binfo, uint32_t ntiles)
{
    const uint32_t b = blockIdx.x, mask = binfo[b] >> 16;
    for (uint32_t l = 1; l <= HFX_MAX_CHARGE; ++l)
        if ((mask >> l) & 1u)
            for (uint32_t t = tbeg[b] + threadIdx.x; t < tend[b]; t += blockDim.x)
                flags[(size_t)(l - 1) * ntiles + t] = 1u;
}

/* ------------------------------------------------------------------ */
/* The contraction                                                        */
/* ------------------------------------------------------------------ */

#define RM_THREADS 768
#define RM_WAVES (RM_THREADS / HFX_WAVE)
#define RM_T 4 /* tiles a wave contracts at once: each B fragment read serves 64 rows */

struct RmArgs {
    float *scores;
    const uint64_t *score_off;
    const uint32_t *begin, *num, *order, *bstart;
    uint32_t B, CT;
    const uint32_t *tbeg, *tend, *binfo;
    const uint64_t *item_off;
    const uint8_t *planes;
    const float *qs;
    uint32_t *counter;
    const uint8_t *rows[HFX_MAX_CHARGE];
    const uint64_t *slots; /* [level - 1][ntiles], or null: tile t at place t */
    const uint8_t *ng;
    uint32_t ntiles, G;
    hfx_spectra sp;
};

/* an even lane: the next lane's value */
__device__ __forceinline__ double rm_next(double h)
{
    const uint64_t u = (uint64_t)__double_as_longlong(h);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0xb1, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0xb1, 0xf, 0xf, false);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

/* Persistent workgroups of twelve waves over (block, level, CT tiles).  The
 * block's planes stay in LDS, laid out so that a fragment read is one
 * contiguous KiB ([k-step][plane][lane]); each wave contracts four tiles at a
 * time over the whole row, its accumulators in registers, the next group's
 * codes loaded while the current one is contracted.  A k-step of four tiles
 * costs 4 x 11 code lookups, 4 x planes matrix instructions and one fragment
 * read a plane.
 * The two kinds add up: vector and matrix instructions take 49 and 39 % of the
 * cycles with three digits, 52 and 39 with six, 70 and 22 in BF16 (20,000 spectra),
 * and interleaving them by hand changes nothing.  So the loop holds lookups
 * alone (no copies of the codes, per-lane addresses or FP64 folds), and a third
 * wave a SIMD fills its waits: three digits, 20,000 spectra, 963 us with two waves
 * and those, 864 so; BF16, 6,000 spectra, 850 and 773.  Six digits take three
 * matrix instructions a k-step and tile as well, for half as many spectra: a plain
 * search of 10,000 866 us, a batch of 4,000 570 (four digits and sixteen spectra,
 * 757 and 547, round the FP32 values below max|x| / 128).  Sixteen
 * waves spill (983 us, three digits); three groups of codes on their way, also
 * across tiles, cost more scalar work than they hide (1,134). */
template <int MODE>
__global__ void __launch_bounds__(RM_THREADS, 3) k_rw_mm(RmArgs a)
{
    constexpr uint32_t NP = MODE == RW_BF16 ? 2 : 3; /* planes in LDS */
    constexpr uint32_t NS = RW_NS(MODE);
    /* a column is half of a spectrum: its high or low digits, its hi or lo */
    constexpr bool HALF = MODE != RW_I8X3;
    extern __shared__ __align__(16) uint8_t rm_lds[];
    rw_u32x4 *Bl = (rw_u32x4 *)rm_lds; /* [k-step][plane][64 lanes] */
    __shared__ uint32_t m_s[16], m_beg[16], m_end[16], m_z[16];
    __shared__ float m_q[16];
    __shared__ uint64_t m_off[16];
    __shared__ uint32_t sh_t[2];
    const uint32_t tid = threadIdx.x, lane = hfx_lane();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / HFX_WAVE);
    const uint32_t col = lane & 15u, kg = lane >> 4;
    const uint32_t g_of = HALF ? col >> 1 : col; /* spectrum of this lane's column */
    const uint32_t nitems = (uint32_t)rw_sload(a.item_off, a.B);
    uint32_t cur = 0xffffffffu;
    if (tid == 0) sh_t[0] = atomicAdd(a.counter, 1u);
    uint32_t next = 0;
    for (uint32_t slot = 0;; slot ^= 1u) {
        __syncthreads(); /* every wave is done with the previous item */
        const uint32_t t0 = __builtin_amdgcn_readfirstlane(sh_t[slot]);
        if (t0 >= nitems) break;
        /* from the last to the first: higher charge levels and heavier
         * precursors (longer rows) come first, the lightest finish the launch */
        const uint32_t it = nitems - 1u - t0;
        if (tid == 0) next = atomicAdd(a.counter, 1u);
        uint32_t lo = 0, hi = a.B;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (rw_sload(a.item_off, mid) <= it) lo = mid; else hi = mid;
        }
        const uint32_t b = lo;
        const uint32_t info = rw_sload(a.binfo, b);
        const uint32_t nks = info & 0xffffu, mask = info >> 16;
        if (b != cur) {
            if (tid < 16) {
                const uint32_t i = a.bstart[b] + tid;
                uint32_t s = 0xffffffffu, be = 0, en = 0, z = 0;
                uint64_t of = 0;
                float q = 0.0f;
                if (tid < NS && i < a.bstart[b + 1]) {
                    s = a.order[i];
                    be = a.begin[s];
                    en = be + a.num[s];
                    z = hfx_zeff(a.sp.d_zmax[s]);
                    of = a.score_off[s];
                    if (MODE != RW_BF16) q = a.qs[s];
                }
                m_s[tid] = s; m_beg[tid] = be; m_end[tid] = en; m_z[tid] = z; m_off[tid] = of;
                m_q[tid] = q;
            }
            __syncthreads();
            /* lanes over columns first: LDS writes are contiguous, and the four
             * k-groups of a column are 64 bytes of its plane */
            const uint32_t nv = nks * NP * 64u;
            constexpr uint32_t U = 6;
            for (uint32_t i0 = tid; i0 < nv; i0 += U * RM_THREADS) {
                rw_u32x4 val[U];
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) {
                    const uint32_t i = i0 + u * RM_THREADS;
                    const uint32_t kd = i >> 6, ks = kd / NP, d = kd - ks * NP;
                    const uint32_t s = m_s[g_of];
                    val[u] = rw_u32x4{0u, 0u, 0u, 0u};
                    if (i < nv && s != 0xffffffffu) {
                        const uint32_t pl = MODE == RW_BF16   ? (col & 1u) * 2u + d
                                            : MODE == RW_I8X6 ? (col & 1u ? d : 3u + d)
                                                              : d;
                        val[u] = *(const rw_u32x4 *)(a.planes +
                                                     ((size_t)s * RW_PLANES(MODE) + pl) * RW_MAXK +
                                                     ks * 64u + kg * 16u);
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    if (i0 + u * RM_THREADS < nv) Bl[i0 + u * RM_THREADS] = val[u];
            }
            cur = b;
            __syncthreads();
        }
        if (tid == 0) sh_t[slot ^ 1u] = next;
        const uint32_t tb = rw_sload(a.tbeg, b), te = rw_sload(a.tend, b);
        const uint32_t nch = (te - tb + a.CT - 1) / a.CT;
        const uint32_t local = (uint32_t)(it - rw_sload(a.item_off, b));
        const uint32_t li = local / nch, chunk = local - li * nch;
        uint32_t m = mask;
        for (uint32_t qq = 0; qq < li; ++qq) m &= m - 1u;
        const uint32_t lvl = (uint32_t)__builtin_ctz(m);
        const uint32_t c0 = tb + chunk * a.CT, c1 = min(c0 + a.CT, te);
        const uint8_t *rows = lvl == 1 ? a.rows[0] : lvl == 2 ? a.rows[1]
                            : lvl == 3 ? a.rows[2] : a.rows[3];
        const uint64_t *slots = a.slots ? a.slots + (size_t)(lvl - 1u) * a.ntiles : nullptr;
        const uint32_t beg = m_beg[g_of], end = m_end[g_of];
        const bool mine = m_z[g_of] == lvl && (!HALF || (col & 1u) == 0u);
        const float qf = MODE == RW_BF16 ? 0.0f : m_q[g_of];
        float *const out = a.scores + m_off[g_of];
        const size_t tile_bytes = (size_t)a.G * 1024u;
        for (uint32_t u0 = c0 + wave * RM_T; u0 < c1; u0 += RM_WAVES * RM_T) {
            const uint8_t *base[RM_T];
            uint32_t ng = 0;
#pragma unroll
            for (uint32_t k = 0; k < RM_T; ++k) {
                const uint32_t t = min(u0 + k, c1 - 1u);
                const uint64_t place = slots ? rw_sload(slots, t) : (uint64_t)t;
                base[k] = rows + place * tile_bytes;
                const uint32_t word = rw_sload((const uint32_t *)a.ng, t >> 2);
                ng = max(ng, (word >> ((t & 3u) * 8u)) & 255u);
            }
            ng = min(ng, (nks + 3u) >> 2);
            /* groups past a tile's own are not written: read as zeros */
            uint32_t own[RM_T];
#pragma unroll
            for (uint32_t k = 0; k < RM_T; ++k) {
                const uint32_t t = min(u0 + k, c1 - 1u);
                own[k] = (rw_sload((const uint32_t *)a.ng, t >> 2) >> ((t & 3u) * 8u)) & 255u;
            }
            const uint32_t own_min = min(min(own[0], own[1]), min(own[2], own[3]));
            static_assert(RM_T == 4, "the least of its tiles' groups");
            auto load = [&](rw_u32x4(&c)[RM_T], uint32_t g) {
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k) {
                    const uint8_t *p = base[k] + min(g, own[k] - 1u) * 1024u; /* uniform */
                    c[k] = *(const rw_u32x4 *)(p + lane * 16u);
                }
            };
            auto past = [&](rw_u32x4(&c)[RM_T], uint32_t g) {
                if (g < own_min) return;
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k)
                    if (g >= own[k]) c[k] = rw_u32x4{0u, 0u, 0u, 0u};
            };
            /* use(codes, group) for every group, the next one's codes on their
             * way meanwhile */
            rw_u32x4 ca[RM_T], cb[RM_T];
            auto groups = [&](auto &&use) {
                load(ca, 0);
                for (uint32_t g = 0; g < ng; g += 2) {
                    load(cb, min(g + 1u, ng - 1u));
                    past(ca, g);
                    use(ca, g);
                    if (g + 1u >= ng) break;
                    load(ca, min(g + 2u, ng - 1u));
                    past(cb, g + 1u);
                    use(cb, g + 1u);
                }
            };
            if constexpr (MODE == RW_BF16) {
                rw_f32x4 acc0[RM_T], acc1[RM_T];
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k) {
                    acc0[k] = rw_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    acc1[k] = acc0[k];
                }
                groups([&](const rw_u32x4(&c)[RM_T], uint32_t g) {
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t ks = g * 4u + j;
                        if (ks < nks) {
                            const rw_u32x4 f0 = Bl[(ks * NP + 0) * 64u + lane];
                            const rw_u32x4 f1 = Bl[(ks * NP + 1) * 64u + lane];
#pragma unroll
                            for (uint32_t k = 0; k < RM_T; ++k) {
                                const uint32_t P = c[k][j];
                                uint32_t w[8];
#pragma unroll
                                for (uint32_t h = 0; h < 4; ++h) {
                                    const uint32_t sel = (P >> (2 * h)) & 0x03030303u;
                                    const uint32_t l8 = __builtin_amdgcn_perm(0u, 0xC8482000u, sel);
                                    const uint32_t h8 = __builtin_amdgcn_perm(0u, 0x41424100u, sel);
                                    w[2 * h] = __builtin_amdgcn_perm(h8, l8, 0x05010400u);
                                    w[2 * h + 1] = __builtin_amdgcn_perm(h8, l8, 0x07030602u);
                                }
                                const rw_u32x4 a0 = {w[0], w[1], w[2], w[3]};
                                const rw_u32x4 a1 = {w[4], w[5], w[6], w[7]};
                                acc0[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    __builtin_bit_cast(rw_bf16x8, a0),
                                    __builtin_bit_cast(rw_bf16x8, f0), acc0[k], 0, 0, 0);
                                acc1[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    __builtin_bit_cast(rw_bf16x8, a1),
                                    __builtin_bit_cast(rw_bf16x8, f1), acc1[k], 0, 0, 0);
                            }
                        }
                    }
                });
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k) {
                    const uint32_t t = u0 + k;
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        const float h = acc0[k][i] + acc1[k][i];
                        /* an even column's lane adds its odd neighbour: hi + lo */
                        const float v = h + __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(
                                                (int)__float_as_uint(h), (int)__float_as_uint(h),
                                                0xb1, 0xf, 0xf, false));
                        const uint32_t p = t * RW_ROWS + 4u * kg + i;
                        if (mine && t < c1 && beg <= p && p < end) out[p - beg] = v;
                    }
                }
            } else {
                rw_i32x4 acc[RM_T][NP];
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k)
#pragma unroll
                    for (uint32_t d = 0; d < NP; ++d) acc[k][d] = rw_i32x4{0, 0, 0, 0};
                groups([&](const rw_u32x4(&c)[RM_T], uint32_t g) {
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t ks = g * 4u + j;
                        if (ks < nks) {
                            rw_i32x4 f[NP];
#pragma unroll
                            for (uint32_t d = 0; d < NP; ++d)
                                f[d] = __builtin_bit_cast(rw_i32x4, Bl[(ks * NP + d) * 64u + lane]);
#pragma unroll
                            for (uint32_t k = 0; k < RM_T; ++k) {
                                const uint32_t P = c[k][j];
                                rw_i32x4 av;
#pragma unroll
                                for (uint32_t h = 0; h < 4; ++h)
                                    av[h] = (int32_t)__builtin_amdgcn_perm(
                                        0u, 0x19320A00u, (P >> (2 * h)) & 0x03030303u);
#pragma unroll
                                for (uint32_t d = 0; d < NP; ++d)
                                    acc[k][d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                        av, f[d], acc[k][d], 0, 0, 0);
                            }
                        }
                    }
                });
                /* Digit sums are below 50 * 128 * RW_MAXK < 2^23.8.  Carries go up until
                 * the highest digit is followed by 16 bits.  Three digits: both parts
                 * are exact in FP32, and the fused sum rounds once.  Six: each half is
                 * exact in FP64, the odd column's (the low one) is fetched, and the
                 * fused sum is rounded to FP32. */
#pragma unroll
                for (uint32_t k = 0; k < RM_T; ++k) {
                    const uint32_t t = u0 + k;
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        int32_t top = acc[k][0][i];
                        uint32_t low = 0;
#pragma unroll
                        for (uint32_t d = 1; d < NP; ++d) {
                            low |= ((uint32_t)top & 255u) << (8 * (d - 1));
                            top = acc[k][d][i] + (top >> 8);
                        }
                        float v;
                        if constexpr (MODE == RW_I8X6) {
                            const double h = __builtin_fma((double)top, 65536.0, (double)low);
                            v = (float)__builtin_fma(h, 16777216.0, rm_next(h)) * qf;
                        } else {
                            v = __builtin_fmaf((float)top, 65536.0f, (float)low) * qf;
                        }
                        const uint32_t p = t * RW_ROWS + 4u * kg + i;
                        if (mine && t < c1 && beg <= p && p < end) out[p - beg] = v;
                    }
                }
            }
        }
    }
}

/* ------------------------------------------------------------------ */
/* Host side                                                              */
/* ------------------------------------------------------------------ */

uint32_t hfx_rows_tiles(uint32_t num_pep) { return (num_pep + RW_ROWS - 1) / RW_ROWS; }
uint32_t hfx_rows_groups(uint32_t x_stride)
{
    return (std::min(x_stride, (uint32_t)RW_MAXK) + 255u) / 256u;
}
/* candidates a work item takes (multiple of RM_T tiles a wave): about four
 * items a CU, but enough rows that the block's planes are worth staging */
uint32_t hfx_rows_chunk(uint64_t rows, uint32_t cus)
{
    const uint64_t c = rows / (4ull * cus);
    const uint64_t step = RM_WAVES * RM_T * RW_ROWS; /* every wave busy */
    return (uint32_t)std::min<uint64_t>(std::max<uint64_t>((c + step - 1) / step * step, step), 8192);
}
/* the tiles of a work item of CH candidates: a round of a workgroup's waves at least.
 * The contraction of 20,000 spectra, three digits, by candidates an item: 512 1,216 us,
 * 768 1,018, 1024 925, 1536 912, 2048 864, 2304 and 3072 897, 4096 911, 6144 975, 8192
 * 1,040; whole rounds past the first gain nothing, 2048 is no multiple of 768. */
uint32_t hfx_rows_item_tiles(uint32_t CH)
{
    return std::max((CH + RW_ROWS - 1) / RW_ROWS, (uint32_t)(RM_WAVES * RM_T));
}

int hfx_rows_split(int mode, const hfx_spectra *sp, uint8_t *planes, float *qs, uint32_t *lvl,
                   const hfx_rest *rest, uint32_t have, float2 *norms, float *scores,
                   const uint64_t *off, const uint32_t *begin, const uint32_t *num, uint32_t num_pep,
                   void *stream)
{
    HFX_REQUIRE(sp->x_stride <= RW_MAXK, HFX_ERR_ARG, "rows: spectra of up to %d bins", RW_MAXK);
    if (sp->num_spec == 0) return HFX_OK;
    const dim3 g(sp->num_spec), t(256);
    hipStream_t st = hfx_stream(stream);
    const auto kernel = mode == RW_I8X3   ? k_rw_split<RW_I8X3>
                        : mode == RW_I8X6 ? k_rw_split<RW_I8X6>
                                          : k_rw_split<RW_BF16>;
    hipLaunchKernelGGL(kernel, g, t, 0, st, planes, qs, lvl, *rest, have, norms, scores, off, begin, num,
                       num_pep, *sp);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

int hfx_rows_build(uint32_t cus, const hfx_db *db, const hfx_rows *r, const uint32_t *flags,
                   void *stream)
{
    RbArgs a{};
    a.db = *db;
    a.ntiles = r->ntiles;
    for (int l = 0; l < HFX_MAX_CHARGE; ++l) a.rows[l] = r->rows[l];
    a.flags = flags;
    a.slots = r->slots;
    a.ng = r->ng;
    a.G = r->G;
    if (r->ntiles)
        hipLaunchKernelGGL(k_rw_build, dim3(std::min(r->ntiles, cus * RB_PER_CU)), dim3(RB_THREADS), 0, hfx_stream(stream), a);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* scratch of the work items of S spectra: tbeg, tend, binfo, items [S] each,
 * item_off [S + 1], counter */
size_t hfx_rows_items_bytes(uint32_t S) { return (size_t)S * 16 + ((size_t)S + 1) * 8 + 64; }

static void rw_items(void *p, uint32_t S, uint32_t **tbeg, uint32_t **tend, uint32_t **binfo,
                     uint32_t **items, uint64_t **off, uint32_t **counter)
{
    *off = (uint64_t *)(((uintptr_t)p + 7) & ~(uintptr_t)7);
    *tbeg = (uint32_t *)(*off + S + 1);
    *tend = *tbeg + S;
    *binfo = *tend + S;
    *items = *binfo + S;
    *counter = *items + S;
}

int hfx_rows_blocks(hfx_ctx *ctx, void *scratch, const uint32_t *order, const uint32_t *bstart,
                    const uint32_t *begin, const uint32_t *num, const hfx_spectra *sp, uint32_t CH,
                    void *stream)
{
    const uint32_t B = sp->num_spec;
    uint32_t *tbeg, *tend, *binfo, *items, *counter;
    uint64_t *off;
    rw_items(scratch, B, &tbeg, &tend, &binfo, &items, &off, &counter);
    hipStream_t st = hfx_stream(stream);
    const uint32_t CT = hfx_rows_item_tiles(CH);
    hipLaunchKernelGGL(k_rw_blocks, dim3((B + 15) / 16), dim3(256), 0, st, tbeg, tend, binfo, items,
                       counter, order, bstart, begin, num, *sp, B, CT);
    int rc = hfx_scan_offsets(ctx, off, items, B, stream);
    if (rc) return rc;
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

int hfx_rows_mark(void *scratch, uint32_t S, uint32_t *flags, uint32_t ntiles, void *stream)
{
    uint32_t *tbeg, *tend, *binfo, *items, *counter;
    uint64_t *off;
    rw_items(scratch, S, &tbeg, &tend, &binfo, &items, &off, &counter);
    hipStream_t st = hfx_stream(stream);
    const uint64_t n = (uint64_t)HFX_MAX_CHARGE * ntiles;
    hipLaunchKernelGGL(k_rw_fill, dim3((uint32_t)std::min<uint64_t>((n + 255) / 256, 2048)),
                       dim3(256), 0, st, flags, n, 0u);
    hipLaunchKernelGGL(k_rw_mark, dim3(S), dim3(256), 0, st, flags, tbeg, tend, binfo, ntiles);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

int hfx_rows_scores(hfx_ctx *ctx, int mode, void *scratch, float *d_scores, const uint64_t *d_off,
                    const uint32_t *begin, const uint32_t *num, const uint32_t *order,
                    const uint32_t *bstart, const hfx_rows *r, const uint8_t *planes,
                    const float *qs, const hfx_spectra *sp, uint32_t CH, void *stream, void **ev)
{
    const uint32_t S = sp->num_spec;
    uint32_t *tbeg, *tend, *binfo, *items, *counter;
    uint64_t *off;
    rw_items(scratch, S, &tbeg, &tend, &binfo, &items, &off, &counter);
    hipStream_t st = hfx_stream(stream);
    RmArgs a{};
    a.scores = d_scores;
    a.score_off = d_off;
    a.begin = begin;
    a.num = num;
    a.order = order;
    a.bstart = bstart;
    a.B = S;
    a.CT = hfx_rows_item_tiles(CH);
    a.tbeg = tbeg;
    a.tend = tend;
    a.binfo = binfo;
    a.item_off = off;
    a.planes = planes;
    a.qs = qs;
    a.counter = counter;
    for (int l = 0; l < HFX_MAX_CHARGE; ++l) a.rows[l] = r->rows[l];
    a.slots = r->slots;
    a.ng = r->ng;
    a.ntiles = r->ntiles;
    a.G = r->G;
    a.sp = *sp;
    const uint32_t lds = RW_NKS * (mode == RW_BF16 ? 2u : 3u) * 1024u;
    const uint32_t per_cu = lds * 2 <= 156u * 1024u ? 2u : 1u;
    const dim3 g((uint32_t)hfx_ctx_num_cus(ctx) * per_cu), t(RM_THREADS);
    const void *fn = mode == RW_I8X3   ? (const void *)k_rw_mm<RW_I8X3>
                     : mode == RW_I8X6 ? (const void *)k_rw_mm<RW_I8X6>
                                       : (const void *)k_rw_mm<RW_BF16>;
    HFX_CHECK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (ev) HFX_CHECK_HIP(hipEventRecord((hipEvent_t)ev[0], st));
    if (mode == RW_I8X3) hipLaunchKernelGGL(k_rw_mm<RW_I8X3>, g, t, lds, st, a);
    else if (mode == RW_I8X6) hipLaunchKernelGGL(k_rw_mm<RW_I8X6>, g, t, lds, st, a);
    else hipLaunchKernelGGL(k_rw_mm<RW_BF16>, g, t, lds, st, a);
    if (ev) HFX_CHECK_HIP(hipEventRecord((hipEvent_t)ev[1], st));
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}
