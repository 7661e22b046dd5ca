/*
 * hfx_db.hip -- database preparation and precursor windows.
 *
 *   prepare_ions       residue byte packing          (prepare_ions.cu:54-132)
 *   sort_idx_f & co    stable LSD radix sort          (sort.cu:20-76, sort_b40c.cu:34-41)
 *   findSpecCandsByMass, hfx_window                   (filter.cu:75-127)
 *   findBeginEnd_f                                    (filter_by_mod.cu:35-143)
 *   prepare_scoring                                   (prepare_scoring.cu:47-67)
 *   hfx_scan_offsets   exclusive scans used by every batched entry point
 */
#include "hfx_common.h"

/* ------------------------------------------------------------------ */
/* prepare_ions                                                          */
/* ------------------------------------------------------------------ */

/* bytes that start head bytes before the first multiple of sixteen: a thread
 * takes sixteen beside each other (9 MB: 18 us with a byte a
 * thread, 5.7 now) */
__global__ void __launch_bounds__(256) k_prepare_ions(uint8_t *ions, uint64_t n, const uint8_t *ma,
                                                      uint32_t num_ma)
{
    __shared__ uint8_t lut[256];
    {
        uint8_t mod = 0;
        for (uint32_t j = 0; j < num_ma; ++j)
            if (ma[j] == threadIdx.x) { mod = (uint8_t)(j + 1); break; }
        lut[threadIdx.x] = mod;
    }
    __syncthreads();
    auto packed = [&](uint32_t c) { return (uint32_t)(uint8_t)((uint8_t)(c - 'A') | (uint8_t)(lut[c] << 5)); };
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t head = min(n, (uint64_t)(-(uintptr_t)ions & 15u)), body = (n - head) / 16;
    if (i < body) {
        uint4 *p = (uint4 *)(ions + head) + i;
        const uint4 v = *p;
        uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t r = 0;
#pragma unroll
            for (int k = 0; k < 32; k += 8) r |= packed((w[q] >> k) & 255u) << k;
            w[q] = r;
        }
        *p = make_uint4(w[0], w[1], w[2], w[3]);
    }
    /* fewer than sixteen bytes at each end */
    const uint64_t tail = head + 16 * body;
    if (i < head) ions[i] = (uint8_t)packed(ions[i]);
    if (i < n - tail) ions[tail + i] = (uint8_t)packed(ions[tail + i]);
}

extern "C" void prepare_ions(uint8_t *d_ions, uint32_t N, uint8_t *d_ma, uint32_t num_ma)
{
    if (N == 0) return;
    if (num_ma > 7) { hfx_set_error("prepare_ions: num_ma %u > 7 (3-bit field)", num_ma); return; }
    const uint32_t blocks = (uint32_t)(((uint64_t)N + 16 * 256 - 1) / (16 * 256));
    const uint8_t *ma = num_ma ? d_ma : nullptr;
    hipLaunchKernelGGL(k_prepare_ions, dim3(blocks), dim3(256), 0, 0, d_ions, (uint64_t)N, ma,
                       num_ma);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("prepare_ions: %s", hipGetErrorString(e));
}

/* ------------------------------------------------------------------ */
/* Stable sorts of float keys with uint32 values                         */
/* ------------------------------------------------------------------ */

/* Exclusive scan of n uint32 in place by one workgroup of 1024 threads. */
__global__ void __launch_bounds__(1024) k_scan_u32_inplace(uint32_t *a, uint32_t n)
{
    __shared__ uint32_t warp_tot[16];
    __shared__ uint32_t carry_s;
    if (threadIdx.x == 0) carry_s = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (uint32_t base = 0; base < n; base += 1024) {
        uint32_t i = base + threadIdx.x;
        uint32_t v = i < n ? a[i] : 0;
        uint32_t x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) warp_tot[wid] = x;
        __syncthreads();
        uint32_t wpre = 0;
        for (uint32_t w = 0; w < wid; ++w) wpre += warp_tot[w];
        uint32_t carry = carry_s;
        if (i < n) a[i] = carry + wpre + x - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry_s = carry + wpre + x;
        __syncthreads();
    }
}

/* keys in radix order: ascending float order, or (desc) its reverse --
 * the complement of an order-preserving key reverses the order, and a
 * stable sort of the complements is a stable descending sort */
__device__ __forceinline__ uint32_t so_key(float f, uint32_t desc)
{
    return desc ? ~hfx_f2key(f) : hfx_f2key(f);
}
__device__ __forceinline__ float so_float(uint32_t k, uint32_t desc)
{
    return hfx_key2f(desc ? ~k : k);
}

/* keys among sk[ja .. jb) that come before key k of position i: smaller, or
 * equal and earlier.  Only the positions of the wave's own 64 keys (from i0 on)
 * need both tests.  Positions count from sk; i0 and i may lie outside it; ja, jb
 * and i0 are multiples of 4. */
__device__ __forceinline__ uint32_t so_before(const uint32_t *sk, int ja, int jb, int i0, int i,
                                              uint32_t k)
{
    uint32_t rk = 0;
    const uint4 *s4 = (const uint4 *)sk;
    const int a1 = min(jb, max(ja, i0)), a2 = min(jb, max(ja, i0 + HFX_WAVE));
    #pragma unroll 4
    for (int j = ja / 4; j < a1 / 4; ++j) {
        const uint4 o = s4[j];
        rk += (o.x <= k ? 1u : 0u) + (o.y <= k ? 1u : 0u) + (o.z <= k ? 1u : 0u) +
              (o.w <= k ? 1u : 0u);
    }
    for (int j = a1 / 4; j < a2 / 4; ++j) {
        const uint4 o = s4[j];
        rk += (o.x < k || (o.x == k && 4 * j < i)) ? 1u : 0u;
        rk += (o.y < k || (o.y == k && 4 * j + 1 < i)) ? 1u : 0u;
        rk += (o.z < k || (o.z == k && 4 * j + 2 < i)) ? 1u : 0u;
        rk += (o.w < k || (o.w == k && 4 * j + 3 < i)) ? 1u : 0u;
    }
    #pragma unroll 4
    for (int j = a2 / 4; j < jb / 4; ++j) {
        const uint4 o = s4[j];
        rk += (o.x < k ? 1u : 0u) + (o.y < k ? 1u : 0u) + (o.z < k ? 1u : 0u) +
              (o.w < k ? 1u : 0u);
    }
    return rk;
}

/* Up to SO_ONE keys: one launch of one workgroup, each key's place counted
 * against all others (key, then position: stable), four keys an LDS read, the
 * other keys shared out among the waves that a short list leaves over.  A call
 * with its synchronisation: 14.8 us for 256 keys, 18.4 for 512, 31.9 for 1024;
 * by k_sort_rank 16.2, 17.0, 18.2; by radix passes 67. */
#define SO_ONE 384u
#define SO_THREADS 1024u
__global__ void __launch_bounds__(SO_THREADS) k_sort_one(float *keys, uint32_t *vals, uint32_t n,
                                                         uint32_t iota, uint32_t init,
                                                         uint32_t desc)
{
    __shared__ __align__(16) uint32_t sk[SO_ONE];
    __shared__ uint32_t rank[SO_ONE];
    const uint32_t t = threadIdx.x;
    const uint32_t n64 = (n + HFX_WAVE - 1) / HFX_WAVE * HFX_WAVE;
    uint32_t k = 0xffffffffu, v = 0;
    if (t < n) {
        k = so_key(keys[t], desc);
        v = iota ? init + t : vals[t];
    }
    if (t < SO_ONE) {
        sk[t] = k; /* past the end: no key before another */
        rank[t] = 0;
    }
    __syncthreads();
    const uint32_t parts = SO_THREADS / n64, part = t / n64, i = t % n64;
    if (part < parts) {
        const uint32_t step = ((n64 + parts - 1) / parts + 3u) & ~3u;
        const uint32_t ja = min(part * step, n64), jb = min(ja + step, n64);
        const uint32_t rk = so_before(sk, (int)ja, (int)jb,
                                      (int)(i & ~(uint32_t)(HFX_WAVE - 1)), (int)i, sk[i]);
        if (i < n) atomicAdd(&rank[i], rk);
    }
    __syncthreads();
    /* every key and value is in registers: in place */
    if (t < n) {
        keys[rank[t]] = so_float(k, desc);
        vals[rank[t]] = v;
    }
}

/* Up to SO_RANK keys: the same count, a workgroup for 64 keys and its sixteen
 * waves a share of all others each, into scratch, which a second launch copies
 * back.  The count grows with n^2: 22.9 us for 4,096 keys, 28.9 for 8,192, 40.7
 * for 16,384, 71 for 24,576; radix passes 67 throughout.  (256 keys a workgroup
 * of four waves, each against all others: 89 for 4,096, 163 for 8,192.) */
#define SO_RANK 16384u
#define SO_CHUNK 8192u
__global__ void __launch_bounds__(SO_THREADS)
    k_sort_rank(const float *keys, const uint32_t *vals, float *okeys, uint32_t *ovals, uint32_t n,
                uint32_t iota, uint32_t init, uint32_t desc)
{
    __shared__ __align__(16) uint32_t sk[SO_CHUNK];
    __shared__ uint32_t rank[HFX_WAVE];
    const uint32_t wave = threadIdx.x / HFX_WAVE, i0 = blockIdx.x * HFX_WAVE;
    const uint32_t i = i0 + hfx_lane();
    const uint32_t k = i < n ? so_key(keys[i], desc) : 0xffffffffu;
    if (threadIdx.x < HFX_WAVE) rank[threadIdx.x] = 0;
    uint32_t rk = 0;
    for (uint32_t b = 0; b < n; b += SO_CHUNK) {
        const uint32_t m = (min(n - b, SO_CHUNK) + HFX_WAVE - 1) / HFX_WAVE * HFX_WAVE;
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < m; j += SO_THREADS)
            sk[j] = b + j < n ? so_key(keys[b + j], desc) : 0xffffffffu;
        __syncthreads();
        constexpr uint32_t W = SO_THREADS / HFX_WAVE;
        const uint32_t step = ((m + W - 1) / W + 3u) & ~3u;
        const uint32_t ja = min(wave * step, m), jb = min(ja + step, m);
        rk += so_before(sk, (int)ja, (int)jb, (int)i0 - (int)b, (int)i - (int)b, k);
    }
    if (rk) atomicAdd(&rank[hfx_lane()], rk);
    __syncthreads();
    if (wave == 0 && i < n) {
        const uint32_t r = rank[hfx_lane()];
        okeys[r] = so_float(k, desc);
        ovals[r] = iota ? init + i : vals[i];
    }
}
__global__ void k_sort_back(const float *k, const uint32_t *v, float *keys, uint32_t *vals,
                            uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        keys[i] = k[i];
        vals[i] = v[i];
    }
}

/* More: stable LSD radix, four passes of eight bits, three launches each:
 *   k_rs_count   a tile's digit counts, hist[digit][tile];
 *   k_rs_scan    one workgroup a digit: the exclusive scan of its row, and the
 *                digit's total;
 *   k_rs_place   a tile's keys ranked by digit (a wave matches its lanes'
 *                digits by eight ballots, wave after wave, so equal digits keep
 *                their order), put in digit order in LDS and written out in
 *                runs.
 * The first pass reads the caller's keys, the last writes them back, so that
 * no conversion or copy pass is left: 2.7 M keys take 130 us, against 560 us
 * with four bits a pass, a single-workgroup scan and separate conversions. */
#define RS_THREADS 512
#define RS_WAVES (RS_THREADS / HFX_WAVE)
#define RS_ITEMS 8
#define RS_TILE (RS_THREADS * RS_ITEMS)
#define RS_BUCKETS 256

struct RsArgs {
    const void *kin;        /* float keys in the first pass, radix keys after */
    const uint32_t *vin;    /* null in the first pass of an index sort */
    void *kout;             /* float keys in the last pass */
    uint32_t *vout;
    uint32_t n, shift, nb, first, last, desc, init;
    uint32_t *hist;         /* [RS_BUCKETS][nb] */
    uint32_t *tot;          /* [RS_BUCKETS] */
};

__device__ __forceinline__ uint32_t rs_load(const RsArgs &a, uint32_t g)
{
    return a.first ? so_key(((const float *)a.kin)[g], a.desc) : ((const uint32_t *)a.kin)[g];
}

__global__ void __launch_bounds__(RS_THREADS) k_rs_count(RsArgs a)
{
    __shared__ uint32_t cnt[RS_BUCKETS];
    if (threadIdx.x < RS_BUCKETS) cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * RS_TILE;
    uint32_t k[RS_ITEMS];
#pragma unroll
    for (uint32_t i = 0; i < RS_ITEMS; ++i) {
        const uint64_t g = base + i * RS_THREADS + threadIdx.x;
        k[i] = g < a.n ? rs_load(a, (uint32_t)g) : 0u;
    }
#pragma unroll
    for (uint32_t i = 0; i < RS_ITEMS; ++i)
        if (base + i * RS_THREADS + threadIdx.x < a.n)
            atomicAdd(&cnt[(k[i] >> a.shift) & 255u], 1u);
    __syncthreads();
    if (threadIdx.x < RS_BUCKETS)
        a.hist[(size_t)threadIdx.x * a.nb + blockIdx.x] = cnt[threadIdx.x];
}

__global__ void __launch_bounds__(256) k_rs_scan(RsArgs a)
{
    __shared__ uint32_t part[4];
    uint32_t *row = a.hist + (size_t)blockIdx.x * a.nb;
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (uint32_t b = 0; b < a.nb; b += 256) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = i < a.nb ? row[i] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) part[wid] = x;
        __syncthreads();
        uint32_t pre = carry, all = 0;
        for (uint32_t w = 0; w < 4; ++w) {
            if (w < wid) pre += part[w];
            all += part[w];
        }
        if (i < a.nb) row[i] = pre + x - v;
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) a.tot[blockIdx.x] = carry;
}

__global__ void __launch_bounds__(RS_THREADS) k_rs_place(RsArgs a)
{
    __shared__ uint32_t wcnt[RS_WAVES][RS_BUCKETS]; /* then: each wave's base in the tile */
    __shared__ uint32_t dbase[RS_BUCKETS];          /* a digit's first place in the tile */
    __shared__ uint32_t gbase[RS_BUCKETS];          /* in the output, less dbase */
    __shared__ uint32_t p1[RS_BUCKETS / HFX_WAVE], p2[RS_BUCKETS / HFX_WAVE];
    __shared__ uint32_t sk[RS_TILE], sv[RS_TILE];
    const uint32_t t = threadIdx.x, lane = hfx_lane(), w = t / HFX_WAVE;
    const uint64_t base = (uint64_t)blockIdx.x * RS_TILE;
    const uint32_t cnt = (uint32_t)min((uint64_t)RS_TILE, a.n - base);
    for (uint32_t i = t; i < RS_WAVES * RS_BUCKETS; i += RS_THREADS) (&wcnt[0][0])[i] = 0;
    /* wave w takes items w * 512 + 64 i + lane: in order over i, then lanes */
    uint32_t k[RS_ITEMS], v[RS_ITEMS], rank[RS_ITEMS];
#pragma unroll
    for (uint32_t i = 0; i < RS_ITEMS; ++i) {
        const uint32_t e = w * (HFX_WAVE * RS_ITEMS) + i * HFX_WAVE + lane;
        k[i] = 0;
        v[i] = 0;
        if (e < cnt) {
            const uint32_t g = (uint32_t)base + e;
            k[i] = rs_load(a, g);
            v[i] = a.vin ? a.vin[g] : a.init + g;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < RS_ITEMS; ++i) {
        const uint32_t e = w * (HFX_WAVE * RS_ITEMS) + i * HFX_WAVE + lane;
        const uint32_t d = (k[i] >> a.shift) & 255u;
        uint64_t same = __ballot(e < cnt);
#pragma unroll
        for (uint32_t b = 0; b < 8; ++b) {
            const uint64_t one = __ballot((d >> b) & 1u);
            same &= (d >> b) & 1u ? one : ~one;
        }
        /* the lanes of a digit count in lane order behind the wave's earlier
         * items; the first of them moves the counter on */
        const uint32_t before = (uint32_t)__builtin_popcountll(same & ((1ull << lane) - 1ull));
        uint32_t seen = 0;
        if (e < cnt) seen = wcnt[w][d];
        hfx_wave_sync();
        if (e < cnt && before == 0) wcnt[w][d] = seen + (uint32_t)__builtin_popcountll(same);
        hfx_wave_sync();
        rank[i] = seen + before;
    }
    __syncthreads();
    uint32_t ex = 0, ey = 0;
    if (t < RS_BUCKETS) {
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t q = 0; q < RS_WAVES; ++q) {
            const uint32_t c = wcnt[q][t];
            wcnt[q][t] = sum;
            sum += c;
        }
        /* exclusive scans over the digits: the tile's counts and the totals */
        const uint32_t tt = a.tot[t];
        uint32_t x = sum, y = tt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t p = __shfl_up(x, o, 64), q = __shfl_up(y, o, 64);
            if (lane >= (uint32_t)o) {
                x += p;
                y += q;
            }
        }
        if (lane == 63) {
            p1[w] = x;
            p2[w] = y;
        }
        ex = x - sum;
        ey = y - tt;
    }
    __syncthreads();
    if (t < RS_BUCKETS) {
        for (uint32_t q = 0; q < w; ++q) {
            ex += p1[q];
            ey += p2[q];
        }
        dbase[t] = ex;
        gbase[t] = ey + a.hist[(size_t)t * a.nb + blockIdx.x] - ex;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < RS_ITEMS; ++i) {
        if (w * (HFX_WAVE * RS_ITEMS) + i * HFX_WAVE + lane < cnt) {
            const uint32_t d = (k[i] >> a.shift) & 255u;
            const uint32_t at = dbase[d] + wcnt[w][d] + rank[i];
            sk[at] = k[i];
            sv[at] = v[i];
        }
    }
    __syncthreads();
    for (uint32_t j = t; j < cnt; j += RS_THREADS) {
        const uint32_t kk = sk[j];
        const uint32_t g = gbase[(kk >> a.shift) & 255u] + j;
        if (a.last) ((float *)a.kout)[g] = so_float(kk, a.desc);
        else ((uint32_t *)a.kout)[g] = kk;
        a.vout[g] = sv[j];
    }
}

/* Sorts float keys ascending (or descending) with values, stably, in place. */
static int radix_sort_f32(hfx_ctx *ctx, float *d_keys, uint32_t *d_vals, uint32_t n, bool iota,
                          uint32_t init, hipStream_t st, uint32_t desc = 0)
{
    if (n == 0) return HFX_OK;
    if (n <= SO_ONE) {
        hipLaunchKernelGGL(k_sort_one, dim3(1), dim3(SO_THREADS), 0, st, d_keys, d_vals, n,
                           (uint32_t)iota, init, desc);
        HFX_CHECK_LAUNCH();
        return HFX_OK;
    }
    const uint32_t nb = (uint32_t)(((uint64_t)n + RS_TILE - 1) / RS_TILE);
    void *p;
    int rc;
    if ((rc = hfx_ctx_scratch(ctx, HFX_SLOT_SORT,
                              (size_t)n * 16 + ((size_t)nb + 1) * RS_BUCKETS * 4, &p)) != HFX_OK)
        return rc;
    uint32_t *ka = (uint32_t *)p, *va = ka + n, *kb = va + n, *vb = kb + n, *hist = vb + n;
    if (n <= SO_RANK) {
        hipLaunchKernelGGL(k_sort_rank, dim3((n + HFX_WAVE - 1) / HFX_WAVE), dim3(SO_THREADS), 0, st,
                           d_keys, d_vals, (float *)ka, va, n, (uint32_t)iota, init, desc);
        hipLaunchKernelGGL(k_sort_back, dim3((n + 255) / 256), dim3(256), 0, st, (float *)ka, va,
                           d_keys, d_vals, n);
        HFX_CHECK_LAUNCH();
        return HFX_OK;
    }
    /* caller -> a -> b -> a -> caller */
    const void *ks[4] = {d_keys, ka, kb, ka};
    const uint32_t *vs[4] = {iota ? nullptr : d_vals, va, vb, va};
    void *kd[4] = {ka, kb, ka, d_keys};
    uint32_t *vd[4] = {va, vb, va, d_vals};
    for (uint32_t q = 0; q < 4; ++q) {
        const RsArgs a{ks[q],   vs[q], kd[q], vd[q], n,    8 * q, nb, q == 0, q == 3, desc,
                       init,    hist,  hist + (size_t)nb * RS_BUCKETS};
        hipLaunchKernelGGL(k_rs_count, dim3(nb), dim3(RS_THREADS), 0, st, a);
        hipLaunchKernelGGL(k_rs_scan, dim3(RS_BUCKETS), dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_rs_place, dim3(nb), dim3(RS_THREADS), 0, st, a);
    }
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

extern "C" void sort_idx_f(float *d_keys_raw, uint32_t *d_idx_raw, uint32_t N, uint32_t init)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    if (radix_sort_f32(ctx, d_keys_raw, d_idx_raw, N, true, init, 0) == HFX_OK)
        (void)hipStreamSynchronize(0);
}

extern "C" void sort_val_f(float *d_keys, uint32_t *d_vals, uint32_t N)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    if (radix_sort_f32(ctx, d_keys, d_vals, N, false, 0, 0) == HFX_OK) (void)hipStreamSynchronize(0);
}

extern "C" void sort_rf(float *d_keys, uint32_t *d_vals, uint32_t N)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    if (radix_sort_f32(ctx, d_keys, d_vals, N, false, 0, 0, 1) == HFX_OK)
        (void)hipStreamSynchronize(0);
}

extern "C" void sort_idx_rf(float *d_keys_raw, uint32_t *d_idx_raw, uint32_t N, uint32_t init)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    if (radix_sort_f32(ctx, d_keys_raw, d_idx_raw, N, true, init, 0, 1) == HFX_OK)
        (void)hipStreamSynchronize(0);
}

/* findIndicesInRange_f (filter.cu:38-73): the indices i, ascending, with
 * min <= d_in[i] <= max; stable compaction (flags, offsets, scatter) */
__global__ void k_range_flags(uint32_t *flag, const float *in, uint32_t n, float lo, float hi)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = (lo <= in[i] && in[i] <= hi) ? 1u : 0u;
}
__global__ void k_range_scatter(uint32_t *out, const uint32_t *flag, const uint64_t *pos, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && flag[i]) out[pos[i]] = i;
}

extern "C" uint32_t findIndicesInRange_f(const float *d_in, uint32_t *d_out, const uint32_t N,
                                         const float min, const float max)
{
    if (N == 0) return 0;
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return 0;
    void *p = nullptr, *h = nullptr;
    const size_t fb = ((size_t)N * 4 + 255) & ~(size_t)255;
    if (hfx_ctx_scratch(ctx, HFX_SLOT_SCAN, fb + ((size_t)N + 1) * 8, &p) != HFX_OK) return 0;
    if (hfx_ctx_pinned(ctx, 16, &h) != HFX_OK) return 0;
    uint32_t *flag = (uint32_t *)p;
    uint64_t *pos = (uint64_t *)((uint8_t *)p + fb);
    const uint32_t g = (N + 255) / 256;
    hipLaunchKernelGGL(k_range_flags, dim3(g), dim3(256), 0, 0, flag, d_in, N, min, max);
    if (hfx_scan_offsets(ctx, pos, flag, N, nullptr) != HFX_OK) return 0;
    hipLaunchKernelGGL(k_range_scatter, dim3(g), dim3(256), 0, 0, d_out, flag, pos, N);
    if (hipMemcpyAsync(h, pos + N, 8, hipMemcpyDeviceToHost, 0) != hipSuccess ||
        hipStreamSynchronize(0) != hipSuccess) {
        hfx_set_error("findIndicesInRange_f: %s", hipGetErrorString(hipGetLastError()));
        return 0;
    }
    return (uint32_t)*(uint64_t *)h;
}

extern "C" void sort_b40c_f(float *d_keys, uint32_t *d_vals, uint32_t N)
{
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    if (radix_sort_f32(ctx, d_keys, d_vals, N, false, 0, 0) == HFX_OK) (void)hipStreamSynchronize(0);
}

/* ------------------------------------------------------------------ */
/* Precursor windows                                                     */
/* ------------------------------------------------------------------ */

/* lower_bound of lo and upper_bound of hi over r[idx[i]] (thrust's
 * permutation_iterator form, filter.cu:101-115); idx == nullptr reads r directly
 * (sorted copy).  Both at once by a wave, a probe a lane: four steps for 2.7 M
 * peptides, where a thread that bisects waits for 44 reads one after the other
 * (250 spectra: 20 -> 5.0 us a launch; 10,000: 18.8 -> 12.8).  All lanes return both. */
__device__ __forceinline__ void db_bounds_wave(const float *r, const uint32_t *idx, uint32_t n,
                                               float lo, float hi, uint32_t *begin, uint32_t *end)
{
    const uint32_t lane = threadIdx.x & 63u;
    /* the result lies in [at, at + left] */
    uint32_t at[2] = {0, 0}, left[2] = {n, n};
    while (left[0] | left[1]) {
        uint32_t k[2], step[2];
        float v[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            step[w] = left[w] / 64 + (left[w] % 64 ? 1u : 0u);
            /* the last of part `lane`; of a search that is done, anything */
            const uint64_t last = min((uint64_t)step[w] * (lane + 1u), (uint64_t)left[w]);
            k[w] = min(at[w] + (last ? (uint32_t)last - 1u : 0u), n - 1u);
        }
        if (idx) {
            k[0] = idx[k[0]];
            k[1] = idx[k[1]];
        }
        v[0] = r[k[0]];
        v[1] = r[k[1]];
        const uint64_t in[2] = {__ballot(v[0] < lo), __ballot(!(hi < v[1]))};
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t c = (uint32_t)__popcll(in[w]);
            const uint32_t go = (uint32_t)min((uint64_t)c * step[w], (uint64_t)left[w]);
            at[w] += go;
            /* into the part whose last is not below */
            left[w] = go == left[w] ? 0u : min(step[w], left[w] - go) - 1u;
        }
    }
    *begin = at[0];
    *end = at[1];
}

/* the same by a thread, seven probes a step of each, all in flight: eight steps
 * for 2.7 M */
template <bool IDX>
__device__ __forceinline__ void db_bounds(const float *r, const uint32_t *idx, uint32_t n, float lo,
                                          float hi, uint32_t *begin, uint32_t *end)
{
    uint32_t at[2] = {0, 0}, left[2] = {n, n};
    while (left[0] | left[1]) {
        uint32_t step[2], k[2][7];
        float v[2][7];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            step[w] = (left[w] + 7) / 8;
#pragma unroll
            for (uint32_t j = 0; j < 7; ++j)
                k[w][j] = min(at[w] + max(min(step[w] * (j + 1), left[w]), 1u) - 1u, n - 1u);
        }
        if constexpr (IDX)
#pragma unroll
            for (uint32_t j = 0; j < 14; ++j) k[j / 7][j % 7] = idx[k[j / 7][j % 7]];
#pragma unroll
        for (uint32_t j = 0; j < 14; ++j) v[j / 7][j % 7] = r[k[j / 7][j % 7]];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint32_t c = 0;
#pragma unroll
            for (uint32_t j = 0; j < 7; ++j) c += (w == 0 ? v[w][j] < lo : !(hi < v[w][j])) ? 1u : 0u;
            const uint32_t go = min(c * step[w], left[w]), rest = left[w] - go;
            at[w] += go;
            /* past seven parts: the eighth; else a part whose last is not below */
            left[w] = c == 7 ? rest : min(step[w], rest) - (rest ? 1u : 0u);
        }
    }
    *begin = at[0];
    *end = at[1];
}

__global__ void __launch_bounds__(256)
    k_window(uint32_t *begin, uint32_t *end, uint32_t *num, const float *r, const uint32_t *idx,
             uint32_t num_pep, const float *mass, uint32_t num_spec, float eps)
{
    const uint32_t s = blockIdx.x * 4 + threadIdx.x / 64;
    if (s >= num_spec) return;
    uint32_t b, e;
    db_bounds_wave(r, idx, num_pep, mass[s] - eps, mass[s] + eps, &b, &e);
    if ((threadIdx.x & 63u) == 0) {
        if (begin) begin[s] = b;
        if (end) end[s] = e;
        num[s] = e - b;
    }
}

/* sum of n uint32 (wrapping, like thrust::reduce on uint32) into *out */
__global__ void __launch_bounds__(1024) k_sum_u32(const uint32_t *a, uint32_t n, uint32_t *out)
{
    __shared__ uint32_t part[16];
    uint32_t s = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024) s += a[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < 16; ++w) t += part[w];
        *out = t;
    }
}

/* partial sums of n uint32: block b adds elements b, b + G*1024, ... (G
 * blocks of 1024 threads) into part[b] */
__global__ void __launch_bounds__(1024) k_sum_part(const uint32_t *a, uint32_t n, uint32_t *part)
{
    __shared__ uint32_t w[16];
    uint32_t s = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * 1024 + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * 1024)
        s += a[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int i = 0; i < 16; ++i) t += w[i];
        part[blockIdx.x] = t;
    }
}

#define SUM_BLOCKS 512u

uint32_t hfx_sum_u32_to_host(hfx_ctx *ctx, const uint32_t *d_a, uint32_t n)
{
    void *p, *h;
    if (hfx_ctx_scratch(ctx, HFX_SLOT_SUM, 16 + 4 * SUM_BLOCKS, &p) != HFX_OK) return 0;
    if (hfx_ctx_pinned(ctx, 16, &h) != HFX_OK) return 0;
    if (n > 65536u) {
        /* many workgroups, then one over their sums (integer: any order) */
        const uint32_t g = min(SUM_BLOCKS, (n + 8191u) / 8192u);
        uint32_t *part = (uint32_t *)p + 4;
        hipLaunchKernelGGL(k_sum_part, dim3(g), dim3(1024), 0, 0, d_a, n, part);
        hipLaunchKernelGGL(k_sum_u32, dim3(1), dim3(1024), 0, 0, part, g, (uint32_t *)p);
    } else {
        hipLaunchKernelGGL(k_sum_u32, dim3(1), dim3(1024), 0, 0, d_a, n, (uint32_t *)p);
    }
    if (hipMemcpyAsync(h, p, 4, hipMemcpyDeviceToHost, 0) != hipSuccess) return 0;
    if (hipStreamSynchronize(0) != hipSuccess) {
        hfx_set_error("sum_to_host: synchronize failed");
        return 0;
    }
    return *(uint32_t *)h;
}

extern "C" uint32_t findSpecCandsByMass(uint32_t *d_spec_begin_raw, uint32_t *d_spec_end_raw,
                                        uint32_t *d_spec_num_pep_raw, const float *d_r_raw,
                                        const uint32_t *d_pep_idx_r_sorted_raw,
                                        const uint32_t num_pep, const float *d_spec_masses_raw,
                                        const uint32_t num_spec, const float eps)
{
    if (num_spec == 0) return 0;
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return 0;
    hipLaunchKernelGGL(k_window, dim3((num_spec + 3) / 4), dim3(256), 0, 0, d_spec_begin_raw,
                       d_spec_end_raw, d_spec_num_pep_raw, d_r_raw, d_pep_idx_r_sorted_raw, num_pep,
                       d_spec_masses_raw, num_spec, eps);
    return hfx_sum_u32_to_host(ctx, d_spec_num_pep_raw, num_spec);
}

extern "C" int hfx_window(hfx_ctx *ctx, uint32_t *d_begin, uint32_t *d_num, const hfx_db *db,
                          const float *d_spec_mass, uint32_t num_spec, float eps, void *stream)
{
    HFX_REQUIRE(ctx && db && d_begin && d_num, HFX_ERR_ARG, "hfx_window: null argument");
    if (num_spec == 0) return HFX_OK;
    const float *r = db->d_r_sorted ? db->d_r_sorted : db->d_r;
    const uint32_t *idx = db->d_r_sorted ? nullptr : db->d_idx_sorted;
    hipLaunchKernelGGL(k_window, dim3((num_spec + 3) / 4), dim3(256), 0, hfx_stream(stream),
                       d_begin, (uint32_t *)nullptr, d_num, r, idx, db->num_pep, d_spec_mass,
                       num_spec, eps);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

__global__ void k_begin_end_mod(uint32_t *begin, uint32_t *end, uint32_t *cnt, const float *r,
                                const uint32_t *idx, uint32_t num_pep, const float *delta,
                                uint32_t num_mod, float lo0, float hi0)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_mod) return;
    uint32_t b, e;
    if (idx) db_bounds<true>(r, idx, num_pep, lo0 - delta[i], hi0 - delta[i], &b, &e);
    else db_bounds<false>(r, idx, num_pep, lo0 - delta[i], hi0 - delta[i], &b, &e);
    begin[i] = b;
    end[i] = e;
    cnt[i] = e - b;
}

extern "C" uint32_t findBeginEnd_f(uint32_t *d_begin_raw, uint32_t *d_end_raw,
                                   uint32_t *d_num_pep_scan_raw, const float *d_r_raw,
                                   const uint32_t *d_pep_idx_r_sorted_raw, const uint32_t num_pep,
                                   const float *d_mod_delta_raw, const uint32_t num_mod,
                                   const float mass_, const float eps)
{
    if (num_mod == 0) return 0;
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return 0;
    float lo0 = mass_ - eps, hi0 = mass_ + eps;
    hipLaunchKernelGGL(k_begin_end_mod, dim3((num_mod + 255) / 256), dim3(256), 0, 0, d_begin_raw,
                       d_end_raw, d_num_pep_scan_raw, d_r_raw, d_pep_idx_r_sorted_raw, num_pep,
                       d_mod_delta_raw, num_mod, lo0, hi0);
    uint32_t total = hfx_sum_u32_to_host(ctx, d_num_pep_scan_raw, num_mod);
    hipLaunchKernelGGL(k_scan_u32_inplace, dim3(1), dim3(1024), 0, 0, d_num_pep_scan_raw, num_mod);
    if (hipStreamSynchronize(0) != hipSuccess) hfx_set_error("findBeginEnd_f: sync failed");
    return total;
}

/* findBeginEnd_f for many spectra in one launch: a wave a spectrum, a lane a
 * modification; the prefix sums of its lanes are the reference's per-spectrum
 * scan.  One thread a spectrum took 205 us for 5,000 spectra and 34
 * modifications, 18 now. */
template <bool IDX>
__global__ void __launch_bounds__(256)
    k_mod_windows(uint32_t *begin, uint32_t *end, uint32_t *scan, uint32_t *spec_cand,
                  const float *r, const uint32_t *idx, uint32_t num_pep, const float *delta,
                  uint32_t num_mod, const float *mass, uint32_t num_spec, float eps)
{
    const uint32_t s = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (s >= num_spec) return;
    const float lo0 = mass[s] - eps, hi0 = mass[s] + eps;
    uint32_t acc = 0;
    for (uint32_t i0 = 0; i0 < num_mod; i0 += 64) {
        const uint32_t i = i0 + lane;
        uint32_t b = 0, e = 0;
        if (i < num_mod) db_bounds<IDX>(r, idx, num_pep, lo0 - delta[i], hi0 - delta[i], &b, &e);
        uint32_t x = e - b;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (i < num_mod) {
            const size_t o = (size_t)s * num_mod + i;
            begin[o] = b;
            end[o] = e;
            scan[o] = acc + x - (e - b);
        }
        acc += (uint32_t)__shfl((int)x, 63, 64);
    }
    if (lane == 0) spec_cand[s] = acc;
}

extern "C" int hfx_mod_windows(hfx_ctx *ctx, uint32_t *d_begin, uint32_t *d_end,
                               uint32_t *d_num_scan, uint32_t *d_spec_cand, const hfx_db *db,
                               const float *d_spec_mass, uint32_t num_spec,
                               const float *d_mod_delta, uint32_t num_mod, float eps,
                               void *stream)
{
    HFX_REQUIRE(ctx && db && d_begin && d_end && d_num_scan && d_spec_cand && d_spec_mass,
                HFX_ERR_ARG, "hfx_mod_windows: null argument");
    HFX_REQUIRE(num_mod == 0 || d_mod_delta, HFX_ERR_ARG, "hfx_mod_windows: null deltas");
    if (num_spec == 0) return HFX_OK;
    const float *r = db->d_r_sorted ? db->d_r_sorted : db->d_r;
    const uint32_t *idx = db->d_r_sorted ? nullptr : db->d_idx_sorted;
    hipLaunchKernelGGL(idx ? k_mod_windows<true> : k_mod_windows<false>, dim3((num_spec + 3) / 4),
                       dim3(256), 0,
                       hfx_stream(stream), d_begin, d_end, d_num_scan, d_spec_cand, r, idx,
                       db->num_pep, d_mod_delta, num_mod, d_spec_mass, num_spec, eps);
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

/* ------------------------------------------------------------------ */
/* Offsets and candidate lists                                           */
/* ------------------------------------------------------------------ */

/* inclusive prefix sum over the wave by lane moves: rows of 16 by shifts of 1,
 * 2, 4 and 8, then across rows */
template <int CTRL, int ROWS>
__device__ __forceinline__ uint64_t sc_step(uint64_t x)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), CTRL, ROWS,
                                                              0xf, false);
    return x + ((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ uint64_t sc_wave_incl(uint64_t x)
{
    x = sc_step<0x111, 0xf>(x);
    x = sc_step<0x112, 0xf>(x);
    x = sc_step<0x114, 0xf>(x);
    x = sc_step<0x118, 0xf>(x);
    x = sc_step<0x142, 0xa>(x);
    x = sc_step<0x143, 0xc>(x);
    return x;
}
__device__ __forceinline__ uint64_t sc_last(uint64_t x)
{
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), 63) << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, 63);
}
/* exclusive prefix sums of a wave's counts v[q], in order of (q, lane); returns
 * their sum */
template <int Q>
__device__ __forceinline__ uint64_t sc_wave_scan(const uint32_t (&v)[Q], uint64_t (&x)[Q])
{
    uint64_t sum = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const uint64_t incl = sc_wave_incl(v[q]);
        x[q] = sum + incl - v[q];
        sum += sc_last(incl);
    }
    return sum;
}

/* four counts / two offsets beside each other, at their own alignment */
typedef uint32_t sc_u4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint64_t sc_l2 __attribute__((ext_vector_type(2), aligned(8)));

/* Exclusive scan of n uint32 counts into n+1 uint64 offsets, one workgroup, Q
 * counts beside each other a thread: one pass for 1024 Q of them.  (A single CU
 * cannot afford a wave scan for each count: 7.5 us for 5000, Q = 1 over five
 * passes 8.5, 4.3 now.) */
template <int Q>
__global__ void __launch_bounds__(1024) k_scan_offsets(uint64_t *off, const uint32_t *cnt, uint32_t n)
{
    __shared__ uint64_t warp_tot[2][16];
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint64_t carry = 0;
    uint32_t turn = 0;
    for (uint64_t base = 0; base < n; base += 1024 * Q, turn ^= 1) {
        const uint64_t first = base + (uint64_t)threadIdx.x * Q;
        const bool all = Q % 4 == 0 && first + Q <= n;
        uint32_t v[Q];
        if (all) {
#pragma unroll
            for (int q = 0; q + 3 < Q; q += 4) {
                const sc_u4 t = *(const sc_u4 *)(cnt + first + q);
                v[q] = t[0];
                v[q + 1] = t[1];
                v[q + 2] = t[2];
                v[q + 3] = t[3];
            }
        } else {
#pragma unroll
            for (int q = 0; q < Q; ++q) v[q] = first + q < n ? cnt[first + q] : 0u;
        }
        uint64_t sum = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) sum += v[q];
        const uint64_t incl = sc_wave_incl(sum);
        if (lane == 63) warp_tot[turn][wid] = incl;
        __syncthreads();
        uint64_t x = carry + incl - sum;
#pragma unroll
        for (uint32_t w = 0; w < 16; ++w) {
            x += w < wid ? warp_tot[turn][w] : 0;
            carry += warp_tot[turn][w];
        }
        if (all) {
#pragma unroll
            for (int q = 0; q + 1 < Q; q += 2) {
                *(sc_l2 *)(off + first + q) = sc_l2{x, x + v[q]};
                x += (uint64_t)v[q] + v[q + 1];
            }
        } else {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                if (first + q < n) off[first + q] = x;
                x += v[q];
            }
        }
    }
    if (threadIdx.x == 0) off[n] = carry;
}

static void scan_offsets_one(uint64_t *off, const uint32_t *cnt, uint32_t n, hipStream_t st)
{
    if (n <= 1024) hipLaunchKernelGGL(k_scan_offsets<1>, dim3(1), dim3(1024), 0, st, off, cnt, n);
    else if (n <= 4096) hipLaunchKernelGGL(k_scan_offsets<4>, dim3(1), dim3(1024), 0, st, off, cnt, n);
    else hipLaunchKernelGGL(k_scan_offsets<16>, dim3(1), dim3(1024), 0, st, off, cnt, n);
}

/* Multi-workgroup form (reduce, then scan), with no scratch: the offsets
 * array itself carries the tile totals between the passes.
 *   k_scan_tile_sums   tile b (SC_TILE counts) writes its sum to
 *                      off[min((b + 1) SC_TILE, n)];
 *   k_scan_tile_bases  one workgroup turns those entries, and off[0] = 0,
 *                      into the exclusive prefix of each tile (inclusive
 *                      prefix of the sums: the entry at (b + 1) SC_TILE is
 *                      tile b + 1's base, the one at n the total);
 *   k_scan_tiles       tile b reads its base from off[b SC_TILE] and writes
 *                      off[b SC_TILE + i] for its counts (the first one
 *                      being the base again); no other tile touches them. */
#define SC_THREADS 1024
#define SC_ITEMS 8
#define SC_TILE (SC_THREADS * SC_ITEMS)
/* below this count one workgroup's passes are quicker than three launches:
 * 10,000 counts take 5.8 us, the launches 4.7 + 2.5 + 6.4 and their gaps; a
 * second pass adds 3 */
#define SC_SMALL 32768u

__device__ __forceinline__ uint64_t sc_block_sum(uint64_t v, uint64_t *part)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (int w = 0; w < SC_THREADS / 64; ++w) t += part[w];
    return t;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_tile_sums(uint64_t *off, const uint32_t *cnt,
                                                               uint32_t n)
{
    __shared__ uint64_t part[SC_THREADS / 64];
    const uint64_t base = (uint64_t)blockIdx.x * SC_TILE;
    uint64_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k) {
        const uint64_t i = base + k * SC_THREADS + threadIdx.x;
        if (i < n) s += cnt[i];
    }
    const uint64_t t = sc_block_sum(s, part);
    if (threadIdx.x == 0) off[min(base + SC_TILE, (uint64_t)n)] = t;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_tile_bases(uint64_t *off, uint32_t n,
                                                                uint32_t ntiles)
{
    __shared__ uint64_t warp_tot[SC_THREADS / 64];
    __shared__ uint64_t carry_s;
    if (threadIdx.x == 0) {
        carry_s = 0;
        off[0] = 0;
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (uint32_t b0 = 0; b0 < ntiles; b0 += SC_THREADS) {
        const uint32_t b = b0 + threadIdx.x;
        const uint64_t at = min((uint64_t)(b + 1) * SC_TILE, (uint64_t)n);
        const uint64_t v = b < ntiles ? off[at] : 0;
        uint64_t x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint64_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) warp_tot[wid] = x;
        __syncthreads();
        uint64_t wpre = 0;
        for (uint32_t w = 0; w < wid; ++w) wpre += warp_tot[w];
        const uint64_t carry = carry_s;
        if (b < ntiles) off[at] = carry + wpre + x;
        __syncthreads();
        if (threadIdx.x == SC_THREADS - 1) carry_s = carry + wpre + x;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(SC_THREADS) k_scan_tiles(uint64_t *off, const uint32_t *cnt,
                                                           uint32_t n)
{
    __shared__ uint64_t warp_tot[SC_THREADS / 64];
    const uint64_t base = (uint64_t)blockIdx.x * SC_TILE;
    const uint64_t tile_base = off[base];
    /* a wave takes SC_ITEMS * 64 counts, its lanes beside each other */
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t first = base + wid * 64 * SC_ITEMS + lane;
    uint32_t v[SC_ITEMS];
    uint64_t x[SC_ITEMS];
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k) v[k] = first + 64 * k < n ? cnt[first + 64 * k] : 0u;
    const uint64_t sum = sc_wave_scan(v, x);
    if (lane == 0) warp_tot[wid] = sum;
    __syncthreads();
    uint64_t pre = tile_base;
    for (uint32_t w = 0; w < wid; ++w) pre += warp_tot[w];
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k)
        if (first + 64 * k < n) off[first + 64 * k] = pre + x[k];
}

/* In-place exclusive scan of n uint32 (wrapping) over many workgroups:
 * tile sums (SC_TILE elements a tile) into scratch, one workgroup scans
 * them, each tile then scans its own elements from its base. */
__global__ void __launch_bounds__(SC_THREADS) k_scan32_tile_sums(const uint32_t *a, uint32_t n,
                                                                 uint32_t *sums)
{
    __shared__ uint64_t part[SC_THREADS / 64];
    const uint64_t base = (uint64_t)blockIdx.x * SC_TILE;
    uint64_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k) {
        const uint64_t i = base + k * SC_THREADS + threadIdx.x;
        if (i < n) s += a[i];
    }
    const uint64_t t = sc_block_sum(s, part);
    if (threadIdx.x == 0) sums[blockIdx.x] = (uint32_t)t;
}

__global__ void __launch_bounds__(SC_THREADS) k_scan32_tiles(uint32_t *a, uint32_t n,
                                                             const uint32_t *sums)
{
    __shared__ uint32_t warp_tot[SC_THREADS / 64];
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t first = (uint64_t)blockIdx.x * SC_TILE + wid * 64 * SC_ITEMS + lane;
    uint32_t v[SC_ITEMS];
    uint64_t x[SC_ITEMS];
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k) v[k] = first + 64 * k < n ? a[first + 64 * k] : 0u;
    const uint64_t sum = sc_wave_scan(v, x);
    if (lane == 0) warp_tot[wid] = (uint32_t)sum;
    __syncthreads();
    uint32_t pre = sums[blockIdx.x];
    for (uint32_t w = 0; w < wid; ++w) pre += warp_tot[w];
#pragma unroll
    for (uint32_t k = 0; k < SC_ITEMS; ++k)
        if (first + 64 * k < n) a[first + 64 * k] = pre + (uint32_t)x[k];
}

int hfx_scan_u32_inplace(uint32_t *d_a, uint32_t n, void *stream)
{
    if (n == 0) return HFX_OK;
    hipStream_t st = hfx_stream(stream);
    if (n < SC_SMALL) {
        hipLaunchKernelGGL(k_scan_u32_inplace, dim3(1), dim3(1024), 0, st, d_a, n);
    } else {
        const uint32_t nt = (uint32_t)(((uint64_t)n + SC_TILE - 1) / SC_TILE);
        hfx_ctx *ctx = hfx_default_ctx();
        HFX_REQUIRE(ctx, HFX_ERR_HIP, "hfx_scan_u32_inplace: no context");
        void *p = nullptr;
        int rc = hfx_ctx_scratch(ctx, HFX_SLOT_SCAN2, (size_t)4 * nt, &p);
        if (rc) return rc;
        uint32_t *sums = (uint32_t *)p;
        hipLaunchKernelGGL(k_scan32_tile_sums, dim3(nt), dim3(SC_THREADS), 0, st, d_a, n, sums);
        hipLaunchKernelGGL(k_scan_u32_inplace, dim3(1), dim3(1024), 0, st, sums, nt);
        hipLaunchKernelGGL(k_scan32_tiles, dim3(nt), dim3(SC_THREADS), 0, st, d_a, n, sums);
    }
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

extern "C" int hfx_scan_offsets(hfx_ctx *ctx, uint64_t *d_off, const uint32_t *d_count, uint32_t n,
                                void *stream)
{
    (void)ctx;
    HFX_REQUIRE(d_off != nullptr, HFX_ERR_ARG, "hfx_scan_offsets: null output");
    hipStream_t st = hfx_stream(stream);
    if (n < SC_SMALL) {
        scan_offsets_one(d_off, d_count, n, st);
    } else {
        const uint32_t nt = (uint32_t)(((uint64_t)n + SC_TILE - 1) / SC_TILE);
        hipLaunchKernelGGL(k_scan_tile_sums, dim3(nt), dim3(SC_THREADS), 0, st, d_off, d_count, n);
        hipLaunchKernelGGL(k_scan_tile_bases, dim3(1), dim3(SC_THREADS), 0, st, d_off, n, nt);
        hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(SC_THREADS), 0, st, d_off, d_count, n);
    }
    HFX_CHECK_LAUNCH();
    return HFX_OK;
}

__global__ void k_prepare_scoring(uint32_t *out, const uint32_t *idx, const uint32_t *begin,
                                  const uint32_t *num, const uint64_t *off)
{
    uint32_t s = blockIdx.x;
    uint32_t b = begin[s], n = num[s];
    uint64_t o = off[s];
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) out[o + i] = idx[b + i];
}

extern "C" void prepare_scoring(uint32_t *d_out_spec_pep_idx, const uint32_t *d_pep_idx_r_sorted_raw,
                                const uint32_t *d_spec_begin, const uint32_t *d_spec_num_pep,
                                const uint32_t num_spec)
{
    if (num_spec == 0) return;
    hfx_ctx *ctx = hfx_default_ctx();
    if (!ctx) return;
    void *p;
    if (hfx_ctx_scratch(ctx, HFX_SLOT_SCAN, ((size_t)num_spec + 1) * 8, &p) != HFX_OK) return;
    uint64_t *off = (uint64_t *)p;
    scan_offsets_one(off, d_spec_num_pep, num_spec, 0);
    hipLaunchKernelGGL(k_prepare_scoring, dim3(num_spec), dim3(256), 0, 0, d_out_spec_pep_idx,
                       d_pep_idx_r_sorted_raw, d_spec_begin, d_spec_num_pep, off);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) hfx_set_error("prepare_scoring: %s", hipGetErrorString(e));
}
