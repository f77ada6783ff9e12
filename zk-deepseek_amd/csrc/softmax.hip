// Fixed-point row softmax over the last dimension of [Bsz,S,H,T] int64 (Q19 truncating, Q21 rounding).
//
// Rows of up to 2048 elements are handled one row per wavefront (or, few rows, per four of them): the row is read once with 16-byte loads
// into registers, the maximum and the weight sum are 64-lane butterfly reductions, and the per-row divide
// is a reciprocal multiply made exact by a remainder test.  HBM traffic is the algorithmic 16 bytes per
// element (24 when the reference's write-back of the weights into the input is switched on).
// Longer rows use one workgroup per row and three passes.
//
// Arithmetic follows inference/int64_gemm.cu:684-746 (Q19) and :605-659 (Q21).
#include "common.h"
#include "../../include/int64gemm.h"

namespace zk {

static bool g_softmax_clobber = false;

struct __attribute__((aligned(16))) i64x2s { int64_t x, y; };
typedef int v4i_s __attribute__((ext_vector_type(4)));

// Streaming 16-byte accesses: every byte is touched exactly once, so the loads and stores are marked
// non-temporal and do not displace anything from the caches.
__device__ __forceinline__ i64x2s ld_stream(const i64x2s *p)
{
    v4i_s t = __builtin_nontemporal_load(reinterpret_cast<const v4i_s *>(p));
    i64x2s r;
    r.x = (int64_t)(((uint64_t)(uint32_t)t[1] << 32) | (uint32_t)t[0]);
    r.y = (int64_t)(((uint64_t)(uint32_t)t[3] << 32) | (uint32_t)t[2]);
    return r;
}

__device__ __forceinline__ void st_stream(i64x2s *p, i64x2s v)
{
    v4i_s t = { (int)(uint32_t)v.x, (int)(uint32_t)((uint64_t)v.x >> 32), (int)(uint32_t)v.y, (int)(uint32_t)((uint64_t)v.y >> 32) };
    __builtin_nontemporal_store(t, reinterpret_cast<v4i_s *>(p));
}

template <int Q>
__device__ __forceinline__ int64_t smx_weight(int64_t x, int64_t rmax, const int64_t *lut)
{
    if (Q == 19) {
        uint64_t d = (uint64_t)rmax - (uint64_t)x;                 // >= 0 by construction
        if (d > ((uint64_t)64 << 19)) return 0;
        uint64_t y = (d * 756388ull) >> 19;                        // d <= 2^25: the product is below 2^45
        uint64_t k = y >> 19;
        uint64_t f = y & 0x7FFFF;
        int64_t t = lut[f >> 11];
        return k >= 64 ? 0 : (t >> (int)k);
    } else {
        int64_t d = (int64_t)((uint64_t)x - (uint64_t)rmax);       // <= 0 unless the subtraction wrapped
        if (d < -((int64_t)64 << 21)) return 0;
        int64_t y = (int64_t)((uint64_t)d * 3025551ull + (1ull << 20)) >> 21;
        int64_t ny = (int64_t)(0 - (uint64_t)y);
        int64_t k = ny >> 21;
        int64_t f = ny & 0x1FFFFF;
        int64_t t = lut[f >> 13];
        if (k >= 64) return 0;
        return k < 0 ? (t >> 63) : (t >> (int)k);
    }
}

template <int Q>
__device__ __forceinline__ int64_t smx_numerator(int64_t w, int64_t s)
{
    int64_t num = (int64_t)((uint64_t)w << Q);
    if (Q == 21) num = (int64_t)((uint64_t)num + (uint64_t)(s / 2));
    return num;
}

// Per-row divide.  fast: 2^12 <= s < 2^52 (true for every row whose maximum has weight LUT[0] = 2^Q).
constexpr int64_t kSmxQuickWeights = (int64_t)1 << 30;

template <int Q>
__device__ __forceinline__ int64_t smx_norm(int64_t w, int64_t s, double inv, bool fast)
{
    const int64_t num = smx_numerator<Q>(w, s);
    if (fast && w >= 0 && w < kSmxQuickWeights) return (int64_t)udiv_by_inv((uint64_t)num, (uint64_t)s, inv);
    return s ? tdiv64(num, s) : 0;
}

constexpr int kSmxThreads = 256;
constexpr long kSmxFewRows = 1024;          // see softmax_wave_kernel

// Optional score preparation fused into the row load (inference/model.py:896-906 does it with three tensor ops):
//   x = floor((s1 + s2) * mul / div) + mask[s][t]
// s2, mask and scores (a copy of x for the witness dump, model.py:911-918) may be null.
struct SmxPre {
    const int64_t *s2;
    const int64_t *mask;      // [S, T], added to every batch and head
    int64_t *scores;
    int64_t mul, div;
    double inv_div;
    int S, H;
};

// floor(x / d) for 0 < d < 2^31 and any x: double estimate (exact to within one for |x| < 2^62, within a few
// otherwise) settled by the remainder
__device__ __forceinline__ int64_t floordiv_small(int64_t x, int64_t d, double inv_d)
{
    int64_t q = (int64_t)floor((double)x * inv_d);
    int64_t rem = (int64_t)((uint64_t)x - (uint64_t)q * (uint64_t)d);
    while (rem < 0) { q--; rem += d; }
    while (rem >= d) { q++; rem -= d; }
    return q;
}

__device__ __forceinline__ int64_t smx_prepare_value(int64_t v, int64_t s2, int64_t m, const SmxPre &pre)
{
    v = (int64_t)((uint64_t)v + (uint64_t)s2);
    v = (int64_t)((uint64_t)v * (uint64_t)pre.mul);
    if (pre.div != 1) v = floordiv_small(v, pre.div, pre.inv_div);
    return (int64_t)((uint64_t)v + (uint64_t)m);
}

template <bool PRE>
__device__ __forceinline__ int64_t smx_prepare(int64_t v, const SmxPre &pre, long row, int idx, int T)
{
    if (!PRE) return v;
    const long e = row * T + idx;
    v = smx_prepare_value(v, pre.s2 ? pre.s2[e] : 0, pre.mask ? pre.mask[(long)((row / pre.H) % pre.S) * T + idx] : 0, pre);
    if (pre.scores) pre.scores[e] = v;
    return v;
}

// One row per wavefront; EPL = elements per lane (even).  VEC: T is even and the pointers are 16-byte aligned, a lane
// owns pairs of adjacent elements; otherwise lanes own every 64th element, so that 8-byte accesses are contiguous over
// the wavefront.  Score preparation: the operands of eight elements (sixteen where a row is short enough for the registers
// and accesses are narrow, without VEC) are loaded before the first of their scores is stored.  Loads and stores taken in
// turn wait for each other, the compiler having to assume that they overlap and the count of what is under way covering
// both: one round trip to memory per element, or per batch.  The scores are stored once the whole row has been loaded, but
// for the two batches of 16-byte accesses of a row of 513 to 1024, where that costs more than it gives (131072 causal rows of
// 1024 734 -> 755 us).  Bound by memory on many rows, by a row's chain of loads, reductions and divisions on few.  Element by
// element / stores behind each batch / as it is, inputs that change from call to call: 128 rows of 779 13.3 / 10.5 / 9.3 us, 31104
// of 243 67 / 53 / 48, 2304 of 1142 22.6 / 25.8 / 20.8, of 2047 58 / 62 / 49, 131072 of 1024 761 / 765 / 765 (5.6 TB/s; 780 with
// sixteen at a time, which takes wavefronts).  Without preparation 4224 of 1999 41.3 -> 30.9.
// RW: wavefronts that share a row.  Few rows (a decoding step has one per head) leave most of the device idle and live on the chain of
// loads, divisions and reductions of one wavefront: four of them per row, meeting twice in LDS, have a quarter of it each.
// One / four wavefronts per row, with preparation: 128 rows of 300 6.3 / 6.0 us, of 779 9.6 / 6.0, of 2047 23.4 / 8.0, 1024 rows of 512 8.1 /
// 6.1, of 1142 15.0 / 10.3; of 243 elements equal; 2048 rows of 512 9.0 / 8.8, of 1500 20.9 / 22.3, 4096 of 1024 25.4 / 27.2.
template <int Q, int EPL, bool VEC, bool PRE, int RW = 1>
__global__ __launch_bounds__(kSmxThreads) void softmax_wave_kernel(int64_t *__restrict__ R, int64_t *__restrict__ C,
                                                                   const int64_t *__restrict__ lut_g, long rows, int T,
                                                                   int clobber, SmxPre pre)
{
    __shared__ int64_t lut[256];
    lut[threadIdx.x] = lut_g[threadIdx.x];
    __syncthreads();
    static_assert(RW == 1 || RW == kSmxThreads / 64, "a row belongs to a wavefront or to the workgroup");
    constexpr int LANES = 64 * RW;
    const int lane = threadIdx.x & (LANES - 1);
    const long row = (long)blockIdx.x * (kSmxThreads / LANES) + threadIdx.x / LANES;
    if (row >= rows) return;
    int64_t *x = R + row * T;
    int64_t *c = C + row * T;

    auto at = [&](int j) { return VEC ? ((j >> 1) * LANES + lane) * 2 + (j & 1) : j * LANES + lane; };     // element j of this lane
    int64_t v[EPL];
    int64_t rmax = INT64_MIN;
    constexpr bool LATE = !VEC || EPL != 16;
    auto store_score = [&](int idx, int j) {
        int64_t *dst = pre.scores + row * T + idx;
        if (VEC) st_stream(reinterpret_cast<i64x2s *>(dst), i64x2s{ v[j], v[j + 1] });
        else *dst = v[j];
    };
    constexpr int MOST = VEC || EPL > 16 ? 8 : 16, BATCH = PRE && EPL > MOST ? MOST : EPL;
#pragma unroll
    for (int j0 = 0; j0 < EPL; j0 += BATCH) {
        int64_t b[PRE ? BATCH : 1], m[PRE ? BATCH : 1];
        const int64_t *s2 = PRE && pre.s2 ? pre.s2 + row * T : nullptr;
        const int64_t *mask = PRE && pre.mask ? pre.mask + (long)((row / pre.H) % pre.S) * T : nullptr;
#pragma unroll
        for (int q = 0; q < BATCH; q += VEC ? 2 : 1) {
            const int idx = at(j0 + q);
            if (PRE) { b[q] = m[q] = 0; if (VEC) b[q + 1] = m[q + 1] = 0; }
            if (idx >= T) continue;
            if (VEC) {
                const i64x2s t = ld_stream(reinterpret_cast<const i64x2s *>(x + idx));
                v[j0 + q] = t.x; v[j0 + q + 1] = t.y;
                if (PRE && s2) { const i64x2s u = ld_stream(reinterpret_cast<const i64x2s *>(s2 + idx)); b[q] = u.x; b[q + 1] = u.y; }
                if (PRE && mask) { const i64x2s u = *reinterpret_cast<const i64x2s *>(mask + idx); m[q] = u.x; m[q + 1] = u.y; }
            } else {
                v[j0 + q] = x[idx];
                if (PRE && s2) b[q] = s2[idx];
                if (PRE && mask) m[q] = mask[idx];
            }
        }
#pragma unroll
        for (int q = 0; q < BATCH; q += VEC ? 2 : 1) {
            const int idx = at(j0 + q);
            if (idx >= T) continue;
#pragma unroll
            for (int h = 0; h < (VEC ? 2 : 1); h++) {
                int64_t &e = v[j0 + q + h];
                if (PRE) e = smx_prepare_value(e, b[q + h], m[q + h], pre);
                rmax = e > rmax ? e : rmax;
            }
            if (PRE && !LATE && pre.scores) store_score(idx, j0 + q);
        }
    }
    if (PRE && LATE && pre.scores) {
#pragma unroll
        for (int j = 0; j < EPL; j += VEC ? 2 : 1)
            if (at(j) < T) store_score(at(j), j);
    }
    rmax = wave_max_i64(rmax);
    __shared__ int64_t red[2][kSmxThreads / 64];
    if (RW > 1) {
        if ((lane & 63) == 0) red[0][lane >> 6] = rmax;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < RW; w++) rmax = red[0][w] > rmax ? red[0][w] : rmax;
    }

    uint64_t sum = 0, all = 0;
#pragma unroll
    for (int j = 0; j < EPL; j++) {
        if (at(j) < T) {
            v[j] = smx_weight<Q>(v[j], rmax, lut);
            sum += (uint64_t)v[j];
            if (!VEC) all |= (uint64_t)v[j];
        }
    }
    sum = wave_sum_u64(sum);
    if (RW > 1) {
        if ((lane & 63) == 0) red[1][lane >> 6] = (int64_t)sum;
        __syncthreads();
        sum = 0;
#pragma unroll
        for (int w = 0; w < RW; w++) sum += (uint64_t)red[1][w];
    }
    const int64_t s = (int64_t)sum;
    const bool fast = s >= ((int64_t)1 << 12) && s < ((int64_t)1 << 52);
    const double inv = fast ? 1.0 / (double)s : 0.0;

    // Without VEC the general division, some 200 instructions of 64-bit arithmetic, is here once, in a loop over weights put where the
    // results go.  Beside every element of a long row it made 69 KB of code with preparation, more than the instruction cache (64 KB)
    // holds, and times that hung on where the code came to lie: 5120 rows of 1301 43.9 us in one build and 47.2 in the next, now 43.5,
    // 12800 of 1999 200, 210, now 207; without preparation 25.9 -> 22.0 and 83.2 -> 81.  The forms with VEC are smaller, and slower
    // this way (131072 rows of 1024 348 -> 365, with preparation 20352 of 1438 177 -> 186).
    constexpr bool ONCE = !VEC;
    const bool quick = fast && all < (uint64_t)kSmxQuickWeights;
    auto result = [&](int64_t w) {
        if (!ONCE) return smx_norm<Q>(w, s, inv, fast);
        return quick ? (int64_t)udiv_by_inv((uint64_t)smx_numerator<Q>(w, s), (uint64_t)s, inv) : w;
    };
#pragma unroll
    for (int j = 0; j < EPL; j += VEC ? 2 : 1) {
        const int idx = at(j);
        if (idx >= T) continue;
        if (VEC) {
            st_stream(reinterpret_cast<i64x2s *>(c + idx), i64x2s{ result(v[j]), result(v[j + 1]) });
            if (clobber) st_stream(reinterpret_cast<i64x2s *>(x + idx), i64x2s{ v[j], v[j + 1] });
        } else {
            c[idx] = result(v[j]);
        }
    }
    if (ONCE && !quick) {
#pragma unroll 1
        for (int j = 0; j < EPL; j++)
            if (at(j) < T) c[at(j)] = smx_norm<Q>(c[at(j)], s, inv, fast);
    }
    if (!VEC && clobber) {
#pragma unroll
        for (int j = 0; j < EPL; j++)
            if (at(j) < T) x[at(j)] = v[j];
    }
}

// One row per workgroup, any T: pass 1 maximum, pass 2 weights (staged in C) and their sum, pass 3 divide.
// Each thread re-reads only what it wrote itself, so the staging needs no fence.
template <int Q>
__global__ __launch_bounds__(kSmxThreads) void softmax_block_kernel(int64_t *__restrict__ R, int64_t *__restrict__ C,
                                                                    const int64_t *__restrict__ lut_g, int T, int clobber)
{
    __shared__ int64_t lut[256];
    __shared__ int64_t red[kSmxThreads / 64];
    lut[threadIdx.x] = lut_g[threadIdx.x];
    const long row = blockIdx.x;
    int64_t *x = R + row * T;
    int64_t *c = C + row * T;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;

    int64_t rmax = INT64_MIN;
    for (int i = threadIdx.x; i < T; i += kSmxThreads) { int64_t a = x[i]; rmax = a > rmax ? a : rmax; }
    rmax = wave_max_i64(rmax);
    if (lane == 0) red[wave] = rmax;
    __syncthreads();
    rmax = red[0];
#pragma unroll
    for (int w = 1; w < kSmxThreads / 64; w++) rmax = red[w] > rmax ? red[w] : rmax;
    __syncthreads();

    uint64_t sum = 0;
    for (int i = threadIdx.x; i < T; i += kSmxThreads) {
        int64_t w = smx_weight<Q>(x[i], rmax, lut);
        c[i] = w;
        if (clobber) x[i] = w;
        sum += (uint64_t)w;
    }
    sum = wave_sum_u64(sum);
    if (lane == 0) red[wave] = (int64_t)sum;
    __syncthreads();
    uint64_t tot = 0;
#pragma unroll
    for (int w = 0; w < kSmxThreads / 64; w++) tot += (uint64_t)red[w];
    const int64_t s = (int64_t)tot;
    const bool fast = s >= ((int64_t)1 << 12) && s < ((int64_t)1 << 52);
    const double inv = fast ? 1.0 / (double)s : 0.0;
    for (int i = threadIdx.x; i < T; i += kSmxThreads) c[i] = smx_norm<Q>(c[i], s, inv, fast);
}

template <int Q, int EPL, int RW = 1>
static void launch_wave(int64_t *R, int64_t *C, const int64_t *lut, long rows, int T, bool vec, int clobber, const SmxPre *pre)
{
    constexpr int PER_BLOCK = kSmxThreads / (64 * RW);
    long blocks = (rows + PER_BLOCK - 1) / PER_BLOCK;
    const dim3 grid((unsigned)blocks), block(kSmxThreads);
    SmxPre none = {};
    if (pre) {
        if (vec) softmax_wave_kernel<Q, EPL, true, true, RW><<<grid, block, 0, 0>>>(R, C, lut, rows, T, clobber, *pre);
        else softmax_wave_kernel<Q, EPL, false, true, RW><<<grid, block, 0, 0>>>(R, C, lut, rows, T, clobber, *pre);
    } else {
        if (vec) softmax_wave_kernel<Q, EPL, true, false, RW><<<grid, block, 0, 0>>>(R, C, lut, rows, T, clobber, none);
        else softmax_wave_kernel<Q, EPL, false, false, RW><<<grid, block, 0, 0>>>(R, C, lut, rows, T, clobber, none);
    }
}

// the score preparation as a pass of its own, for rows too long for the one-row-per-wavefront kernel
__global__ __launch_bounds__(256) void smx_prepare_kernel(const int64_t *__restrict__ s1, int64_t *__restrict__ out, long rows, int T, SmxPre pre)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= rows * T) return;
    SmxPre q = pre;
    q.scores = nullptr;
    out[e] = smx_prepare<true>(s1[e], q, e / T, (int)(e % T), T);
}

template <int Q>
static void launch_softmax(const char *name, int64_t *R, int64_t *C, const int64_t *lut, int Bsz, int S, int H, int T,
                           const SmxPre *pre = nullptr)
{
    if (Bsz < 0 || S < 0 || H < 0 || T < 0) { set_error(kBadArgument, "%s: negative dimension", name); return; }
    long rows = (long)Bsz * S * H;
    if (rows == 0 || T == 0) return;
    if (!R || !C || !lut) { set_error(kBadArgument, "%s: null pointer", name); return; }
    if (rows > 0x7FFFFFFFL) { set_error(kUnsupportedSize, "%s: more than 2^31-1 rows", name); return; }
    int clobber = g_softmax_clobber && !pre ? 1 : 0;
    bool vec = (T % 2 == 0) && ((((uintptr_t)R | (uintptr_t)C) & 15) == 0);
    if (pre && ((((uintptr_t)pre->s2 | (uintptr_t)pre->mask | (uintptr_t)pre->scores) & 15) != 0)) vec = false;
    if (rows <= kSmxFewRows && T > 256 && T <= 2048) {
        if (T <= 512) launch_wave<Q, 2, 4>(R, C, lut, rows, T, vec, clobber, pre);
        else if (T <= 1024) launch_wave<Q, 4, 4>(R, C, lut, rows, T, vec, clobber, pre);
        else launch_wave<Q, 8, 4>(R, C, lut, rows, T, vec, clobber, pre);
    } else if (T <= 128) launch_wave<Q, 2>(R, C, lut, rows, T, vec, clobber, pre);
    else if (T <= 256) launch_wave<Q, 4>(R, C, lut, rows, T, vec, clobber, pre);
    else if (T <= 512) launch_wave<Q, 8>(R, C, lut, rows, T, vec, clobber, pre);
    else if (T <= 1024) launch_wave<Q, 16>(R, C, lut, rows, T, vec, clobber, pre);
    else if (T <= 2048) launch_wave<Q, 32>(R, C, lut, rows, T, vec, clobber, pre);
    else {
        if (pre) {
            // long rows: prepared scores go to the scores buffer if there is one, else through C (the block kernel
            // reads all of a row before it writes any of it only when input and output differ, so C cannot serve as both)
            if (!pre->scores) { set_error(kBadArgument, "%s: rows longer than 2048 need a scores buffer", name); return; }
            const long n = rows * T;
            smx_prepare_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0>>>(R, pre->scores, rows, T, *pre);
            R = pre->scores;
        }
        softmax_block_kernel<Q><<<dim3((unsigned)rows), dim3(kSmxThreads), 0, 0>>>(R, C, lut, T, clobber);
    }
    check_launch(name);
}

}  // namespace zk

extern "C" {

void softmax_q19(int64_t *R, int64_t *C, int64_t *lut, int Bsz, int S, int H, int T)
{
    zk::launch_softmax<19>("softmax_q19", R, C, lut, Bsz, S, H, T);
}

void softmax_q21(int64_t *R, int64_t *C, int64_t *lut, int Bsz, int S, int H, int T)
{
    zk::launch_softmax<21>("softmax_q21", R, C, lut, Bsz, S, H, T);
}

void zk_softmax_clobber_input(int on) { zk::g_softmax_clobber = on != 0; }

void softmax_q19_scores(const int64_t *s1, const int64_t *s2, const int64_t *mask, int64_t *scores, int64_t *C,
                        const int64_t *lut, int Bsz, int S, int H, int T, int64_t mul, int64_t div)
{
    const char *name = "softmax_q19_scores";
    if (div <= 0 || div >= ((int64_t)1 << 31)) { zk::set_error(zk::kBadArgument, "%s: div must be in [1, 2^31)", name); return; }
    zk::SmxPre pre;
    pre.s2 = s2; pre.mask = mask; pre.scores = scores; pre.mul = mul; pre.div = div; pre.inv_div = 1.0 / (double)div;
    pre.S = S > 0 ? S : 1; pre.H = H > 0 ? H : 1;
    zk::launch_softmax<19>(name, const_cast<int64_t *>(s1), C, lut, Bsz, S, H, T, &pre);
}

}  // extern "C"
