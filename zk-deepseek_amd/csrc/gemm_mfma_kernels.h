// Device side of the limb-decomposed i8 MFMA GEMM (see gemm_mfma.hip for the scheme): digit split, loaders, the GEMM
// kernel, the split-K finish, the range kernels, and the table type that pairs a digit-count combination with its
// kernels.  The combinations are instantiated in several translation units (gemm_mfma_inst_*.hip) so that they
// compile side by side.
#pragma once
#include "gemm.h"
#include "../../include/int64gemm.h"

#include <type_traits>
#include <vector>

// Tuning knob: how many vector-ALU instructions of the digit split are scheduled behind each MFMA of a step's last depth.  (A 32x32x32 MFMA holds the
// matrix pipe for 32 cycles, a vector instruction its own for 4; with two wavefronts on a SIMD up to four or five
// vector instructions per MFMA run in its shade, eight cost a quarter more time per MFMA: measured with a probe, and
// on the 512 x 7168 x 18432 product 0.631-0.638 ms with 5 against 0.642-0.643 with 8.)
#ifndef ZK_VALU_PER_MFMA
#define ZK_VALU_PER_MFMA 5
#endif

namespace zk {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct MfmaParams {
    const int64_t *A;
    const void *B;
    int64_t *C, *R;
    long lda, sA, ldbn, ldbk, sB, ldc, sC;
    int M, N, K, shift;
    int64_t init;
    int tiles_m, tiles_n;
    unsigned long long *range;      // sampling only: [minA, maxA, minB, maxB], order-preserving unsigned images of int64
    unsigned *seen;                 // one word per workgroup: digits its share of A (byte 0) and of B (byte 1) needs, 0 = nothing seen; may be null
    unsigned *verdict;              // 0 unless some workgroup met an element its digit counts do not hold (see raise_verdict)
    int fail_class;                 // what such a workgroup reports at least: 1, or 2 when a digit count of this launch is above five
    int verify_b_all_batches;       // B differs per batch: every batch's first tile row tracks its range
    const unsigned char *a_planes;  // pre-split digits of A (planes variants only)
    int a_msub, a_ksteps;           // 32-row groups and 32-k steps the planes were written for
    int b_nsub, b_ksteps;           // BPL kernels: B (or every group's B) is digit planes of that geometry
    long b_gstride;                 // ... and this many bytes from one batch's planes to the next one's (0: shared)
    const int *row_steps;           // 32-k steps of a row tile (128 rows) of A up to its last non-zero one (null: all of them; pipelined kernel only)
    int row_order, items, batches;  // pipelined kernel: items walked row tile by row tile, how many there are, and batches
    int col_parts;                  // row-tile kernel: an item is a row tile and one of this many parts of its tile columns
    // split-K tail: workgroup ids below main_tiles are whole tiles; the rest are `split` workgroups per tile that
    // each cover a slice of K and leave raw 128-bit partial sums in `partials`
    int main_tiles, split;
    int tail_xcd;                             // split tiles: deal (tile column, K slice) pairs over the 8 XCDs (see the kernel)
    int n_fastest;                            // tile order inside a batch: 0 = tile rows move fastest (the workgroups that run together share a B tile), 1 = tile columns (they share an A tile)
    unsigned long long *partials;
    int part64;                     // the partial sums fit 64 bits: only the low words are kept
    // grouped mode (GRP kernels): rows of A and C form one segment per group, each group has its own B.
    // Workgroup (mt, tn) looks up 32-row tile mt in grp_tiles = {group, first row} and stops at the segment's end.
    const int *grp_seg;             // [groups + 1] first row of every segment
    const int *grp_tiles;           // [2 * tiles] group and first row of every 32-row tile
    const int *grp_ntiles;          // how many of them exist (the grid is sized for the worst case)
    const void *const *grp_b;       // [groups] B of every group
    int b_shift;                    // BRS kernels: every element of B is divided by 2^b_shift first, truncating toward zero
    int finish_rq;                  // workgroups per tile of the finishing kernel (4 or 16)
    // guarded launches (the fallback behind a speculative launch): the kernel does nothing unless the verdict is non-zero,
    // and its workgroups, one per compute unit, walk the `walk_blocks` workgroup ids of an ordinary launch
    GuardArgs guard;
    int walk_blocks;
};

constexpr unsigned long long kSignFlip = 0x8000000000000000ull;

// ---- digit split -------------------------------------------------------------------------------
template <int N>
struct Limb {
    static constexpr uint64_t kBias = N >= 9 ? 0x8080808080808080ull
                                             : (N == 1 ? 0ull : (0x0080808080808080ull >> (8 * (8 - N))));
};

// 4x4 byte transpose: out[i] = bytes (y0.b_i, y1.b_i, y2.b_i, y3.b_i)
__device__ __forceinline__ void transpose4(uint32_t y0, uint32_t y1, uint32_t y2, uint32_t y3, uint32_t (&o)[4])
{
    uint32_t p01l = __builtin_amdgcn_perm(y1, y0, 0x05010400u);
    uint32_t p01h = __builtin_amdgcn_perm(y1, y0, 0x07030602u);
    uint32_t p23l = __builtin_amdgcn_perm(y3, y2, 0x05010400u);
    uint32_t p23h = __builtin_amdgcn_perm(y3, y2, 0x07030602u);
    o[0] = __builtin_amdgcn_perm(p23l, p01l, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(p23l, p01l, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(p23h, p01h, 0x05040100u);
    o[3] = __builtin_amdgcn_perm(p23h, p01h, 0x07060302u);
}

// x[0..7] (8 consecutive k of one row) -> out[i] = 8 bytes of digit i, k ascending.
template <int N>
__device__ __forceinline__ void limb_split8(const int64_t (&x)[8], uint2 (&out)[N])
{
    uint32_t lo[8], hi[8], e[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
        uint64_t u = (uint64_t)x[q] + Limb<N>::kBias;
        if (N >= 9) e[q] = (x[q] >= 0 && u < Limb<N>::kBias) ? 1u : 0u;
        u ^= Limb<N>::kBias;
        lo[q] = (uint32_t)u;
        hi[q] = (uint32_t)(u >> 32);
    }
    uint32_t t0[4], t1[4];
    transpose4(lo[0], lo[1], lo[2], lo[3], t0);
    transpose4(lo[4], lo[5], lo[6], lo[7], t1);
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (i < N) out[i] = make_uint2(t0[i], t1[i]);
    if (N > 4) {
        transpose4(hi[0], hi[1], hi[2], hi[3], t0);
        transpose4(hi[4], hi[5], hi[6], hi[7], t1);
#pragma unroll
        for (int i = 4; i < 8; i++)
            if (i < N) out[i] = make_uint2(t0[i - 4], t1[i - 4]);
    }
    if (N >= 9)
        out[N - 1] = make_uint2(e[0] | (e[1] << 8) | (e[2] << 16) | (e[3] << 24),
                                e[4] | (e[5] << 8) | (e[6] << 16) | (e[7] << 24));
}

// Smallest digit count whose range holds every value in [lo, hi].
__host__ __device__ static inline int limbs_needed(int64_t lo, int64_t hi)
{
    if (lo > hi) return 1;                   // nothing was seen
    for (int n = 1; n <= 8; n++) {
        // x + bias_n in [-2^(8n-1), 2^(8n-1))
        i128 bias = n == 1 ? 0 : (i128)(0x0080808080808080ull >> (8 * (8 - n)));
        i128 half = (i128)1 << (8 * n - 1);
        if ((i128)lo + bias >= -half && (i128)hi + bias < half) return n;
    }
    return 9;
}

// C++ division by 2^s (truncation toward zero) as shifts: the bias makes the arithmetic shift round negative values up
__device__ __forceinline__ int64_t tdiv_pow2(int64_t x, int s)
{
    const uint64_t bias = (uint64_t)(x >> 63) & (((uint64_t)1 << s) - 1);
    return (int64_t)((uint64_t)x + bias) >> s;
}

// ---- range tracking ------------------------------------------------------------------------------
struct MinMax { int64_t lo, hi; };

__device__ __forceinline__ void mm_update(MinMax &r, int64_t v)
{
    r.lo = v < r.lo ? v : r.lo;
    r.hi = v > r.hi ? v : r.hi;
}

// What the hot loop tracks instead of a 64-bit minimum and maximum (two quarter-rate compares and four selects per
// element; measured on the 512 x 7168 x 18432 product, 5.5 % of the kernel's time went into tracking B that way): the
// digit count itself.  In balanced base-256 digits x + 0x8080...80 has byte j equal to 0x80 wherever digit j is zero,
// so the OR over all elements of (x + 0x80..80) ^ 0x80..80 has its highest non-zero byte at the highest digit any
// element needs: six full-rate 32-bit instructions per element.  (An element beyond eight digits wraps the sum; it leaves
// a non-zero top byte like one that needs eight, and both count as nine digits.)
struct DigitsSeen {
    uint32_t lo = 0, hi = 0;
    bool seen = false;
    __device__ __forceinline__ void add(int64_t v)
    {
        const uint64_t t = ((uint64_t)v + 0x8080808080808080ull) ^ 0x8080808080808080ull;
        lo |= (uint32_t)t;
        hi |= (uint32_t)(t >> 32);
    }
    // digits that hold everything added (0: nothing was)
    __device__ __forceinline__ int digits() const
    {
        if (!seen) return 0;
        const uint64_t e = ((uint64_t)hi << 32) | lo;
        if (e >> 56) return 9;
        return e ? (71 - __clzll((long long)e)) >> 3 : 1;                 // bytes up to the highest non-zero one
    }
};

// the same for int32 values between lo and hi (0: lo > hi, nothing was seen)
__device__ __forceinline__ int digits_i32(int lo, int hi)
{
    if (lo > hi) return 0;
    if (lo >= -0x80 && hi <= 0x7F) return 1;
    if (lo >= -0x8080 && hi <= 0x7F7F) return 2;
    if (lo >= -0x808080 && hi <= 0x7F7F7F) return 3;
    return hi <= 0x7F7F7F7F ? 4 : 5;
}

__device__ __forceinline__ int wave_max_i32(int v)
{
    wave_steps([&](auto off) {
        unsigned a, b;
        lane_pair<decltype(off)::value>((unsigned)v, a, b);
        v = (int)a > (int)b ? (int)a : (int)b;
    });
    return v;
}

__device__ __forceinline__ MinMax mm_wave(MinMax r)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        int64_t ol = __shfl_xor(r.lo, off, kWave), oh = __shfl_xor(r.hi, off, kWave);
        r.lo = ol < r.lo ? ol : r.lo;
        r.hi = oh > r.hi ? oh : r.hi;
    }
    return r;
}

__device__ __forceinline__ void mm_publish(MinMax r, unsigned long long *slot)
{
    r = mm_wave(r);
    // The slots only ever move one way, so a plain (possibly stale) read is enough to skip the atomic when this
    // wave cannot improve them; that keeps thousands of waves from serialising on two addresses.
    if ((threadIdx.x & 63) == 0) {
        const unsigned long long lo = (unsigned long long)r.lo ^ kSignFlip, hi = (unsigned long long)r.hi ^ kSignFlip;
        if (lo < __atomic_load_n(slot, __ATOMIC_RELAXED)) atomicMin(slot, lo);
        if (hi > __atomic_load_n(slot + 1, __ATOMIC_RELAXED)) atomicMax(slot + 1, hi);
    }
}

static __global__ void range_reset_kernel(unsigned long long *range)
{
    if (threadIdx.x < 4) range[threadIdx.x] = (threadIdx.x & 1) ? 0ull : ~0ull;
}

// What a workgroup leaves about the digits of its share: its word for the report (see guard_report), and, only when an
// element did not fit the launch's digit counts, the verdict that makes the guarded launch behind compute everything
// again: 1 when five digits hold what it saw (and every digit count of the launch is at most five), else 2.  Nothing is
// written to the shared word in the ordinary case, so thousands of workgroups do not queue up for one address.
__device__ __forceinline__ void leave_digits(unsigned *seen_slot, unsigned *verdict, int fail_class, int na, int nb, int need_a, int need_b)
{
    if (seen_slot) *seen_slot = (unsigned)need_a | ((unsigned)need_b << 8);
    if (need_a > na || need_b > nb) {
        const unsigned v = (need_a > 5 || need_b > 5) ? 2u : (unsigned)fail_class;
        atomicMax(verdict, v);
    }
}

// Strided sample of both operands for the first guess (at most `rows_s` rows x `cols_s` k each).
static __global__ __launch_bounds__(256) void range_sample_kernel(MfmaParams p, int b32, int G, int which)
{
    MinMax r = { INT64_MAX, INT64_MIN };
    const long rows = which == 0 ? (long)p.M : (long)p.N;
    const long rstep = rows > 32 ? rows / 32 : 1;
    const long kstep = p.K > 256 ? p.K / 256 : 1;
    for (long ri = threadIdx.x >> 6; ri * rstep < rows && ri < 32; ri += 4) {
        long row = ri * rstep;
        for (long ki = threadIdx.x & 63; ki * kstep < p.K && ki < 256; ki += 64) {
            long k = ki * kstep;
            for (int g = 0; g < G; g += (G > 2 ? G / 2 : 1)) {
                int64_t v;
                if (which == 0) v = p.A[(long)g * p.sA + row * p.lda + k];
                else {
                    long off = (long)g * p.sB + row * p.ldbn + k * p.ldbk;
                    v = b32 ? (int64_t)reinterpret_cast<const int32_t *>(p.B)[off]
                            : reinterpret_cast<const int64_t *>(p.B)[off];
                    v = tdiv_pow2(v, p.b_shift);
                }
                mm_update(r, v);
            }
        }
    }
    mm_publish(r, p.range + 2 * which);
}

// ---- element ownership ---------------------------------------------------------------------------
// Within a pipeline step of BK = 8*OCTS k-values, thread j (0 <= j < OCTS) of a row owns elements
//     k(e) = RUN*OCTS*(e / RUN) + RUN*j + e % RUN,   e = 0..7,
// i.e. 8/RUN runs of RUN consecutive k.  RUN = 2 for int64 B (a run is one 16-byte load), 4 for int32 B.
template <int RUN, int OCTS>
__device__ __forceinline__ int owned_k(int j, int e) { return RUN * OCTS * (e / RUN) + RUN * j + e % RUN; }

// Loads the 8 owned int64 elements of one row; `src` points at the row's first k of this step.
template <int RUN, int OCTS>
__device__ __forceinline__ void load_owned_i64(const int64_t *src_generic, int j, bool row_ok, int k_left, bool vec, int64_t (&x)[8])
{
    const ZK_GLOBAL_MEM int64_t *src = (const ZK_GLOBAL_MEM int64_t *)src_generic;
    if (row_ok && owned_k<RUN, OCTS>(j, 7) < k_left && vec) {
#pragma unroll
        for (int q = 0; q < 8 / RUN; q++) {
#pragma unroll
            for (int h = 0; h < RUN / 2; h++) {
                const v4i t = *(const ZK_GLOBAL_MEM v4i *)(src + owned_k<RUN, OCTS>(j, q * RUN + 2 * h));
                x[q * RUN + 2 * h] = (int64_t)(((uint64_t)(uint32_t)t[1] << 32) | (uint32_t)t[0]);
                x[q * RUN + 2 * h + 1] = (int64_t)(((uint64_t)(uint32_t)t[3] << 32) | (uint32_t)t[2]);
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = owned_k<RUN, OCTS>(j, e);
            x[e] = (row_ok && k < k_left) ? src[k] : 0;
        }
    }
}

template <int RUN, int OCTS>
__device__ __forceinline__ void load_owned_i32(const int32_t *src_generic, int j, bool row_ok, int k_left, bool vec, int64_t (&x)[8])
{
    const ZK_GLOBAL_MEM int32_t *src = (const ZK_GLOBAL_MEM int32_t *)src_generic;
    if (RUN == 4 && row_ok && owned_k<RUN, OCTS>(j, 7) < k_left && vec) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const v4i t = *(const ZK_GLOBAL_MEM v4i *)(src + owned_k<RUN, OCTS>(j, q * 4));
#pragma unroll
            for (int z = 0; z < 4; z++) x[q * 4 + z] = (int64_t)t[z];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = owned_k<RUN, OCTS>(j, e);
            x[e] = (row_ok && k < k_left) ? (int64_t)src[k] : 0;
        }
    }
}

// Byte offset, inside one operand region of an LDS stage (or of a plane step), of the 8 digit bytes that
// thread j of `row` produces: 1 KB fragment blocks, lane slot = row%32 + 32*(k-half), 16 bytes per slot.
__device__ __forceinline__ int frag_offset(int row, int j, int n_limbs, int substage_bytes)
{
    const int o4 = j & 3;
    return (j >> 2) * substage_bytes + ((row >> 5) * n_limbs) * 1024 + ((row & 31) + 32 * (o4 >> 1)) * 16 + (o4 & 1) * 8;
}

// ---- A digit planes (pre-pass) ------------------------------------------------------------------
// When A is reused by many column tiles it is split once, into digit planes stored in MFMA fragment order:
// block (g, sub, ks32, i) of 1 KB holds digit i of rows [32*sub, 32*sub+32) for the 32 owned-k slots of MFMA
// depth ks32, lane-major.  Rows >= M and k >= K are written as zero digits.  Each workgroup also leaves the
// digits of what it read needs in seen[block] (when that is given; 0: it was all zeros).
// IN32: the matrix holds int32 elements (weights prepared once; lda and sA count elements as they do for int64).
template <int NA, int RUN, int KK, bool IN32 = false>
__global__ __launch_bounds__(256) void a_planes_kernel(MfmaParams p, unsigned char *planes, int msub, int ksteps32, unsigned *seen)
{
    constexpr int OCTS = 4 * KK, ROWS = 256 / OCTS;
    __shared__ int red[4];
    const int tid = threadIdx.x;
    const int g = blockIdx.z, ks = blockIdx.x;
    const int row = blockIdx.y * ROWS + tid / OCTS, j = tid % OCTS;
    const int k0 = ks * (8 * OCTS);
    const bool vec = (((uintptr_t)p.A | (uintptr_t)(p.lda * 8) | (uintptr_t)(p.sA * 8)) & 15) == 0;
    int64_t x[8];
    if (IN32) load_owned_i32<RUN, OCTS>(reinterpret_cast<const int32_t *>(p.A) + (long)g * p.sA + (long)row * p.lda + k0, j, row < p.M, p.K - k0, false, x);
    else load_owned_i64<RUN, OCTS>(p.A + (long)g * p.sA + (long)row * p.lda + k0, j, row < p.M, p.K - k0, vec, x);
    DigitsSeen bound;
#pragma unroll
    for (int q = 0; q < 8; q++) bound.add(x[q]);
    bound.seen = true;
    uint2 dg[NA];
    limb_split8<NA>(x, dg);
    // plane step layout: [g][sub][ks32][digit][1 KB]; a step of KK depths is contiguous per sub
    unsigned char *dst = planes + (((long)g * msub + (row >> 5)) * ksteps32 + ks * KK + (j >> 2)) * (NA * 1024) +
                         ((row & 31) + 32 * ((j & 3) >> 1)) * 16 + (j & 1) * 8;
    if (row < msub * 32) {                  // a workgroup may reach past the last 32-row group (skinny tiles)
#pragma unroll
        for (int i = 0; i < NA; i++) *reinterpret_cast<uint2 *>(dst + i * 1024) = dg[i];
    }
    if (!seen) return;
    const int need = wave_max_i32((bound.lo | bound.hi) == 0 ? 0 : bound.digits());
    if ((tid & 63) == 0) red[tid >> 6] = need;
    __syncthreads();
    if (tid == 0) {
        int n = red[0];
#pragma unroll
        for (int w = 1; w < 4; w++) n = red[w] > n ? red[w] : n;
        const long b = ((long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        leave_digits(seen + b, p.verdict, p.fail_class, NA, NA, n, 0);
    }
}

// The same for a B that is small next to the product (pipe_b_planes in gemm_mfma.hip): its rows (columns of the output) for
// A's, either layout, both element types, one depth per step.  It runs behind the pass over A and, with `row_steps`,
// finds the last step of every 128 rows of A that is not all zeros from the words that pass has left.
struct BPlanesParams {
    const void *B;
    long ldn, ldk, sB;              // B[g * sB + n * ldn + k * ldk]
    int N, K, nsub, ksteps;
    long gstride;                   // bytes of planes per batch
    unsigned char *planes;
    unsigned *seen, *verdict;
    int fail_class;
    int *row_steps;                 // may be null
    const unsigned *a_seen;         // [row tiles][2][ksteps]
    long row_tiles;
};

template <int NB, bool KMAJOR, bool IN32>
__global__ __launch_bounds__(256) void b_planes_kernel(BPlanesParams p)
{
    __shared__ int red[4];
    const int tid = threadIdx.x, g = blockIdx.z, ks = blockIdx.x;
    // adjacent lanes read adjacent elements: of k where k is contiguous, of n where n is
    const int row = blockIdx.y * 64 + (KMAJOR ? (tid & 63) : tid >> 2), j = KMAJOR ? tid >> 6 : tid & 3;
    int64_t x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int k = ks * 32 + owned_k<2, 4>(j, e);
        const long at = (long)g * p.sB + (long)row * p.ldn + (long)k * p.ldk;
        x[e] = row < p.N && k < p.K ? (IN32 ? (int64_t)reinterpret_cast<const int32_t *>(p.B)[at] : reinterpret_cast<const int64_t *>(p.B)[at]) : 0;
    }
    DigitsSeen bound;
#pragma unroll
    for (int e = 0; e < 8; e++) bound.add(x[e]);
    bound.seen = true;
    uint2 dg[NB];
    limb_split8<NB>(x, dg);
    if ((row >> 5) < p.nsub) {
        unsigned char *dst = p.planes + (long)g * p.gstride + ((long)(row >> 5) * p.ksteps + ks) * (NB * 1024) + ((row & 31) + 32 * (j >> 1)) * 16 + (j & 1) * 8;
#pragma unroll
        for (int i = 0; i < NB; i++) *reinterpret_cast<uint2 *>(dst + i * 1024) = dg[i];
    }
    const int need = wave_max_i32(bound.digits());
    if ((tid & 63) == 0) red[tid >> 6] = need;
    __syncthreads();
    const long block = ((long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (tid == 0) {
        int n = red[0];
#pragma unroll
        for (int w = 1; w < 4; w++) n = red[w] > n ? red[w] : n;
        leave_digits(p.seen + block, p.verdict, p.fail_class, NB, NB, 0, n);
    }
    if (!p.row_steps) return;
    // a wavefront per row tile
    const long waves = 4L * gridDim.x * gridDim.y * gridDim.z;
    for (long t = block * 4 + (tid >> 6); t < p.row_tiles; t += waves) {
        const unsigned *w = p.a_seen + t * 2 * p.ksteps;
        int last = 0;
        for (int i = tid & 63; i < p.ksteps; i += 64)
            if ((w[i] | w[p.ksteps + i]) & 0xFFu) last = i + 1;
        last = wave_max_i32(last);
        if ((tid & 63) == 0) p.row_steps[t] = last;
    }
}

// The report of a launch that has no guarded launch behind it (its caller waits for the digits instead).
static __global__ __launch_bounds__(256) void digits_report_kernel(GuardArgs g) { guard_report(g, 0, __atomic_load_n(g.verdict, __ATOMIC_RELAXED)); }

// One output from its D int32 diagonals: init + sum_d dg(d) * 2^(8d) as the words of a 128-bit sum.  A diagonal keeps its
// low byte and hands the rest to the next one, so everything is 32-bit: two instructions per diagonal and a byte permute
// per byte, where adding the diagonals up in 64 and 128 bits took some forty per output with wait states between the
// carries (a 128x128 tile of six diagonals: 13k cycles, as long as eight steps of its MFMAs).
// kMaxDiagonal: what a diagonal may reach for that; 0 <= init < 2^20.
constexpr long kMaxDiagonal = 0x7F000000L;
struct Words { uint32_t w[4]; };
template <int D, class F>
__device__ __forceinline__ Words sum_diagonals(F &&dg, int init)
{
    int c[D];
    c[0] = dg(0) + init;
#pragma unroll
    for (int d = 1; d < D; d++) c[d] = dg(d) + (c[d - 1] >> 8);
    // bytes 0 .. D-2 are the low bytes of c; from byte D-1 on the sum is c[D-1], sign-extended
    Words s;
    constexpr int TOP = D - 1;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (4 * q + 3 < TOP) {
            const uint32_t p01 = __builtin_amdgcn_perm((uint32_t)c[4 * q + 1], (uint32_t)c[4 * q], 0x0c0c0400u);
            const uint32_t p23 = __builtin_amdgcn_perm((uint32_t)c[4 * q + 3], (uint32_t)c[4 * q + 2], 0x04000c0cu);
            s.w[q] = p01 | p23;
        } else if (4 * q <= TOP) {
            constexpr int n = TOP & 3;                       // whole bytes below c[TOP] in this word
            uint32_t v = (uint32_t)c[TOP] << (8 * n);
            if (n == 1) v = __builtin_amdgcn_perm(v, (uint32_t)c[TOP - 1], 0x07060500u);
            if (n >= 2) v = __builtin_amdgcn_perm(v, __builtin_amdgcn_perm((uint32_t)c[TOP - n + 1], (uint32_t)c[TOP - n], 0x0c0c0400u), 0x07060100u);
            if (n == 3) v = __builtin_amdgcn_perm(v, __builtin_amdgcn_perm((uint32_t)c[TOP - 1], v, 0x0c040100u), 0x07020100u);
            s.w[q] = v;
        } else {
            s.w[q] = 4 * (q - 1) <= TOP ? (uint32_t)((TOP & 3) ? c[TOP] >> (32 - 8 * (TOP & 3)) : c[TOP] >> 31) : (uint32_t)((int)s.w[q - 1] >> 31);
        }
    }
    return s;
}

// bits [sh, sh + 64) of the sum, and the bits below sh; sh (0..63) is the same in every lane
__device__ __forceinline__ int64_t shifted_sum(const Words &s, int sh)
{
    const bool upper = sh >= 32;
    const uint32_t a = upper ? s.w[1] : s.w[0], b = upper ? s.w[2] : s.w[1], c = upper ? s.w[3] : s.w[2];
    const uint32_t lo = __builtin_amdgcn_alignbit(b, a, (uint32_t)sh & 31), hi = __builtin_amdgcn_alignbit(c, b, (uint32_t)sh & 31);
    return (int64_t)((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ int64_t sum_below(const Words &s, uint64_t mask)
{
    return (int64_t)((uint64_t)(s.w[1] & (uint32_t)(mask >> 32)) << 32 | (s.w[0] & (uint32_t)mask));
}

// Number of digit pairs (i', j') with i' + j' < d that come before (i, j) in row order (i' < i, or i' == i and j' < j).
__host__ __device__ constexpr int kept_pairs_before(int na, int nb, int d, int i, int j)
{
    int n = 0;
    for (int r = 0; r < i && r < na; r++) {
        const int row = d - r < 0 ? 0 : (d - r > nb ? nb : d - r);
        n += row;
    }
    if (i < na) {
        const int row = d - i < 0 ? 0 : (d - i > nb ? nb : d - i);
        n += j < row ? j : row;
    }
    return n;
}

// ---- the GEMM kernel -------------------------------------------------------------------------------
// WVM x WVN waves per workgroup, WM x WN 32x32 MFMA tiles per wave, KK MFMA k-depths (32 k each) per pipeline
// step.  APL: A comes from pre-split digit planes (plain copy into LDS); otherwise it is split on the fly like B.
// BPL: so does B (weights prepared once, in the layout of the A planes with columns for rows); nothing of B is tracked then,
// its digit count was fixed exactly when the planes were made.
//
// The hot loop is branch-free: rows past M or N are clamped to the last valid row (their products land in
// outputs that are never stored), only a final partial k-step uses guarded loads, and every thread walks its
// own row pointers.  Loads of step s+1 are issued first, the MFMAs of the step's leading depths give them time
// to land, and the MFMAs of the last depth are interleaved with the digit split of the loaded data.
// (the body of the kernels below: `block` is the workgroup id of an ordinary launch, one tile or one slice of a split tile)
template <int NA, int NB, int WVM, int WVN, int WM, int WN, int KK, bool B32, bool BKM, bool APL, bool GRP = false, bool BRS = false, int DMAX = 16,
          bool BPL = false>
__device__ __forceinline__ void gemm_mfma_block(const MfmaParams &p, const int block)
{
    constexpr int T = 64 * WVM * WVN;
    constexpr int BM = 32 * WM * WVM, BN = 32 * WN * WVN, BK = 32 * KK, OCTS = BK / 8;
    constexpr int RUN = B32 ? 4 : 2;
    // Diagonal d carries weight 2^(8d).  Diagonal 16 (2^128) never matters; a launch whose shift + 64 result bits
    // end below 2^(8 DMAX) leaves out the digit pairs of the diagonals from DMAX up as well.
    constexpr int D = (NA + NB - 1) > DMAX ? DMAX : (NA + NB - 1);
    static_assert(DMAX >= 8 && DMAX <= 16, "the low 64 bits of the sum need diagonals 0..7");
    constexpr int A_BLOCKS = (BM / 32) * NA, B_BLOCKS = (BN / 32) * NB;
    constexpr int SUBSTAGE = (A_BLOCKS + B_BLOCKS) * 1024;
    constexpr int STAGE = KK * SUBSTAGE;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WVN, wn = wave % WVN;

    // workgroup -> tile.  Consecutive workgroup ids go to different XCDs (8 of them, each with its own L2), so
    // ids are regrouped to give each XCD a contiguous run of tiles; within a run the tile-row index moves
    // fastest, so the workgroups that share a B tile sit on the same L2.
    const int per_batch = p.tiles_m * p.tiles_n;
    int lin = block, sidx = 0, nsplit = 1;
    int tail_tile = 0, g = 0, tn, tm, m0, m_lim = p.M;
    const void *b_base = p.B;
    if (GRP) {
        // Consecutive workgroup ids go round the 8 XCDs, each with its own L2: the tile columns of one 32-row tile go to
        // ONE of them, so that its rows of A come from memory once and not once per tile column (the routed experts'
        // w1/w3 launch fetched 15.68 GB for 14.86 that way).  The grid is a multiple of 8 * tiles_n workgroups.
        const int xcd = lin & 7, w = lin >> 3, wq = w / p.tiles_n;
        const int mt = wq * 8 + xcd;
        if (mt >= *p.grp_ntiles) {                 // the grid covers the worst case: nothing to do, an empty range
            if (tid == 0 && p.seen) p.seen[block] = 0;
            return;
        }
        tn = w - wq * p.tiles_n;
        tm = 0;
        const int e = p.grp_tiles[2 * mt];
        m0 = p.grp_tiles[2 * mt + 1];
        m_lim = p.grp_seg[e + 1];
        b_base = p.grp_b[e];
    } else {
        if (lin < p.main_tiles) {
            if ((p.main_tiles & 7) == 0) lin = (lin & 7) * (p.main_tiles >> 3) + (lin >> 3);
        } else {
            const int t = lin - p.main_tiles;
            if (p.tail_xcd) {
                // Workgroup ids go round the 8 XCDs.  Each XCD takes whole (tile column, K slice) pairs and runs the
                // tiles_m workgroups of a pair one after the other, so that they find the pair's B data in their L2.
                const int x = t & 7, q = t >> 3;
                const int pair = (q / p.tiles_m) * 8 + x;
                lin = p.main_tiles + (pair / p.split) * p.tiles_m + q % p.tiles_m;
                sidx = pair % p.split;
            } else {
                lin = p.main_tiles + t / p.split;
                sidx = t % p.split;
            }
            nsplit = p.split;
        }
        tail_tile = lin - p.main_tiles;            // index among the split tiles (when nsplit > 1)
        g = lin / per_batch;
        const int rem = lin - g * per_batch;
        if (p.n_fastest) { tm = rem / p.tiles_n; tn = rem - tm * p.tiles_n; }
        else { tn = rem / p.tiles_m; tm = rem - tn * p.tiles_m; }
        m0 = tm * BM;
    }
    const int n0 = tn * BN;
    // A wavefront whose rows all lie past the last one (the last tile of a row count that is no multiple of the tile)
    // loads and splits its share and leaves the matrix pipe to the others.
    const bool rows_live = __builtin_amdgcn_readfirstlane(m0 + wm * (32 * WM) < m_lim ? 1 : 0) != 0;

    // Range tracking is shared out: the tiles_m workgroups that load the same B tile each check every
    // tiles_m-th k-step of it (likewise for A across the workgroups of a tile row), so no workgroup is slower
    // than its neighbours and every element is still seen once.
    const int vmod_b = p.tiles_m < 8 ? p.tiles_m : 8, vmod_a = p.tiles_n < 8 ? p.tiles_n : 8;
    const bool verify_a = !APL && tn < vmod_a;
    const bool verify_b = !BPL && tm < vmod_b && (g == 0 || p.verify_b_all_batches);
    DigitsSeen oa, ob;
    int rb32_lo = INT32_MAX, rb32_hi = INT32_MIN;        // the range of an int32 B is tracked in 32 bits and joins rb at the end

    // Work items of the loaders: (row, j) pairs owning 8 elements each, or 16-byte chunks of digit planes.
    constexpr int A_ITEMS = BM * OCTS, B_ITEMS = BN * OCTS;
    constexpr int A_IT = APL ? 1 : (A_ITEMS + T - 1) / T, B_IT = BPL ? 1 : (B_ITEMS + T - 1) / T;
    constexpr int A_CHUNKS = KK * A_BLOCKS * 64, A_CIT = APL ? (A_CHUNKS + T - 1) / T : 1;
    constexpr int B_CHUNKS = KK * B_BLOCKS * 64, B_CIT = BPL ? (B_CHUNKS + T - 1) / T : 1;
    // Where the blocks of A's planes come out even, a wavefront loads those of its own rows (and of the depth that its column
    // group has the number of): one without rows then loads its share of B alone.
    constexpr bool OWN_ROWS = APL && WM == 1 && WVM > 1 && KK == WVN;
    static_assert(!OWN_ROWS || A_CIT == NA, "two depths of 32 rows between the wavefronts of a row");
    static_assert(!BPL || (!B32 && !BKM && !BRS), "prepared planes of B go with the int64 forms (and are made for the kernel's KK: the owned-k order depends on it)");
    int64_t sa[A_IT][8], sb[B_IT][8];
    v4i pa[A_CIT], pb[B_CIT];

    const bool a_vec = (((uintptr_t)p.A | (uintptr_t)(p.lda * 8) | (uintptr_t)(p.sA * 8)) & 15) == 0;
    const bool b_vec = BPL || (!BKM && (((uintptr_t)b_base | (uintptr_t)(p.ldbn * (B32 ? 4 : 8)) | (uintptr_t)(p.sB * (B32 ? 4 : 8))) & 15) == 0);

    // per-thread source pointers (advanced by BK per step) and LDS destinations
    const int64_t *a_src[A_IT];
    const unsigned char *a_pl[A_CIT];
    const char *b_src[B_IT];
    const unsigned char *b_pl[B_CIT];
    // LDS destinations are stage-relative; threads with no work in an iteration aim at a dummy area behind the two
    // stages (and a zero stage stride), which keeps the loop body free of branches.
    constexpr int DUMMY = 2 * STAGE;
    bool a_pad[A_IT];
    int a_j[A_IT], b_j[B_IT], a_dst[A_IT], b_dst[B_IT], pl_dst[A_CIT], plb_dst[B_CIT];
    int a_stride[A_IT], b_stride[B_IT], pl_stride[A_CIT], plb_stride[B_CIT];
    if (APL) {
#pragma unroll
        for (int it = 0; it < A_CIT; it++) {
            const int c = it * T + tid;
            const bool live = A_CHUNKS % T == 0 || c < A_CHUNKS;
            const int cc0 = live ? c : 0;
            // LDS order inside a stage is [kk][sub][digit]; planes are [sub][ks32][digit]
            const int kk = OWN_ROWS ? wn : cc0 / (A_BLOCKS * 64);
            const int cc = OWN_ROWS ? (wm * NA + it) * 64 + lane : cc0 - kk * (A_BLOCKS * 64);
            const int sub_i = cc / (NA * 64), within = cc - sub_i * (NA * 64);
            a_pl[it] = p.a_planes + (((long)g * p.a_msub + (m0 >> 5) + sub_i) * p.a_ksteps + kk) * (NA * 1024) + within * 16;
            pl_dst[it] = live ? kk * SUBSTAGE + cc * 16 : DUMMY;
            pl_stride[it] = live ? STAGE : 0;
        }
    } else {
#pragma unroll
        for (int it = 0; it < A_IT; it++) {
            const int idx = it * T + tid;
            const bool live = A_ITEMS % T == 0 || idx < A_ITEMS;
            const int row = (live ? idx : 0) / OCTS;
            a_j[it] = idx % OCTS;
            int m = m0 + row;
            // (rows past the end are loaded from the last row, a valid address, and multiplied as zeros: the device is
            // power managed and what the matrix pipe draws depends on the bits it is fed; an expert's tile has some
            // 8 real rows of 32)
            a_pad[it] = m >= m_lim;
            m = m < m_lim ? m : m_lim - 1;
            a_src[it] = p.A + (long)g * p.sA + (long)m * p.lda;
            a_dst[it] = live ? frag_offset(row, a_j[it], NA, SUBSTAGE) : DUMMY;
            a_stride[it] = live ? STAGE : 0;
        }
    }
    if (BPL) {
#pragma unroll
        for (int it = 0; it < B_CIT; it++) {
            const int c = it * T + tid;
            const bool live = B_CHUNKS % T == 0 || c < B_CHUNKS;
            const int cc0 = live ? c : 0;
            // as for the planes of A: LDS order inside a stage is [kk][sub][digit], planes are [sub][ks32][digit]
            const int kk = cc0 / (B_BLOCKS * 64), cc = cc0 - kk * (B_BLOCKS * 64);
            const int sub_i = cc / (NB * 64), within = cc - sub_i * (NB * 64);
            int sub = (n0 >> 5) + sub_i;
            sub = sub < p.b_nsub ? sub : p.b_nsub - 1;          // column groups past N: any valid data, never stored
            b_pl[it] = reinterpret_cast<const unsigned char *>(b_base) + (GRP ? 0 : (long)g * p.b_gstride) + ((long)sub * p.b_ksteps + kk) * (NB * 1024) + within * 16;
            plb_dst[it] = live ? A_BLOCKS * 1024 + kk * SUBSTAGE + cc * 16 : DUMMY;
            plb_stride[it] = live ? STAGE : 0;
        }
    }
#pragma unroll
    for (int it = 0; it < (BPL ? 0 : B_IT); it++) {
        const int idx = it * T + tid;
        const bool live = B_ITEMS % T == 0 || idx < B_ITEMS;
        const int idx0 = live ? idx : 0;
        int row;
        if (BKM) { row = (idx0 & 63) + 64 * (idx0 / (64 * OCTS)); b_j[it] = (idx0 >> 6) % OCTS; }
        else { row = idx0 / OCTS; b_j[it] = idx0 % OCTS; }
        int n = n0 + row;
        n = n < p.N ? n : p.N - 1;
        const long off = (long)g * p.sB + (long)n * p.ldbn;
        b_src[it] = reinterpret_cast<const char *>(b_base) + off * (B32 ? 4 : 8);
        b_dst[it] = live ? A_BLOCKS * 1024 + frag_offset(row, b_j[it], NB, SUBSTAGE) : DUMMY;
        b_stride[it] = live ? STAGE : 0;
    }

    // The staged data of a step can be handled in two parts, so that a kernel with two MFMA depths per step splits,
    // stores and reloads one half behind each depth (its loads are then spread over the step instead of leaving in one
    // burst at its end): PART 0 = A and the first half of B's items, 1 = the rest of B, -1 = everything.
    typedef std::integral_constant<int, -1> PAll;
    typedef std::integral_constant<int, 0> PFirst;
    typedef std::integral_constant<int, 1> PSecond;
    constexpr int B_N = BPL ? B_CIT : B_IT;          // items (or chunks of planes) of B per thread

    // FAST: the whole step lies inside K and the pointers allow 16-byte loads: no guards at all.
    // WITH_A: false in a wavefront whose rows of A nobody multiplies.
    auto fetch = [&](int ks, auto fast_tag, auto part_tag, auto a_tag) {
        constexpr bool WITH_A = decltype(a_tag)::value;
        constexpr bool FAST = decltype(fast_tag)::value;
        constexpr int PART = decltype(part_tag)::value;
        constexpr int B_LO = PART == 1 ? B_N / 2 : 0, B_HI = PART == 0 ? B_N / 2 : B_N;
        const int k0 = ks * BK;
        if (PART == 1 || !WITH_A) {
        } else if (APL) {
#pragma unroll
            for (int it = 0; it < A_CIT; it++)
                pa[it] = *reinterpret_cast<const v4i *>(a_pl[it] + (long)ks * (KK * NA * 1024));
        } else {
#pragma unroll
            for (int it = 0; it < A_IT; it++) {
                if (FAST) load_owned_i64<RUN, OCTS>(a_src[it] + k0, a_j[it], true, BK, true, sa[it]);
                else load_owned_i64<RUN, OCTS>(a_src[it] + k0, a_j[it], true, p.K - k0, false, sa[it]);
            }
        }
        if (BPL) {
#pragma unroll
            for (int it = B_LO; it < B_HI; it++)
                pb[it] = *(const ZK_GLOBAL_MEM v4i *)(b_pl[it] + (long)ks * (KK * NB * 1024));
        }
#pragma unroll
        for (int it = (BPL ? 0 : B_LO); it < (BPL ? 0 : B_HI); it++) {
            if (BKM) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int k = k0 + owned_k<RUN, OCTS>(b_j[it], e);
                    const long off = (long)k * p.ldbk;
                    int64_t v = 0;
                    if (FAST || k < p.K)
                        v = B32 ? (int64_t)((const ZK_GLOBAL_MEM int32_t *)b_src[it])[off] : ((const ZK_GLOBAL_MEM int64_t *)b_src[it])[off];
                    sb[it][e] = v;
                }
            } else if (B32) {
                const int32_t *src = reinterpret_cast<const int32_t *>(b_src[it]) + k0;
                if (FAST) load_owned_i32<RUN, OCTS>(src, b_j[it], true, BK, true, sb[it]);
                else load_owned_i32<RUN, OCTS>(src, b_j[it], true, p.K - k0, false, sb[it]);
            } else {
                const int64_t *src = reinterpret_cast<const int64_t *>(b_src[it]) + k0;
                if (FAST) load_owned_i64<RUN, OCTS>(src, b_j[it], true, BK, true, sb[it]);
                else load_owned_i64<RUN, OCTS>(src, b_j[it], true, p.K - k0, false, sb[it]);
            }
        }
    };

    // staged elements -> digits -> LDS stage `buf`, fragment order
    auto stash = [&](int buf, auto part_tag, auto a_tag) {
        constexpr bool WITH_A = decltype(a_tag)::value;
        constexpr int PART = decltype(part_tag)::value;
        constexpr int B_LO = PART == 1 ? B_N / 2 : 0, B_HI = PART == 0 ? B_N / 2 : B_N;
        if (PART == 1 || !WITH_A) {
        } else if (APL) {
#pragma unroll
            for (int it = 0; it < A_CIT; it++)
                *reinterpret_cast<v4i *>(smem + pl_dst[it] + buf * pl_stride[it]) = pa[it];
        } else {
#pragma unroll
            for (int it = 0; it < A_IT; it++) {
                uint2 dg[NA];
                limb_split8<NA>(sa[it], dg);
#pragma unroll
                for (int i = 0; i < NA; i++)
                    *reinterpret_cast<uint2 *>(smem + a_dst[it] + buf * a_stride[it] + i * 1024) = a_pad[it] ? make_uint2(0u, 0u) : dg[i];
            }
        }
        if (BPL) {
#pragma unroll
            for (int it = B_LO; it < B_HI; it++)
                *reinterpret_cast<v4i *>(smem + plb_dst[it] + buf * plb_stride[it]) = pb[it];
        }
#pragma unroll
        for (int it = (BPL ? 0 : B_LO); it < (BPL ? 0 : B_HI); it++) {
            uint2 dg[NB];
            if (BRS) {
                int64_t y[8];
#pragma unroll
                for (int q = 0; q < 8; q++) y[q] = tdiv_pow2(sb[it][q], p.b_shift);
                limb_split8<NB>(y, dg);
            } else {
                limb_split8<NB>(sb[it], dg);
            }
#pragma unroll
            for (int i = 0; i < NB; i++)
                *reinterpret_cast<uint2 *>(smem + b_dst[it] + buf * b_stride[it] + i * 1024) = dg[i];
        }
    };

    // Fragments of one MFMA depth, and the MFMAs of a slice [LO, HI) of the depth's (i, j, tile) list.
    auto load_frags = [&](int buf, int kk, v4i (&fa)[WM][NA], v4i (&fb)[WN][NB]) {
        const unsigned char *base = smem + buf * STAGE + kk * SUBSTAGE;
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int i = 0; i < NA; i++)
                fa[a][i] = *reinterpret_cast<const v4i *>(base + (((wm * WM + a) * NA + i) * 1024) + lane * 16);
#pragma unroll
        for (int b = 0; b < WN; b++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                fb[b][j] = *reinterpret_cast<const v4i *>(base + ((A_BLOCKS + (wn * WN + b) * NB + j) * 1024) + lane * 16);
    };
    const int ksteps = (p.K + BK - 1) / BK;
    const int full_steps = (a_vec || APL) && (b_vec || BKM) ? p.K / BK : 0;     // steps that can use unguarded loads
    // this workgroup's slice of the k-steps (everything unless it is one of the split workgroups of a tail tile)
    const int ks_begin = (int)((long)sidx * ksteps / nsplit), ks_end = (int)((long)(sidx + 1) * ksteps / nsplit);

    // Range tracking of the staged elements of data step d, done while the registers still hold them.
    // (called once per data step, in order: the turn counters stand for d % vmod_a and d % vmod_b without a division)
    int turn_a = ks_begin % vmod_a, turn_b = ks_begin % vmod_b;
    bool my_a = false, my_b = false;
    auto track = [&](auto part_tag) {
        constexpr int PART = decltype(part_tag)::value;
        constexpr int B_LO = PART == 1 ? B_IT / 2 : 0, B_HI = PART == 0 ? B_IT / 2 : B_IT;
        if (PART != 1) {            // (the turns advance once per data step, with its first part)
            my_a = turn_a == tn;
            my_b = turn_b == tm;
            turn_a = turn_a + 1 == vmod_a ? 0 : turn_a + 1;
            turn_b = turn_b + 1 == vmod_b ? 0 : turn_b + 1;
        }
        if (PART != 1 && verify_a && my_a) {
#pragma unroll
            for (int it = 0; it < A_IT; it++)
#pragma unroll
                for (int q = 0; q < 8; q++) oa.add(sa[it][q]);
            oa.seen = true;
        }
        if (verify_b && my_b) {
#pragma unroll
            for (int it = B_LO; it < B_HI; it++)
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    if (B32 && !BRS) {
                        // int32 values: one min and one max instruction each, against four for a 64-bit pair
                        const int v = (int)sb[it][q];
                        rb32_lo = v < rb32_lo ? v : rb32_lo;
                        rb32_hi = v > rb32_hi ? v : rb32_hi;
                    } else {
                        ob.add(BRS ? tdiv_pow2(sb[it][q], p.b_shift) : sb[it][q]);     // what the digits are taken from
                    }
                }
            ob.seen = true;
        }
    };

    // every workgroup leaves the digits of what it saw in its own word; the waves meet in LDS (the stages are free by now)
    auto leave = [&]() {
        int need_a = 0, need_b = 0;
        if (verify_a || verify_b) {
            __syncthreads();
            int *red = reinterpret_cast<int *>(smem);
            need_a = wave_max_i32(oa.digits());
            need_b = wave_max_i32(B32 && !BRS ? digits_i32(rb32_lo, rb32_hi) : ob.digits());
            if (lane == 0) { red[2 * wave] = need_a; red[2 * wave + 1] = need_b; }
            __syncthreads();
            if (tid == 0) {
                for (int w = 1; w < T / 64; w++) {
                    need_a = red[2 * w] > need_a ? red[2 * w] : need_a;
                    need_b = red[2 * w + 1] > need_b ? red[2 * w + 1] : need_b;
                }
            }
        }
        if (tid == 0) leave_digits(p.seen ? p.seen + block : nullptr, p.verdict, p.fail_class, NA, NB, need_a, need_b);
    };

    // prologue: stage 0 holds the first step, the staging registers hold the second
    if (ks_begin < full_steps) fetch(ks_begin, std::true_type(), PAll(), std::true_type()); else fetch(ks_begin, std::false_type(), PAll(), std::true_type());
    track(PAll());
    stash(0, PAll(), std::true_type());
    if (ks_begin + 1 < ks_end) {
        if (ks_begin + 1 < full_steps) fetch(ks_begin + 1, std::true_type(), PAll(), std::true_type()); else fetch(ks_begin + 1, std::false_type(), PAll(), std::true_type());
    }
    __syncthreads();
    int ks = ks_begin;
    const int fast_end = full_steps < ks_end ? full_steps : ks_end;
    // (411 rows x [18432,7168] int32, (4,4): 846 -> 805 us, and 824 -> 803 on another device without its share of
    // A's planes, too; 192 rows 427 -> 418, 300 rows 619 -> 606.  The 128x128 tiles keep the one loop: with two, the registers of
    // the hot one were dealt worse and 512 x 7168 x 18432 went from 622 to 634.)
    if (WM == 1 && WVM > 1 && !rows_live) {
        typedef std::integral_constant<bool, !OWN_ROWS> DeadA;
        auto dead_step = [&](int step, auto fast_tag) {
            stash(((step - ks_begin) & 1) ^ 1, PAll(), DeadA());
            track(PAll());
            if (step + 2 < ks_end) fetch(step + 2, fast_tag, PAll(), DeadA());
            __syncthreads();
        };
        for (; ks + 2 < fast_end; ks++) dead_step(ks, std::true_type());
        for (; ks + 1 < ks_end; ks++) dead_step(ks, std::false_type());
        leave();
        return;
    }
    v16i acc[WM][WN][D];
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
        for (int b = 0; b < WN; b++)
#pragma unroll
            for (int d = 0; d < D; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[a][b][d][r] = 0;
    // the digit pairs (i, j) with i + j < D are numbered in row order; a slice issues those numbered LO..HI-1
    constexpr int MFMAS = WM * WN * kept_pairs_before(NA, NB, D, NA, 0);
    auto mfma_slice = [&](auto lo_tag, auto hi_tag, const v4i (&fa)[WM][NA], const v4i (&fb)[WN][NB]) {
        constexpr int LO = decltype(lo_tag)::value, HI = decltype(hi_tag)::value;
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int a = 0; a < WM; a++)
#pragma unroll
                    for (int b = 0; b < WN; b++) {
                        const int idx = (kept_pairs_before(NA, NB, D, i, j) * WM + a) * WN + b;
                        if (idx >= LO && idx < HI && i + j < D)
                            acc[a][b][i + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][i], fb[b][j], acc[a][b][i + j], 0, 0, 0);
                    }
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, MFMAS / 2> IH;
    typedef std::integral_constant<int, MFMAS> IF;
    auto compute_all = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < KK; kk++) {
            v4i fa[WM][NA], fb[WN][NB];
            load_frags(buf, kk, fa, fb);
            mfma_slice(I0(), IF(), fa, fb);
        }
    };

    // One pipeline step, three fenced phases:
    //   A  fragment reads of stage `cur` and the first half of its MFMAs (time for the staged loads to land);
    //   B  the second half of the MFMAs interleaved, in one scheduling region, with the digit split of the
    //      elements staged for step ks+1 and their LDS writes into the other stage;
    //   C  the loads of step ks+2 into the now free staging registers, then the barrier.
    // Two depths per step, B split on the fly: one depth's MFMAs carry the split of one half of the staged data, whose
    // registers are reloaded right behind it.  Each half's loads then have a whole step to land and some are under way
    // at every moment (with one burst per step nothing is for the part of the step between their arrival and the next
    // burst: the routed experts' int32 weights streamed at 5.3 TB/s that way).
    constexpr bool SPREAD = KK == 2 && !BKM && B_N >= 2 && B_N % 2 == 0;
    auto step_body = [&](int ks, auto fast_tag) {
        const int cur = (ks - ks_begin) & 1;
        if constexpr (SPREAD) {
            {
                v4i fa[WM][NA], fb[WN][NB];
                load_frags(cur, 0, fa, fb);
                mfma_slice(I0(), IF(), fa, fb);
                stash(cur ^ 1, PFirst(), std::true_type());
#pragma unroll
                for (int i = 0; i < MFMAS; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, ZK_VALU_PER_MFMA, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                track(PFirst());
                if (ks + 2 < ks_end) fetch(ks + 2, fast_tag, PFirst(), std::true_type());
                __builtin_amdgcn_sched_barrier(0);
            }
            {
                v4i fa[WM][NA], fb[WN][NB];
                load_frags(cur, 1, fa, fb);
                mfma_slice(I0(), IF(), fa, fb);
                stash(cur ^ 1, PSecond(), std::true_type());
#pragma unroll
                for (int i = 0; i < MFMAS; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, ZK_VALU_PER_MFMA, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                track(PSecond());
                if (ks + 2 < ks_end) fetch(ks + 2, fast_tag, PSecond(), std::true_type());
            }
            __syncthreads();
            return;
        }
#pragma unroll
        for (int kk = 0; kk < KK - 1; kk++) {
            v4i fa[WM][NA], fb[WN][NB];
            load_frags(cur, kk, fa, fb);
            mfma_slice(I0(), IF(), fa, fb);
        }
        v4i fa[WM][NA], fb[WN][NB];
        load_frags(cur, KK - 1, fa, fb);
        mfma_slice(I0(), IH(), fa, fb);
        __builtin_amdgcn_sched_barrier(0);
        mfma_slice(IH(), IF(), fa, fb);
        stash(cur ^ 1, PAll(), std::true_type());
#pragma unroll
        for (int i = 0; i < MFMAS - MFMAS / 2; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, ZK_VALU_PER_MFMA, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        track(PAll());
        if (ks + 2 < ks_end) fetch(ks + 2, fast_tag, PAll(), std::true_type());
        __syncthreads();
    };

    for (; ks + 2 < fast_end; ks++) step_body(ks, std::true_type());
    for (; ks + 1 < ks_end; ks++) step_body(ks, std::false_type());
    compute_all((ks_end - 1 - ks_begin) & 1);

    leave();

    // epilogue: diagonals -> 128-bit sum -> shift.  Accumulator register r of lane l holds
    // row 8*(r/4) + 4*(l/32) + r%4, column l%32 of its 32x32 tile.
    auto combine = [&](int a, int b, int r, int init) { return sum_diagonals<D>([&](int d) { return acc[a][b][d][r]; }, init); };
    if (nsplit > 1) {
        // raw partial sums (without the rounding term), finished by gemm_split_finish_kernel: 64 lanes' low words, then
        // (unless 64 bits hold the sums) their high words, per (slice, wave, tile, register)
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int b = 0; b < WN; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    // rows of this register that all lie past M (uniform over the wave): nothing to keep
                    if (m0 + (wm * WM + a) * 32 + 8 * (r >> 2) + (r & 3) >= m_lim) continue;
                    const Words sum = combine(a, b, r, 0);
                    const long q = (((long)tail_tile * p.split + sidx) * (T / 64) + wave) * (WM * WN * 16) + (a * WN + b) * 16 + r;
                    const uint64_t lo = (uint64_t)sum.w[1] << 32 | sum.w[0];
                    if (p.part64) p.partials[q * 64 + lane] = lo;
                    else { p.partials[q * 128 + lane] = lo; p.partials[q * 128 + 64 + lane] = (uint64_t)sum.w[3] << 32 | sum.w[2]; }
                }
        return;
    }
    // Whole tiles: the loops carry no uniform branches (tiles that reach past M or N, and calls that want the remainder,
    // have their own copy), and a row's address is the tile's plus a scalar multiple of the row stride.
    const uint64_t rmask = p.shift ? ((1ull << p.shift) - 1) : 0;
    const int sum0 = (int)p.init;
    const int sh = p.shift;
    auto store_tile = [&](auto edge_tag, auto rem_tag) {
        constexpr bool EDGE = decltype(edge_tag)::value, REM = decltype(rem_tag)::value;
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int b = 0; b < WN; b++) {
                const int n = n0 + (wn * WN + b) * 32 + (lane & 31);
                const int mrow = m0 + (wm * WM + a) * 32 + 4 * (lane >> 5);
                const long o0 = (long)g * p.sC + (long)mrow * p.ldc + n;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int dr = 8 * (r >> 2) + (r & 3);
                    const Words sum = combine(a, b, r, sum0);
                    if (EDGE && !(mrow + dr < m_lim && n < p.N)) continue;
                    const long o = o0 + (long)dr * p.ldc;
                    p.C[o] = shifted_sum(sum, sh);
                    if (REM) p.R[o] = sum_below(sum, rmask);
                }
            }
    };
    const bool edge = m0 + BM > m_lim || n0 + BN > p.N;
    if (p.R) { if (edge) store_tile(std::true_type(), std::true_type()); else store_tile(std::false_type(), std::true_type()); }
    else { if (edge) store_tile(std::true_type(), std::false_type()); else store_tile(std::false_type(), std::false_type()); }
}

template <int NA, int NB, int WVM, int WVN, int WM, int WN, int KK, bool B32, bool BKM, bool APL, bool GRP = false, bool BRS = false, int DMAX = 16,
          bool BPL = false>
__global__ __launch_bounds__(64 * WVM * WVN) void gemm_mfma_kernel(MfmaParams p)
{
    gemm_mfma_block<NA, NB, WVM, WVN, WM, WN, KK, B32, BKM, APL, GRP, BRS, DMAX, BPL>(p, (int)blockIdx.x);
}

// The same product on 64x64 tiles of four wavefronts, two workgroups to a compute unit (see short_k_tiles in gemm_mfma.hip).
template <int NA, int NB, int KK, bool B32, bool BKM>
__global__ __launch_bounds__(256, 2) void gemm_mfma_short_kernel(MfmaParams p)
{
    gemm_mfma_block<NA, NB, 2, 2, 1, 1, KK, B32, BKM, false>(p, (int)blockIdx.x);
}

// The same product behind a guard word: nothing happens unless *p.guard is non-zero (the verdict of the speculative launch
// in front of it: its digit counts did not cover the operands), and then the grid, one workgroup per compute unit, walks
// the workgroup ids of an ordinary launch.  A guarded launch almost always finds nothing to do, and thousands of
// workgroups with 80 KB of LDS each would take tens of microseconds to find that out.
template <int NA, int NB, int WVM, int WVN, int WM, int WN, int KK, bool B32, bool BKM, int DMAX = 16>
__global__ __launch_bounds__(64 * WVM * WVN) void gemm_mfma_guarded_kernel(MfmaParams p)
{
    const unsigned verdict = __atomic_load_n(p.guard.verdict, __ATOMIC_RELAXED);            // (the same for every thread of the launch)
    if ((int)blockIdx.x < p.guard.parts) guard_report(p.guard, (int)blockIdx.x, verdict);
    if (verdict == 0) return;
    if (verdict == 1 && (NA > 5 || NB > 5)) {
        // five digits cover both operands (every workgroup that met a wider element would have raised the verdict to 2): a
        // third of the digit pairs of (9,9)
        constexpr int NA5 = NA > 5 ? 5 : NA, NB5 = NB > 5 ? 5 : NB;
        for (int block = (int)blockIdx.x; block < p.walk_blocks; block += (int)gridDim.x) {
            gemm_mfma_block<NA5, NB5, WVM, WVN, WM, WN, KK, B32, BKM, false, false, false, 16, false>(p, block);
            __syncthreads();
        }
        return;
    }
    for (int block = (int)blockIdx.x; block < p.walk_blocks; block += (int)gridDim.x) {
        gemm_mfma_block<NA, NB, WVM, WVN, WM, WN, KK, B32, BKM, false, false, false, DMAX, false>(p, block);
        __syncthreads();            // (the LDS stages and the range words in them are used again)
    }
}

// Adds the `split` partial sums of every tail tile, applies the rounding term and the shift, and stores C and R.
// Thread layout and element order are those of the GEMM kernel's epilogue.  The first p.guard.parts workgroups leave the report
// instead, beside the sums: in the guarded launch behind, the stores to host memory are all that a launch with nothing to do waits for (report there / here, us:
// 128 rows x [2048,7168] int64 38.9 / 37.0, 243 x [512,7168] int32 38.9 / 35.2, 40 x [2048,7168] 39.2 / 36.2, 128 x [576,7168] 24.7 / 23.1).
template <int WVM, int WVN, int WM, int WN>
__global__ __launch_bounds__(64 * WVM * WVN) void gemm_split_finish_kernel(MfmaParams p)
{
    constexpr int T = 64 * WVM * WVN, BM = 32 * WM * WVM, BN = 32 * WN * WVN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WVN, wn = wave % WVN;
    const int per_batch = p.tiles_m * p.tiles_n;
    if ((int)blockIdx.x < p.guard.parts) {
        guard_report(p.guard, (int)blockIdx.x, __atomic_load_n(p.guard.verdict, __ATOMIC_RELAXED));
        return;
    }
    const int item = (int)blockIdx.x - p.guard.parts;
    const int tail_tile = item / p.finish_rq, rq = item % p.finish_rq, lin = p.main_tiles + tail_tile;
    const int r_per = 16 / p.finish_rq;
    const int g = lin / per_batch, rem = lin - g * per_batch;
    const int tn = p.n_fastest ? rem % p.tiles_n : rem / p.tiles_m, tm = p.n_fastest ? rem / p.tiles_n : rem - tn * p.tiles_m;
    const int m0 = tm * BM, n0 = tn * BN;
    const uint64_t rmask = p.shift ? ((1ull << p.shift) - 1) : 0;
    const long qs = (long)(T / 64) * (WM * WN * 16);          // from one slice to the next
    // the registers of this workgroup's share, RPER at a time with all their slices' loads under way together (one
    // output at a time, a thread has `split` loads in flight and the launch lives on latency)
    auto finish = [&](auto rper_tag) {
        constexpr int RPER = decltype(rper_tag)::value;
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int b = 0; b < WN; b++) {
                const int n = n0 + (wn * WN + b) * 32 + (lane & 31);
                const int r0 = rq * RPER;
                const long q0 = ((long)tail_tile * p.split * (T / 64) + wave) * (WM * WN * 16) + (a * WN + b) * 16 + r0;
                uint64_t lo[RPER], hi[RPER];
                bool live[RPER];
#pragma unroll
                for (int r4 = 0; r4 < RPER; r4++) {
                    const int r = r0 + r4;
                    lo[r4] = (uint64_t)p.init;
                    hi[r4] = (uint64_t)(p.init >> 63);
                    live[r4] = m0 + (wm * WM + a) * 32 + 8 * (r >> 2) + (r & 3) < p.M;      // (uniform over the wave; the others were never written)
                }
                if (p.part64) {
                    uint64_t s[RPER];
#pragma unroll
                    for (int r4 = 0; r4 < RPER; r4++) s[r4] = 0;
#pragma unroll 4
                    for (int sidx = 0; sidx < p.split; sidx++)
#pragma unroll
                        for (int r4 = 0; r4 < RPER; r4++)
                            s[r4] += p.partials[(q0 + r4 + sidx * qs) * 64 + lane];      // (rows past M: slots nobody wrote, read and dropped)
#pragma unroll
                    for (int r4 = 0; r4 < RPER; r4++) {
                        const uint64_t t = lo[r4] + s[r4];
                        hi[r4] += (uint64_t)((int64_t)s[r4] >> 63) + (t < lo[r4] ? 1 : 0);
                        lo[r4] = t;
                    }
                } else {
#pragma unroll 2
                    for (int sidx = 0; sidx < p.split; sidx++)
#pragma unroll
                        for (int r4 = 0; r4 < RPER; r4++)
                        {
                            const uint64_t plo = p.partials[(q0 + r4 + sidx * qs) * 128 + lane];
                            const uint64_t phi = p.partials[(q0 + r4 + sidx * qs) * 128 + 64 + lane];
                            const uint64_t t = lo[r4] + plo;
                            hi[r4] += phi + (t < lo[r4] ? 1 : 0);
                            lo[r4] = t;
                        }
                }
#pragma unroll
                for (int r4 = 0; r4 < RPER; r4++) {
                    const int r = r0 + r4;
                    const int m = m0 + (wm * WM + a) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (live[r4] && m < p.M && n < p.N) {
                        const long o = (long)g * p.sC + (long)m * p.ldc + n;
                        p.C[o] = (int64_t)(p.shift == 0 ? lo[r4] : ((lo[r4] >> p.shift) | (hi[r4] << (64 - p.shift))));
                        if (p.R) p.R[o] = (int64_t)(lo[r4] & rmask);
                    }
                }
            }
    };
    if (r_per == 4) finish(std::integral_constant<int, 4>());
    else if (r_per == 2) finish(std::integral_constant<int, 2>());
    else finish(std::integral_constant<int, 1>());
}

// ---- kernel tables -------------------------------------------------------------------------------------
typedef void (*MfmaKernel)(MfmaParams);
typedef void (*FinishKernel)(MfmaParams);
typedef void (*PlanesKernel)(MfmaParams, unsigned char *, int, int, unsigned *);

enum Variant { kB64Fly = 0, kB64Planes, kB32Fly, kB32Planes, kB64KmajorFly, kB32KmajorFly, kB64Group, kB32Group, kB64FlyRs, kB32FlyRs,
               kB64PlanesBoth, kB64FlyBPlanes, kB64GroupBPlanes, kVariants };     // the last three: B from prepared digit planes

struct Instance {
    int na, nb, bm, bn, threads, kk;
    bool skinny;                 // 32-row tiles for M <= 32
    int dmax;                    // diagonals from this one up are left out (16: none but the 2^128 one)
    bool alt;                    // 128x64 tiles for digit counts that also have 128x128 ones: taken by launch size (see smaller_tiles)
    bool short_k;                // 64x64 tiles for digit counts that also have larger ones: taken by K (see short_k_tiles)
    MfmaKernel fn[kVariants];
    PlanesKernel planes[2];      // [b32]: the owned-k pattern follows the element size of B
    FinishKernel finish;         // adds up the partial sums of split tail tiles
    MfmaKernel guarded[2][2];    // [b32][n-contiguous B]: the guarded form, A split on the fly (the widest instances only)
};


// Tile shapes by diagonals kept (= int32 accumulator sets): up to 5, eight waves as 2x4 with 64x32 outputs each (128x128);
// up to 10, 4x2 with 32x32 each (128x64); beyond, four waves as 2x2 (64x64, one wave per SIMD because of the accumulators).
// kRows32 (few rows): 1x8 waves (32x256).
enum Tile { kTileAuto = 0, kTileRows32, kTile128x64 };
// What an instance is for: everything, int32 B alone, grouped launches on prepared planes of B alone, or ungrouped launches
// with planes on both sides alone.
enum Use { kUseAll = 0, kUseB32, kUseGroupPlanes, kUsePlanesBoth };

// KK: MFMA k-depths (of 32) per pipeline step.  Two of them halve the barriers and double the bytes under way.  The
// 32-row kernels live on the latter: a step of int32 weights is half the bytes of a step of int64 weights, and with two
// depths streams as much.  The 128x64 tiles have the registers for it (at most 256 with (5,5), no more than one spilled)
// and gain on every shape: 243 rows x [7168,16384] int32, (3,4) digits, 413 -> 353 us; 411 x [18432,7168], (4,4),
// 908 -> 846; 100 x [18432,7168] 269 -> 248; 131072 x [1024,512] int64, (3,4), 1343 -> 1184.  The 128x128 tiles do not
// (they spill: 0.74 against 0.67 ms on 512 x 7168 x 18432).
template <int NA, int NB, int TILE = kTileAuto, int DMAX = 16, int KK = 1, int USE = kUseAll>
static Instance make_instance()
{
    constexpr int DD = (NA + NB - 1) > DMAX ? DMAX : (NA + NB - 1);      // diagonals kept = accumulator sets
    constexpr bool SKINNY = TILE == kTileRows32, B32ONLY = USE == kUseB32;
    constexpr bool NARROW = !SKINNY && TILE != kTile128x64 && DD <= 5, MID = !SKINNY && !NARROW && DD <= 10;
    static_assert(!SKINNY || DD <= 10, "skinny tiles keep two waves per SIMD");
    constexpr int WVM = SKINNY ? 1 : (NARROW ? 2 : (MID ? 4 : 2));
    constexpr int WVN = SKINNY ? 8 : (NARROW ? 4 : 2);
    constexpr int WM = NARROW ? 2 : 1, WN = 1;
    static_assert(!B32ONLY || NB <= 5, "int32 values never need more than five digits");
    Instance s;
    s.na = NA; s.nb = NB; s.bm = 32 * WM * WVM; s.bn = 32 * WN * WVN; s.threads = 64 * WVM * WVN; s.kk = KK;
    s.skinny = SKINNY;
    s.dmax = DMAX;
    s.alt = TILE == kTile128x64;
    s.short_k = false;
    for (int v = 0; v < kVariants; v++) s.fn[v] = nullptr;
    s.guarded[0][0] = s.guarded[0][1] = s.guarded[1][0] = s.guarded[1][1] = nullptr;
    // every operand fits nine digits, every int32 five: these instances can stand behind any speculative launch
    if constexpr (NA == 9 && !SKINNY && DMAX == 16 && USE == kUseAll) {
        if constexpr (NB == 9) {
            s.guarded[0][0] = gemm_mfma_guarded_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, DMAX>;
            s.guarded[0][1] = gemm_mfma_guarded_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, true, DMAX>;
        }
        if constexpr (NB == 5) {
            s.guarded[1][0] = gemm_mfma_guarded_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, false, DMAX>;
            s.guarded[1][1] = gemm_mfma_guarded_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, true, DMAX>;
        }
    }
    if constexpr (USE == kUsePlanesBoth) {
        static_assert(!SKINNY && KK == 1, "prepared planes of one matrix are in the order of one depth per step");
        s.fn[kB64PlanesBoth] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, true, false, false, DMAX, true>;
        s.finish = gemm_split_finish_kernel<WVM, WVN, WM, WN>;
        s.planes[0] = a_planes_kernel<NA, 2, KK>;
        s.planes[1] = a_planes_kernel<NA, 4, KK>;
        return s;
    }
    if constexpr (USE == kUseGroupPlanes) {
        static_assert(SKINNY, "grouped launches run on the 32-row tiles");
        s.fn[kB64GroupBPlanes] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, true, false, DMAX, true>;
        s.finish = gemm_split_finish_kernel<WVM, WVN, WM, WN>;
        s.planes[0] = a_planes_kernel<NA, 2, KK>;
        s.planes[1] = a_planes_kernel<NA, 4, KK>;
        return s;
    }
    if constexpr (!B32ONLY) {
        s.fn[kB64Fly] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, false, false, DMAX>;
        s.fn[kB64Planes] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, true, false, false, DMAX>;
        s.fn[kB64KmajorFly] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, true, false, false, false, DMAX>;
    }
    if constexpr (!B32ONLY && KK == 1 && !SKINNY)
        s.fn[kB64PlanesBoth] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, true, false, false, DMAX, true>;
    if constexpr (!B32ONLY && KK == 1 && SKINNY) {
        s.fn[kB64FlyBPlanes] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, false, false, DMAX, true>;
        s.fn[kB64GroupBPlanes] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, true, false, DMAX, true>;
    }
    if constexpr (NB <= 5) {          // int32 values never need more than five digits
        s.fn[kB32Fly] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, false, false, false, false, DMAX>;
        s.fn[kB32Planes] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, false, true, false, false, DMAX>;
        s.fn[kB32KmajorFly] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, true, false, false, false, DMAX>;
    }
    if constexpr (SKINNY) {          // grouped launches (one B per segment of rows) run on the 32-row tiles only
        if constexpr (!B32ONLY) s.fn[kB64Group] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, true, false, DMAX>;
        if constexpr (NB <= 5) s.fn[kB32Group] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, false, false, true, false, DMAX>;
        // and so do products whose B is divided by a power of two first (the model's head projection)
        if constexpr (!B32ONLY) s.fn[kB64FlyRs] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, false, false, false, false, true, DMAX>;
        if constexpr (NB <= 5) s.fn[kB32FlyRs] = gemm_mfma_kernel<NA, NB, WVM, WVN, WM, WN, KK, true, false, false, false, true, DMAX>;
    }
    s.finish = gemm_split_finish_kernel<WVM, WVN, WM, WN>;
    s.planes[0] = a_planes_kernel<NA, 2, KK>;
    s.planes[1] = a_planes_kernel<NA, 4, KK>;
    return s;
}

// 64x64 tiles, A always split on the fly
template <int NA, int NB, int KK>
static Instance make_short_instance()
{
    static_assert(NA + NB <= 8, "two workgroups' LDS and registers fit a compute unit up to seven diagonals");
    Instance s = {};
    s.na = NA; s.nb = NB; s.bm = 64; s.bn = 64; s.threads = 256; s.kk = KK;
    s.dmax = 16;
    s.short_k = true;
    s.fn[kB64Fly] = gemm_mfma_short_kernel<NA, NB, KK, false, false>;
    s.fn[kB64KmajorFly] = gemm_mfma_short_kernel<NA, NB, KK, false, true>;
    s.fn[kB32Fly] = gemm_mfma_short_kernel<NA, NB, KK, true, false>;
    s.fn[kB32KmajorFly] = gemm_mfma_short_kernel<NA, NB, KK, true, true>;
    s.finish = gemm_split_finish_kernel<2, 2, 1, 1>;
    return s;
}

// the instance lists of the translation units
void mfma_instances_short(std::vector<Instance> &out);
void mfma_instances_narrow(std::vector<Instance> &out);
void mfma_instances_mid(std::vector<Instance> &out);
void mfma_instances_wide(std::vector<Instance> &out);
void mfma_instances_both(std::vector<Instance> &out);
void mfma_instances_pruned(std::vector<Instance> &out);
void mfma_instances_rows32(std::vector<Instance> &out);
void mfma_instances_rows32b(std::vector<Instance> &out);
void mfma_instances_rows32c(std::vector<Instance> &out);
void mfma_instances_rows32d(std::vector<Instance> &out);
void mfma_instances_rows32e(std::vector<Instance> &out);

}  // namespace zk
