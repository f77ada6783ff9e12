// Products so small that launches and latencies are all they cost (the attention of a decoding step: 128 heads against
// the cache): one launch, nothing guessed.  What bounds them is one round trip to memory per step of a wavefront.
//
// On the general kernel such a product is three dependent launches (tiles cut along K, the sum of the slices, the guarded
// launch behind a guess of digit counts) of 4 to 11 us each.  Here a workgroup owns a tile of 16 x 16 outputs and all of K: its
// eight (or four) wavefronts take every eighth (fourth) step of 64 k, load their fragments straight into registers (the four lanes of a
// row read 64 contiguous bytes per load), take the digit counts that those need (3, 4 or 5 per operand, gemm_frag16.h),
// split, multiply, and meet in LDS with their 128-bit sums.  A wavefront that meets values beyond five digits (2^38 and up) goes on with
// nine digits for the side that needs them, from the step it holds.  Its share read again with nine digits on both sides / so, a cache of 44 bits, us
// a call: 128 rows x [779,512] k-contiguous 14.8 / 11.4 (13.2 with eight wavefronts of one step each), x [779,576] 16.5 / 13.2, x
// [300,576] 12.1 / 8.8, n-contiguous x [576,512] 12.9 / 9.8, x [576,779] 16.3 / 14.2.  Narrow values are level (n-contiguous 0.05-0.2 us more).
// Where no wavefront has more than one step (K up to 512, or 256) there is no loop around it: narrow and 44 bits, loop / this, 128 rows x
// [512,257] n-contiguous 5.8 / 4.9 and 6.8 / 5.9, x [300,512] k-contiguous 7.2 / 6.9 and 8.2 / 7.6.
#include "gemm_frag16.h"

#include <atomic>

namespace zk {

struct SmallParams {
    const int64_t *A, *B;
    int64_t *C;
    long lda, sA, ldbn, ldbk, sB, ldc, sC;
    int M, N, K, shift, tiles_m, tiles_n;
    int64_t init;
};

constexpr int kSmallTile = 16, kSmallDiagonals = 9, kSmallWideDiagonals = 16;   // of five digits a side, of nine (what lies at 2^128 and above does not matter)
// Where it pays, against the general and the 16-row kernels over 250 shapes of 5 to 600 rows and 16 to 2048 columns (those / this, us):
// one round of tiles 0.3-0.8 of their time up to K = 2048 (128 rows x [512,779] n-contiguous 20.0 / 8.9, 50 x [94,321] (5,5)
// 24.9 / 7.1, 32 x [1513,759] 23.2 / 8.7, 274 x [161,2145] 22.6 / 16.2) and level at 4000; two rounds up to K = 1024 (128 x
// [779,512] 18.8 / 10.4, 128 x [1024,512] 19.4 / 10.9; 66 x [1398,1454] 26.5 / 30.4); three rounds no longer (256 x [779,512]
// 19.4 / 21.1).  Offered to it are scores and values of up to eight positions (kFewPositions).
constexpr int kSmallMaxK = 2048, kSmallMaxKTwoRounds = 1024;

template <int NA, int NB, int D>
__device__ __forceinline__ void small_step(const RawFrag<false> &fa_raw, const RawFrag<false> &fb_raw, v4i (&acc)[D])
{
    v4i fa[NA], fb[NB];
    split_frag<NA, false>(fa_raw, fa);
    split_frag<NB, false>(fb_raw, fb);
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (i + j < D) acc[i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i], fb[j], acc[i + j], 0, 0, 0);
}

// up to five digits a side
__device__ __forceinline__ void small_narrow_step(int na, int nb, const RawFrag<false> &fa, const RawFrag<false> &fb, v4i (&acc)[kSmallDiagonals])
{
    switch ((na - 3) * 3 + (nb - 3)) {
    case 0: small_step<3, 3>(fa, fb, acc); break;
    case 1: small_step<3, 4>(fa, fb, acc); break;
    case 2: small_step<3, 5>(fa, fb, acc); break;
    case 3: small_step<4, 3>(fa, fb, acc); break;
    case 4: small_step<4, 4>(fa, fb, acc); break;
    case 5: small_step<4, 5>(fa, fb, acc); break;
    case 6: small_step<5, 3>(fa, fb, acc); break;
    case 7: small_step<5, 4>(fa, fb, acc); break;
    default: small_step<5, 5>(fa, fb, acc); break;
    }
}

__device__ __forceinline__ u128 words_value(const Words &t) { return (u128)((uint64_t)t.w[3] << 32 | t.w[2]) << 64 | ((uint64_t)t.w[1] << 32 | t.w[0]); }

// any width
__device__ __forceinline__ void small_wide_step(int na, int nb, const RawFrag<false> &fa, const RawFrag<false> &fb, v4i (&acc)[kSmallWideDiagonals])
{
    if (na <= 5) small_step<5, 9>(fa, fb, acc);
    else if (nb <= 5) small_step<9, 5>(fa, fb, acc);
    else small_step<9, 9>(fa, fb, acc);
}

// A fragment element by element: byte b of the fragment is k = frag_k(q, b) of the step, `lane_at` the lane's offset with its
// first k, `step_at` the step's first element, `ldk` elements from one k to the next; k of `k_left` and up are zeros.  (Offsets
// that all lanes share stay in scalar registers.)
__device__ __forceinline__ void load_elements(RawFrag<false> &f, const int64_t *base, long lane_at, long step_at, long ldk, int k_left)
{
#pragma unroll
    for (int b = 0; b < 16; b++) {
        const int k = frag_k<false>(0, b);
        const int64_t *at = base + (step_at + k * ldk);
        const int64_t x = k < k_left ? ((const ZK_GLOBAL_MEM int64_t *)at)[lane_at] : 0;
        f.v[b >> 1][2 * (b & 1)] = (int)(uint32_t)x;
        f.v[b >> 1][2 * (b & 1) + 1] = (int)(uint32_t)((uint64_t)x >> 32);
    }
}

// BKM: B is contiguous along n.  ONE: no wavefront has more than one step
template <bool BKM, bool ONE, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2))) void gemm_small_kernel(SmallParams p)
{
    __shared__ Words red[WAVES][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, q = lane >> 4;
    const int per_batch = p.tiles_m * p.tiles_n;
    const int g = blockIdx.x / per_batch, rem = blockIdx.x - g * per_batch;
    const int m0 = rem % p.tiles_m * kSmallTile, n0 = rem / p.tiles_m * kSmallTile;

    // this lane's rows (clamped: what lies past the end lands in outputs that are never stored)
    const long a_at = (long)g * p.sA + (long)(m0 + li < p.M ? m0 + li : p.M - 1) * p.lda;
    const long ldbk = BKM ? p.ldbk : 1;
    const int nc = n0 + li < p.N ? n0 + li : p.N - 1;
    const long b_at = (long)g * p.sB + (long)nc * p.ldbn;
    const bool a_vec = (((uintptr_t)p.A | (uintptr_t)(p.lda * 8) | (uintptr_t)(p.sA * 8)) & 15) == 0;
    const bool b_vec = !BKM && (((uintptr_t)p.B | (uintptr_t)(p.ldbn * 8) | (uintptr_t)(p.sB * 8)) & 15) == 0;

    const int steps = (p.K + 63) / 64;
    auto load = [&](int ks, RawFrag<false> &fa, RawFrag<false> &fb) {
        const int k0 = ks * 64, k_left = p.K - k0, kq = frag_k<false>(q, 0);
        const bool whole = k_left >= 64;
        if (whole && b_vec) {
#pragma unroll
            for (int j = 0; j < 8; j++) fb.v[j] = *(const ZK_GLOBAL_MEM v4i *)(p.B + b_at + k0 + frag_k<false>(q, 2 * j));
        } else if (whole) {
            load_elements(fb, p.B, b_at + kq * ldbk, k0 * ldbk, ldbk, 64);
        } else {
            load_elements(fb, p.B, b_at + kq * ldbk, k0 * ldbk, ldbk, k_left - kq);
        }
        if (whole && a_vec) {
#pragma unroll
            for (int j = 0; j < 8; j++) fa.v[j] = *(const ZK_GLOBAL_MEM v4i *)(p.A + a_at + k0 + frag_k<false>(q, 2 * j));
        } else if (whole) {
            load_elements(fa, p.A, a_at + kq, k0, 1, 64);
        } else {
            load_elements(fa, p.A, a_at + kq, k0, 1, k_left - kq);
        }
    };
    // accumulator register r of lane (li, q) holds row 4*q + r, column li of the tile
    auto store_sums = [&](auto &acc) {
        constexpr int D = sizeof(acc) / sizeof(v4i);
#pragma unroll
        for (int o = 0; o < 4; o++) red[wave][o][lane] = sum_diagonals<D>([&](int d) { return acc[d][o]; }, 0);
    };
    // HELD: the step that shows values beyond five digits outlives the loop in its registers.  Eight wavefronts with B contiguous along n read
    // their share again instead: holding it costs them 0.15 us of 8.6 on 128 rows x [512,779] of narrow values (it would save 2.4 of 12.1 with
    // 44 bits), and values are narrow in the model.
    constexpr bool HELD = !BKM || WAVES == 4;
    // (5 pairs, of nine digits 9, x 64 products of 2^14 a step)
    static_assert((kSmallMaxK / 64 + WAVES - 1) / WAVES * 9L * 64 * 16384 <= kMaxDiagonal, "the int32 accumulators hold a wavefront's share");
    if (ONE) {
        RawFrag<false> fa, fb;
        int na = 0, nb = 0;
        if (wave < steps) {
            load(wave, fa, fb);
            na = wave_digits(magnitude_or<false>(fa));
            nb = wave_digits(magnitude_or<false>(fb));
        }
        // (each width adds up its own sums: with a choice between the two sets of accumulators in front of the sums a call took 0.9 us
        // more, 128 rows x [779,512] on eight wavefronts)
        if (na == 0) {
#pragma unroll
            for (int o = 0; o < 4; o++) red[wave][o][lane] = Words{};
        } else if (na <= 5 && nb <= 5) {
            v4i acc[kSmallDiagonals];
#pragma unroll
            for (int d = 0; d < kSmallDiagonals; d++) acc[d] = v4i{ 0, 0, 0, 0 };
            small_narrow_step(na, nb, fa, fb, acc);
            store_sums(acc);
        } else {
            v4i acc[kSmallWideDiagonals];
#pragma unroll
            for (int d = 0; d < kSmallWideDiagonals; d++) acc[d] = v4i{ 0, 0, 0, 0 };
            small_wide_step(na, nb, fa, fb, acc);
            store_sums(acc);
        }
    } else if constexpr (HELD) {
        v4i acc[kSmallDiagonals];
#pragma unroll
        for (int d = 0; d < kSmallDiagonals; d++) acc[d] = v4i{ 0, 0, 0, 0 };
        RawFrag<false> fa, fb;
        int na = 0, nb = 0, ks = wave;
        for (; ks < steps; ks += WAVES) {
            load(ks, fa, fb);
            na = wave_digits(magnitude_or<false>(fa));
            nb = wave_digits(magnitude_or<false>(fb));
            if (na > 5 || nb > 5) break;
            small_narrow_step(na, nb, fa, fb, acc);
        }
        if (ks >= steps) {
            store_sums(acc);
        } else {
            // (the sums so far are the lower diagonals of the wide ones)
            v4i wide[kSmallWideDiagonals];
#pragma unroll
            for (int d = 0; d < kSmallWideDiagonals; d++) wide[d] = d < kSmallDiagonals ? acc[d] : v4i{ 0, 0, 0, 0 };
            for (;;) {
                small_wide_step(na, nb, fa, fb, wide);
                ks += WAVES;
                if (ks >= steps) break;
                load(ks, fa, fb);
                na = wave_digits(magnitude_or<false>(fa));
                nb = wave_digits(magnitude_or<false>(fb));
            }
            store_sums(wide);
        }
    } else {
        v4i acc[kSmallDiagonals];
#pragma unroll
        for (int d = 0; d < kSmallDiagonals; d++) acc[d] = v4i{ 0, 0, 0, 0 };
        bool wide = false;
        for (int ks = wave; ks < steps; ks += WAVES) {
            RawFrag<false> fa, fb;
            load(ks, fa, fb);
            const int na = wave_digits(magnitude_or<false>(fa));
            const int nb = wave_digits(magnitude_or<false>(fb));
            if (na > 5 || nb > 5) { wide = true; break; }
            small_narrow_step(na, nb, fa, fb, acc);
        }
        store_sums(acc);
        if (wide) {
            v4i wacc[kSmallWideDiagonals];
#pragma unroll
            for (int d = 0; d < kSmallWideDiagonals; d++) wacc[d] = v4i{ 0, 0, 0, 0 };
            for (int ks = wave; ks < steps; ks += WAVES) {
                RawFrag<false> fa, fb;
                load(ks, fa, fb);
                small_step<9, 9>(fa, fb, wacc);
            }
            store_sums(wacc);
        }
    }
    __syncthreads();
    const int m = m0 + 4 * q + (wave & 3), n = n0 + li;
    if (wave >= 4 || m >= p.M || n >= p.N) return;
    u128 s = (u128)(i128)p.init;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        s += words_value(red[w][wave][lane]);
    }
    const uint64_t lo = (uint64_t)s, hi = (uint64_t)(s >> 64);
    p.C[(long)g * p.sC + (long)m * p.ldc + n] = (int64_t)((lo >> p.shift) | ((hi << 1) << (63 - p.shift)));
}

static std::atomic<long> g_small_calls(0);
long gemm_small_calls() { return g_small_calls; }

bool gemm_small_launch(const GemmDesc &d)
{
    const long tiles_m = (d.M + kSmallTile - 1) / kSmallTile, tiles_n = (d.N + kSmallTile - 1) / kSmallTile, tiles = tiles_m * tiles_n * d.G;
    if (d.b32 || d.R || d.a_rs != 1 || d.b_rs != 1 || d.K < 1 || d.K > kSmallMaxK || d.M < 1 || d.N < 1 || d.G < 1) return false;
    if (tiles > (d.K <= kSmallMaxKTwoRounds ? 2 : 1) * (long)device_cus()) return false;
    SmallParams p = {};
    p.A = d.A; p.B = reinterpret_cast<const int64_t *>(d.B); p.C = d.C;
    p.lda = d.lda; p.sA = d.sA; p.ldbn = d.ldbn; p.ldbk = d.ldbk; p.sB = d.sB; p.ldc = d.ldc; p.sC = d.sC;
    p.M = d.M; p.N = d.N; p.K = d.K; p.shift = d.shift; p.init = d.init;
    p.tiles_m = (int)tiles_m; p.tiles_n = (int)tiles_n;
    const dim3 grid((unsigned)tiles);
    // More tiles than compute units: four wavefronts each, two workgroups to a unit (their registers leave room for no more than two of
    // four), so that all tiles run at once and one loads while the other multiplies.  Eight / four wavefronts, us: 128 rows x [779,512] 11.7 / 10.4, x
    // [779,64] 6.5 / 6.1, x [1024,576] 15.9 / 13.3, n-contiguous x [1024,779] 18.0 / 14.9, 256 rows x [512,779] 15.2 / 11.9.
    const int waves = tiles > device_cus() ? 4 : 8;
    const bool one = d.K <= 64 * waves;
#define ZK_SMALL(BKM) do { if (waves == 4) { if (one) gemm_small_kernel<BKM, true, 4><<<grid, dim3(256), 0, 0>>>(p); else gemm_small_kernel<BKM, false, 4><<<grid, dim3(256), 0, 0>>>(p); } \
                           else if (one) gemm_small_kernel<BKM, true, 8><<<grid, dim3(512), 0, 0>>>(p); else gemm_small_kernel<BKM, false, 8><<<grid, dim3(512), 0, 0>>>(p); } while (0)
    if (d.ldbk != 1) ZK_SMALL(true); else ZK_SMALL(false);
#undef ZK_SMALL
    g_small_calls++;
    return true;
}

}  // namespace zk
