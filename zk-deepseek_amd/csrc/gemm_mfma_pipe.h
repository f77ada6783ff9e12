// Products whose operands are BOTH digit planes (A pre-split by the pass in front; B prepared once, or pre-split like A where
// it is small next to the product): nothing is split, tracked or staged in registers, so a step is loads, fragment reads
// and MFMAs only, and it is written as a software pipeline instead of the fenced phases of gemm_mfma_block:
//   * the planes of a step are blocks of 1 KB, already in fragment order; every wavefront sends its share of them from
//     global memory straight into a ring of LDS stages (global_load_lds_dwordx4), kPipeStages - 1 steps before they are
//     multiplied, one load at a time between MFMAs;
//   * the fragments of step s+1 are read into registers while the MFMAs of step s run, each into the registers whose last
//     use has just been issued (the MFMAs go through A's digits in order and through B's within each), so that the
//     matrix pipe has its operands when the step's one barrier opens;
//   * a workgroup walks several tiles (one workgroup per compute unit), and the ring runs on across them: the first steps
//     of the next tile are loaded while this one is multiplied and stored.  With a short K (512: sixteen steps) a tile's
//     first loads and its epilogue are a third of its time.
// What bounds it: the matrix pipe at the clock the device grants it.  A step takes 0.81 / 1.11 us on 128x128 tiles with
// (3,3) / (3,4) digits and 0.79 / 1.04 on 128x64 with (4,4) / (5,5): 2.7-3.2 POP/s of i8 products while steps run, where the
// probe that multiplies random bytes out of LDS and loads nothing does 2.9.  A tile's epilogue, in which all eight wavefronts of
// a compute unit's only workgroup combine and store, comes on top and leaves the matrix pipe idle: 8-9 us against 18 of steps at
// K = 512, so that 131072 rows x [1024,512] take 800-850 us, 2.0 POP/s.  Then LDS (108 KB per 1536 cycles of (3,4) MFMAs).  128x128 tiles need 16 (NA + NB - 1) x 2
// accumulator registers per lane: up to six diagonals fit beside two wavefronts per SIMD, more take 128x64 tiles.
// Against gemm_mfma_block on planes of A alone: see pipe_b_planes in gemm_mfma.hip.
//
// All of a row tile's later steps may hold nothing but zeros in A (the probabilities of a causal prompt: a token's rows
// end at its own position): p.row_steps then says how many steps of a row tile there are to multiply.
#pragma once
#include "lds_dma.h"

namespace zk {

constexpr int kPipeStages = 5;

// tile shape by diagonals: 128x128 as 2x4 wavefronts of 64x32, or 128x64 as 4x2 of 32x32
constexpr bool pipe_wide(int na, int nb) { return na + nb - 1 <= 6; }
constexpr size_t pipe_lds_bytes(int na, int nb) { return (size_t)kPipeStages * (4 * na + (pipe_wide(na, nb) ? 4 : 2) * nb) * 1024; }

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<I + 1, N>(f);
    }
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t uniform64(uint64_t v)
{
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32;
}

// one tile, or one slice of K of a split tile
struct PipeItem {
    int g, tm, tn, ks_begin, nsteps, tail_tile, sidx, i;      // i: its number
};

// The launch's arguments, read again wherever a tile begins or ends.  (Kept in scalar registers through the steps, they and
// what the compiler derives from them took 110 more than there are; the spills' reloads were then waited for inside the
// steps, and every such wait drained the ring: 1.30 us per step of (3,4) digits where 1.11 is what the matrix pipe takes
// at the clock it is given.)
typedef const __attribute__((address_space(4))) MfmaParams ConstParams;
__device__ __forceinline__ ConstParams &launch_args()
{
    ConstParams *q = (ConstParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return *q;
}

template <int NA, int NB>
__global__ __launch_bounds__(512) void gemm_mfma_pipe_kernel(MfmaParams)
{
    constexpr bool WIDE = pipe_wide(NA, NB);
    constexpr int D = NA + NB - 1, STG = kPipeStages, AHEAD = STG - 1, T = 512;
    constexpr int WVN = WIDE ? 4 : 2, WM = WIDE ? 2 : 1, BN = 32 * WVN;
    constexpr int A_BLOCKS = 4 * NA, BLOCKS = A_BLOCKS + WVN * NB, STAGE = BLOCKS * 1024;
    constexpr int LOADS = (BLOCKS + 7) / 8;                 // per wavefront and step (the last wavefront's may repeat the last block)
    static_assert(WM * D * 16 + WM * NA * 4 + NB * 4 <= 240, "two wavefronts share a SIMD");
    static_assert(LOADS * AHEAD < 64, "vmcnt is a 6-bit counter");
    static_assert(NA * NB >= LOADS, "the loads ride behind the MFMAs");
    extern __shared__ __attribute__((aligned(16))) unsigned char pipe_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int wm = wave / WVN, wn = wave % WVN;
    const unsigned ring_lds = (unsigned)(uintptr_t)pipe_smem, lane16 = (unsigned)lane * 16;

    // ---- work items: number i of this workgroup's walk, i = blockIdx.x + n * gridDim.x; false: no such item ----
    auto decode = [](int i) {
        ConstParams &p = launch_args();
        const int per_batch = p.tiles_m * p.tiles_n, tiles_m = p.tiles_m, tiles_n = p.tiles_n;
        const int ksteps = (p.K + 31) / 32;                 // (the planes are padded with zeros to whole steps)
        int g, tm, tn, tail_tile = 0, sidx = 0, nsplit = 1;
        if (p.row_order) {
            // Consecutive ids go round the 8 XCDs: an XCD takes every eighth row tile and all its tile columns, so that its
            // planes of A come from memory once and row tiles of different lengths are dealt evenly.
            const int q = i >> 3, r = q / tiles_n * 8 + (i & 7);
            tn = q % tiles_n;
            g = r / tiles_m;
            tm = r - g * tiles_m;
            if (g >= p.batches) g = -1;
        } else {
            int lin = i;
            if (lin < p.main_tiles) {
                if ((p.main_tiles & 7) == 0) lin = (lin & 7) * (p.main_tiles >> 3) + (lin >> 3);
            } else {
                const int t = lin - p.main_tiles;
                if (p.tail_xcd) {
                    const int x = t & 7, q = t >> 3;
                    const int pair = (q / tiles_m) * 8 + x;
                    lin = p.main_tiles + (pair / p.split) * tiles_m + q % tiles_m;
                    sidx = pair % p.split;
                } else {
                    lin = p.main_tiles + t / p.split;
                    sidx = t % p.split;
                }
                nsplit = p.split;
            }
            tail_tile = lin - p.main_tiles;
            g = lin / per_batch;
            const int rem = lin - g * per_batch;
            if (p.n_fastest) { tm = rem / tiles_n; tn = rem % tiles_n; }
            else { tn = rem / tiles_m; tm = rem % tiles_m; }
        }
        const int ks_begin = (int)((long)sidx * ksteps / nsplit);
        int ks_end = (int)((long)(sidx + 1) * ksteps / nsplit);
        if (p.row_steps && g >= 0) {
            // (a scalar load: were it a vector load, the compiler would keep waiting for it, and with it for the whole ring)
            const int live = *(const __attribute__((address_space(4))) int *)(p.row_steps + uniform64((uint64_t)((long)g * tiles_m + tm)));
            ks_end = live < ks_end ? live : ks_end;
        }
        // (at least one step, of zeros if need be: the accumulators are set by it)
        return PipeItem{ uniform(g), uniform(tm), uniform(tn), uniform(ks_begin), uniform(ks_end > ks_begin ? ks_end - ks_begin : 1),
                         uniform(tail_tile), uniform(sidx), i };
    };
    auto next_item = [&](int i) {                           // the first item from i on; its g is negative if there is none
        const int items = launch_args().items;
        PipeItem it{ -1, 0, 0, 0, 1, 0, 0, i };
        while (it.i < items && (it = decode(it.i)).g < 0) it.i += gridDim.x;
        return it;
    };

    // ---- loading: this wavefront's blocks of a step, numbers wave * LOADS + l of [A: 32-row group 0..3][digit], [B: 32-column group][digit] ----
    PipeItem li;
    int l_left;
    uint64_t l_src[LOADS];
    auto aim = [&]() {
        ConstParams &p = launch_args();
#pragma unroll
        for (int l = 0; l < LOADS; l++) {
            int b = wave * LOADS + l;
            b = b < BLOCKS ? b : BLOCKS - 1;
            if (b < A_BLOCKS) {
                const int grp = b / NA, dig = b - grp * NA;
                l_src[l] = uniform64((uint64_t)p.a_planes + ((((long)li.g * p.a_msub + li.tm * 4 + grp) * p.a_ksteps + li.ks_begin) * NA + dig) * 1024);
            } else {
                const int bb = b - A_BLOCKS, grp = bb / NB, dig = bb - grp * NB;
                int sub = li.tn * WVN + grp;
                sub = sub < p.b_nsub ? sub : p.b_nsub - 1;  // column groups past N: any valid data, never stored
                l_src[l] = uniform64((uint64_t)p.B + (uint64_t)li.g * p.b_gstride + (((long)sub * p.b_ksteps + li.ks_begin) * NB + dig) * 1024);
            }
        }
    };
    auto issue_one = [&](unsigned stage, auto l_tag) {
        constexpr int L = decltype(l_tag)::value;
        int b = wave * LOADS + L;
        b = b < BLOCKS ? b : BLOCKS - 1;
        lds_dma16_uniform(l_src[L], lane16, ring_lds + stage * STAGE + b * 1024);
    };
    // the loads move on to the next step (past the last one they repeat it, into stages nobody reads any more)
    auto advance = [&]() {
        if (--l_left > 0) {
#pragma unroll
            for (int l = 0; l < LOADS; l++) {
                const int b = wave * LOADS + l;
                l_src[l] += (b < A_BLOCKS ? NA : NB) * 1024;
            }
            return;
        }
        l_left = 1;
        if (li.g >= 0) {
            li = next_item(li.i + gridDim.x);
            if (li.g >= 0) { l_left = li.nsteps; aim(); }
        }
    };

    PipeItem it = next_item((int)blockIdx.x);
    if (it.g < 0) return;
    li = it;
    l_left = li.nsteps;
    aim();

    v16i acc[WM][D];
    v4i fa[WM][NA], fb[NB];
    auto read_a = [&](unsigned st, int a, int i) {
        return *reinterpret_cast<const v4i *>(pipe_smem + st * STAGE + ((wm * WM + a) * NA + i) * 1024 + lane16);
    };
    auto read_b = [&](unsigned st, int j) {
        return *reinterpret_cast<const v4i *>(pipe_smem + st * STAGE + (A_BLOCKS + wn * NB + j) * 1024 + lane16);
    };

    // prologue: AHEAD steps under way, the first one's fragments in registers
#pragma unroll 1
    for (unsigned t = 0; t < AHEAD; t++) {
        static_for<0, LOADS>([&](auto l) { issue_one(t, l); });
        advance();
    }
    wait_vmcnt<LOADS * (AHEAD - 1)>();                     // step 0 has landed (my share)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    unsigned st_next = 1, st_load = AHEAD;                  // stages of step s+1 and of step s+AHEAD
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
        for (int i = 0; i < NA; i++) fa[a][i] = read_a(0, a, i);
#pragma unroll
    for (int j = 0; j < NB; j++) fb[j] = read_b(0, j);

    // Step s: the MFMAs of step s on the fragments in registers; beside them the fragment reads of step s+1 (landed and
    // fenced by the barrier at the top) and the loads of step s+AHEAD into the stage step s-1 was read from (those reads
    // were waited for by the MFMAs of step s-1, so the barrier need not wait for LDS).
    auto step = [&](auto first_tag) {
        constexpr bool FIRST = decltype(first_tag)::value;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, NA>([&](auto i_tag) {
            constexpr int I = decltype(i_tag)::value;
            static_for<0, NB>([&](auto j_tag) {
                constexpr int J = decltype(j_tag)::value;
                constexpr bool ZERO = FIRST && (I == 0 || J == NB - 1);      // the first pair of diagonal I + J
                const v16i zero = {};
#pragma unroll
                for (int a = 0; a < WM; a++)
                    acc[a][I + J] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][I], fb[J], ZERO ? zero : acc[a][I + J], 0, 0, 0);
                constexpr int L = I * NB + J;
                if constexpr (L < LOADS) {
                    __builtin_amdgcn_sched_barrier(0);
                    issue_one(st_load, std::integral_constant<int, (L < LOADS ? L : 0)>());
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (I == NA - 1) {                // digit J of B has been issued for the last time this step
                    fb[J] = read_b(st_next, J);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
#pragma unroll
            for (int a = 0; a < WM; a++) fa[a][I] = read_a(st_next, a, I);   // and so has digit I of A
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto move_on = [&]() {
        advance();
        st_next = st_next + 1 == STG ? 0 : st_next + 1;
        st_load = st_load + 1 == STG ? 0 : st_load + 1;
    };

    int landed = 0;                                         // steps whose loads are known to have landed beyond what a step needs
    for (;;) {
        // before a step: the one behind it has landed (my share), the AHEAD - 2 after that may be under way
        if (landed > 0) landed--; else wait_vmcnt<LOADS * (AHEAD - 2)>();
        step(std::true_type());
        for (int s = it.nsteps; s > 1; s--) {
            move_on();
            if (landed > 0) landed--; else wait_vmcnt<LOADS * (AHEAD - 2)>();
            step(std::false_type());
        }
        move_on();
        // The stores below count like loads and may complete out of turn with them: everything issued so far is waited for
        // here, and the next tile's first steps, which that covers, wait for nothing (by the time a later one does, the
        // stores are through).
        wait_vmcnt<0>();
        landed = AHEAD - 1;

        // epilogue: diagonals -> 128-bit sum -> shift, as in gemm_mfma_block (accumulator register r of lane l holds
        // row 8*(r/4) + 4*(l/32) + r%4, column l%32 of its 32 x 32 tile)
        ConstParams &p = launch_args();
        const int m0 = it.tm * 128, n0 = it.tn * BN, sh = p.shift, sum0 = (int)p.init;
        const uint64_t rmask = sh ? ((1ull << sh) - 1) : 0;
        auto combine = [&](int a, int r, int init) { return sum_diagonals<D>([&](int d) { return acc[a][d][r]; }, init); };
        if (!p.row_order && it.tail_tile >= 0 && p.split > 1) {
            // raw partial sums in the layout gemm_split_finish_kernel<8 / WVN, WVN, WM, 1> adds up
#pragma unroll
            for (int a = 0; a < WM; a++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    if (m0 + (wm * WM + a) * 32 + 8 * (r >> 2) + (r & 3) >= p.M) continue;
                    const Words sum = combine(a, r, 0);
                    const long q = (((long)it.tail_tile * p.split + it.sidx) * (T / 64) + wave) * (WM * 16) + a * 16 + r;
                    const uint64_t lo = (uint64_t)sum.w[1] << 32 | sum.w[0];
                    if (p.part64) p.partials[q * 64 + lane] = lo;
                    else { p.partials[q * 128 + lane] = lo; p.partials[q * 128 + 64 + lane] = (uint64_t)sum.w[3] << 32 | sum.w[2]; }
                }
        } else {
            auto store_tile = [&](auto edge_tag, auto rem_tag) {
                constexpr bool EDGE = decltype(edge_tag)::value, REM = decltype(rem_tag)::value;
                const int n = n0 + wn * 32 + (lane & 31);
#pragma unroll
                for (int a = 0; a < WM; a++) {
                    const int mrow = m0 + (wm * WM + a) * 32 + 4 * (lane >> 5);
                    const long o0 = (long)it.g * p.sC + (long)mrow * p.ldc + n;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int dr = 8 * (r >> 2) + (r & 3);
                        const Words sum = combine(a, r, sum0);
                        if (EDGE && !(mrow + dr < p.M && n < p.N)) continue;
                        const long o = o0 + (long)dr * p.ldc;
                        p.C[o] = shifted_sum(sum, sh);
                        if (REM) p.R[o] = sum_below(sum, rmask);
                    }
                }
            };
            const bool edge = m0 + 128 > p.M || n0 + BN > p.N;
            if (p.R) { if (edge) store_tile(std::true_type(), std::true_type()); else store_tile(std::false_type(), std::true_type()); }
            else { if (edge) store_tile(std::true_type(), std::false_type()); else store_tile(std::false_type(), std::false_type()); }
        }
        it = next_item(it.i + gridDim.x);
        if (it.g < 0) break;
        // the fragments of its first step once more (read beside the last step's MFMAs already, but no register keeps them
        // through the epilogue)
        const unsigned st = st_next == 0 ? STG - 1 : st_next - 1;
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int i = 0; i < NA; i++) fa[a][i] = read_a(st, a, i);
#pragma unroll
        for (int j = 0; j < NB; j++) fb[j] = read_b(st, j);
    }
    wait_vmcnt<0>();                                       // (the loads past the end)
}

// Digit counts (A, B) that this kernel and the one that splits A itself (gemm_mfma_rowtile.h) exist for: one list, since a product that
// finds the first may be given to the second.
#define ZK_PIPE_DIGITS(X) X(3, 3) X(3, 4) X(4, 3) X(4, 4) X(3, 5) X(6, 3) X(5, 4) X(4, 5) X(5, 5)

// the kernel for digit counts (na, nb) or null, its dynamic LDS, its tile columns and its finishing kernel
struct PipeForm {
    MfmaKernel fn;
    FinishKernel finish;
    int bn;
    size_t lds;
};
PipeForm pipe_form(int na, int nb);

}  // namespace zk
