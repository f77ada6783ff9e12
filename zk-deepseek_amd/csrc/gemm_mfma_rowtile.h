// Products of many rows with a B that is small next to them (a KV cache against the queries of a whole prompt, one head's
// weights): B is split into digit planes by a pass in front (b_planes_kernel), A by this kernel itself, row tile by row tile.
//   * A workgroup owns 64 rows of A at a time.  It reads them once, splits them into digit planes in a slot of scratch memory of
//     its own (a slot is written and read by one workgroup only; the slots outgrow the L2s, and the cache behind those serves the loads), and
//     multiplies all tile columns, or a part of them, from there.  A share of the next row tile is split behind every tile.  As a pass
//     of its own the split writes its planes to memory and reads them back: 435 of 2500 us of the attention core on 1024
//     tokens.
//   * Two workgroups of four wavefronts share a compute unit, and nothing ties them to one another: while one splits, or combines
//     and stores a tile, the other has the matrix pipe.
//   * Steps are those of gemm_mfma_pipe.h: planes travel straight into a ring of LDS stages, the fragments of step s+1 are
//     read beside the MFMAs of step s, each into the registers whose last use has just been issued.  Half of a compute
//     unit's LDS leaves three to five stages, so a stage is loaded again as soon as its fragments are in registers.
// Row tiles whose later steps hold nothing but zeros in A (the probabilities of a causal prompt: a token's rows end at its
// own position) end there; the split sees it.
// What bounds it: stores and splits that the steps do not hide, and the steps themselves.  131072 rows x [1024,512], (3,4) digits, 780-790
// us: 630 with neither stores nor splits (2.6 POP/s of i8 products, what the pipelined kernel reaches on ready planes), 595 with every load at
// one address on top; the stores add 105 and the splits 110-130, overlapped or not.  As a whole the matrix pipe is busy 53 % of the
// time at 1.88 GHz, for the values of 1024 causal tokens 33 % at 2.17 GHz; each tile column reads the planes of A again from beyond
// the L2s (1.6 GB beside 0.54 of A).  Whole calls, pass over A and pipelined kernel / this, both on one device, medians of six runs in turn: 131072 x
// [1024,512] 876 / 833 us (869-885 / 827-896), x [1024,64] 266 / 239, values of 1024 causal tokens 643 / 579, 31104 x [243,512] 85 / 76.
#pragma once
#include "gemm_mfma_pipe.h"

namespace zk {

// tiles of 64x128 (1x4 wavefronts of 64x32) up to six diagonals, else 64x64 (2x2 of 32x32): what fits 256 registers
constexpr int rowtile_cols(int na, int nb) { return pipe_wide(na, nb) ? 128 : 64; }
constexpr int rowtile_blocks(int na, int nb) { return 2 * na + rowtile_cols(na, nb) / 32 * nb; }
constexpr int rowtile_stages(int na, int nb) { return 80 / rowtile_blocks(na, nb) < 5 ? 80 / rowtile_blocks(na, nb) : 5; }
constexpr size_t rowtile_lds_bytes(int na, int nb) { return (size_t)rowtile_stages(na, nb) * rowtile_blocks(na, nb) * 1024; }

constexpr int kRowtileRows = 64;

// One item: row tile `tm` of batch `g`, or a part of its tile columns.  p.a_planes: slots of `a_ksteps` steps of planes of 64 rows, `a_msub` per
// workgroup: two, or one where no workgroup has a second item.
template <int NA, int NB>
__global__ __launch_bounds__(256, 2) void gemm_mfma_rowtile_kernel(MfmaParams)
{
    constexpr bool WIDE = pipe_wide(NA, NB);
    constexpr int D = NA + NB - 1, STG = rowtile_stages(NA, NB);
    constexpr int WVN = WIDE ? 4 : 2, WM = WIDE ? 2 : 1, BN = 32 * WVN;
    constexpr int A_BLOCKS = 2 * NA, BLOCKS = rowtile_blocks(NA, NB), STAGE = BLOCKS * 1024;
    constexpr int LOADS = (BLOCKS + 3) / 4;                 // per wavefront and step (the last wavefront's may repeat the last block)
    static_assert(WM * D * 16 + WM * NA * 4 + NB * 4 <= 240, "two wavefronts share a SIMD");
    static_assert(STG >= 3 && LOADS * STG < 64, "vmcnt is a 6-bit counter");
    static_assert(NA * NB >= LOADS, "the loads ride behind the MFMAs");
    extern __shared__ __attribute__((aligned(16))) unsigned char rowtile_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = uniform(tid >> 6);
    const int wm = wave / WVN, wn = wave % WVN;
    const unsigned ring_lds = (unsigned)(uintptr_t)rowtile_smem, lane16 = (unsigned)lane * 16;

    int it_g, it_tm, tn_begin, tn_end, nsteps;
    uint64_t slot;                                          // the planes of the row tile that is multiplied: one of this workgroup's slots
    auto slot_of = [&](int turn) {
        ConstParams &p = launch_args();
        return uniform64((uint64_t)p.a_planes + (uint64_t)(blockIdx.x * p.a_msub + (turn & 1)) * (2 * NA * 1024) * p.a_ksteps);
    };

    // ---- the split: 64 rows of A -> planes [32-row group][step][digit] of 1 KB; a thread owns 8 elements of a row and step ----
    int last = 0, need = 0;                                 // this wavefront's last step that is not all zeros, and the digits of all it has split
    auto split_rows = [&](int item, uint64_t to, int ks, int ks_end) {
        ConstParams &p = launch_args();
        int t = tid;
        asm volatile("" : "+v"(t));                         // (nothing derived from it is kept, and spilled, through the steps)
        const int row = t >> 2, j = t & 3, ksteps = p.a_ksteps, K = p.K;
        const int tile = item / p.col_parts, g = tile / p.tiles_m, m = (tile - g * p.tiles_m) * kRowtileRows + row;
        const bool row_ok = m < p.M;
        const bool vec = (((uintptr_t)p.A | (uintptr_t)(p.lda * 8) | (uintptr_t)(p.sA * 8)) & 15) == 0;
        // (rows past the end are read from the last row, a valid address, and taken for zeros)
        const int64_t *src = p.A + (long)g * p.sA + (long)(row_ok ? m : p.M - 1) * p.lda;
        unsigned char *dst = (unsigned char *)to + (long)(row >> 5) * ksteps * (NA * 1024) + ((row & 31) + 32 * (j >> 1)) * 16 + (j & 1) * 8;
        DigitsSeen bound;
        int live = 0;
        auto put = [&](int64_t (&x)[8], int step) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = row_ok ? x[e] : 0;
            DigitsSeen here;
#pragma unroll
            for (int e = 0; e < 8; e++) here.add(x[e]);
            bound.lo |= here.lo;
            bound.hi |= here.hi;
            live = (here.lo | here.hi) ? step + 1 : live;
            uint2 dg[NA];
            limb_split8<NA>(x, dg);
#pragma unroll
            for (int i = 0; i < NA; i++) *(ZK_GLOBAL_MEM uint64_t *)(dst + (long)step * (NA * 1024) + i * 1024) = (uint64_t)dg[i].y << 32 | dg[i].x;
        };
        constexpr int AT_ONCE = 4;                          // steps whose loads are under way together
        const int whole = vec ? K / 32 : 0;
        for (; ks + AT_ONCE <= whole && ks + AT_ONCE <= ks_end; ks += AT_ONCE) {
            int64_t x[AT_ONCE][8];
#pragma unroll
            for (int u = 0; u < AT_ONCE; u++) load_owned_i64<2, 4>(src + (ks + u) * 32, j, true, 32, true, x[u]);
#pragma unroll
            for (int u = 0; u < AT_ONCE; u++) put(x[u], ks + u);
        }
        for (; ks < ks_end; ks++) {
            int64_t x[8];
            load_owned_i64<2, 4>(src + ks * 32, j, true, K - ks * 32, ks < whole, x);
            put(x, ks);
        }
        live = uniform(wave_max_i32(live));
        last = live > last ? live : last;
        bound.seen = true;
        const int n = uniform(wave_max_i32((bound.lo | bound.hi) == 0 ? 0 : bound.digits()));
        need = n > need ? n : need;
    };
    // every wavefront's part of a row tile has been split: its length (the ring has drained, its first words serve the maximum)
    auto settle = [&]() {
        int *red = reinterpret_cast<int *>(rowtile_smem);
        if (lane == 0) red[wave] = last;
        asm volatile("" ::: "memory");
        wait_vmcnt<0>();                                    // the planes are written before another wavefront loads them
        __syncthreads();
        int n = red[0];
#pragma unroll
        for (int w = 1; w < 4; w++) n = red[w] > n ? red[w] : n;
        __syncthreads();
        nsteps = uniform(n > 1 ? n : 1);                    // (at least one step: the accumulators are set by it)
        last = 0;
    };

    // ---- loading: this wavefront's blocks of a step, numbers wave * LOADS + l of [A: 32-row group][digit], [B: 32-column group][digit] ----
    int l_left, l_tn;
    uint64_t l_src[LOADS];
    auto aim = [&]() {
        ConstParams &p = launch_args();
#pragma unroll
        for (int l = 0; l < LOADS; l++) {
            int b = wave * LOADS + l;
            b = b < BLOCKS ? b : BLOCKS - 1;
            if (b < A_BLOCKS) {
                const int grp = b / NA, dig = b - grp * NA;
                l_src[l] = uniform64(slot + ((uint64_t)grp * p.a_ksteps * NA + dig) * 1024);
            } else {
                const int bb = b - A_BLOCKS, grp = bb / NB, dig = bb - grp * NB;
                int sub = l_tn * WVN + grp;
                sub = sub < p.b_nsub ? sub : p.b_nsub - 1;  // column groups past N: any valid data, never stored
                l_src[l] = uniform64((uint64_t)p.B + (uint64_t)it_g * p.b_gstride + (((long)sub * p.b_ksteps) * NB + dig) * 1024);
            }
        }
    };
    auto issue_one = [&](unsigned stage, auto l_tag) {
        constexpr int L = decltype(l_tag)::value;
        int b = wave * LOADS + L;
        b = b < BLOCKS ? b : BLOCKS - 1;
        lds_dma16_uniform(l_src[L], lane16, ring_lds + stage * STAGE + b * 1024);
    };
    // the loads move on to the next step (past the row tile's last one they repeat it, into stages nobody reads any more)
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
        if (l_tn + 1 < tn_end) { l_tn++; l_left = nsteps; aim(); }
    };

    typedef v16i Acc[WM][D];
    struct Frags { v4i a[WM][NA], b[NB]; };
    auto read_a = [&](unsigned st, int a, int i) {
        return *reinterpret_cast<const v4i *>(rowtile_smem + st * STAGE + ((wm * WM + a) * NA + i) * 1024 + lane16);
    };
    auto read_b = [&](unsigned st, int j) {
        return *reinterpret_cast<const v4i *>(rowtile_smem + st * STAGE + (A_BLOCKS + wn * NB + j) * 1024 + lane16);
    };
    auto read_all = [&](unsigned st, Frags &f) {
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int i = 0; i < NA; i++) f.a[a][i] = read_a(st, a, i);
#pragma unroll
        for (int j = 0; j < NB; j++) f.b[j] = read_b(st, j);
    };
    unsigned st_cur, st_next;                               // stages of steps s and s+1
    // Step s: the MFMAs of step s on the fragments in registers; beside them the fragment reads of step s+1 (landed and
    // fenced by the barrier at the top) and the loads of step s+STG into this step's own stage (whose reads every wavefront
    // has waited for before the barrier).
    auto step = [&](auto first_tag, Acc &acc, Frags &f) {
        constexpr bool FIRST = decltype(first_tag)::value;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);                 // lgkmcnt(0), the others at their maxima
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
                for (int t = 0; t < WM; t++) {
                    const int a = (I * NB + J) & 1 ? WM - 1 - t : t;         // (one operand changes from one MFMA to the next)
                    acc[a][I + J] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[a][I], f.b[J], ZERO ? zero : acc[a][I + J], 0, 0, 0);
                }
                constexpr int L = I * NB + J;
                if constexpr (L < LOADS) {
                    __builtin_amdgcn_sched_barrier(0);
                    issue_one(st_cur, std::integral_constant<int, (L < LOADS ? L : 0)>());
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (I == NA - 1) {                // digit J of B has been issued for the last time this step
                    f.b[J] = read_b(st_next, J);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
#pragma unroll
            for (int a = 0; a < WM; a++) f.a[a][I] = read_a(st_next, a, I);   // and so has digit I of A
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto move_on = [&]() {
        advance();
        st_cur = st_next;
        st_next = st_next + 1 == STG ? 0 : st_next + 1;
    };

    // Row tiles are dealt in rounds of alternating direction: where their lengths grow with their number (a causal prompt),
    // a workgroup's tiles of two rounds add up to the same length.
    auto item_of = [&](int round) {                         // negative: none
        const int items = launch_args().items, base = round * (int)gridDim.x;
        const int i = base + ((round & 1) ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
        return i < items ? i : -1;
    };
    int item = item_of(0);
    split_rows(item, slot_of(0), 0, launch_args().a_ksteps);
    settle();
    for (int round = 0;; round++) {
        {
            ConstParams &p = launch_args();
            const int tile = item / p.col_parts, part = item - tile * p.col_parts;
            it_g = uniform(tile / p.tiles_m);
            it_tm = uniform(tile - it_g * p.tiles_m);
            tn_begin = uniform((int)((long)part * p.tiles_n / p.col_parts));
            tn_end = uniform((int)((long)(part + 1) * p.tiles_n / p.col_parts));
        }
        slot = slot_of(round);
        const int next = item_of(round + 1);

        l_tn = tn_begin;
        l_left = nsteps;
        aim();
#pragma unroll 1
        for (unsigned t = 0; t < STG; t++) {
            static_for<0, LOADS>([&](auto l) { issue_one(t, l); });
            advance();
        }
        wait_vmcnt<LOADS * (STG - 1)>();                    // step 0 has landed (my share)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        st_cur = 0;
        st_next = 1;

        int landed = 0;                                     // steps whose loads are known to have landed beyond what a step needs
        for (int tn = tn_begin; tn < tn_end; tn++) {
            // (the fragments of a tile's first step are read again: no register keeps them through the epilogue)
            Acc acc;
            Frags f;
            read_all(st_cur, f);
            // before a step: the one behind it has landed (my share), the STG - 2 after that may be under way
            if (landed > 0) landed--; else wait_vmcnt<LOADS * (STG - 2)>();
            step(std::true_type(), acc, f);
            for (int s = nsteps; s > 1; s--) {
                move_on();
                if (landed > 0) landed--; else wait_vmcnt<LOADS * (STG - 2)>();
                step(std::false_type(), acc, f);
            }
            move_on();
            // (as in gemm_mfma_pipe_kernel: the stores below count like loads)
            wait_vmcnt<0>();
            landed = STG - 1;

            ConstParams &p = launch_args();
            int m0 = it_tm * kRowtileRows;
            asm volatile("" : "+s"(m0));                    // (a tile's addresses are its own: kept from tile to tile, they took 60 registers that the steps have no room for)
            const int n0 = tn * BN, sh = p.shift, sum0 = (int)p.init;
            const uint64_t rmask = sh ? ((1ull << sh) - 1) : 0;
            // (STREAM: rows of C in whole lines of memory, which nobody reads before they have left the caches; stores that fill
            // parts of lines take twice the time this way)
            auto store_tile = [&](auto edge_tag, auto rem_tag, auto stream_tag) {
                constexpr bool EDGE = decltype(edge_tag)::value, REM = decltype(rem_tag)::value, STREAM = decltype(stream_tag)::value;
                const int n = n0 + wn * 32 + (lane & 31);
#pragma unroll
                for (int a = 0; a < WM; a++) {
                    const int mrow = m0 + (wm * WM + a) * 32 + 4 * (lane >> 5);
                    const long o0 = (long)it_g * p.sC + (long)mrow * p.ldc + n;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int dr = 8 * (r >> 2) + (r & 3);
                        const Words sum = sum_diagonals<D>([&](int d) { return acc[a][d][r]; }, sum0);
                        if (EDGE && !(mrow + dr < p.M && n < p.N)) continue;
                        const long o = o0 + (long)dr * p.ldc;
                        if (STREAM) {
                            __builtin_nontemporal_store(shifted_sum(sum, sh), p.C + o);
                            asm volatile("; streamed");     // (keeps the compiler from making one copy, without the hint, of the two)
                        } else {
                            p.C[o] = shifted_sum(sum, sh);
                        }
                        if (REM) p.R[o] = sum_below(sum, rmask);
                    }
                }
            };
            typedef std::true_type Yes;
            typedef std::false_type No;
            const bool edge = m0 + kRowtileRows > p.M || n0 + BN > p.N;
            if (p.R) { if (edge) store_tile(Yes(), Yes(), No()); else store_tile(No(), Yes(), No()); }
            else if (edge) store_tile(Yes(), No(), No());
            else if ((((uintptr_t)p.C | (uintptr_t)(p.ldc * 8) | (uintptr_t)(p.sC * 8)) & 127) == 0) store_tile(No(), No(), Yes());
            else store_tile(No(), No(), No());
            // a share of the next row tile's split behind every tile: all of it at once would have its loads in front of the
            // other workgroup's, and every workgroup's at the same time
            if (next >= 0) {
                const int ksteps = p.a_ksteps;
                split_rows(next, slot_of(round + 1), (int)((long)(tn - tn_begin) * ksteps / (tn_end - tn_begin)), (int)((long)(tn + 1 - tn_begin) * ksteps / (tn_end - tn_begin)));
            }
        }
        // the loads past the end have landed (waited for in front of the stores), and no wavefront reads the ring any more
        __syncthreads();
        if (next < 0) break;
        settle();
        item = next;
    }

    // what this workgroup saw of A
    ConstParams &p = launch_args();
    int *red = reinterpret_cast<int *>(rowtile_smem);
    if (lane == 0) red[wave] = need;
    __syncthreads();
    if (tid == 0) {
        int n = red[0];
#pragma unroll
        for (int w = 1; w < 4; w++) n = red[w] > n ? red[w] : n;
        leave_digits(p.seen + blockIdx.x, p.verdict, p.fail_class, NA, NB, n, 0);
    }
}

// the kernel for digit counts (na, nb) or null, its dynamic LDS and its tile columns
struct RowtileForm {
    MfmaKernel fn;
    int bn;
    size_t lds;
};
RowtileForm rowtile_form(int na, int nb);

}  // namespace zk
