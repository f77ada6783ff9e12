// One descriptor for every GEMM-shaped entry point (the two bmm launchers and the four MLA einsums):
//
//   C[g][m][n] = (init + sum_k (A[g][m][k] / a_rs) * (B[g][n,k] / b_rs)) >> shift      (128-bit wrapping sum)
//   R[g][m][n] = (that sum) mod 2^shift                                                 (optional)
//
// A is always k-contiguous.  B is either k-contiguous ("n-major", ldbk == 1: weights [N,K], K^T of the
// attention scores) or n-contiguous ("k-major", ldbn == 1: V of P.V, wkv_b_1 [D,C]).
#pragma once
#include "common.h"

namespace zk {

struct GemmDesc {
    const int64_t *A;
    long lda, sA;             // A[g][m][k] = A[g * sA + m * lda + k]
    const void *B;
    int b32;                  // 1: B holds int32, 0: int64
    long ldbn, ldbk, sB;      // B[g][n,k] = B[g * sB + n * ldbn + k * ldbk]; exactly one of ldbn, ldbk is 1
    int64_t *C, *R;           // R may be null
    long ldc, sC;             // C[g][m][n] = C[g * sC + m * ldc + n]
    int G, M, N, K;
    int shift;                // 0..63
    int64_t init;             // added to the sum before the shift
    int64_t a_rs, b_rs;       // operand divisors (truncating), 1 = none
    bool few_positions = false;       // the attention of a decoding step or a handful of positions (gemm_small_launch)
};

enum GemmPath { kPathAuto = 0, kPathValu = 1, kPathMfma = 2 };

// A guarded launch stands behind a speculative one on the stream and computes every output again if some workgroup of
// that launch raised the verdict; otherwise its workgroups return at once.  Its first workgroup also reports what the
// speculative launch saw, so that no launch, no event and no wait is needed for that alone.
struct GuardArgs {
    const unsigned *verdict;         // device word; null: an unconditional launch
    unsigned *next;                  // device word cleared for the next speculative launch (the calls take turns with two)
    const unsigned *seen;            // per-workgroup digit counts of the speculative launch: byte 0 A, byte 1 B
    long seen_count;
    unsigned long long *host;        // [parts] words; each receives seq << 32 | verdict << 16 | digits of B << 8 | digits of A in one store (may be null)
    unsigned seq;
    int parts;                       // the first `parts` workgroups share the words of `seen`, see guard_parts
};

// One workgroup for every 1024 words of `seen` (a load or four per thread), at most 32: a product of 131072 rows leaves
// 50000 words, for which one workgroup took 44 us.
constexpr int kGuardParts = 32;
// kReported in place of the count: a launch in between has left the report.
constexpr long kReported = -1;
inline int guard_parts(long seen_count, long grid)
{
    if (seen_count == kReported) return 0;
    const long n = (seen_count + 1023) / 1024, most = grid < kGuardParts ? grid : kGuardParts;
    return (int)(n < 1 ? 1 : (n > most ? most : n));
}

// by whole workgroups of at most 1024 threads, number `part` of g.parts; `verdict`: what the verdict word holds
__device__ __forceinline__ void guard_report(const GuardArgs &g, int part, unsigned verdict)
{
    __shared__ int report_red[16];
    unsigned a = 0, b = 0;
    // (four loads under way per thread: the launch waits for this workgroup)
    const long stride = (long)g.parts * blockDim.x;
    for (long i0 = (long)part * blockDim.x + threadIdx.x; i0 < g.seen_count; i0 += 4 * stride) {
        unsigned w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const long i = i0 + j * stride;
            w[j] = i < g.seen_count ? g.seen[i] : 0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const unsigned wa = w[j] & 0xFFu, wb = (w[j] >> 8) & 0xFFu;
            a = wa > a ? wa : a;
            b = wb > b ? wb : b;
        }
    }
    unsigned ab = a << 16 | b;
    wave_steps([&](auto off) {
        unsigned x, y;
        lane_pair<decltype(off)::value>(ab, x, y);
        const unsigned xa = x >> 16, xb = x & 0xFFFFu, ya = y >> 16, yb = y & 0xFFFFu;
        ab = (xa > ya ? xa : ya) << 16 | (xb > yb ? xb : yb);
    });
    if ((threadIdx.x & 63) == 0) report_red[threadIdx.x >> 6] = (int)ab;
    __syncthreads();
    if (threadIdx.x != 0) return;
    a = b = 0;
    for (unsigned w = 0; w < blockDim.x / 64; w++) {
        const unsigned o = (unsigned)report_red[w];
        a = (o >> 16) > a ? (o >> 16) : a;
        b = (o & 0xFFFFu) > b ? (o & 0xFFFFu) : b;
    }
    if (g.host) __hip_atomic_store(g.host + part, (unsigned long long)g.seq << 32 | verdict << 16 | b << 8 | a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (g.next && part == 0) __atomic_store_n(g.next, 0u, __ATOMIC_RELAXED);
}

// Native 64-bit multiply-add chains on the vector ALU; handles every descriptor.
// (A guarded launcher settles guard->parts by its grid.)
void gemm_valu_launch(const GemmDesc &d, GuardArgs *guard = nullptr);

// Matrix-vector kernel of the same family for one or two rows of A against k-contiguous B: one launch, nothing
// guessed.  Returns false (nothing launched) for any other descriptor.
bool gemm_gemv_launch(const GemmDesc &d);

// Small products in one launch, nothing guessed (gemm_small.hip).  Returns false (nothing launched) for any other descriptor.
bool gemm_small_launch(const GemmDesc &d);
long gemm_small_calls();                   // launches so far

// Limb-decomposed i8 MFMA.  Returns 0 when the product was launched, 1 when the descriptor is outside what it
// supports or memory for its buffers is short (nothing was launched; the caller falls back to the VALU path), -1 on an
// error (recorded).  The outcome describes this call only, whatever the sticky error channel holds from earlier ones.
int gemm_mfma_launch(const GemmDesc &d, int *limbs_a, int *limbs_b);

// A handful of rows (M <= 16) against k-contiguous B on the 16-row MFMA tiles: every wavefront on its own, digit counts
// taken from the data (nothing guessed, nothing read back), K split over wavefronts when the launch would not fill the
// device otherwise (a second, small launch then adds the slices' partial sums).  acc: scratch for those sums (`max_slots`
// slots of 8 KB: one per output tile of 16 x 32 and workgroup of slices; nothing in it needs clearing); null: the library's
// own, grown on demand.  Returns 0 when launched, 1 when the descriptor is outside what it takes (nothing launched), -1
// on an error (recorded).
int gemm_rows16_launch(const GemmDesc &d, unsigned long long *acc = nullptr, size_t max_slots = 0);
size_t gemm_rows16_workspace_bytes();
void gemm_rows16_release_workspace();
void gemm_rows16_reload_switches();

// Calls of the MFMA path that returned before their verdict was known and turned out to need the guarded
// vector-ALU recomputation (known once their range has reached the host).
long gemm_mfma_guard_hits();
// weights prepared once as digit planes (an int64 or int32 matrix, or a device table of `groups` of them): 0 on success
int gemm_mfma_prepare(const void *B, int b32, int groups, int N, int K);
void gemm_mfma_release(const void *B);
bool gemm_mfma_is_prepared(const void *B);
int gemm_mfma_last_pairs();       // digit pairs multiplied per element of K by the last MFMA launch
int gemm_mfma_last_prepared();    // 1 when the last MFMA launch read B from prepared planes
long gemm_mfma_grouped_streamed_calls();   // grouped launches so far that ran on the streamed int32 kernel
long gemm_mfma_pipe_calls();               // launches so far that ran on the software-pipelined kernels for planes on both sides
long gemm_mfma_rowtile_calls();            // ... and those of them on the kernel that splits A itself (gemm_mfma_rowtile.h)
long gemm_mfma_short_calls();              // launches so far on the 64x64 tiles for a short K
long gemm_mfma_sum_reports();              // reports so far that left with the sum of a product's slices

// Grouped product: the rows of A and C form one contiguous segment per group and every group has its own
// k-contiguous B[N,K] (the experts of a MoE layer after the tokens have been sorted by expert):
//   C[r][n] = (init + sum_k A[r][k] * B_group(r)[n][k]) >> shift,   R likewise.
// Everything that describes the segments lives on the device, so the host never learns the segment sizes.
struct GroupedDesc {
    const int64_t *A;
    long lda;
    const void *const *B;     // device array of `groups` device pointers
    int b32;
    int64_t *C, *R;           // R may be null
    long ldc;
    const int *seg;           // device [groups + 1]: first row of every segment, seg[groups] = rows
    const int *tiles;         // device [2 * (rows / 32 + groups)]: {group, first row} of every 32-row tile
    const int *ntiles;        // device [1]: how many of those tiles exist
    int groups, rows, N, K, shift;
    int64_t init;
};

// The grouped product row by row on the matrix-vector kernel: one launch, every row of A against the B of its segment.
// Streams a B once per row of its segment, so it is for a handful of rows (a decoding step's routed experts).
// Returns false (nothing launched) when the descriptor is outside what it takes.
bool gemm_gemv_grouped_launch(const GroupedDesc &d);

// The grouped product on the 16-row MFMA tiles (see gemm_rows16_launch): one launch, no wait.  0 / 1 / -1 as there.
// `guard`: see GuardArgs (the fallback behind a speculative launch of the 32-row kernels).
int gemm_rows16_grouped(const GroupedDesc &d, GuardArgs *guard = nullptr);

// One launch of the 32-row-tile MFMA kernels over all groups.  Returns 0 when done, 1 when the operands need
// more digits than those kernels are built for (nothing valid was written: the caller takes another route),
// -1 on an error (recorded).
int gemm_mfma_grouped(const GroupedDesc &d, int *limbs_a, int *limbs_b);

// Grouped product through the MFMA launch above or, where that does not apply (path forced to VALU, K = 0,
// operands wider than its kernels take), group by group through gemm_dispatch after one read-back of the segments.
void gemm_grouped_dispatch(const char *name, const GroupedDesc &d);

// Top-level dispatch used by the extern "C" launchers.  False when this call failed (the error is recorded).
bool gemm_dispatch(const char *name, const GemmDesc &d);

}  // namespace zk
