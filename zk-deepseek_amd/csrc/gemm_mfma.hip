// GEMM path (b): limb-decomposed i8 MFMA.
//
// Every int64 operand x is written in balanced base-256 digits, x = sum_j d_j * 256^j with d_j in [-128,127].
// The digits come from one 64-bit add and one xor: with bias_n = 0x80 in bytes 0..n-2,
//     d_j = byte_j(x + bias_n) - 128  (j < n-1),   d_{n-1} = signed byte_{n-1}(x + bias_n),
// which is exact whenever x + bias_n fits n signed bytes; n = 9 covers all of int64 (d_8 in {0,1}).
// The product sum then splits into digit-pair GEMMs that run on v_mfma_i32_32x32x32_i8,
//     sum_k a*b = sum_{i,j} 256^(i+j) * (sum_k da_i * db_j),
// all pairs with the same i+j share one int32 accumulator tile, and the epilogue recombines the
// NA+NB-1 diagonals with carries into the 128-bit sum before the shift.  Nothing is approximated.
//
// Operand tiles are converted on the fly: a thread gathers 8 elements of one row, splits them into digits with
// v_perm_b32 byte transposes and stores each digit plane to LDS already in MFMA fragment order (lane l of a
// fragment = row l%32, k-half l/32, 16 bytes), so the inner loop is ds_read_b128 + MFMA.
// A dot product does not care about the order of k as long as both operands use the same one, so the 8
// elements a thread owns are NOT consecutive: thread j of a row owns runs of RUN consecutive k spaced
// RUN*OCTS apart.  Adjacent lanes then read adjacent 16-byte pieces and every 64-byte line of the tile is
// fetched by exactly one load instruction.
//
// The digit counts are speculated from a cached or sampled range.  The kernels track the digits that everything they
// load needs.  A workgroup that meets an element its digit counts do not hold raises the verdict, a word on the device
// that nobody writes otherwise; a guarded launch follows on the stream, which recomputes everything if the verdict is
// raised and returns at once otherwise.  Its first workgroups also fold what every workgroup saw into 8-byte stores
// to pinned host memory, marked with the call's number: that refreshes the cache at a later call.  (A fold kernel
// between the two and an event behind them cost 10 us per call: 5 for the kernel, 5.5 of idle device at the event.)
// Results never depend on the guess, and a call whose operands were seen before never blocks the host.
#include "gemm_mfma_kernels.h"
#include "gemm_mfma_pipe.h"
#include "gemm_mfma_rowtile.h"
#include "report_ring.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <set>
#include <tuple>

namespace zk {

// the streamed form of the grouped launch for int32 weights (gemm_stream32.h), by digit counts; null: none
MfmaKernel stream32_grouped_kernel(int na, int nb, size_t *lds);
MfmaKernel stream32_grouped_kernel_wide(int na, int nb, size_t *lds);

// Digit-count combinations that are compiled.  A request is rounded up to the cheapest one that covers it.
static const Instance *instances(int *count)
{
    static const std::vector<Instance> table = [] {
        std::vector<Instance> t;
#ifdef ZK_PROBE
        const Instance probe[] = { ZK_PROBE };
        t.assign(probe, probe + sizeof(probe) / sizeof(probe[0]));
#else
        mfma_instances_narrow(t);
        mfma_instances_mid(t);
        mfma_instances_wide(t);
        mfma_instances_short(t);
        mfma_instances_both(t);
        mfma_instances_pruned(t);
        mfma_instances_rows32(t);
        mfma_instances_rows32b(t);
        mfma_instances_rows32c(t);
        mfma_instances_rows32d(t);
        mfma_instances_rows32e(t);
#endif
        return t;
    }();
    *count = (int)table.size();
    return table.data();
}

// need_diag: the result's top bit is below 2^(8 need_diag), so diagonals from need_diag up cannot reach it
// exact_nb / variant: for B from prepared planes the instance must have exactly the planes' digit count and that kernel
static const Instance *pick_instance(int na, int nb, bool b32, bool skinny, int need_diag = 16, int exact_nb = 0, int variant = -1, int exact_kk = 1)
{
    int count;
    const Instance *t = instances(&count);
    const Instance *best = nullptr;
    long best_cost = 0;
    for (int i = 0; i < count; i++) {
        if (t[i].na < na || t[i].nb < nb || t[i].skinny != skinny || t[i].alt || t[i].short_k) continue;
        if (t[i].dmax < 16 && t[i].dmax < need_diag) continue;
        if (exact_nb && (t[i].nb != exact_nb || t[i].kk != exact_kk)) continue;
        if (variant >= 0 && !t[i].fn[variant]) continue;
        if (variant < 0 && b32 && !t[i].fn[kB32Fly]) continue;
        if (variant < 0 && !b32 && !t[i].fn[kB64Fly]) continue;
        long cost = kept_pairs_before(t[i].na, t[i].nb, t[i].dmax, t[i].na, 0);     // MFMAs per 32x32x32 block
        // at equal MFMA count the deeper step wins (only instances made for int32 B have one)
        if (!best || cost < best_cost || (cost == best_cost && t[i].kk > best->kk)) { best = &t[i]; best_cost = cost; }
    }
    return best;
}

// The 128x64 form of an instance with 128x128 tiles, for launches of fewer 128x128 tiles than compute units: twice the
// tiles, so half the slices of K per tile (half the partial sums), and two depths per step.  With (3,3) digits on int64
// weights, 128x128 against 128x64 tiles, both on planes of A: 128 rows x [2048,7168] (16 tiles) 39.0 / 36.9 us, 128 x
// [7168,2048] (56) 41.7 / 38.0, 200 x [7168,7168] (112) 159 / 147, 300 x [7168,7168] (168) 217 / 202.  Not where the
// halves fill a round and three quarters (their last round is then not split): 500 x [7168,2048] (224) 69.5 / 80; nor for
// launches larger than the device, which are bound by operand traffic: 512 x [18432,7168] 607 / 666.  Halves that take a
// second round need a long K, too (300 x [7168,1024] 39 / 45, 700 x [4096,2048] 68 / 77), and tall products of a long K and
// one or two tile columns stay as they are, where the slices of the halves no longer fall into step with the XCDs (1100 x [256,7168] 45 /
// 58, 2400 x [256,16384] 150 / 196).
static const Instance *smaller_tiles(const Instance *inst, const GemmDesc &d, int cus)
{
    const long tiles = (long)((d.M + inst->bm - 1) / inst->bm) * ((d.N + inst->bn - 1) / inst->bn) * d.G;
    if (inst->bm != 128 || inst->bn != 128 || tiles >= cus) return inst;
    const long halves = (long)((d.M + inst->bm - 1) / inst->bm) * ((d.N + 63) / 64) * d.G;        // (fewer than twice as many where the last column is)
    if (2 * tiles - cus > cus / 2 || (halves > cus && d.K < 4096)) return inst;
    if (d.N <= 256 && d.M > 1024 && d.K >= 4096) return inst;
    int count;
    const Instance *t = instances(&count);
    for (int i = 0; i < count; i++)
        if (t[i].alt && t[i].na == inst->na && t[i].nb == inst->nb) return t + i;
    return inst;
}

typedef std::tuple<const void *, long, long, int> OperandKey;     // (pointer, rows, K, element size)

// Whose digit counts are on their way from the device to the host behind the stream (calls that do not wait for their verdict).
struct PendingRange {
    OperandKey key_a, key_b;
    int nb_fixed = 0;                        // B came from prepared planes with this many digits (nothing of it was tracked)
};

constexpr unsigned kPendingSlots = 256;      // (a host this many calls ahead of the device skips the report, not the check)

struct RangeCache {
    std::mutex mu;
    std::map<OperandKey, int> limbs;         // operand -> digits its values needed when last seen
    std::map<OperandKey, int> partner_a;     // B operand -> digits of the A operand it was last multiplied with
    std::map<std::tuple<long, long, int>, int> by_shape;      // (rows, K, element size) -> digits of the last operand of that shape, wherever it lay
    unsigned long long *dev = nullptr;       // [minA, maxA, minB, maxB] of a sample, [4] a report that is waited for, [5] the two verdict words
    int turn = 0;                            // which verdict word the next speculative launch uses; it is clear
    unsigned char *planes = nullptr;         // digit planes of A, grown on demand, kept for the process lifetime
    size_t planes_bytes = 0;
    unsigned *seen = nullptr;                // per-workgroup digit counts of the GEMM kernel and of the plane pre-pass
    size_t seen_count = 0;
    unsigned long long *partials = nullptr;  // partial sums of split tiles
    size_t partials_bytes = 0;
    unsigned char *b_planes = nullptr;       // digit planes of a small B
    size_t b_planes_bytes = 0;
    int64_t *b_rows = nullptr;               // a small n-contiguous B of many digits rewritten with contiguous rows
    size_t b_rows_count = 0;
    int *row_steps = nullptr;                // per row tile of A: its steps up to the last one that is not all zeros
    size_t row_steps_count = 0;
    int cus = 0;                             // compute units of the device
    ReportRing<PendingRange, kPendingSlots, kGuardParts> reports;       // its words are pinned memory; without any, calls wait
    long guard_hits = 0;                     // calls whose speculation failed after they had returned
    int lookup(const OperandKey &k)
    {
        auto it = limbs.find(k);
        return it == limbs.end() ? 0 : it->second;
    }
    void store(const OperandKey &k, int n)
    {
        if (limbs.size() > 4096) limbs.clear();
        limbs[k] = n;
        if (by_shape.size() > 4096) by_shape.clear();
        by_shape[std::make_tuple(std::get<1>(k), std::get<2>(k), std::get<3>(k))] = n;
    }
    // An operand at an address never seen (or seen with another shape): what the last operand of its shape needed.  The
    // weights of one kind of projection need the same digits in every layer, and so do the activations that meet them.
    int lookup_shape(const OperandKey &k)
    {
        auto it = by_shape.find(std::make_tuple(std::get<1>(k), std::get<2>(k), std::get<3>(k)));
        return it == by_shape.end() ? 0 : it->second;
    }
    void store_pair(const OperandKey &ka, int na, const OperandKey &kb, int nb)
    {
        store(ka, na);
        store(kb, nb);
        if (partner_a.size() > 4096) partner_a.clear();
        partner_a[kb] = na;
    }
};

static RangeCache g_cache;

// Diagnosis switches, read from the environment once when the library is loaded (and again on zk_reload_env):
// ZK_GEMM_SYNC: every call waits for its own digit verdict; ZK_NO_TAIL_SPLIT: no split-K; ZK_VALU_FALLBACK: the guarded launch
// behind a speculative one is always the vector-ALU kernel; ZK_NO_STREAM32: grouped launches on int32 weights keep the general
// 32-row kernel; ZK_NO_PIPE: no pipelined kernel for planes on both sides; ZK_NO_ROWTILE: none that splits A itself; ZK_B_ROWS_MIN_MACS: product
// size from which a B that is small next to it is split into digit planes or rewritten first; ZK_SKINNY_MAX_M: rows up to
// which the 32-row tiles are used; ZK_SCRATCH_LIMIT: bytes a scratch buffer may grow to, as if the device had no more.
struct Switches { bool sync_verdict, no_tail_split, valu_fallback, no_stream32, no_pipe, no_rowtile; double b_rows_min_macs, scratch_limit; int skinny_max_m, planes_min_tiles_n, stream32_min_pairs; };
constexpr long kBRowsMinMacs = 1L << 30;
constexpr double kShapeGuessMaxMacs = 17179869184.0;        // 2^34: about 0.15 ms on the matrix pipe
// Rows up to which a product runs on the 32-row tiles (two of them from 33 rows on): measured against the 128-row tiles,
// 48 rows x [1536,7168] int32 34.1 against 38.1 us, 64 x [2048,7168] int64 37.6-39.4 against 41.2, 128 rows 56.8 against 45.1.
constexpr int kSkinnyMaxRows = 64;
static Switches read_switches()
{
    Switches s;
    s.sync_verdict = getenv("ZK_GEMM_SYNC") != nullptr;
    s.no_tail_split = getenv("ZK_NO_TAIL_SPLIT") != nullptr;
    s.valu_fallback = getenv("ZK_VALU_FALLBACK") != nullptr;
    s.no_stream32 = getenv("ZK_NO_STREAM32") != nullptr;
    s.no_pipe = getenv("ZK_NO_PIPE") != nullptr;
    s.no_rowtile = getenv("ZK_NO_ROWTILE") != nullptr;
    const char *sp = getenv("ZK_STREAM32_MIN_PAIRS");
    s.stream32_min_pairs = sp ? atoi(sp) : 16;
    const char *m = getenv("ZK_B_ROWS_MIN_MACS");
    s.b_rows_min_macs = m ? atof(m) : (double)kBRowsMinMacs;
    const char *sl = getenv("ZK_SCRATCH_LIMIT");
    s.scratch_limit = sl ? atof(sl) : 1e30;
    const char *sk = getenv("ZK_SKINNY_MAX_M");
    s.skinny_max_m = sk ? atoi(sk) : kSkinnyMaxRows;
    const char *pt = getenv("ZK_PLANES_MIN_TILES_N");
    s.planes_min_tiles_n = pt ? atoi(pt) : 4;
    return s;
}
static Switches g_switches = read_switches();
void gemm_mfma_reload_switches() { g_switches = read_switches(); }

// Outcome of a launcher, derived from the call itself (never from the sticky error channel, which may still hold an
// error of an earlier, unrelated call): done, declined (nothing launched that the caller may not overwrite: it takes
// another route) or failed (an error was recorded).
enum Outcome { kDone = 0, kDeclined = 1, kFailed = -1 };

// Grows a device buffer kept until gemm_mfma_release_workspace.  kDeclined (buffer left empty) when memory is short.
template <typename T>
static Outcome grow(T *&buf, size_t &have, size_t need, const char *what)
{
    if (need <= have) return kDone;
    if ((double)need * sizeof(T) > g_switches.scratch_limit) return kDeclined;
    if (buf && hipFree(buf) != hipSuccess) { set_error(kLaunchFailure, "gemm: cannot release the %s", what); return kFailed; }
    buf = nullptr;
    have = 0;
    if (hipMalloc(&buf, need * sizeof(T)) != hipSuccess) { (void)hipGetLastError(); buf = nullptr; return kDeclined; }
    have = need;
    return kDone;
}

static bool read_range(unsigned long long *dev, int64_t (&out)[4])
{
    unsigned long long h[4];
    if (hipMemcpy(h, dev, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return false;
    for (int i = 0; i < 4; i++) out[i] = (int64_t)(h[i] ^ kSignFlip);
    return true;
}

// Takes in the reports that have arrived since the last call.
static void drain_pending()
{
    g_cache.reports.drain([](const PendingRange &s, const volatile unsigned long long *words, int parts) {
        int na = 0, nb = 0, verdict = 0;
        for (int i = 0; i < parts; i++) {
            const unsigned long long w = words[i];
            na = (int)(w & 0xFF) > na ? (int)(w & 0xFF) : na;
            nb = (int)(w >> 8 & 0xFF) > nb ? (int)(w >> 8 & 0xFF) : nb;
            verdict |= (int)(w >> 16 & 0xFF);
        }
        if (nb) g_cache.store_pair(s.key_a, na ? na : 1, s.key_b, nb);
        else if (s.nb_fixed) g_cache.store_pair(s.key_a, na ? na : 1, s.key_b, s.nb_fixed);      // (a grouped launch on prepared planes)
        else g_cache.store(s.key_a, na ? na : 1);        // B came from prepared planes: nothing of it was tracked
        if (verdict) g_cache.guard_hits++;
    });
}

// The guard of the call being launched: its verdict word, the word cleared for the next call, and, while a slot is free,
// where the report goes.  guard_taken() once the guarded launch is on the stream.
static GuardArgs make_guard(long seen_count)
{
    unsigned *words = reinterpret_cast<unsigned *>(g_cache.dev + 5);
    GuardArgs g = {};
    g.verdict = words + g_cache.turn;
    g.next = words + (g_cache.turn ^ 1);
    g.seen = g_cache.seen;
    g.seen_count = seen_count;
    g.host = g_cache.reports.open(&g.seq);
    return g;
}

static void guard_taken(const GuardArgs &g, const OperandKey &key_a, const OperandKey &key_b, int nb_fixed)
{
    g_cache.turn ^= 1;
    if (!g.host) return;
    PendingRange s;
    s.key_a = key_a;
    s.key_b = key_b;
    s.nb_fixed = nb_fixed;
    g_cache.reports.push(s, g.seq, g.parts);
}

// Waits for the digits the launch just issued has seen, and clears its verdict word (its caller launches again).
static bool wait_digits(long first, long seen_count, int *need_a, int *need_b)
{
    GuardArgs g = {};
    unsigned *word = reinterpret_cast<unsigned *>(g_cache.dev + 5) + g_cache.turn;
    g.verdict = word; g.next = word; g.seen = g_cache.seen + first; g.seen_count = seen_count;
    g.host = g_cache.dev + 4;
    g.parts = 1;
    digits_report_kernel<<<1, 256, 0, 0>>>(g);
    unsigned long long w;
    if (hipMemcpy(&w, g_cache.dev + 4, sizeof(w), hipMemcpyDeviceToHost) != hipSuccess) return false;
    *need_a = (int)(w & 0xFF);
    *need_b = (int)(w >> 8 & 0xFF);
    if (!*need_a) *need_a = 1;
    if (!*need_b) *need_b = 1;
    return true;
}

static int g_last_pairs = 0, g_last_prepared = 0;
static long g_streamed_calls = 0, g_pipe_calls = 0, g_rowtile_calls = 0, g_short_calls = 0, g_sum_reports = 0;
int gemm_mfma_last_pairs() { return g_last_pairs; }
int gemm_mfma_last_prepared() { return g_last_prepared; }
long gemm_mfma_grouped_streamed_calls() { return g_streamed_calls; }
long gemm_mfma_pipe_calls() { return g_pipe_calls; }
long gemm_mfma_rowtile_calls() { return g_rowtile_calls; }
long gemm_mfma_short_calls() { return g_short_calls; }
long gemm_mfma_sum_reports() { return g_sum_reports; }

long gemm_mfma_guard_hits()
{
    std::lock_guard<std::mutex> lock(g_cache.mu);
    drain_pending();
    return g_cache.guard_hits;
}

static bool init_cache()
{
    if (g_cache.dev) return true;
    const size_t dev_bytes = 8 * sizeof(unsigned long long);
    if (hipMalloc(&g_cache.dev, dev_bytes) != hipSuccess || hipMemset(g_cache.dev, 0, dev_bytes) != hipSuccess) {
        g_cache.dev = nullptr;
        set_error(kLaunchFailure, "gemm: cannot allocate the range buffer");
        return false;
    }
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    g_cache.cus = n;
    // without the pinned words every call simply waits for its own verdict
    void *pinned = nullptr;
    if (hipHostMalloc(&pinned, kPendingSlots * kGuardParts * sizeof(unsigned long long), hipHostMallocDefault) == hipSuccess) {
        volatile unsigned long long *words = reinterpret_cast<volatile unsigned long long *>(pinned);
        for (unsigned i = 0; i < kPendingSlots * kGuardParts; i++) words[i] = 0;
        g_cache.reports.words = words;
    } else {
        (void)hipGetLastError();
    }
    return true;
}

// ---- weights prepared once ------------------------------------------------------------------------------
// Model weights do not change between calls.  `gemm_mfma_prepare` splits an int64 weight matrix (or every matrix of a
// device table of pointers, the experts of a layer) into digit planes in MFMA fragment order once, with the digit
// count its exact range needs; later launches whose B is that pointer copy the planes into LDS instead of splitting B
// in every tile (and read NB bytes per weight instead of 8).  The original matrix stays the caller's and is what the
// guarded vector-ALU fallback reads; the caller must not change it while it is prepared.
struct PreparedB {
    unsigned char *planes = nullptr;     // per matrix: [nsub][ksteps][nb] blocks of 1 KB
    const void **table = nullptr;        // device array: the planes of every group (tables only)
    int groups = 0, N = 0, K = 0, nb = 0, nsub = 0, ksteps = 0, b32 = 0;
    int kk = 1;                          // MFMA depths per step of the kernels the planes were ordered for
};
static std::map<const void *, PreparedB> g_prepared;

template <typename T>
static __global__ __launch_bounds__(256) void range_exact_kernel(const T *__restrict__ x, long n, unsigned long long *out)
{
    MinMax r = { INT64_MAX, INT64_MIN };
    // 16-byte pieces, four in flight per thread, then whatever is left (n and the pointer need not be aligned)
    constexpr int PER = 16 / sizeof(T);
    const long head = ((uintptr_t)x & 15) ? n : 0;                       // unaligned: everything goes element by element
    const long pieces = (n - head) / PER;
    const v4i *xv = reinterpret_cast<const v4i *>(x);
    for (long q0 = (long)blockIdx.x * 1024 + threadIdx.x; q0 < pieces; q0 += (long)gridDim.x * 1024) {
        v4i t[4];
#pragma unroll
        for (int u = 0; u < 4; u++) t[u] = q0 + 256 * u < pieces ? __builtin_nontemporal_load(xv + q0 + 256 * u) : xv[0];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (sizeof(T) == 8) {
                mm_update(r, (int64_t)(((uint64_t)(uint32_t)t[u][1] << 32) | (uint32_t)t[u][0]));
                mm_update(r, (int64_t)(((uint64_t)(uint32_t)t[u][3] << 32) | (uint32_t)t[u][2]));
            } else {
#pragma unroll
                for (int z = 0; z < 4; z++) mm_update(r, (int64_t)t[u][z]);
            }
        }
    }
    for (long i = (head ? 0 : pieces * PER) + (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) mm_update(r, (int64_t)x[i]);
    r = mm_wave(r);
    if ((threadIdx.x & 63) == 0 && r.lo <= r.hi) {
        atomicMin(out, (unsigned long long)r.lo ^ kSignFlip);
        atomicMax(out + 1, (unsigned long long)r.hi ^ kSignFlip);
    }
}

static void release_prepared(PreparedB &pb)
{
    if (pb.planes) (void)hipFree(pb.planes);
    if (pb.table) (void)hipFree((void *)pb.table);
    pb = PreparedB();
}

bool gemm_mfma_is_prepared(const void *B)
{
    std::lock_guard<std::mutex> lock(g_cache.mu);
    return g_prepared.count(B) != 0;
}

void gemm_mfma_release(const void *B)
{
    std::lock_guard<std::mutex> lock(g_cache.mu);
    auto it = g_prepared.find(B);
    if (it == g_prepared.end()) return;
    (void)hipDeviceSynchronize();              // launches that read the planes may still be under way
    release_prepared(it->second);
    g_prepared.erase(it);
}

int gemm_mfma_prepare(const void *B, int b32, int groups, int N, int K)
{
    const char *name = "zk_gemm_prepare_weights";
    if (!B || groups < 0 || groups > 65535 || N < 1 || K < 1) { set_error(kBadArgument, "%s: bad argument", name); return 1; }
    std::lock_guard<std::mutex> lock(g_cache.mu);
    if (!init_cache()) return 1;
    {
        auto it = g_prepared.find(B);
        if (it != g_prepared.end()) { (void)hipDeviceSynchronize(); release_prepared(it->second); g_prepared.erase(it); }
    }
    const int count = groups > 0 ? groups : 1;
    std::vector<const void *> mats((size_t)count, B);
    if (groups > 0 && hipMemcpy(mats.data(), B, (size_t)count * sizeof(void *), hipMemcpyDeviceToHost) != hipSuccess) {
        set_error(kLaunchFailure, "%s: cannot read the pointer table", name);
        return 1;
    }
    for (int i = 0; i < count; i++)
        if (!mats[i]) { set_error(kBadArgument, "%s: null matrix in the table", name); return 1; }
    // the exact range of all the matrices fixes one digit count for them
    const long elems = (long)N * K;
    range_reset_kernel<<<1, 64, 0, 0>>>(g_cache.dev);
    const unsigned rgrid = (unsigned)(elems / 256 + 1 < 2048 ? elems / 256 + 1 : 2048);
    for (int i = 0; i < count; i++) {
        if (b32) range_exact_kernel<int32_t><<<rgrid, 256, 0, 0>>>(reinterpret_cast<const int32_t *>(mats[i]), elems, g_cache.dev);
        else range_exact_kernel<int64_t><<<rgrid, 256, 0, 0>>>(reinterpret_cast<const int64_t *>(mats[i]), elems, g_cache.dev);
    }
    int64_t r[4];
    if (!read_range(g_cache.dev, r)) { set_error(kLaunchFailure, "%s: range readback failed", name); return 1; }
    const int need = limbs_needed(r[0], r[1]);
    PreparedB pb;
    pb.groups = groups; pb.N = N; pb.K = K; pb.b32 = b32 ? 1 : 0;
    pb.nb = need <= 3 ? 3 : (need <= 5 ? need : 9);              // digit counts the kernels are built for
    // the experts' three- and four-digit planes go to kernels with two depths per step (the k-order inside a step follows it)
    pb.kk = (groups > 0 && pb.nb <= 4) ? 2 : 1;
    pb.nsub = (N + 31) / 32;
    pb.ksteps = ((K + 32 * pb.kk - 1) / (32 * pb.kk)) * pb.kk;
    const size_t per = (size_t)pb.nsub * pb.ksteps * pb.nb * 1024;
    if (hipMalloc(&pb.planes, per * count) != hipSuccess) {
        (void)hipGetLastError();
        set_error(kLaunchFailure, "%s: cannot allocate %zu bytes of digit planes", name, per * count);
        return 1;
    }
    if (groups > 0) {
        std::vector<const void *> bases((size_t)count);
        for (int i = 0; i < count; i++) bases[i] = pb.planes + per * i;
        if (hipMalloc((void **)&pb.table, (size_t)count * sizeof(void *)) != hipSuccess ||
            hipMemcpy((void *)pb.table, bases.data(), (size_t)count * sizeof(void *), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipGetLastError();
            release_prepared(pb);
            set_error(kLaunchFailure, "%s: cannot allocate the table of planes", name);
            return 1;
        }
    }
    // the pre-pass that splits A in fragment order does the same for the rows of a weight matrix (64 rows per workgroup)
    const int rows_per_wg = 256 / (4 * pb.kk);
    const dim3 grid((unsigned)(pb.ksteps / pb.kk), (unsigned)((pb.nsub * 32 + rows_per_wg - 1) / rows_per_wg), 1);
    MfmaParams q = {};
    q.lda = K; q.sA = 0; q.M = N; q.K = K;
    for (int i = 0; i < count; i++) {
        q.A = reinterpret_cast<const int64_t *>(mats[i]);
        unsigned char *dst = pb.planes + per * i;
#define ZK_PLANES(NB_) do { if (b32) a_planes_kernel<NB_, 2, 1, true><<<grid, dim3(256), 0, 0>>>(q, dst, pb.nsub, pb.ksteps, nullptr); \
                           else a_planes_kernel<NB_, 2, 1, false><<<grid, dim3(256), 0, 0>>>(q, dst, pb.nsub, pb.ksteps, nullptr); } while (0)
        switch (pb.nb) {
#define ZK_PLANES2(NB_) do { if (b32) a_planes_kernel<NB_, 2, 2, true><<<grid, dim3(256), 0, 0>>>(q, dst, pb.nsub, pb.ksteps, nullptr); \
                            else a_planes_kernel<NB_, 2, 2, false><<<grid, dim3(256), 0, 0>>>(q, dst, pb.nsub, pb.ksteps, nullptr); } while (0)
        case 3: if (pb.kk == 2) ZK_PLANES2(3); else ZK_PLANES(3); break;
        case 4: if (pb.kk == 2) ZK_PLANES2(4); else ZK_PLANES(4); break;
#undef ZK_PLANES2
        case 5: ZK_PLANES(5); break;
        default: ZK_PLANES(9); break;
        }
#undef ZK_PLANES
    }
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
        release_prepared(pb);
        set_error(kLaunchFailure, "%s: the plane pre-pass failed", name);
        return 1;
    }
    g_prepared[B] = pb;
    return 0;
}

// Device memory the GEMM path holds right now: its scratch buffers, and the digit planes of prepared weights.
size_t gemm_mfma_workspace_bytes(size_t *prepared_bytes)
{
    std::lock_guard<std::mutex> lock(g_cache.mu);
    size_t scratch = g_cache.dev ? 8 * sizeof(unsigned long long) : 0;
    scratch += g_cache.planes_bytes + g_cache.seen_count * sizeof(unsigned) + g_cache.partials_bytes * sizeof(unsigned long long) +
               g_cache.b_planes_bytes + g_cache.b_rows_count * sizeof(int64_t) + g_cache.row_steps_count * sizeof(int);
    size_t prepared = 0;
    for (const auto &kv : g_prepared) {
        const PreparedB &pb = kv.second;
        const size_t count = pb.groups > 0 ? (size_t)pb.groups : 1;
        prepared += (size_t)pb.nsub * pb.ksteps * pb.nb * 1024 * count + (pb.table ? count * sizeof(void *) : 0);
    }
    if (prepared_bytes) *prepared_bytes = prepared;
    return scratch;
}

// Gives the scratch buffers back (they grow again on demand).  Waits for the device first: launches that use them may
// still be under way.  Prepared weights stay (zk_gemm_release_weights returns those).
void gemm_mfma_release_workspace()
{
    std::lock_guard<std::mutex> lock(g_cache.mu);
    (void)hipDeviceSynchronize();
    drain_pending();
    if (g_cache.planes) (void)hipFree(g_cache.planes);
    if (g_cache.seen) (void)hipFree(g_cache.seen);
    if (g_cache.partials) (void)hipFree(g_cache.partials);
    if (g_cache.b_planes) (void)hipFree(g_cache.b_planes);
    if (g_cache.b_rows) (void)hipFree(g_cache.b_rows);
    if (g_cache.row_steps) (void)hipFree(g_cache.row_steps);
    g_cache.planes = nullptr; g_cache.planes_bytes = 0;
    g_cache.seen = nullptr; g_cache.seen_count = 0;
    g_cache.partials = nullptr; g_cache.partials_bytes = 0;
    g_cache.b_planes = nullptr; g_cache.b_planes_bytes = 0;
    g_cache.b_rows = nullptr; g_cache.b_rows_count = 0;
    g_cache.row_steps = nullptr; g_cache.row_steps_count = 0;
}

// A B that is small next to the product (a KV cache against the queries of a whole prompt, one head's weights) is split
// into digit planes like A, and the product runs on the pipelined kernel for planes on both sides (gemm_mfma_pipe.h),
// or on the one that splits A itself (gemm_mfma_rowtile.h, see rowtile_parts).
// One more launch in front and the general kernel's time, against its own split of B in every tile.  Whole calls, (3,4)
// digits, general against this: k-contiguous int64 B, 131072 rows x [1024,512] 1124 / 864 us, x [1024,64] 379 / 268, 31104 x
// [243,512] 95.8 / 84.0, 8192 x [512,512] (3,3) 35.2 / 36.7, (4,4) 49.8 / 49.0; the heads' int32 weights (128 heads, 1024
// rows each) 248 / 310.  n-contiguous B, which the general kernel reads element by element: 512 values of 1024 tokens 1250 /
// 630 (860 without the causal zeros), of 243 tokens 109 / 68, of 100 tokens 37.7 / 32.5, the heads' int32 weights at 400
// rows 134 / 132, at 500 169 / 149.
// Few columns do not pay for the pass over A: 131072 rows x [64,512], (3,3) 167 / 230 us, (4,4) 148 / 236, x [192,512] 243 /
// 305 and 304 / 345, x [256,512] (3,3) 259 / 308, from 384 columns equal; 64000 x [64,1024] n-contiguous (3,4) 116 / 227,
// [256,1024] (3,3) 243 / 275; int32 n-contiguous, 500 rows of 128 heads [512,64] 72 / 144, [512,128] 130 / 158, [256,256]
// 126 / 134 (675 rows of 128 heads [70,300] 121 / 107).  Nor do launches of hardly more than one tile per compute unit, where the ring has no next tile to run on to:
// 8192 x [256,512] n-contiguous (4,4) 28 / 37, 16384 x [192,512] (3,3) 31 / 46 (with the 128x128 tiles of six diagonals a
// long K makes up for it: 8192 x [512,1024] (3,4) 76 / 66).
constexpr long kPipeBMaxElements = 8L << 20;         // 40 MB of planes at most
constexpr int kPipeMinRows = 16384, kPipeMinRowsKmajor = 385;
constexpr int kPipeMinCols = 193, kPipeMinColsWide = 257;        // (a fourth column of 64; wide: (3,3) digits, a third of 128, and int32 weights)
static bool pipe_b_planes(const GemmDesc &d, bool kmajor, long b_batches)
{
    if (g_switches.no_pipe || b_batches * d.N * d.K > kPipeBMaxElements) return false;
    return d.M >= (kmajor ? kPipeMinRowsKmajor : kPipeMinRows) && (double)d.G * d.M * d.N * d.K >= g_switches.b_rows_min_macs;
}

// ... by digit counts, with `tiles` tiles of its kernel.  (With the product size lowered by its switch, whatever fills the device.)
static bool pipe_b_pays(const GemmDesc &d, int na, int nb, long tiles, int cus)
{
    if (g_switches.b_rows_min_macs < kBRowsMinMacs) return tiles >= cus;
    if (d.N < (na + nb <= 6 || d.b32 ? kPipeMinColsWide : kPipeMinCols)) return false;
    return 2 * tiles >= 3L * cus || (tiles >= cus && na + nb == 7 && d.K >= 512);
}

// How the row-tile kernel (gemm_mfma_rowtile.h) would run a product that b_planes_kernel serves: the parts that a row tile's
// columns are dealt in, or 0 where the pass over A in front of the pipelined kernel is expected to be as fast.  In us: a tile
// of the row-tile kernel's two workgroups, or of the pipelined kernel's one twice as tall, has its steps and 3 for the sums and
// stores; 64 rows of A are split at 11.7 KB per us when every workgroup does it; the pass over A moves 5.5 TB/s behind a
// launch of 5.  What decides is how well the items fill whole rounds: pass and pipelined kernel / row tiles in one part, 17024 rows x
// [1746,512] 209 / 265 us, 622 rows of 64 heads [457,128] 82 / 100, 61184 x [512,209] 151 / 115.
static int rowtile_parts(const GemmDesc &d, int na, int nb, int bn, int cus)
{
    const long row_tiles = (long)((d.M + kRowtileRows - 1) / kRowtileRows) * d.G, tiles_n = (d.N + bn - 1) / bn, slots = 2L * cus;
    const double steps = (d.K + 31) / 32, tile = steps * na * nb * (bn == 128 ? 0.104 : 0.052) + 3, split = d.K * (8.0 * kRowtileRows / 11700);
    const long old_tiles = (long)((d.M + 127) / 128) * d.G * tiles_n;
    double best = (double)((old_tiles + cus - 1) / cus) * tile + (double)d.G * d.M * d.K * (8 + na) / 5.5e6 + 5;
    int parts = 0;
    // It has to be expected to win by more than the estimate is off.  Tiles of 64x64 read twice the planes per product of the pipelined
    // kernel's 128x64 ((6,3) digits 20096 x [1760,542] 352 / 374, (5,4) 46464 x [512,214] 158 / 166, 79104 x [512,1081] 984 / 906, (4,4) 584
    // rows of 128 heads [350,80] 126 / 147), and nine products a step leave less to hide the splits behind ((3,3) 94976 x [1903,512] 958 /
    // 1022, 54144 x [588,98] 97 / 111, 29568 x [512,244] 72 / 61).
    if (bn != 128 && d.K < 128) return 0;
    // Two workgroups per compute unit store parts of lines, and remainders, at a lower rate than one, once the outputs are more than the
    // 256 MB of the memory-side cache hold: 3.5 against 4.5 TB/s.  With remainder, pass over A and pipelined kernel / row tiles: 127714
    // x [743,76] 371 / 519 us, 129713 x [692,334] 592 / 691, 121446 x [492,96] 260 / 317, (6,3) 122597 x [398,246] 363 / 393, but 25409
    // x [356,223] (145 MB) 76 / 60; without, 126912 x [635,61] 191 / 228, 47202 x [1225,55] 139 / 166, but 60551 x [441,55] 80 / 63.
    const bool lines = (((uintptr_t)d.C | (uintptr_t)d.R | (uintptr_t)(d.ldc * 8) | (uintptr_t)(d.sC * 8)) & 127) == 0;
    const double beyond = std::max(0.0, (double)d.G * d.M * d.N * (d.R ? 16 : 8) - 256e6);
    if (beyond > 0 && d.K < 96 && (d.R || !lines)) return 0;
    if (d.R && !lines && na == 6) return 0;
    const double stores = d.R && !lines ? beyond / 3.5e6 : 0;
    best += stores * (3.5 / 4.5);
    best *= bn != 128 ? 0.93 : (na * nb <= 9 ? 0.88 : 0.97);
    for (long n = 1; n <= tiles_n && n <= 8; n++) {
        const double t = (double)((row_tiles * n + slots - 1) / slots) * (split + (double)((tiles_n + n - 1) / n) * tile) + stores;
        if (t < best) { best = t; parts = (int)n; }
    }
    return parts;
}

// The 64x64 form of an instance with 128x64 tiles, for a K of a few steps.  A tile is then bound by its first loads and its epilogue, and
// a workgroup of eight wavefronts has its compute unit to itself, so nothing runs beside them; of these workgroups of four two run to a unit, one
// loading while the other combines and stores, and fewer rows are padding.  What it costs is B split twice as often.
// 128x64 tiles / this, us, all with A split in the kernel but the last.  One B per head, int32 n-contiguous, 128 heads [128,512]: 129 rows
// (3,4) 54.6 / 45.5, 192 rows (4,4) 64.0 / 52.6, 243 rows 65.4 / 61.5, 300 rows 84.6 / 74.1, 384 rows 113 / 108; 64 heads [64,300], 65 rows 16.0 /
// 14.2; not where they fill two rounds at most (64 heads [128,512], 65 rows 20.7 / 21.2, 16 heads, 192 rows 13.4 / 14.4).  k-contiguous, 128
// heads, K = 512, 128 columns: 192 rows 44.6 / 38.7, 243 rows 49.5 / 46.7, 500 rows 124 / 110; not in one round (64 heads 25.1 / 26.1), nor up
// to 128 rows (70 rows 25.9 / 26.8).  A shared B of many columns: not at K = 512 (20480 rows x [160,512] 43.2 / 44.8), but tall at K = 64, where the
// pass that splits A in front goes as well: 25600 rows x [200,64] 31.1 / 25.9, 31104 x [243,64] 35.4 / 27.8, and at any K below (64000 x [277,8]
// 64.6 / 56.1, 19968 x [960,48] 63.3 / 57.7).  With (3,3) digits, 128x128 tiles, it is slower throughout (243 rows of 128 heads [128,512] 52.7 / 59.4).
// Splitting B twice as often shows where nothing is won by it, n-contiguous and K > 256, (4,4), [512,512]: rows that fill their tiles in
// rounds that fill the device, 32 heads 243 rows 48.3 / 50.7, 384 rows 70.1 / 73.7, 64 heads 243 rows 91.3 / 95.3; half a last round is enough to
// win (48 heads, 384 rows x [256,512] 67.0 / 61.9), and so are many rounds (64 heads, 500 rows 201 / 190; 256 columns from four: 128 heads, 500
// rows x [128,512] 128 / 119).  And two workgroups store at a lower rate than one where A and the outputs are more than the memory-side cache holds next to
// each other (256 MB): K <= 64 and k-contiguous or tall, 16384 x [1924,32] (242 MB) 84.1 / 80.5, 64000 x [621,24] (315) 107 / 123, 19968 x
// [2328,16] (357) 117 / 137, with remainder 65536 x [243,64] (275) 72.6 / 82.3, 16 heads, 8000 rows x [300,64] (355) 131 / 144.
static const Instance *short_k_tiles(const Instance *inst, const GemmDesc &d, int cus)
{
    const long tiles_n = (d.N + 63) / 64, tiles = (long)((d.M + 127) / 128) * tiles_n * d.G;
    if (inst->bm != 128 || inst->bn != 64 || inst->dmax != 16) return inst;
    const bool in_cache = (double)d.G * d.M * (8.0 * d.K + (d.R ? 16.0 : 8.0) * d.N) <= 252.0 * (1 << 20);
    const long last = tiles % cus;
    const bool gaps = (d.M - 1) % 128 < 64 || (last != 0 && 2 * last <= cus) || tiles > (d.N <= 256 ? 3L : 6L) * cus;
    const bool heads = d.G > 1 && d.sB != 0 && (d.K <= 64 ? tiles >= cus && (in_cache || d.ldbk != 1) : d.K <= 128 ? tiles > 2L * cus
                       : d.K <= 512 && d.M > 128 && 2 * tiles >= 3L * cus && (d.K <= 256 || d.ldbk == 1 || gaps));
    const bool tall = d.K <= 64 && d.M >= kPipeMinRows && tiles_n >= 4 && in_cache;
    if (!heads && !tall) return inst;
    int count;
    const Instance *t = instances(&count);
    for (int i = 0; i < count; i++)
        if (t[i].short_k && t[i].na == inst->na && t[i].nb == inst->nb) return t + i;
    return inst;
}

// B[g][k][n] (n contiguous) -> out[g][n][k]: 32x32 tiles through LDS, both sides coalesced
__global__ __launch_bounds__(256) void b_rows_kernel(const int64_t *__restrict__ B, long ldbk, long sB, int64_t *__restrict__ out, int N, int K)
{
    __shared__ int64_t tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int n0 = blockIdx.x * 32, k0 = blockIdx.y * 32;
    const int64_t *src = B + (long)blockIdx.z * sB;
    int64_t *dst = out + (long)blockIdx.z * N * K;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int k = k0 + ty + 8 * i, n = n0 + tx;
        tile[ty + 8 * i][tx] = (k < K && n < N) ? src[(long)k * ldbk + n] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int n = n0 + ty + 8 * i, k = k0 + tx;
        if (n < N && k < K) dst[(long)n * K + k] = tile[tx][ty + 8 * i];
    }
}

// An n-contiguous int64 B that is small next to the product and needs more digits than the pipelined kernel has instances
// for is rewritten with contiguous rows: the kernels of many digits then read it with 16-byte loads and take A from digit
// planes.  As it lies / rewritten, (5,9) digits, the values of 128 heads: 16 tokens x [4096,512] 169 / 161 us, 32 x [4096,512]
// 332 / 309, 63 x [8192,512] 1307 / 1220, 200 x [779,512] 539 / 475, 100 x [2048,1000] 1062 / 927.  (Of up to five digits the
// kernels with two depths per step read it as it lies in the same time: 32 x [4096,512], (3,4), 161 rewritten, 159.)
constexpr double kBCopyMinMacs = 4294967296.0;       // 2^32
static bool b_copy_pays(const GemmDesc &d, int nb, long b_batches)
{
    if (d.b32 || nb <= 5 || d.M <= 32 || b_batches * d.N * d.K > kPipeBMaxElements) return false;
    return (double)d.G * d.M * d.N * d.K >= (g_switches.b_rows_min_macs < kBRowsMinMacs ? g_switches.b_rows_min_macs : kBCopyMinMacs);
}

// The launch behind a speculative one: it does nothing unless the verdict word says that the digit counts did not cover
// the operands, and then computes every output again.  B without a divisor: the widest MFMA instance (nine
// digits hold every int64, five every int32; config 4 with stale three-digit guesses: 4 ms where the vector-ALU tiles
// take 35), one workgroup per compute unit walking the tiles.  Everything else, and a K beyond what its int32
// accumulators take in one piece: the vector-ALU tiles.
static Outcome launch_guarded_fallback(const GemmDesc &d, const MfmaParams &spec, int b_shift, GuardArgs *guard)
{
    const bool kmajor = d.ldbn == 1 && d.ldbk != 1;
    const Instance *wide = (b_shift == 0 && !g_switches.valu_fallback) ? pick_instance(9, d.b32 ? 5 : 9, d.b32 != 0, false, 16) : nullptr;
    MfmaKernel fn = wide ? wide->guarded[d.b32 ? 1 : 0][kmajor ? 1 : 0] : nullptr;
    if (fn) {
        const long pairs = wide->na < wide->nb ? wide->na : wide->nb;
        const int ksteps = ((d.K + 32 * wide->kk - 1) / (32 * wide->kk)) * wide->kk;
        if (pairs * ksteps * 32 * 16384 > kMaxDiagonal) fn = nullptr;
    }
    MfmaParams q = spec;
    if (fn) {
        // the caller's operands, not digit planes
        q.A = d.A; q.lda = d.lda; q.sA = d.sA;
        q.B = d.B; q.ldbn = d.ldbn; q.ldbk = d.ldbk; q.sB = d.sB;
        q.a_planes = nullptr; q.a_msub = 0; q.a_ksteps = 0; q.b_nsub = 0; q.b_ksteps = 0; q.b_gstride = 0; q.row_steps = nullptr;
        q.tiles_m = (d.M + wide->bm - 1) / wide->bm;
        q.tiles_n = (d.N + wide->bn - 1) / wide->bn;
        const long total = (long)q.tiles_m * q.tiles_n * d.G;
        if (total > 0x7FFFFFFFL / 8) fn = nullptr;
        else {
            q.main_tiles = (int)total; q.split = 1; q.tail_xcd = 0; q.partials = nullptr; q.part64 = 0; q.n_fastest = 0;
            q.seen = nullptr;                  // (its digit counts hold whatever raised the verdict)
            q.walk_blocks = (int)total;
        }
    }
    if (!fn) {
        gemm_valu_launch(d, guard);
        if (hipGetLastError() != hipSuccess) { set_error(kLaunchFailure, "gemm: guarded vector-ALU launch failed"); return kFailed; }
        return kDone;
    }
    const size_t lds = 2 * (size_t)wide->kk * ((wide->bm / 32) * wide->na + (wide->bn / 32) * wide->nb) * 1024 + 9 * 1024 + 16;
    static std::set<const void *> lds_raised;
    if (lds > 64 * 1024 && !lds_raised.count((const void *)fn)) {
        if (hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
            set_error(kLaunchFailure, "gemm: cannot raise the LDS limit to %zu bytes", lds);
            return kFailed;
        }
        lds_raised.insert((const void *)fn);
    }
    const long grid = q.walk_blocks < g_cache.cus ? q.walk_blocks : g_cache.cus;
    guard->parts = guard_parts(guard->seen_count, grid);
    q.guard = *guard;
    fn<<<dim3((unsigned)grid), dim3((unsigned)wide->threads), lds, 0>>>(q);
    if (hipGetLastError() != hipSuccess) { set_error(kLaunchFailure, "gemm: guarded MFMA launch failed"); return kFailed; }
    return kDone;
}

int gemm_mfma_launch(const GemmDesc &d, int *limbs_a, int *limbs_b)
{
    // Operand divisors: a power of two on B is folded into the digit split of the 32-row kernels (the head projection
    // divides its weights by 256, inference/model.py:1519, and runs on the last token only); anything else: VALU path.
    int b_shift = 0;
    if (d.a_rs != 1) return kDeclined;
    if (d.b_rs != 1) {
        if (d.b_rs <= 0 || (d.b_rs & (d.b_rs - 1)) != 0 || d.M > 32) return kDeclined;
        while (((int64_t)1 << b_shift) < d.b_rs) b_shift++;
    }
    if (d.K <= 0 || d.M <= 0 || d.N <= 0 || d.G <= 0) return kDeclined;
    if (d.G > 65535) return kDeclined;
    const bool kmajor = d.ldbn == 1 && d.ldbk != 1;
    std::lock_guard<std::mutex> lock(g_cache.mu);
    if (!init_cache()) return kFailed;
    drain_pending();

    MfmaParams p = {};
    p.A = d.A; p.B = d.B; p.C = d.C; p.R = d.R;
    p.lda = d.lda; p.sA = d.sA; p.ldbn = d.ldbn; p.ldbk = d.ldbk; p.sB = d.sB; p.ldc = d.ldc; p.sC = d.sC;
    // B prepared beforehand: its planes stand in for it, its digit count is exact
    const PreparedB *prep = nullptr;
    {
        auto it = g_prepared.find(d.B);
        if (it != g_prepared.end() && it->second.groups == 0 && it->second.b32 == (d.b32 ? 1 : 0) && !kmajor && b_shift == 0 && d.sB == 0 &&
            d.ldbk == 1 && d.ldbn == d.K && it->second.N == d.N && it->second.K == d.K)
            prep = &it->second;
    }
    const long b_batches = d.sB != 0 ? d.G : 1;
    p.M = d.M; p.N = d.N; p.K = d.K; p.shift = d.shift; p.init = d.init;
    p.range = g_cache.dev;
    p.verify_b_all_batches = d.sB != 0;
    p.b_shift = b_shift;

    // (a divided B has another range than the raw one: the shift is part of its key)
    const OperandKey key_a(d.A, (long)d.G * d.M, d.K, 8), key_b(d.B, d.N, d.K, (d.b32 ? 4 : 8) | (b_shift << 8));
    int na = g_cache.lookup(key_a), nb = prep ? prep->nb : g_cache.lookup(key_b);
    // Activations gathered into a fresh buffer for a known weight matrix (the experts of a MoE layer): guess the
    // digits the last activations multiplied with that matrix needed.  A wrong guess costs one guarded recomputation.
    if (!na && nb) {
        auto it = g_cache.partner_a.find(key_b);
        if (it != g_cache.partner_a.end()) na = it->second;
    }
    // Operands at addresses never seen: for products below kShapeGuessMaxMacs the digits of the last operands of the
    // same shapes stand in (a wrong guess costs such a product less than the wait for a sample would: the reference's
    // driver builds every layer anew, generate.py:227-238, so most of its calls come with new or recycled addresses);
    // larger products, and shapes never seen, are sampled, which waits for the stream once.
    if ((!na || !nb) && (double)d.G * d.M * d.N * d.K < kShapeGuessMaxMacs) {
        if (!na) na = g_cache.lookup_shape(key_a);
        if (!nb) nb = g_cache.lookup_shape(key_b);
    }
    // No call waits for its verdict (unless there is no pinned memory, or ZK_GEMM_SYNC asks for it): a guarded launch
    // behind the product redoes it with digits that cover everything if the verdict is raised.
    const bool speculate = g_cache.reports.words && !g_switches.sync_verdict;
    if (!na || !nb) {
        p.tiles_m = p.tiles_n = 1;
        range_reset_kernel<<<1, 64, 0, 0>>>(p.range);
        range_sample_kernel<<<1, 256, 0, 0>>>(p, d.b32, d.G, 0);
        range_sample_kernel<<<1, 256, 0, 0>>>(p, d.b32, d.G, 1);
        int64_t r[4];
        if (!read_range(p.range, r)) { set_error(kLaunchFailure, "gemm: range readback failed"); return kFailed; }
        if (!na) na = limbs_needed(r[0], r[1]);
        if (!nb) nb = limbs_needed(r[2], r[3]);
    }
    if (prep) { p.B = prep->planes; p.b_nsub = prep->nsub; p.b_ksteps = prep->ksteps; }

    // Everything an attempt allocates is allocated before its first launch: memory that is short for digit planes then
    // sends the call to the kernels that split both operands themselves (which need none), and nothing it has launched
    // can have raised the verdict that the next call relies on being clear.
    bool planes_fit = true, slots_fit = true;
    for (int attempt = 0; attempt < 3; attempt++) {
        // the stored bits are [shift, shift + 64) of the sum (the remainder lies below them)
        const int need_diag = (d.shift + 64 + 7) / 8;
        // (the kernels that read planes never see B's element type: they are the int64 forms)
        const Instance *inst = d.M <= g_switches.skinny_max_m ? pick_instance(na, nb, d.b32 != 0 && !prep, true, need_diag, prep ? prep->nb : 0, prep ? kB64FlyBPlanes : -1) : nullptr;
        if (!inst) inst = pick_instance(na, nb, d.b32 != 0 && !prep, false, need_diag, prep ? prep->nb : 0, prep ? kB64PlanesBoth : -1);
        if (!inst && prep) {
            // no kernel with exactly the planes' digit count covers A: this call splits the original B like any other
            // (nb, the planes' count, covers B)
            prep = nullptr;
            p.B = d.B;
            inst = d.M <= g_switches.skinny_max_m ? pick_instance(na, nb, d.b32 != 0, true, need_diag) : nullptr;
            if (!inst) inst = pick_instance(na, nb, d.b32 != 0, false, need_diag);
        }
        if (!inst) return kDeclined;
        if (!prep && !inst->skinny) inst = smaller_tiles(inst, d, g_cache.cus);
        if (!prep) { p.B = d.B; p.b_gstride = 0; }
        p.ldbn = d.ldbn; p.ldbk = d.ldbk; p.sB = d.sB;
        p.row_steps = nullptr;
        // planes on both sides: the pipelined kernel, where there is one for the digit counts
        PipeForm pipe = {};
        if (prep && !inst->skinny && inst->kk == 1 && !g_switches.no_pipe) pipe = pipe_form(inst->na, inst->nb);
        RowtileForm rowtile = {};
        bool pre_b = false;
        if (planes_fit && !prep && b_shift == 0 && pipe_b_planes(d, kmajor, b_batches)) {
            const Instance *both = pick_instance(na, nb, false, false, need_diag, 0, kB64PlanesBoth);
            const PipeForm f = both ? pipe_form(both->na, both->nb) : PipeForm{};
            const long fewer = both && both->na < both->nb ? both->na : (both ? both->nb : 0);
            if (f.fn && fewer * ((d.K + 31) / 32) * 32 * 16384 <= kMaxDiagonal &&
                pipe_b_pays(d, both->na, both->nb, (long)((d.M + 127) / 128) * ((d.N + f.bn - 1) / f.bn) * d.G, g_cache.cus)) {
                inst = both;
                pipe = f;
                pre_b = true;
                p.col_parts = g_switches.no_rowtile || !slots_fit ? 0 : rowtile_parts(d, inst->na, inst->nb, f.bn, g_cache.cus);
                if (p.col_parts) { rowtile = rowtile_form(inst->na, inst->nb); pipe = PipeForm{}; }
            }
        }
        if (!prep && !pre_b && b_shift == 0) inst = short_k_tiles(inst, d, g_cache.cus);
        bool b_copied = false;
        if (kmajor && !pre_b && b_copy_pays(d, inst->nb, b_batches)) {
            // (without memory for the copy the n-contiguous kernels run as they are)
            const Outcome got = grow(g_cache.b_rows, g_cache.b_rows_count, (size_t)(b_batches * d.N * d.K), "row-major copy of B");
            if (got == kFailed) return kFailed;
            b_copied = got == kDone;
        }
        const bool by_columns = kmajor && !b_copied;         // the kernels read B along n
        // int32 accumulators: at most min(NA,NB) digit pairs per diagonal, each product at most 2^14 in magnitude
        const long pairs = inst->na < inst->nb ? inst->na : inst->nb;
        const int ksteps = ((d.K + 32 * inst->kk - 1) / (32 * inst->kk)) * inst->kk;     // 32-k steps, padded
        // (a K beyond that bound is cut into slices that respect it: every tile is then split, see below)
        const bool k_over = pairs * ksteps * 32 * 16384 > kMaxDiagonal;
        const int BM = rowtile.fn ? kRowtileRows : inst->bm, BN = rowtile.fn ? rowtile.bn : pipe.fn ? pipe.bn : inst->bn;
        p.tiles_m = (d.M + BM - 1) / BM;
        p.tiles_n = (d.N + BN - 1) / BN;
        // A B operand that stays in L2 whatever the order (the MLA einsums: a KV cache or one head's weights against
        // a hundred thousand rows) lets the tile columns move fastest, so that each A tile is streamed once
        const size_t b_bytes = (size_t)d.N * d.K * (d.b32 ? 4 : 8);
        p.n_fastest = (b_bytes <= ((size_t)8 << 20) && p.tiles_n > 1 && p.tiles_m > 1) ? 1 : 0;
        const long per_batch = (long)p.tiles_m * p.tiles_n;
        if (per_batch > 0x7FFFFFFFL) return kDeclined;
        const long total = per_batch * d.G;
        if (total > 0x7FFFFFFFL / 8) return kDeclined;
        const int steps = (d.K + 32 * inst->kk - 1) / (32 * inst->kk);
        // slices of K per tile of a launch smaller than the device
        int small_split = total < g_cache.cus ? (int)(g_cache.cus / total) : 1;
        if (small_split > 64) small_split = 64;
        // At least four steps a slice: every one more leaves a tile of partial sums to write and to read (100 rows x
        // [1000,2048] int32: eight slices of 16 tiles 25.7 us, sixteen 33.5; 300 x [600,1536] six of 30 24.2, eight 29.0).
        // While all of that stays small (64 workgroups), down to 128 k: the launch is then as long as one slice.  128 rows
        // against a cache of 779: scores 19.5 -> 18.4 us, values 23.9 -> 19.7; of 64: 18.4 -> 15.3; 128 x [512,512] int64
        // 18.6 -> 17.1.
        int most_slices = steps / 4;
        if (total * most_slices < 64) most_slices = (int)std::max<long>(most_slices, std::min<long>(steps * inst->kk / 4, 64 / total));
        if (small_split > most_slices) small_split = most_slices;
        // A is pre-split into digit planes when enough column tiles reuse it to pay for the extra pass (never for the
        // 32-row tiles: splitting a handful of rows on the fly is cheaper than another kernel in front; nor where the
        // slices of a small launch are so short that the launch in front costs more than three bytes instead of eight per
        // element of A save.  On the fly against planes, by K per workgroup: 256 (512 rows x [1024,1024] int32) 34.6 / 36.6
        // us, 448 (243 x [512,7168]) 35.6 / 39.4, 896 (128 x [2048,7168]) 46.7 / 46.2, 1024 (128 x [7168,2048]) 49.5 /
        // 47.1, 1434 (243 x [1536,7168]) 54.7 / 52.2, 16384 (243 x [7168,16384]) 449 / 353.)
        // Four tile columns of a small launch are too few: 909 x [256,7168] 37 on the fly, 42 on planes, (5,4) digits 50 / 59,
        // 500 x [256,16384] (4,4) 47 / 55; but for three digits of A and slices that do not fall into step with the eight
        // XCDs, so that each of them reads every slice: 1100 x [256,16384] (3,4), seven slices, 117 / 99.
        const bool in_step = small_split > 1 && (small_split % 8 == 0 || 8 % small_split == 0);
        const bool few_columns = p.tiles_n <= 4 && (inst->na > 3 || in_step);
        const bool long_slices = !few_columns && (long)steps * 32 * inst->kk >= 800L * (small_split > 1 ? small_split : 1);
        const bool use_planes = !rowtile.fn && !inst->short_k && (pre_b || (planes_fit && !by_columns && !inst->skinny && (prep || (p.tiles_n >= g_switches.planes_min_tiles_n && (total >= g_cache.cus || long_slices)))));
        if (b_shift && (by_columns || !inst->skinny)) return kDeclined;
        const int variant = pre_b ? kB64PlanesBoth : prep ? (inst->skinny ? kB64FlyBPlanes : kB64PlanesBoth)
                          : b_shift ? (d.b32 ? kB32FlyRs : kB64FlyRs)
                          : by_columns ? (d.b32 ? kB32KmajorFly : kB64KmajorFly)
                                   : (d.b32 ? (use_planes ? kB32Planes : kB32Fly) : (use_planes ? kB64Planes : kB64Fly));
        MfmaKernel fn = inst->fn[variant];
        if (!fn) return kDeclined;
        if (pipe.fn) fn = pipe.fn;
        if (rowtile.fn) fn = rowtile.fn;

        // Split-K: a launch smaller than the device is cut into `split` slices of K per tile, each a workgroup of
        // its own; with more tiles than compute units the same is done for the tiles of the last, partial round
        // only.  The slices leave raw partial sums and a small kernel adds them.
        int tail = (int)(total % g_cache.cus), split = 1;
        p.main_tiles = (int)total;
        p.split = 1;
        p.tail_xcd = 0;
        p.partials = nullptr;
        p.part64 = 0;
        p.finish_rq = 4;
        if (!g_switches.no_tail_split && !pre_b) {
            if (total < g_cache.cus) {
                tail = (int)total;
                split = small_split;
                p.finish_rq = 16;
            } else if (inst->skinny && total < 8L * g_cache.cus) {
                // a few rows against many columns is a weight stream: more, shorter workgroups keep more of it in
                // flight and even out the last round (the partial sums of so few rows cost next to nothing)
                tail = (int)total;
                split = (int)((8L * g_cache.cus + total - 1) / total);
                if (split > 64) split = 64;
                if (split > steps / 4) split = steps / 4;
                p.finish_rq = 16;
            } else if (tail > 0 && tail <= g_cache.cus / 2) {
                split = g_cache.cus / tail;
                if (split > 8) split = 8;
                if (split > steps / 8) split = steps / 8;
            }
        }
        if (k_over) {
            // every tile in slices short enough for the int32 accumulators; without room for the partial sums (or with
            // the split switched off) the vector-ALU path takes the product
            int min_split = 2;
            while (pairs * ((steps + min_split - 1) / min_split) * 32 * inst->kk * 16384 > kMaxDiagonal) min_split++;
            if (g_switches.no_tail_split || min_split > steps) return kDeclined;
            if (tail != (int)total || split < min_split) {
                tail = (int)total;
                split = min_split;
                p.finish_rq = 4;
            }
            if ((size_t)tail * split * BM * BN * 16 > ((size_t)2 << 30)) return kDeclined;
        }
        if (split >= 2) {
            // |sum| < K * 2^(8(NA+NB)-2): below 2^62 the low word alone carries a partial sum
            int kbits = 0;
            while ((1L << kbits) < (long)ksteps * 32) kbits++;
            const bool part64 = 8 * (inst->na + inst->nb) - 2 + kbits <= 62;
            const size_t need = (size_t)tail * split * BM * BN * (part64 ? 1 : 2);
            const Outcome got = grow(g_cache.partials, g_cache.partials_bytes, need, "partial-sum buffer");
            if (got == kDone) {
                p.main_tiles = (int)(total - tail);
                p.split = split;
                p.tail_xcd = (!p.n_fastest && d.G == 1 && tail % p.tiles_m == 0 && p.main_tiles % 8 == 0 &&
                              ((long)tail * split) % (8L * p.tiles_m) == 0) ? 1 : 0;
                p.partials = g_cache.partials;
                p.part64 = part64 ? 1 : 0;
            } else if (got == kFailed) return kFailed;
            else if (k_over) return kDeclined;
        }
        const long row_items = rowtile.fn ? (long)p.tiles_m * d.G * p.col_parts : 0;
        const int row_slots = row_items > 2L * g_cache.cus ? 2 : 1;
        const long blocks = rowtile.fn ? std::min<long>(row_items, 2L * g_cache.cus) : (long)p.main_tiles + (total - p.main_tiles) * p.split;
        long plane_wgs = 0, b_plane_wgs = 0;
        p.fail_class = inst->na > 5 || inst->nb > 5 ? 2 : 1;
        p.verdict = reinterpret_cast<unsigned *>(g_cache.dev + 5) + g_cache.turn;
        p.a_planes = nullptr; p.a_msub = 0; p.a_ksteps = 0;
        const int msub = p.tiles_m * (BM / 32), rows_per_wg = 256 / (4 * inst->kk);
        const dim3 pgrid((unsigned)(ksteps / inst->kk), (unsigned)((msub * 32 + rows_per_wg - 1) / rows_per_wg), (unsigned)d.G);
        const dim3 bgrid((unsigned)ksteps, (unsigned)((d.N + 63) / 64), (unsigned)b_batches);
        BPlanesParams b = {};
        {
            Outcome got = kDone;
            if (use_planes) {
                plane_wgs = (long)pgrid.x * pgrid.y * pgrid.z;
                got = grow(g_cache.planes, g_cache.planes_bytes, (size_t)d.G * msub * ksteps * inst->na * 1024, "digit-plane buffer");
            }
            if (pre_b && got == kDone) {
                b_plane_wgs = (long)bgrid.x * bgrid.y * bgrid.z;
                b.B = d.B; b.ldn = d.ldbn; b.ldk = d.ldbk; b.sB = d.sB; b.N = d.N; b.K = d.K;
                b.nsub = (d.N + 31) / 32; b.ksteps = ksteps;
                b.gstride = (long)b.nsub * ksteps * inst->nb * 1024;
                // (the one product of the model with zeros in A worth finding: a causal prompt's probabilities times the values)
                b.row_tiles = kmajor && !d.b32 && !rowtile.fn ? (long)p.tiles_m * d.G : 0;
                got = grow(g_cache.b_planes, g_cache.b_planes_bytes, (size_t)(b.gstride * b_batches), "digit planes of B");
                // (slots for the digit planes of its row tiles, two per workgroup that has more than one)
                if (got == kDone && rowtile.fn) got = grow(g_cache.planes, g_cache.planes_bytes, (size_t)blocks * row_slots * (kRowtileRows / 32) * ksteps * inst->na * 1024, "digit-plane buffer");
                if (got == kDone && b.row_tiles) got = grow(g_cache.row_steps, g_cache.row_steps_count, (size_t)b.row_tiles, "step counts");
            }
            if (got == kDone) got = grow(g_cache.seen, g_cache.seen_count, (size_t)(blocks + plane_wgs + b_plane_wgs), "digit counts");
            if (got == kFailed) return kFailed;
            if (got == kDeclined) {
                if (!use_planes && !pre_b) return kDeclined;
                // (row tiles dealt in parts take more room than the planes of A in one piece)
                if (rowtile.fn) slots_fit = false;
                else { planes_fit = false; prep = nullptr; }
                attempt--;
                continue;
            }
        }
        if (b_copied) {
            const dim3 grid((unsigned)((d.N + 31) / 32), (unsigned)((d.K + 31) / 32), (unsigned)b_batches);
            b_rows_kernel<<<grid, dim3(256), 0, 0>>>(reinterpret_cast<const int64_t *>(d.B), d.ldbk, d.sB, g_cache.b_rows, d.N, d.K);
            p.B = g_cache.b_rows; p.ldbn = d.K; p.ldbk = 1; p.sB = d.sB != 0 ? (long)d.N * d.K : 0;
        }
        if (use_planes) {
            p.a_planes = g_cache.planes; p.a_msub = msub; p.a_ksteps = ksteps;
            // (the owned-k pattern of the planes of A follows the kernel that reads them: planes of B go with the int64 forms)
            inst->planes[(d.b32 && !prep && !pre_b) ? 1 : 0]<<<pgrid, dim3(256), 0, 0>>>(p, g_cache.planes, msub, ksteps, g_cache.seen + blocks);
        }
        if (pre_b) {
            if (b.row_tiles) {
                b.row_steps = g_cache.row_steps;
                b.a_seen = g_cache.seen + blocks;
            }
            b.planes = g_cache.b_planes; b.seen = g_cache.seen + blocks + plane_wgs; b.verdict = p.verdict; b.fail_class = p.fail_class;
#define ZK_BPL(NB_) do { if (d.b32) { if (kmajor) b_planes_kernel<NB_, true, true><<<bgrid, 256, 0, 0>>>(b); else b_planes_kernel<NB_, false, true><<<bgrid, 256, 0, 0>>>(b); } \
                         else { if (kmajor) b_planes_kernel<NB_, true, false><<<bgrid, 256, 0, 0>>>(b); else b_planes_kernel<NB_, false, false><<<bgrid, 256, 0, 0>>>(b); } } while (0)
            if (inst->nb == 3) ZK_BPL(3); else if (inst->nb == 4) ZK_BPL(4); else ZK_BPL(5);
#undef ZK_BPL
            p.B = b.planes; p.b_nsub = b.nsub; p.b_ksteps = ksteps; p.b_gstride = d.sB != 0 ? b.gstride : 0;
            p.row_steps = b.row_steps;
            if (rowtile.fn) { p.a_planes = g_cache.planes; p.a_msub = row_slots; p.a_ksteps = ksteps; p.items = (int)row_items; }
        }
        p.seen = pipe.fn ? nullptr : g_cache.seen;
        const size_t lds = rowtile.fn ? rowtile.lds : pipe.fn ? pipe.lds : 2 * (size_t)inst->kk * ((BM / 32) * inst->na + (BN / 32) * inst->nb) * 1024 + 9 * 1024 + 16;
        static std::set<const void *> lds_raised;
        if (lds > 64 * 1024 && !lds_raised.count((const void *)fn)) {
            if (hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
                set_error(kLaunchFailure, "gemm: cannot raise the LDS limit to %zu bytes", lds);
                return kFailed;
            }
            lds_raised.insert((const void *)fn);
        }
        unsigned grid = (unsigned)blocks;
        if (pipe.fn) {
            // one workgroup per compute unit walks the items; without split tiles they go row tile by row tile
            p.batches = d.G;
            p.row_order = pre_b ? 1 : 0;
            p.items = pre_b ? (int)(((long)p.tiles_m * d.G + 7) / 8 * 8 * p.tiles_n) : (int)blocks;
            grid = (unsigned)(p.items < g_cache.cus ? p.items : g_cache.cus);
        }
        const unsigned threads = rowtile.fn ? 256 : (unsigned)inst->threads;
        fn<<<dim3(grid), dim3(threads), lds, 0>>>(p);
        g_last_pairs = kept_pairs_before(inst->na, inst->nb, inst->dmax, inst->na, 0);
        g_last_prepared = prep ? 1 : 0;
        if (pipe.fn || rowtile.fn) g_pipe_calls++;
        if (rowtile.fn) g_rowtile_calls++;
        if (inst->short_k) g_short_calls++;
        {
            const hipError_t err = hipGetLastError();
            if (err != hipSuccess) {
                set_error(kLaunchFailure, "gemm: MFMA kernel launch failed (%s; digits %d,%d, %ld workgroups of %d threads, %zu bytes of LDS)",
                          hipGetErrorString(err), inst->na, inst->nb, blocks, (int)threads, lds);
                return kFailed;
            }
        }
        // no waiting: a guarded launch redoes the product if the verdict is raised, the digits seen follow later
        GuardArgs guard = {};
        if (speculate) {
            guard = make_guard((p.seen ? blocks : 0) + plane_wgs + b_plane_wgs);
            if (!p.seen) guard.seen += blocks;
        }
        if (p.split > 1) {
            if (speculate) {
                guard.parts = guard_parts(guard.seen_count, kGuardParts);
                p.guard = guard;
                g_sum_reports++;
            }
            (pipe.fn ? pipe.finish : inst->finish)<<<dim3((unsigned)((total - p.main_tiles) * p.finish_rq + p.guard.parts)), dim3((unsigned)inst->threads), 0, 0>>>(p);
            if (hipGetLastError() != hipSuccess) { set_error(kLaunchFailure, "gemm: split finish launch failed"); return kFailed; }
        }
        *limbs_a = inst->na;
        *limbs_b = inst->nb;
        if (speculate) {
            GuardArgs behind = guard;
            if (p.split > 1) behind.seen_count = kReported;
            if (const Outcome got = launch_guarded_fallback(d, p, b_shift, &behind)) return got;
            if (p.split <= 1) guard.parts = behind.parts;
            guard_taken(guard, key_a, key_b, prep ? prep->nb : 0);       // (the slots are shared with the grouped launches, which set it too)
            return kDone;
        }
        int need_a, need_b;
        if (!wait_digits(p.seen ? 0 : blocks, (p.seen ? blocks : 0) + plane_wgs + b_plane_wgs, &need_a, &need_b)) { set_error(kLaunchFailure, "gemm: digit readback failed"); return kFailed; }
        if (prep) need_b = prep->nb;
        g_cache.store_pair(key_a, need_a, key_b, need_b);
        if (need_a <= inst->na && need_b <= inst->nb) return kDone;
        na = need_a;
        nb = need_b;
    }
    set_error(kLaunchFailure, "gemm: digit count did not settle");
    return kFailed;
}

int gemm_mfma_grouped(const GroupedDesc &d, int *limbs_a, int *limbs_b)
{
    if (d.K <= 0 || d.N <= 0 || d.rows <= 0 || d.groups <= 0) return 1;
    std::lock_guard<std::mutex> lock(g_cache.mu);
    if (!init_cache()) return -1;
    drain_pending();

    MfmaParams p = {};
    p.A = d.A; p.B = nullptr; p.C = d.C; p.R = d.R;
    p.lda = d.lda; p.sA = 0; p.ldbn = d.K; p.ldbk = 1; p.sB = 0; p.ldc = d.ldc; p.sC = 0;
    p.M = d.rows; p.N = d.N; p.K = d.K; p.shift = d.shift; p.init = d.init;
    p.range = g_cache.dev;
    p.tiles_m = 1;
    p.split = 1; p.finish_rq = 4;
    p.grp_seg = d.seg; p.grp_tiles = d.tiles; p.grp_ntiles = d.ntiles; p.grp_b = d.B;

    // digits: what these operands needed last time, else the widest the 32-row kernels have
    const OperandKey key_a(d.A, (long)d.rows, d.K, 8), key_b(d.B, (long)d.groups * d.N, d.K, d.b32 ? 4 : 8);
    // the experts' weights prepared beforehand (the table pointer is the key): planes instead of B, an exact digit count
    const PreparedB *prep = nullptr;
    {
        auto it = g_prepared.find((const void *)d.B);
        if (it != g_prepared.end() && it->second.groups == d.groups && it->second.b32 == (d.b32 ? 1 : 0) && it->second.N == d.N && it->second.K == d.K)
            prep = &it->second;
    }
    if (prep) { p.grp_b = prep->table; p.b_nsub = prep->nsub; p.b_ksteps = prep->ksteps; }
    int na = g_cache.lookup(key_a), nb = prep ? prep->nb : g_cache.lookup(key_b);
    bool na_guessed = false, informed = nb != 0;
    if (!na) {
        auto it = g_cache.partner_a.find(key_b);
        na = it != g_cache.partner_a.end() ? it->second : 5;
        informed = informed && it != g_cache.partner_a.end();
        na_guessed = true;
    }
    if (!nb) nb = 5;
    // Both digit counts come from what these weights met before: speculate, do not wait.  A guarded launch of the
    // 16-row kernels follows on the stream (they guess nothing and take every operand); its workgroups return at once
    // unless the verdict is bad, in which case they compute every output again.  What the kernels saw is
    // stored to pinned host memory by the guarded launch and reaches the cache at a later call.  Otherwise (first sight
    // of the weights) the verdict is read back before the call returns.
    bool speculate = informed && g_cache.reports.words && !g_switches.sync_verdict;

    for (int attempt = 0; attempt < 3; attempt++) {
        const Instance *inst = nullptr;
        for (int tries = 0; tries < 2 && !inst; tries++) {
            inst = pick_instance(na, nb, d.b32 != 0 && !prep, true, 16, prep ? prep->nb : 0, prep ? kB64GroupBPlanes : -1, prep ? prep->kk : 1);
            if (!inst && prep && (inst = pick_instance(na, nb, d.b32 != 0, true)) != nullptr) {
                // no kernel with exactly the planes' digit count covers A: this call splits the original weights
                prep = nullptr;
                p.grp_b = d.B;
            }
            // a guess taken over from other activations that no 32-row kernel covers: try the widest they have (the
            // digit check settles it, and the guess would otherwise never be replaced)
            if (!inst && na_guessed && na > 5) na = 5; else break;
        }
        if (!inst) return 1;
        MfmaKernel fn = inst->fn[prep ? kB64GroupBPlanes : (d.b32 ? kB32Group : kB64Group)];
        if (!fn) return 1;
        // int32 weights, whole steps, rows of A on 16-byte boundaries, sixteen digit pairs or more: the form that streams the
        // weights through LDS rings.  (Measured on 256 experts, one box, streamed against general: (3,4) digits 5.64
        // against 5.86 TB/s at K = 7168 and level at K = 2048; (4,4) level at K = 7168 and 5.08 against 3.15 at K = 2048;
        // (5,5) 4.18 against 3.87.  ZK_STREAM32_MIN_PAIRS moves the limit.)
        size_t stream_lds = 0;
        if (d.b32 && !prep && !g_switches.no_stream32 && d.K % 32 == 0 && (((uintptr_t)d.A | (uintptr_t)(d.lda * 8)) & 15) == 0 && inst->bn == 256 &&
            inst->na * inst->nb >= g_switches.stream32_min_pairs) {
            MfmaKernel sfn = stream32_grouped_kernel(inst->na, inst->nb, &stream_lds);
            if (!sfn) sfn = stream32_grouped_kernel_wide(inst->na, inst->nb, &stream_lds);
            if (sfn) fn = sfn; else stream_lds = 0;
        }
        const long pairs = inst->na < inst->nb ? inst->na : inst->nb;
        const int ksteps = (d.K + 31) / 32;
        if (pairs * ksteps * 32 * 16384 > kMaxDiagonal) return 1;
        p.tiles_n = (d.N + inst->bn - 1) / inst->bn;
        const long max_mtiles = (long)d.rows / 32 + d.groups;
        const long blocks = (max_mtiles + 7) / 8 * 8 * p.tiles_n;       // (whole rounds of the 8 XCDs: see the kernels' tile order)
        if (blocks > 0x7FFFFFFFL / 8) return 1;
        p.main_tiles = (int)blocks;
        if (const Outcome got = grow(g_cache.seen, g_cache.seen_count, (size_t)blocks, "digit counts")) return got;
        p.seen = g_cache.seen;
        p.fail_class = inst->na > 5 || inst->nb > 5 ? 2 : 1;
        p.verdict = reinterpret_cast<unsigned *>(g_cache.dev + 5) + g_cache.turn;
        const size_t lds = stream_lds ? stream_lds : 2 * (size_t)inst->kk * ((inst->bm / 32) * inst->na + (inst->bn / 32) * inst->nb) * 1024 + 9 * 1024 + 16;
        static std::set<const void *> lds_raised;
        if (lds > 64 * 1024 && !lds_raised.count((const void *)fn)) {
            if (hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
                set_error(kLaunchFailure, "grouped gemm: cannot raise the LDS limit to %zu bytes", lds);
                return -1;
            }
            lds_raised.insert((const void *)fn);
        }
        fn<<<dim3((unsigned)blocks), dim3((unsigned)inst->threads), lds, 0>>>(p);
        if (stream_lds) g_streamed_calls++;
        g_last_pairs = kept_pairs_before(inst->na, inst->nb, inst->dmax, inst->na, 0);
        g_last_prepared = prep ? 1 : 0;
        {
            const hipError_t err = hipGetLastError();
            if (err != hipSuccess) {
                set_error(kLaunchFailure, "grouped gemm: launch failed (%s; digits %d,%d, %ld workgroups)", hipGetErrorString(err), inst->na, inst->nb, blocks);
                return -1;
            }
        }
        if (speculate) {
            GuardArgs guard = make_guard(blocks);
            const int rc = gemm_rows16_grouped(d, &guard);
            if (rc < 0) return -1;
            if (rc == 0) {
                *limbs_a = inst->na;
                *limbs_b = inst->nb;
                guard_taken(guard, key_a, key_b, prep ? prep->nb : 0);
                return 0;
            }
            speculate = false;      // the 16-row kernels do not take this product: wait for the verdict after all
        }
        int need_a, need_b;
        if (!wait_digits(0, blocks, &need_a, &need_b)) { set_error(kLaunchFailure, "grouped gemm: digit readback failed"); return -1; }
        if (prep) need_b = prep->nb;
        g_cache.store_pair(key_a, need_a, key_b, need_b);
        *limbs_a = inst->na;
        *limbs_b = inst->nb;
        if (need_a <= inst->na && need_b <= inst->nb) return 0;
        na = need_a;
        nb = need_b;
        na_guessed = false;
    }
    set_error(kLaunchFailure, "grouped gemm: digit count did not settle");
    return -1;
}

}  // namespace zk
