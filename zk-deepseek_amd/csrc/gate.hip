// Expert routing of the MoE gate in exact integers: one wavefront per token.
//
// Restates the tensor ops of Gate.forward (inference/model.py:1143-1208) on the sigmoid scores the gate's kernel
// part produced: add the bias, score every group of experts by the sum of its two largest biased scores (by its
// maximum when there is no bias), keep the `topk_groups` best groups, take the `topk` largest biased scores among
// the kept groups (the others count as -2^42), gather the UNBIASED scores of the winners, and normalise them:
// w = floor(floor(w * 2^23 / sum w) * 5 / 2).  Winners come out in descending order of biased score.
// Where values tie, torch.topk leaves the order to its implementation; here the lower index wins.
#include "common.h"
#include "act_one.h"
#include "../../include/int64gemm.h"

#include <atomic>

namespace zk {

struct Best { int64_t v; int idx; };
struct __attribute__((aligned(16))) i64x2g { int64_t x, y; };

// larger value wins; on equal values the lower index
__device__ __forceinline__ Best better(Best a, Best b)
{
    const bool take_b = b.v > a.v || (b.v == a.v && b.idx < a.idx);
    return take_b ? b : a;
}

__device__ __forceinline__ Best wave_best(Best x)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        Best o;
        o.v = __shfl_xor(x.v, off, kWave);
        o.idx = __shfl_xor(x.idx, off, kWave);
        x = better(x, o);
    }
    return x;
}

__device__ __forceinline__ int64_t floordiv64(int64_t a, int64_t b)
{
    if (b == 0) return 0;
    int64_t q = tdiv64(a, b);
    if ((uint64_t)q * (uint64_t)b != (uint64_t)a && ((a < 0) != (b < 0))) q--;
    return q;
}

// the two largest of both sides: the larger first, then the best of the rest
template <int OFF>
__device__ __forceinline__ void lane_best2(int64_t &b1, int64_t &b2)
{
    int64_t a1, o1, a2, o2;
    lane_pair<OFF>(b1, a1, o1);
    lane_pair<OFF>(b2, a2, o2);
    const int64_t lo = a1 > o1 ? o1 : a1, rest = a2 > o2 ? a2 : o2;
    b1 = a1 > o1 ? a1 : o1;
    b2 = lo > rest ? lo : rest;
}
__device__ __forceinline__ int64_t from_lane(int64_t v, int lane)      // (the same lane for the whole wavefront)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(uint64_t)v, lane), hi = (unsigned)__builtin_amdgcn_readlane((int)((uint64_t)v >> 32), lane);
    return (int64_t)((uint64_t)hi << 32 | lo);
}

constexpr int64_t kMasked = -((int64_t)1 << 42);
constexpr int kNone = 0x7FFFFFFF;

// EPL elements per lane, element e = lane * EPL + j.  FUSED: `scores` holds the gate's logits; their sigmoid (Q23, table
// `lut`) is taken here and stored to `sig` when that is not null.
template <int EPL, bool FUSED>
__global__ __launch_bounds__(256) void gate_route_kernel(const int64_t *__restrict__ scores, const int64_t *__restrict__ lut,
                                                         int64_t *__restrict__ sig, const int32_t *__restrict__ bias,
                                                         int64_t *__restrict__ weights, int64_t *__restrict__ indices,
                                                         int64_t *__restrict__ raw, int T, int E, int n_groups,
                                                         int topk_groups, int topk)
{
    const int lane = threadIdx.x & 63;
    const long tok = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tok >= T) return;
    const int64_t *row = scores + tok * E;
    int64_t orig[EPL], s[EPL];
    bool live[EPL];
#pragma unroll
    for (int j = 0; j < EPL; j++) {
        const int e = lane * EPL + j;
        live[j] = e < E;
        orig[j] = live[j] ? row[e] : 0;
        if (FUSED && live[j]) {
            orig[j] = act_one<23, true>(orig[j], lut);
            if (sig) sig[tok * E + e] = orig[j];
        }
        s[j] = live[j] ? (int64_t)((uint64_t)orig[j] + (uint64_t)(int64_t)(bias ? bias[e] : 0)) : 0;
    }

    if (n_groups > 1) {
        // lane g ends up holding the score of group g
        const int gsize = E / n_groups;
        int grp[EPL];                                     // group of every element (one division each, not one per test)
#pragma unroll
        for (int j = 0; j < EPL; j++) grp[j] = live[j] ? (lane * EPL + j) / gsize : -1;
        int64_t my_group_score = 0;
        for (int g = 0; g < n_groups; g++) {
            Best b1 = { INT64_MIN, kNone };
#pragma unroll
            for (int j = 0; j < EPL; j++) {
                const int e = lane * EPL + j;
                if (grp[j] == g) b1 = better(b1, Best{ s[j], e });
            }
            b1 = wave_best(b1);
            int64_t gs = b1.v;
            if (bias) {                                   // top-2 sum: the best of the rest of the group
                Best b2 = { INT64_MIN, kNone };
#pragma unroll
                for (int j = 0; j < EPL; j++) {
                    const int e = lane * EPL + j;
                    if (grp[j] == g && e != b1.idx) b2 = better(b2, Best{ s[j], e });
                }
                b2 = wave_best(b2);
                gs = (int64_t)((uint64_t)gs + (uint64_t)(b2.idx == kNone ? 0 : b2.v));
            }
            if (lane == g) my_group_score = gs;
        }
        // rank of group `lane` among the groups (ties: the lower group first), then every element asks its group
        int rank = 0;
        for (int h = 0; h < n_groups; h++) {
            const int64_t o = __shfl(my_group_score, h, kWave);
            if (o > my_group_score || (o == my_group_score && h < lane)) rank++;
        }
        const int keep = (lane < n_groups && rank < topk_groups) ? 1 : 0;
#pragma unroll
        for (int j = 0; j < EPL; j++) {
            const int kept = __shfl(keep, live[j] ? grp[j] : 0, kWave);
            if (live[j] && !kept) s[j] = kMasked;
        }
    }

    // the topk largest, one wave-wide arg-max per winner
    int64_t wsum = 0, my_w = 0;                     // lane i < topk keeps the unbiased score of winner i
    int my_idx = 0;
    bool taken[EPL];
#pragma unroll
    for (int j = 0; j < EPL; j++) taken[j] = !live[j];
    for (int i = 0; i < topk; i++) {
        Best b = { INT64_MIN, kNone };
#pragma unroll
        for (int j = 0; j < EPL; j++)
            if (!taken[j]) b = better(b, Best{ s[j], lane * EPL + j });
        b = wave_best(b);
        int64_t w = 0;
#pragma unroll
        for (int j = 0; j < EPL; j++)
            if (lane * EPL + j == b.idx) { taken[j] = true; w = orig[j]; }
        w = __shfl(w, b.idx / EPL, kWave);
        wsum = (int64_t)((uint64_t)wsum + (uint64_t)w);
        if (lane == i) { my_w = w; my_idx = b.idx; }
    }
    if (lane < topk) {
        if (raw) raw[tok * topk + lane] = my_w;
        int64_t w = floordiv64((int64_t)((uint64_t)my_w << 23), wsum);      // (w * 2^23) // sum  (model.py:1203)
        w = floordiv64((int64_t)((uint64_t)w * 5ull), 2);                    // w * 5 // 2         (model.py:1208)
        weights[tok * topk + lane] = w;
        indices[tok * topk + lane] = my_idx;
    }
}

// The same routing with the experts of a token spread over LT = NG * LPG lanes: lane l holds the GS consecutive scores
// from l * GS on in registers, LPG neighbouring lanes make up a group.  The groups' two best, the masking and most of the
// arg-max over a token's experts (GS comparisons per lane, log2(LT) exchanges) stay inside a lane; the wave-wide form
// above pays six exchanges per group and per winner.  LPG = 1 gives the most tokens per wavefront (throughput when
// there are many tokens), LPG = 4 the shorter chain of dependent work per token (fewer tokens; the fewest: gate_route_few_kernel).
template <int GS, int LPG, int NG, bool FUSED>
__global__ __launch_bounds__(256) void gate_route_groups_kernel(const int64_t *__restrict__ scores, const int64_t *__restrict__ lut,
                                                                int64_t *__restrict__ sig, const int32_t *__restrict__ bias,
                                                                int64_t *__restrict__ weights, int64_t *__restrict__ indices,
                                                                int64_t *__restrict__ raw, int T, int topk_groups, int topk)
{
    constexpr int LT = NG * LPG, E = GS * LT, kTokens = 64 / LT;
    static_assert(LT <= 64 && GS % 2 == 0, "a token fits a wavefront; 16-byte loads");
    const int lane = threadIdx.x & 63, l = lane % LT, g = l / LPG, first = lane - l;
    const long tok_raw = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * kTokens + lane / LT;
    const bool tok_live = tok_raw < T;
    const long tok = tok_live ? tok_raw : T - 1;          // lanes past the end walk the last token along and store nothing
    const int64_t *row = scores + tok * E + l * GS;
    int64_t s[GS];
#pragma unroll
    for (int j = 0; j < GS; j += 2) {
        const i64x2g v = *reinterpret_cast<const i64x2g *>(row + j);
        s[j] = v.x;
        s[j + 1] = v.y;
    }
    if (FUSED) {
#pragma unroll
        for (int j = 0; j < GS; j++) s[j] = act_one<23, true>(s[j], lut);
        if (sig && tok_live) {
#pragma unroll
            for (int j = 0; j < GS; j += 2) *reinterpret_cast<i64x2g *>(sig + tok * E + l * GS + j) = i64x2g{ s[j], s[j + 1] };
        }
    }
    if (bias) {
#pragma unroll
        for (int j = 0; j < GS; j++) s[j] = (int64_t)((uint64_t)s[j] + (uint64_t)(int64_t)bias[l * GS + j]);
    }

    // the group's score: its two largest biased scores (its largest without bias); then the group's rank
    int64_t b1 = s[0], b2 = INT64_MIN;
#pragma unroll
    for (int j = 1; j < GS; j++) {
        const bool first_j = s[j] > b1;
        const int64_t lower = first_j ? b1 : s[j];
        b1 = first_j ? s[j] : b1;
        b2 = lower > b2 ? lower : b2;
    }
#pragma unroll
    for (int off = LPG / 2; off > 0; off >>= 1) {          // the two best of both halves: the larger first, then the best of the rest
        const int64_t o1 = __shfl_xor(b1, off, kWave), o2 = __shfl_xor(b2, off, kWave);
        const int64_t lo = b1 > o1 ? o1 : b1, rest = b2 > o2 ? b2 : o2;
        b1 = b1 > o1 ? b1 : o1;
        b2 = lo > rest ? lo : rest;
    }
    const int64_t gs = bias ? (int64_t)((uint64_t)b1 + (uint64_t)b2) : b1;
    int rank = 0;
#pragma unroll
    for (int h = 0; h < NG; h++) {
        const int64_t o = __shfl(gs, first + h * LPG, kWave);
        if (o > gs || (o == gs && h < g)) rank++;
    }
    const bool masked = rank >= topk_groups;               // every score of this lane counts as -2^42

    unsigned taken = 0;                                    // bit j: s[j] has won already
    int64_t wsum = 0;
    for (int i = 0; i < topk; i++) {
        // this lane's candidate: its largest score not taken (the lowest index on ties; a masked lane's scores all tie)
        Best b = { INT64_MIN, kNone };
#pragma unroll
        for (int j = 0; j < GS; j++) {
            const int64_t v = masked ? kMasked : s[j];
            if (!((taken >> j) & 1) && (b.idx == kNone || v > b.v)) b = Best{ v, l * GS + j };
        }
#pragma unroll
        for (int off = LT / 2; off > 0; off >>= 1) {
            Best o;
            o.v = __shfl_xor(b.v, off, kWave);
            o.idx = __shfl_xor(b.idx, off, kWave);
            b = better(b, o);
        }
        // the owner gives the winner's unbiased score
        int64_t w = 0;
        if (b.idx / GS == l) {
            const int jw = b.idx % GS;
            taken |= 1u << jw;
            int64_t sv = 0;
#pragma unroll
            for (int j = 0; j < GS; j++) sv = j == jw ? s[j] : sv;
            w = bias ? (int64_t)((uint64_t)sv - (uint64_t)(int64_t)bias[b.idx]) : sv;
        }
        w = __shfl(w, first + b.idx / GS, kWave);
        wsum = (int64_t)((uint64_t)wsum + (uint64_t)w);
        if (l == i % LT && tok_live) {                     // parked in the outputs until the sum is known
            weights[tok * topk + i] = w;
            indices[tok * topk + i] = b.idx;
            if (raw) raw[tok * topk + i] = w;
        }
    }
    if (!tok_live) return;
    for (int i = l; i < topk; i += LT) {                   // (a lane reads back what it stored itself)
        int64_t w = floordiv64((int64_t)((uint64_t)weights[tok * topk + i] << 23), wsum);    // (w * 2^23) // sum  (model.py:1203)
        w = floordiv64((int64_t)((uint64_t)w * 5ull), 2);                                      // w * 5 // 2         (model.py:1208)
        weights[tok * topk + i] = w;
    }
}

// Tokens up to which a token has a wavefront to itself, or four lanes per group.  What bounds one token is the chain of dependent work,
// what bounds many their instructions.
// (One token of 256 experts in 8 groups, with sigmoid, in the lane groups / as a wavefront 12.4 / 7.0 us; of 512, which had six exchanges through LDS per group
// and winner, 24.0 / 9.8, 8192 tokens 119 / 38.)
constexpr int kFewTokens = 8192;

// ... and the line between the two, where the lane groups have the shape: a wavefront to a token is ahead while the chain is what counts, the
// lane groups once there are more wavefronts than the device runs at once, sooner without the sigmoid and its table.  Kernels alone, with
// bias, lane groups / a wavefront, us.  Without sigmoid, 6 winners: 128 experts in 8 groups, 4096 tokens 8.8 / 8.0, 6144 9.3 / 10.1, 8192 10.5 /
// 12.1, in 4 groups 8.4 / 7.7, 9.2 / 9.7, 9.3 / 11.7; 256 in 8 groups 10.0 / 9.3, 11.2 / 11.7, 12.9 / 14.0, of 32 winners 7168 tokens 42.6 / 38.1.
// With it: 128 in 8 groups 10.9 / 9.6, 12.2 / 12.2, 14.1 / 14.8; 256 in 8 groups 15.9 / 12.7, 19.3 / 16.6, 22.5 / 20.8.  In 16 groups a wavefront is ahead all
// through (128 experts, 8192 tokens 21.6 / 16.0, 256 25.3 / 21.8; 512 37.0 / 36.4, without sigmoid 23.3 / 24.2 with bias, 22.3 / 17.5 without).
static int wave_per_token_up_to(int E, int gsize, int topk, bool fused)
{
    if (E == 512 || gsize == 8 || (E == 256 && gsize == 16)) return kFewTokens;
    if (fused) return E == 256 ? kFewTokens : 7168;
    return E == 256 ? (topk <= 8 ? 5120 : 7168) : (topk <= 8 ? 4096 : 5120);
}

// Few tokens: a wavefront each, EPL consecutive experts per lane, 64 / n_groups lanes per group (a power of two).  What takes
// the time is the chain of dependent work per token, so nothing in it leaves the registers: maxima go through lane_pair, a
// winner's lane is found by a ballot (the lowest lane, and in it the lowest expert, wins a tie) and its unbiased score is read
// from that lane; the sigmoid's table waits in LDS, loaded beside the logits.
template <int EPL, bool FUSED>
__global__ __launch_bounds__(64) void gate_route_few_kernel(const int64_t *__restrict__ scores, const int64_t *__restrict__ lut,
                                                            int64_t *__restrict__ sig, const int32_t *__restrict__ bias,
                                                            int64_t *__restrict__ weights, int64_t *__restrict__ indices,
                                                            int64_t *__restrict__ raw, int n_groups, int topk_groups, int topk)
{
    __shared__ int64_t table[256];
    const int lane = threadIdx.x;
    const long tok = blockIdx.x;
    const int64_t *row = scores + (tok * 64 + lane) * EPL;
    int64_t orig[EPL], s[EPL];
#pragma unroll
    for (int j = 0; j < EPL; j += 2) {
        const i64x2g v = *reinterpret_cast<const i64x2g *>(row + j);
        orig[j] = v.x;
        orig[j + 1] = v.y;
    }
    int add[EPL];
#pragma unroll
    for (int j = 0; j < EPL; j++) add[j] = bias ? bias[lane * EPL + j] : 0;
    if (FUSED) {
#pragma unroll
        for (int q = 0; q < 4; q++) table[lane + 64 * q] = lut[lane + 64 * q];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < EPL; j++) orig[j] = act_one<23, true>(orig[j], table);
        if (sig) {
#pragma unroll
            for (int j = 0; j < EPL; j += 2) *reinterpret_cast<i64x2g *>(sig + (tok * 64 + lane) * EPL + j) = i64x2g{ orig[j], orig[j + 1] };
        }
    }
#pragma unroll
    for (int j = 0; j < EPL; j++) s[j] = (int64_t)((uint64_t)orig[j] + (uint64_t)(int64_t)add[j]);

    if (n_groups > 1) {
        // the group's score: its two largest biased scores (its largest without bias); then the group's rank
        const int lanes = 64 / n_groups, g = lane / lanes;
        int64_t b1 = s[0], b2 = INT64_MIN;
#pragma unroll
        for (int j = 1; j < EPL; j++) {
            const bool first_j = s[j] > b1;
            const int64_t lower = first_j ? b1 : s[j];
            b1 = first_j ? s[j] : b1;
            b2 = lower > b2 ? lower : b2;
        }
        if (lanes > 1) lane_best2<1>(b1, b2);
        if (lanes > 2) lane_best2<2>(b1, b2);
        if (lanes > 4) lane_best2<4>(b1, b2);
        if (lanes > 8) lane_best2<8>(b1, b2);
        if (lanes > 16) lane_best2<16>(b1, b2);
        const int64_t gs = bias ? (int64_t)((uint64_t)b1 + (uint64_t)b2) : b1;
        int rank = 0;
        for (int h = 0; h < n_groups; h++) {
            const int64_t o = from_lane(gs, h * lanes);
            if (o > gs || (o == gs && h < g)) rank++;
        }
        if (rank >= topk_groups) {
#pragma unroll
            for (int j = 0; j < EPL; j++) s[j] = kMasked;
        }
    }

    unsigned taken = 0;                                    // bit j: s[j] has won already
    int64_t wsum = 0, my_w = 0;                            // lane i < topk keeps winner i
    int my_idx = 0;
    for (int i = 0; i < topk; i++) {
        int64_t v = INT64_MIN, w = 0;
        int slot = -1;
#pragma unroll
        for (int j = 0; j < EPL; j++) {
            const bool better_j = !((taken >> j) & 1) && (slot < 0 || s[j] > v);
            v = better_j ? s[j] : v;
            w = better_j ? orig[j] : w;
            slot = better_j ? j : slot;
        }
        const int64_t best = wave_max_i64(v);
        const int owner = __ffsll((unsigned long long)__ballot(slot >= 0 && v == best)) - 1;
        w = from_lane(w, owner);
        wsum = (int64_t)((uint64_t)wsum + (uint64_t)w);
        const int idx = owner * EPL + __builtin_amdgcn_readlane(slot, owner);
        if (lane == owner) taken |= 1u << slot;
        if (lane == i) { my_w = w; my_idx = idx; }
    }
    if (lane >= topk) return;
    if (raw) raw[tok * topk + lane] = my_w;
    const int64_t w = floordiv64((int64_t)((uint64_t)my_w << 23), wsum);           // (w * 2^23) // sum  (model.py:1203)
    weights[tok * topk + lane] = (int64_t)((uint64_t)w * 5ull) >> 1;                // w * 5 // 2         (model.py:1208)
    indices[tok * topk + lane] = my_idx;
}

static std::atomic<long> g_gate_wave_calls(0);

template <bool FUSED>
static void gate_launch(const char *name, const int64_t *scores, const int64_t *lut, int64_t *sig, const int32_t *bias,
                        int64_t *weights, int64_t *indices, int64_t *raw, int T, int E, int n_groups, int topk_groups, int topk)
{
    if (T < 0 || E <= 0 || n_groups <= 0 || topk_groups <= 0 || topk <= 0) { set_error(kBadArgument, "%s: bad dimension", name); return; }
    if (T == 0) return;
    if (!scores || !weights || !indices || (FUSED && !lut)) { set_error(kBadArgument, "%s: null pointer", name); return; }
    if (E > 1024) { set_error(kUnsupportedSize, "%s: more than 1024 experts", name); return; }
    if (n_groups > 64 || E % n_groups != 0 || topk_groups > n_groups || topk > 64 || topk > E) {
        set_error(kBadArgument, "%s: groups must divide the experts (at most 64), topk at most 64 and E", name);
        return;
    }
    const int gsize = E / n_groups;
    const bool aligned = (((uintptr_t)scores | (uintptr_t)sig) & 15) == 0;
    const bool pow2 = (n_groups & (n_groups - 1)) == 0;
    const bool lane_groups = aligned && pow2 && n_groups >= 2 && (gsize == 32 || gsize == 16 || gsize == 8) && n_groups <= 16;
    if (aligned && pow2 && T <= (lane_groups ? wave_per_token_up_to(E, gsize, topk, FUSED) : kFewTokens) && (E == 128 || E == 256 || E == 512) && gsize >= E / 64) {
#define ZK_GATE_F(EPL) gate_route_few_kernel<EPL, FUSED><<<dim3((unsigned)T), dim3(64), 0, 0>>>(scores, lut, sig, bias, weights, indices, raw, n_groups, topk_groups, topk)
        if (E == 128) ZK_GATE_F(2);
        else if (E == 256) ZK_GATE_F(4);
        else ZK_GATE_F(8);
#undef ZK_GATE_F
        g_gate_wave_calls++;
        check_launch(name);
        return;
    }
    if (lane_groups) {
        // what the kernel for few tokens does not take: four lanes per group while tokens are few, then one
        const bool spread = T <= kFewTokens;
        const int per_wave = 64 / (n_groups * (spread ? 4 : 1));
        const dim3 grid((unsigned)((T + 4 * per_wave - 1) / (4 * per_wave))), block(256);
#define ZK_GATE_G(GS, LPG, NG) gate_route_groups_kernel<GS, LPG, NG, FUSED><<<grid, block, 0, 0>>>(scores, lut, sig, bias, weights, indices, raw, T, topk_groups, topk)
        // (groups of 8, 16 and 32 out of more than 64, 128 and 256 experts come here with many tokens only)
#define ZK_GATE_NG(GSIZE, NG) do { if constexpr (GSIZE * NG <= (GSIZE == 32 ? 256 : GSIZE == 16 ? 128 : 64)) { if (spread) { ZK_GATE_G(GSIZE / 4, 4, NG); break; } } ZK_GATE_G(GSIZE, 1, NG); } while (0)
#define ZK_GATE_GS(GSIZE) do { if (n_groups == 2) ZK_GATE_NG(GSIZE, 2); else if (n_groups == 4) ZK_GATE_NG(GSIZE, 4); \
                               else if (n_groups == 8) ZK_GATE_NG(GSIZE, 8); else ZK_GATE_NG(GSIZE, 16); } while (0)
        if (gsize == 32) ZK_GATE_GS(32);
        else if (gsize == 16) ZK_GATE_GS(16);
        else ZK_GATE_GS(8);
#undef ZK_GATE_GS
#undef ZK_GATE_NG
#undef ZK_GATE_G
        check_launch(name);
        return;
    }
    const dim3 grid((unsigned)((T + 3) / 4)), block(256);
#define ZK_GATE(EPL) gate_route_kernel<EPL, FUSED><<<grid, block, 0, 0>>>(scores, lut, sig, bias, weights, indices, raw, T, E, n_groups, topk_groups, topk)
    if (E <= 64) ZK_GATE(1);
    else if (E <= 128) ZK_GATE(2);
    else if (E <= 256) ZK_GATE(4);
    else if (E <= 512) ZK_GATE(8);
    else ZK_GATE(16);
#undef ZK_GATE
    check_launch(name);
}

}  // namespace zk

extern "C" void gate_route_q23(const int64_t *scores, const int32_t *bias, int64_t *weights, int64_t *indices,
                               int64_t *raw_weights, int T, int E, int n_groups, int topk_groups, int topk)
{
    zk::gate_launch<false>("gate_route_q23", scores, nullptr, nullptr, bias, weights, indices, raw_weights, T, E, n_groups, topk_groups, topk);
}

extern "C" void gate_sigmoid_route_q23(const int64_t *logits, const int64_t *lut, const int32_t *bias, int64_t *scores,
                                       int64_t *weights, int64_t *indices, int64_t *raw_weights, int T, int E,
                                       int n_groups, int topk_groups, int topk)
{
    zk::gate_launch<true>("gate_sigmoid_route_q23", logits, lut, scores, bias, weights, indices, raw_weights, T, E, n_groups, topk_groups, topk);
}

extern "C" long zk_gate_wave_calls(void) { return zk::g_gate_wave_calls; }
