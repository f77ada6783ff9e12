// Float checkpoint -> fixed-point weights on the device.
//
// The reference builds its integer weights in inference/convert2.py with tensor ops around a Triton kernel:
//   fp8 weights:   w = weight_dequant(w_fp8, scale)                     (inference/kernel.py:67-117: e4m3 value times
//                  the float32 scale of its 128x128 block, stored in the default dtype, bfloat16: convert2.py:185)
//                  w_int = (w.to(float32) * 2^k).round().to(int32)      (convert2.py:144-147, 308-311, 325-328, ...)
//   bf16 params:   p_int = (p.to(float32) * 2^k).round().to(int32|int64) (convert2.py:250-262, 290-295, 353-359)
// Each step is one IEEE operation, restated here per element: exact fp8 -> float32, one float32 multiply (round to
// nearest even), float32 -> bfloat16 (round to nearest even), an exact power-of-two scaling, round half to even, and
// the float -> integer conversion of the device the reference runs on (saturating, NaN -> 0).
// One pass: 1 byte read and 4 written per fp8 weight, instead of six tensor-sized round trips.
#include "common.h"
#include "../../include/int64gemm.h"

namespace zk {

constexpr int kScaleBlock = 128;      // weight_dequant's block_size default (inference/kernel.py:96)

// OCP e4m3fn byte `sel` of a packed word -> float32, exact (1 sign, 4 exponent with bias 7, 3 mantissa bits; no
// infinities, S.1111.111 is NaN): gfx950's own conversion instruction
template <int SEL>
__device__ __forceinline__ float e4m3fn_to_f32(uint32_t packed)
{
    return __builtin_amdgcn_cvt_f32_fp8((int)packed, SEL);
}

// float32 -> bfloat16 -> float32, round to nearest even (NaN stays NaN): the hardware conversion, as a cast
__device__ __forceinline__ float round_to_bf16(float v)
{
    return (float)(__bf16)v;
}

// round half to even, then convert as the reference's device does: saturate, NaN -> 0.  That is what v_cvt_i32_f32
// does on its own; the instruction is named because a C++ cast is undefined outside the int32 range.
__device__ __forceinline__ int32_t round_to_i32(float z)
{
    int32_t o;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(o) : "v"(rintf(z)));
    return o;
}

__device__ __forceinline__ int64_t round_to_i64(float z)
{
    const float r = rintf(z);
    if (!(r == r)) return 0;
    if (r >= 9223372036854775808.0f) return INT64_MAX;
    if (r <= -9223372036854775808.0f) return INT64_MIN;
    return (int64_t)r;
}

typedef int v4i_q __attribute__((ext_vector_type(4)));

// Four consecutive weights per thread and round (cols % 4 == 0, aligned pointers): a 4-byte load and a 16-byte store, adjacent
// lanes on adjacent pieces so that both are contiguous over the wave, and over the launch: workgroup after workgroup takes the next
// U * 256 pieces of the matrix, whatever the rows.  A 128-wide scale block covers whole 4-element pieces, so one scale serves a
// piece.  Bound by its stores, four fifths of the bytes.  A workgroup per row, four rounds of 1024 pieces one after the other /
// as it is: [18432,7168] 148.6 / 103.7 us (6.4 TB/s), [2048,7168] 17.9 / 14.3, [7168,2048] 16.0 / 13.8, [576,7168] 7.4 / 5.3,
// [1536,1536] 3.9 / 3.6, [100,16000] 9.0 / 3.3.
template <int U>
__global__ __launch_bounds__(256) void fp8_to_int32_vec_kernel(const uint32_t *__restrict__ w, const float *__restrict__ scale,
                                                               v4i_q *__restrict__ out, long begin, long pieces, int pieces_per_row, int scale_cols, float mult)
{
    const long first = begin + (long)blockIdx.x * (256 * U);
    const long row0 = first / pieces_per_row;
    const unsigned col0 = (unsigned)(first - row0 * pieces_per_row) + threadIdx.x;
    uint32_t in[U];
    float s[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (first + u * 256 + threadIdx.x >= pieces) continue;
        unsigned col = col0 + u * 256;
        long row = row0;
        if (col >= (unsigned)pieces_per_row) { const unsigned n = col / (unsigned)pieces_per_row; row += n; col -= n * (unsigned)pieces_per_row; }
        in[u] = __builtin_nontemporal_load(w + first + u * 256 + threadIdx.x);
        s[u] = scale[(row / kScaleBlock) * scale_cols + col / (kScaleBlock / 4)];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (first + u * 256 + threadIdx.x >= pieces) continue;
        v4i_q o;
        o[0] = round_to_i32(round_to_bf16(e4m3fn_to_f32<0>(in[u]) * s[u]) * mult);
        o[1] = round_to_i32(round_to_bf16(e4m3fn_to_f32<1>(in[u]) * s[u]) * mult);
        o[2] = round_to_i32(round_to_bf16(e4m3fn_to_f32<2>(in[u]) * s[u]) * mult);
        o[3] = round_to_i32(round_to_bf16(e4m3fn_to_f32<3>(in[u]) * s[u]) * mult);
        __builtin_nontemporal_store(o, out + first + u * 256 + threadIdx.x);
    }
}

// The same for rows of any length from four on: a piece's four weights may lie in two rows and in two scale blocks, and what is left
// behind the last whole piece goes one by one.  Bound by memory where the matrix is large.  Element by element with a division each, as below / this, us:
// 2048 x 7169 26.5 / 17.2, 18432 x 7171 277 / 125 (5.3 TB/s), 16384 x 513 16.5 / 11.9, 576 x 7166 8.6 / 6.3, 1535 x 1537 5.7 / 4.4;
// 100 x 101, 5000 x 130 and 100000 x 5 the same.
template <int U>
__global__ __launch_bounds__(256) void fp8_to_int32_any_kernel(const uint8_t *__restrict__ w, const float *__restrict__ scale, int32_t *__restrict__ out,
                                                               long begin, long n, int cols, int scale_cols, float mult)
{
    const long first = begin + (long)blockIdx.x * (256 * U), pieces = n >> 2;
    const long row0 = 4 * first / cols;
    const unsigned col0 = (unsigned)(4 * first - row0 * cols) + 4 * threadIdx.x;
    uint32_t in[U];
    float s[U][4];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const long piece = first + u * 256 + threadIdx.x;
        if (piece >= pieces) continue;
        unsigned col = col0 + u * 1024;
        const unsigned over = col / (unsigned)cols;
        long row = row0 + over;
        col -= over * (unsigned)cols;
        in[u] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(w) + piece);
#pragma unroll
        for (int z = 0; z < 4; z++) {
            s[u][z] = scale[(row / kScaleBlock) * scale_cols + col / kScaleBlock];
            if (++col == (unsigned)cols) { col = 0; row++; }
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const long piece = first + u * 256 + threadIdx.x;
        if (piece >= pieces) continue;
        v4i_q o;
        o[0] = round_to_i32(round_to_bf16(e4m3fn_to_f32<0>(in[u]) * s[u][0]) * mult);
        o[1] = round_to_i32(round_to_bf16(e4m3fn_to_f32<1>(in[u]) * s[u][1]) * mult);
        o[2] = round_to_i32(round_to_bf16(e4m3fn_to_f32<2>(in[u]) * s[u][2]) * mult);
        o[3] = round_to_i32(round_to_bf16(e4m3fn_to_f32<3>(in[u]) * s[u][3]) * mult);
        __builtin_nontemporal_store(o, reinterpret_cast<v4i_q *>(out) + piece);
    }
    const long rest = 4 * pieces + threadIdx.x;
    if (first == 0 && rest < n)
        out[rest] = round_to_i32(round_to_bf16(e4m3fn_to_f32<0>(w[rest]) * scale[(rest / cols / kScaleBlock) * scale_cols + rest % cols / kScaleBlock]) * mult);
}

// Launches of 256 threads over `pieces` pieces: launch(grid, first piece, two pieces a thread).
// Two pieces per thread once the launch is long enough to be bound by memory (one / two, us: 1536 x 1536 3.6 / 4.4, 576 x 7168
// 5.3 / 5.1, 2048 x 7168 15.7 / 14.3, 18432 x 7168 122.7 / 103.7; four: 110.9).  A grid of 2^32 threads or more runs only what is
// left of their number in 32 bits, with no error: a matrix of 2^35 weights and more takes several launches.
template <typename Launch>
static void for_stretches(long pieces, Launch launch)
{
    constexpr long kMost = 1L << 23;
    const bool two = pieces > (1L << 20);
    const long per_block = two ? 512 : 256, blocks = (pieces + per_block - 1) / per_block;
    for (long b = 0; b < blocks; b += kMost) launch(dim3((unsigned)(blocks - b < kMost ? blocks - b : kMost)), b * per_block, two);
}

constexpr long kPiecesMin = 512;

// element by element: rows of one to three weights, matrices so small that a thread per piece is a longer chain for nothing (in
// pieces / so, kernel alone, us: 1 x 7 1.55 / 1.36, 1 x 101 1.60 / 1.36, 1 x 333 1.60 / 1.48, but 128 x 5 1.46 / 1.72, 1 x 1537 1.68 / 2.20), and
// pointers that are not aligned to the vectors
__global__ __launch_bounds__(256) void fp8_to_int32_kernel(const uint8_t *__restrict__ w, const float *__restrict__ scale,
                                                           int32_t *__restrict__ out, long n, int cols, int scale_cols, float mult)
{
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const long row = i / cols;
        const int col = (int)(i - row * cols);
        const float s = scale[(row / kScaleBlock) * scale_cols + col / kScaleBlock];
        out[i] = round_to_i32(round_to_bf16(e4m3fn_to_f32<0>(w[i]) * s) * mult);
    }
}

template <typename OT>
__global__ __launch_bounds__(256) void bf16_round_kernel(const uint16_t *__restrict__ in, OT *__restrict__ out, long n, float mult)
{
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const float z = __uint_as_float((uint32_t)in[i] << 16) * mult;
        if (sizeof(OT) == 4) out[i] = (OT)round_to_i32(z);
        else out[i] = (OT)round_to_i64(z);
    }
}

static unsigned grid_for(long items)
{
    const long blocks = (items + 255) / 256;
    return (unsigned)(blocks < 1 ? 1 : (blocks > 65536 * 4 ? 65536 * 4 : blocks));
}

// 2^k as a float32, the scalar the reference multiplies by; k in [0,127] keeps it finite
static bool pow2_ok(const char *name, int k, float *mult)
{
    if (k < 0 || k > 127) { set_error(kBadArgument, "%s: exponent %d outside 0..127", name, k); return false; }
    *mult = ldexpf(1.0f, k);
    return true;
}

template <typename OT>
static void launch_bf16_round(const char *name, const uint16_t *in, OT *out, long n, int k)
{
    float mult;
    if (n < 0) { set_error(kBadArgument, "%s: negative size", name); return; }
    if (!pow2_ok(name, k, &mult) || n == 0) return;
    if (!in || !out) { set_error(kBadArgument, "%s: null pointer", name); return; }
    bf16_round_kernel<OT><<<dim3(grid_for(n)), dim3(256), 0, 0>>>(in, out, n, mult);
    check_launch(name);
}

}  // namespace zk

extern "C" {

void fp8_block_scaled_to_int32(const uint8_t *w, const float *scale, int32_t *out, int rows, int cols, int k)
{
    const char *name = "fp8_block_scaled_to_int32";
    float mult;
    if (rows < 0 || cols < 0) { zk::set_error(zk::kBadArgument, "%s: negative dimension", name); return; }
    if (!zk::pow2_ok(name, k, &mult) || (long)rows * cols == 0) return;
    if (!w || !scale || !out) { zk::set_error(zk::kBadArgument, "%s: null pointer", name); return; }
    const int scale_cols = (cols + zk::kScaleBlock - 1) / zk::kScaleBlock;
    const long n = (long)rows * cols;
    if (cols % 4 == 0 && ((uintptr_t)w & 3) == 0 && ((uintptr_t)out & 15) == 0) {
        const int ppr = cols / 4;
        const uint32_t *wp = reinterpret_cast<const uint32_t *>(w);
        zk::v4i_q *op = reinterpret_cast<zk::v4i_q *>(out);
        zk::for_stretches(n / 4, [&](dim3 grid, long begin, bool two) {
            if (two) zk::fp8_to_int32_vec_kernel<2><<<grid, dim3(256), 0, 0>>>(wp, scale, op, begin, n / 4, ppr, scale_cols, mult);
            else zk::fp8_to_int32_vec_kernel<1><<<grid, dim3(256), 0, 0>>>(wp, scale, op, begin, n / 4, ppr, scale_cols, mult);
        });
    } else if (cols >= 4 && n >= zk::kPiecesMin && ((uintptr_t)w & 3) == 0 && ((uintptr_t)out & 15) == 0) {
        zk::for_stretches(n / 4, [&](dim3 grid, long begin, bool two) {
            if (two) zk::fp8_to_int32_any_kernel<2><<<grid, dim3(256), 0, 0>>>(w, scale, out, begin, n, cols, scale_cols, mult);
            else zk::fp8_to_int32_any_kernel<1><<<grid, dim3(256), 0, 0>>>(w, scale, out, begin, n, cols, scale_cols, mult);
        });
    } else {
        zk::fp8_to_int32_kernel<<<dim3(zk::grid_for(n)), dim3(256), 0, 0>>>(w, scale, out, n, cols, scale_cols, mult);
    }
    zk::check_launch(name);
}

void bf16_scaled_round_to_int32(const uint16_t *in, int32_t *out, long n, int k)
{
    zk::launch_bf16_round<int32_t>("bf16_scaled_round_to_int32", in, out, n, k);
}

void bf16_scaled_round_to_int64(const uint16_t *in, int64_t *out, long n, int k)
{
    zk::launch_bf16_round<int64_t>("bf16_scaled_round_to_int64", in, out, n, k);
}

}  // extern "C"
