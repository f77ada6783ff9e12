// Operand fragments of v_mfma_i32_16x16x64_i8 held by the lanes that loaded them: digit counts from the data, digit split in
// registers (gemm_rows16.hip, gemm_small.hip).
#pragma once
#include "gemm_mfma_kernels.h"
#include "lds_dma.h"

namespace zk {

// The 64 k of a step are dealt to (lane quarter q, fragment byte b) so that every load is 16 bytes and the four lanes
// of a row read 64 contiguous bytes:
//   int64 weights: byte b <-> k = 8*(b/2) + 2*q + b%2      (A and B: eight loads of two elements)
//   int32 weights: byte b <-> k = 16*(b/4) + 4*q + b%4     (B: four loads of four elements; A: eight loads of two)
template <bool B32>
__device__ __forceinline__ int frag_k(int q, int b) { return B32 ? 16 * (b >> 2) + 4 * q + (b & 3) : 8 * (b >> 1) + 2 * q + (b & 1); }

// One operand fragment as loaded: 16 elements of 64 bits (A, int64 weights) or of 32 bits (int32 weights), as the
// 16-byte pieces the loads delivered.
template <bool W32> struct RawFrag { v4i v[W32 ? 4 : 8]; };

template <bool W32>
__device__ __forceinline__ uint64_t magnitude_or(const RawFrag<W32> &f)
{
    // OR of x for x >= 0 and ~x otherwise: below 2^(8n-2) means n digits hold every element
    if (W32) {
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int z = 0; z < 4; z++) m |= (uint32_t)(f.v[j][z] ^ (f.v[j][z] >> 31));
        return m;
    }
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int j = 0; j < 8; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int s = f.v[j][2 * h + 1] >> 31;
            lo |= (uint32_t)(f.v[j][2 * h] ^ s);
            hi |= (uint32_t)(f.v[j][2 * h + 1] ^ s);
        }
    return ((uint64_t)hi << 32) | lo;
}

// digits (3, 4, 5, or 9 for "more") that hold every element of the wavefront whose magnitudes OR to m in some lane
__device__ __forceinline__ int wave_digits(uint64_t m)
{
    if (__builtin_amdgcn_ballot_w64(m >> 22 != 0) == 0) return 3;
    if (__builtin_amdgcn_ballot_w64(m >> 30 != 0) == 0) return 4;
    if (__builtin_amdgcn_ballot_w64(m >> 38 != 0) == 0) return 5;
    return 9;
}

template <int N, bool W32>
__device__ __forceinline__ void split_frag(const RawFrag<W32> &f, v4i (&out)[N])
{
    if (W32) {
        int x[16];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int z = 0; z < 4; z++) x[4 * j + z] = f.v[j][z];
        split16_w32<N>(x, out);
    } else if (N <= 4) {
        int x[16];                  // values below 2^(8N-2): the low words say it all
#pragma unroll
        for (int j = 0; j < 8; j++) { x[2 * j] = f.v[j][0]; x[2 * j + 1] = f.v[j][2]; }
        split16_w32<N>(x, out);
    } else {
        int64_t x[16];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            x[2 * j] = (int64_t)(((uint64_t)(uint32_t)f.v[j][1] << 32) | (uint32_t)f.v[j][0]);
            x[2 * j + 1] = (int64_t)(((uint64_t)(uint32_t)f.v[j][3] << 32) | (uint32_t)f.v[j][2]);
        }
        split16<N>(x, out);
    }
}

}  // namespace zk
