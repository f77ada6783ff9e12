// Shared declarations of libint64gemm.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

typedef __int128 i128;
typedef unsigned __int128 u128;

namespace zk {

enum ErrorCode { kOk = 0, kBadArgument = 1, kLaunchFailure = 2, kUnsupportedSize = 3 };

// Records the first error since zk_clear_error(); later ones are dropped so the cause is kept.
void set_error(int code, const char *fmt, ...);
// hipGetLastError() after a launch; records kLaunchFailure and returns false on failure.
bool check_launch(const char *what);
int device_cus();                          // compute units of the current device

// Errors detected on the device: a pinned host flag per kind (null when pinned memory is not to be had) that a kernel
// sets to 1; zk_last_error() turns a set flag into a recorded error.
enum DeferredError { kDeferredMoeIndex = 0, kDeferredCount };
int *deferred_error_flag(int which);

// Device memory the library holds between calls (per module), and its release.
size_t gemm_mfma_workspace_bytes(size_t *prepared_bytes);
void gemm_mfma_release_workspace();
void gemm_mfma_reload_switches();
size_t act_workspace_bytes();
void act_release_workspace();

constexpr int kWave = 64;

// A pointer that came out of memory itself (an expert's matrix from the table of a grouped launch) could point anywhere
// as far as the compiler knows, and a load through it counts as an LDS access as well: every wait for LDS then waits
// for the weights under way.  Loads of operands name their address space: (const ZK_GLOBAL_MEM T *)ptr.
#define ZK_GLOBAL_MEM __attribute__((address_space(1)))

// ---- wave-level helpers --------------------------------------------------------------------
// The values of a lane and of its partner OFF lanes away, as a reduction over 1, 2, 4 ... lanes needs them (lanes that have met
// already hold the same): through the vector pipe alone, where a shuffle goes through LDS.  Within sixteen lanes by row permutes
// (neighbours, pairs, mirrored eights, mirrored sixteens), beyond by swapping rows of sixteen and halves of the wavefront.  Everything
// that uses it through shuffles / so, kernels alone, us: softmax with preparation of 128 rows of 779 5.2 / 4.9, of 1024 rows of 1024 9.6 / 9.1, RMSNorm
// of one row of 7168 5.7 / 5.1, of 500 rows 12.5 / 11.9, routing of one token 8.1 / 6.7, one row x [576,7168] int64 8.7 / 8.4, 243 rows x [512,1536]
// int32 (the report) 19.2 / 18.9; long streams are level.
template <int OFF>
__device__ __forceinline__ void lane_pair(unsigned v, unsigned &a, unsigned &b)
{
    if constexpr (OFF <= 8) {
        constexpr int CTRL = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x140;
        a = v;
        b = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
    } else {
        const auto t = OFF == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false) : __builtin_amdgcn_permlane32_swap(v, v, false, false);
        a = t[0];
        b = t[1];
    }
}
template <int OFF>
__device__ __forceinline__ void lane_pair(uint64_t v, uint64_t &a, uint64_t &b)
{
    unsigned al, bl, ah, bh;
    lane_pair<OFF>((unsigned)v, al, bl);
    lane_pair<OFF>((unsigned)(v >> 32), ah, bh);
    a = (uint64_t)ah << 32 | al;
    b = (uint64_t)bh << 32 | bl;
}
template <int OFF>
__device__ __forceinline__ void lane_pair(int64_t v, int64_t &a, int64_t &b)
{
    uint64_t ua, ub;
    lane_pair<OFF>((uint64_t)v, ua, ub);
    a = (int64_t)ua;
    b = (int64_t)ub;
}

// f(offset) for the six steps of a reduction over a wavefront, nearest lanes first
template <class F>
__device__ __forceinline__ void wave_steps(F &&f)
{
    f(std::integral_constant<int, 1>());
    f(std::integral_constant<int, 2>());
    f(std::integral_constant<int, 4>());
    f(std::integral_constant<int, 8>());
    f(std::integral_constant<int, 16>());
    f(std::integral_constant<int, 32>());
}

// 64-lane reductions.  Every lane ends up with the result.
__device__ __forceinline__ int64_t wave_max_i64(int64_t v)
{
    wave_steps([&](auto off) {
        int64_t a, b;
        lane_pair<decltype(off)::value>(v, a, b);
        v = a > b ? a : b;
    });
    return v;
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v)
{
    wave_steps([&](auto off) {
        uint64_t a, b;
        lane_pair<decltype(off)::value>(v, a, b);
        v = a + b;
    });
    return v;
}

// ---- exact integer division helpers -----------------------------------------------------------
// C++ signed division with the two undefined corners fixed (b == 0 -> 0, INT64_MIN / -1 wraps).
__device__ __forceinline__ int64_t tdiv64(int64_t a, int64_t b)
{
    if (b == 0) return 0;
    if (b == -1) return (int64_t)(0 - (uint64_t)a);
    return a / b;
}

// floor(num / den) for 0 <= num < 2^53, 0 < den < 2^53 and quotient < 2^40, given inv = 1.0 / (double)den.
// The double estimate is within one of the quotient; the remainder test makes it exact.
__device__ __forceinline__ uint64_t udiv_by_inv(uint64_t num, uint64_t den, double inv)
{
    uint64_t q = (uint64_t)((double)num * inv);
    int64_t rem = (int64_t)(num - q * den);
    if (rem < 0) { q -= 1; rem += (int64_t)den; }
    if (rem >= (int64_t)den) q += 1;
    return q;
}

}  // namespace zk
