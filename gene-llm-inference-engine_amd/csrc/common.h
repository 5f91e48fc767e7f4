// Shared declarations of the gfx950 kernel library: element types, error reporting, wave helpers.
//
// Every entry point is `extern "C"`, takes raw device pointers and a HIP stream, checks on the host
// that the operand shapes fit what its kernel assumes, launches, and returns 0 or a negative code
// whose text `gi_last_error()` gives.  Nothing here allocates device memory.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define GI_API extern "C" __attribute__((visibility("default")))

enum GiDtype : int { GI_F32 = 0, GI_BF16 = 1 };

typedef uint16_t bf16_t;   // storage of a bfloat16: the high half of a float

// Records the message and returns -1 (defined in elementwise.hip).
int gi_fail(const char* fmt, ...);

// Compute units of the current device (defined in elementwise.hip).
GI_API int gi_compute_units();

#define GI_REQUIRE(cond, ...)                  \
    do {                                       \
        if (!(cond)) return gi_fail(__VA_ARGS__); \
    } while (0)

#define GI_CHECK_LAUNCH(name)                                                        \
    do {                                                                             \
        hipError_t e_ = hipGetLastError();                                           \
        if (e_ != hipSuccess) return gi_fail("%s: launch failed: %s", name, hipGetErrorString(e_)); \
    } while (0)

__device__ __forceinline__ float bf16_to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// Round to nearest, ties to even; NaN stays NaN.  gfx950 converts in hardware (v_cvt_pk_bf16_f32).
typedef __bf16 gi_bf16x2 __attribute__((ext_vector_type(2)));
typedef float gi_floatx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float lo, float hi) {
    const gi_floatx2 f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, gi_bf16x2));
}
__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return (bf16_t)(f32x2_to_bf16x2(f, 0.f) & 0xffffu); }

__device__ __forceinline__ float load_f32(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float load_f32(const bf16_t* p, size_t i) { return bf16_to_f32(p[i]); }
__device__ __forceinline__ void store_f32(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void store_f32(bf16_t* p, size_t i, float v) { p[i] = f32_to_bf16(v); }

// The gated feed-forwards' activations, act(gate) * up with the float32 products of a row:
//   0  SiLU(g) * u
//   1  the tanh form of GELU, 0.5 g (1 + tanh(sqrt(2/pi) (g + 0.044715 g^3))), times u
//   2  both halves clamped first, g <- min(g, limit), u <- clamp(u, -limit, limit): g * sigmoid(1.702 g) * (u + 1)
constexpr int GI_N_ACTIVATIONS = 3;
__device__ __forceinline__ float gated_act(float g, float u, int act, float limit) {
    if (act == 2) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g * (1.0f / (1.0f + expf(-1.702f * g))) * (u + 1.0f);
    }
    if (act == 1) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
    return g * (1.0f / (1.0f + expf(-g))) * u;
}

// The two-parameter activation "xielu": with a = softplus(p) and b = 1/2 + softplus(q),
//   z > 0:  a z^2 + z / 2          z <= 0:  b (exp(z) - 1 - z) + z / 2
// (quadratic on the right, bounded below on the left, slope 1/2 on both sides of 0).
__device__ __forceinline__ float softplus_f32(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float xielu(float z, float a, float b) { return z > 0.f ? fmaf(a * z, z, 0.5f * z) : fmaf(b, expm1f(z) - z, 0.5f * z); }

// 16 bytes that a launch reads no second time: they go past the caches, which is faster where the lanes of one load take whole cache lines of 128 bytes
// (67 MB of weights 12.8 -> 11.4 us in a bare read) and slower where they take half lines (14.1 -> 14.8).
// Weights that the next pass reads again go the same way, though 256 MB behind the L2s could hold a small model's till then: in whole models that is worth next to nothing.  Past the caches and through them, us a pass:
// 768 wide with 200 MB at 1 / 8 rows 298, 298 / 322, 322; 1,024 wide with 213 MB at 4 rows 236, 234; 512 wide with 70 MB 187, 185; 256 wide with 11 MB 136, 131; in 32 bits 462, 466 and 303, 308; two or three
// models of 200 MB in turn 303, 324 and 238, 251; 1.1 GB, some of whose matrices have 2 million numbers, with these through the caches 1 % slower.  (A chain of one shape of product, 200 MB of weights in all, tells
// otherwise: 768 x 768 2.5, 2.3.)
__device__ __forceinline__ uint4 load16_once(const bf16_t* p) {              // of bytes that this launch reads no second time
    typedef uint32_t gi_load4 __attribute__((ext_vector_type(4)));
    const gi_load4 v = __builtin_nontemporal_load(reinterpret_cast<const gi_load4*>(p));
    return uint4{v.x, v.y, v.z, v.w};
}

// Two loads of 8 rows' 128 bytes each, lane l of either with row l % 8 and the 16 bytes l / 16 + 4 (l / 8 % 2) of it (`low`: rows 0 to 7, `high`: 8 to 15), become operands
// of two products: lane l with row l % 16 and the 16 bytes l / 16 (`low`) and those 64 bytes further (`high`).  Within 16 lanes the upper half of `low` and the lower half of
// `high` change places.
__device__ __forceinline__ void rows_of_halves(uint4& low, uint4& high) {
    auto swap = [](uint32_t& a, uint32_t& b) {
        const uint32_t was = a;
        a = __builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);        // (rotated by 8 within 16 lanes; lanes 8 to 15 take it)
        b = __builtin_amdgcn_update_dpp(b, was, 0x128, 0xf, 0x3, false);      // (lanes 0 to 7)
    };
    swap(low.x, high.x);
    swap(low.y, high.y);
    swap(low.z, high.z);
    swap(low.w, high.w);
}

// A workgroup barrier that waits for this wave's LDS traffic only.  __syncthreads() also waits for every load
// from global memory the wave has in flight, which undoes a prefetch into registers; use this one where the
// barrier orders LDS reads and writes and nothing else.
__device__ __forceinline__ void barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Butterfly reductions over the 64 lanes of a wave: every lane ends with the same value, and the
// order of the additions is fixed by the lane numbers alone.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// Sum over a workgroup of `NT` threads (a multiple of 64, at most 1024); `red` holds NT/64 floats of LDS.
// All threads get the result; the order of additions depends on NT only.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) t += red[w];
    return t;
}

// For workgroups of one launch that meet: waits (one thread of a workgroup) until `counter` says that `n` others have come.  A wait ends whatever the counter
// held at the start: false after so many polls of about a microsecond each, of which a meeting takes some dozens at most, for a caller whose counters were
// not 0 or that gave them to two launches at once.  The workgroup then leaves no numbers (NaN) where its sums would have gone.
constexpr int MEETING_POLLS = 1 << 18;
__device__ __forceinline__ bool others_came(unsigned* counter, int n) {
    for (int polls = 0; (int)__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n; ++polls) {
        if (polls == MEETING_POLLS) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}
