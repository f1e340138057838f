// Shared helpers of the HIP sources: error reporting, dtype codes, bf16 conversion,
// wave64 reductions.  Every exported function returns 0 on success; on failure it
// returns nonzero and leaves a message that <family>_last_error() returns, the way
// the reference's HIP layer turns a status into code + message
// (rocml-hip/src/error.rs:32-48).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstdint>
#include <cstdio>

#define ROCML_EXPORT extern "C" __attribute__((visibility("default")))

enum RocmlDtype : int { ROCML_F32 = 0, ROCML_BF16 = 1 };

static thread_local char g_rocml_err[1024] = "";

static int rocml_fail(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_rocml_err, sizeof(g_rocml_err), fmt, ap);
    va_end(ap);
    return 1;
}

#define ROCML_REQUIRE(cond, ...)                       \
    do {                                               \
        if (!(cond)) return rocml_fail(__VA_ARGS__);   \
    } while (0)

#define ROCML_CHECK_LAUNCH(name)                                                         \
    do {                                                                                 \
        hipError_t e_ = hipGetLastError();                                               \
        if (e_ != hipSuccess)                                                            \
            return rocml_fail("%s: launch failed: %s (%d)", name, hipGetErrorString(e_), \
                              (int)e_);                                                  \
    } while (0)

#define ROCML_LAST_ERROR_FN(family) \
    ROCML_EXPORT const char* family##_last_error() { return g_rocml_err; }

// Compute units of the current device (256 on an MI355X).  Launch sizes are phrased in it: how
// many blocks fill the chip, how many tiles leave CUs idle.
static int cu_count() {
    static int cached[64] = {0};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
    if (cached[device] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) n = 256;
        cached[device] = n;
    }
    return cached[device];
}

// ---- bf16 as raw 16 bits ------------------------------------------------------
typedef uint16_t bf16_t;

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
    return __uint_as_float(((uint32_t)v) << 16);
}

// Round to nearest even; NaN stays NaN.  gfx950 has the conversion in hardware
// (v_cvt_pk_bf16_f32), which the compiler picks for these casts.
__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }

// two values in one instruction: a in the low half
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2_t_;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t_;
    f32x2_t_ v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t_));
}

template <typename T> struct Elem;
template <> struct Elem<float> {
    static __device__ __forceinline__ float load(const float* p) { return *p; }
    static __device__ __forceinline__ void store(float* p, float v) { *p = v; }
};
template <> struct Elem<bf16_t> {
    static __device__ __forceinline__ float load(const bf16_t* p) { return bf16_to_f32(*p); }
    static __device__ __forceinline__ void store(bf16_t* p, float v) { *p = f32_to_bf16(v); }
};

// ---- buffers --------------------------------------------------------------------
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ga_buffer(const void* base, long long bytes) {
    // raw buffer (stride 0), 32-bit data format; the range check is on the byte offset
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)min(bytes, (long long)0x7fffffff), 0x00020000);
}
constexpr uint32_t BUF_NOWHERE = 0x80000000u;         // an offset beyond every such buffer: the load gives zeros

// ---- wave64 reductions --------------------------------------------------------
constexpr int WAVE = 64;

// Exchanges that stay in the vector registers (a shuffle is a trip through LDS, some 50 ns one after the other).  All 64 lanes are
// active.  lane_xor1, lane_xor2: the neighbour's value one and two lanes across.
template <int CTRL> __device__ __forceinline__ float lane_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_xor1(float v) { return lane_dpp<0xB1>(v); }
__device__ __forceinline__ float lane_xor2(float v) { return lane_dpp<0x4E>(v); }

// sum over the 16 lanes of a row, the same in every lane: lanes 1 apart, 2 apart, mirrored inside a
// half row, mirrored inside the row
__device__ __forceinline__ float row16_sum(float v) {
    v += lane_xor1(v);
    v += lane_xor2(v);
    v += lane_dpp<0x141>(v);
    v += lane_dpp<0x140>(v);
    return v;
}

__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, lane_xor1(v));
    v = fmaxf(v, lane_xor2(v));
    v = fmaxf(v, lane_dpp<0x141>(v));
    return fmaxf(v, lane_dpp<0x140>(v));
}

// The two values of lanes 16 (32) apart, in both: swapping the odd rows (the upper half) of one copy with the even rows (the lower half) of the other.
struct LanePair { float a, b; };
__device__ __forceinline__ LanePair lane_pair16(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ LanePair lane_pair32(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}

// sum and maximum over the four rows' lanes of the same place
__device__ __forceinline__ float rows4_sum(float v) {
    LanePair p = lane_pair16(v);
    p = lane_pair32(p.a + p.b);
    return p.a + p.b;
}
__device__ __forceinline__ float rows4_max(float v) {
    LanePair p = lane_pair16(v);
    p = lane_pair32(fmaxf(p.a, p.b));
    return fmaxf(p.a, p.b);
}

// and over all lanes, in the order of a butterfly of shuffles from 32 lanes apart to 1: turns by 8 and by 4 in a row bring the value
// 8 and 4 lanes across, as all rows are alike by then and a row repeats itself after 8.  A sum of 64 values waits for six
// vector operations instead of six trips through LDS, some 50 ns each (of a whole request at most 1 %, little more than two runs of one
// side differ by).
__device__ __forceinline__ float row16_sum_far(float v) {
    v += lane_dpp<0x128>(v);
    v += lane_dpp<0x124>(v);
    v += lane_xor2(v);
    return v + lane_xor1(v);
}
__device__ __forceinline__ float wave_sum(float v) {
    LanePair p = lane_pair32(v);
    p = lane_pair16(p.a + p.b);
    return row16_sum_far(p.a + p.b);
}
__device__ __forceinline__ float wave_max(float v) { return rows4_max(row16_max(v)); }

static inline int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
