// Shared device/host helpers for the gfx950 kernels of the ATA beamforming path.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <string>

#include "blade_amd.h"

namespace bl {

// Vector types used by the MFMA builtins.
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWave = 64;

// Error plumbing: the C-ABI returns a Result code and keeps a thread-local
// message for blade_amd_last_error().
void set_error(const std::string& msg);

inline int fail(const std::string& msg) {
    set_error(msg);
    return BLADE_ERROR;
}

inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string(what) + ": " + hipGetErrorString(e));
        return BLADE_HIP_ERROR;
    }
    return BLADE_SUCCESS;
}

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Compute units of the current device (cached per device).
inline int device_cus() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

// Library-owned scratch for launches that need it, one buffer per (device,
// stream, consumer) so that calls on different streams never share one;
// grown on demand (the old buffer is released after the stream drains).
enum WorkspaceUser { WS_BEAMFORMER_SINK = 0, WS_ADJOINT = 1, WS_CHANNELIZER_BIG = 2 };
int library_workspace(int user, size_t bytes, hipStream_t s, unsigned char** out);

// The library's own stream on the current device, for filling tables: created on
// first use, kept for the life of the process.
hipError_t table_stream(hipStream_t* out);

// A library-owned table of the current device, whole when this returns: `fill`
// queues its kernels on the library's stream, which is waited for.  Filled on the
// caller's stream it would be ready there only, while calls on other streams find
// the same pointer; and a stream under capture would record the fill instead of
// running it.  Once per table, so the wait costs nothing later.
template <typename Fill>
int device_table(const char* what, size_t bytes, void** out, Fill fill) {
    void* p = nullptr;
    hipStream_t s = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipSuccess) e = table_stream(&s);
    if (e == hipSuccess) {
        fill(p, s);
        e = hipGetLastError();
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
    }
    if (e != hipSuccess) {
        (void)hipFree(p);
        set_error(std::string(what) + ": " + hipGetErrorString(e));
        return BLADE_HIP_ERROR;
    }
    *out = p;
    return BLADE_SUCCESS;
}

// Number of scalar components and bytes per element of a blade_type.
inline int type_components(int t) {
    switch (t) {
        case BLADE_CI8: case BLADE_CF16: case BLADE_CF32: case BLADE_CF64: return 2;
        default: return 1;
    }
}

inline int type_scalar_bytes(int t) {
    switch (t) {
        case BLADE_I8: case BLADE_CI8: return 1;
        case BLADE_F16: case BLADE_CF16: return 2;
        case BLADE_F32: case BLADE_CF32: case BLADE_I32: return 4;
        case BLADE_F64: case BLADE_CF64: return 8;
        default: return 0;
    }
}

inline int type_bytes(int t) { return type_components(t) * type_scalar_bytes(t); }

__device__ __forceinline__ floatx4 mfma_f16(halfx8 a, halfx8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ floatx4 mfma_bf16(uint4 a, uint4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The high halves of two floats as one dword (lo in bits 0-15): the pair of
// BF16 values (lo, hi) when both are exact in BF16.
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// Exact CI8 -> BF16 (an int8 needs 8 significant bits, BF16 has 8): the
// (re, im) pair of polarization p of one voltage dword.
__device__ __forceinline__ uint32_t ci8_to_bf16(uint32_t d, int p) {
    return bf16_pair((float)(int8_t)(d >> (16 * p)), (float)(int8_t)(d >> (16 * p + 8)));
}

// v = part[0] + part[1] + part[2] exactly, each part with the 8 significant
// bits of BF16 (in the high half of its float): an FP32 value has 24, so
// cutting 8 off the top three times leaves nothing.  As BF16 pairs the parts end
// at 2^-133, so this holds from |v| = 2^-110 on; smaller values lose what they
// hold below 2^-133 (relative error 2^-15 at 2^-118).  Infinities and NaN stay in part 0 (CHECKED; otherwise they
// become NaN).
template <bool CHECKED = true>
__device__ __forceinline__ void split_bf16x3(float v, float (&part)[3]) {
    const uint32_t u = __float_as_uint(v);
    if (CHECKED && (u & 0x7f800000u) == 0x7f800000u) {
        part[0] = __uint_as_float((u & 0x007fffffu) ? (u | 0x00400000u) : u);
        part[1] = part[2] = 0.f;
        return;
    }
    part[0] = __uint_as_float(u & 0xffff0000u);
    const float r = v - part[0];
    part[1] = __uint_as_float(__float_as_uint(r) & 0xffff0000u);
    part[2] = r - part[1];
}

// Exact CI8 -> FP16: int8 b becomes the biased byte u = b + 128, placed in the
// mantissa of 1024.0 (0x6400) to give 1024 + u exactly; subtracting 1152 gives b.
// Both pols of a dword at once: v_perm_b32 places each biased byte below a
// 0x64 byte (0x64uu = 1024 + u in FP16), one packed subtract removes the bias.
// {src0, src1} is read as bytes 7..4 = src0, 3..0 = src1.
__device__ __forceinline__ void ci8_to_half2x2(uint32_t d, halfx2& p0, halfx2& p1) {
    const uint32_t u = d ^ 0x80808080u;
    const uint32_t b0 = __builtin_amdgcn_perm(u, 0x64646464u, 0x00050004u);   // (u0, 64, u1, 64)
    const uint32_t b1 = __builtin_amdgcn_perm(u, 0x64646464u, 0x00070006u);   // (u2, 64, u3, 64)
    const halfx2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    p0 = __builtin_bit_cast(halfx2, b0) - bias;
    p1 = __builtin_bit_cast(halfx2, b1) - bias;
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
    return make_float2(a.x + b.x, a.y + b.y);
}

__device__ __forceinline__ float2 csub(float2 a, float2 b) {
    return make_float2(a.x - b.x, a.y - b.y);
}

}  // namespace bl
