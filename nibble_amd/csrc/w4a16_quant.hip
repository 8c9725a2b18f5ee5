// Round-to-nearest group quantizer on the device: fp16 / fp32 weights [N, K]
// -> packed INT4 codes [N, K / 2] and fp16 scales [N, K / G], byte-identical to
// nibble_amd/quantization.py's torch ops (reference
// w4a16/quantization.py:65-113): s = amax|w| / 7 in fp32 (1.0 for a zero
// group), code = clamp(round_half_even(fl(w / s)), -7, 7), stored scale
// fp16(s).
//
// Bound: memory (2 or 4 bytes read and 0.5 written per weight, each once).
// K is a multiple of G, so groups lie end to end over the whole matrix and
// rows do not matter: lane i of a wavefront holds 8 consecutive weights, a
// group is G / 8 neighbouring lanes, and its maximum is a DPP reduction in
// registers. Four vectors a lane are in flight before the first is used.
// 14336 x 4096 from fp16 (148 MB): 32.7 us, 4.5 TB/s of the 5.1 a copy reaches;
// 901 us as 14 torch passes and a host check.
#include "w4a16_hip.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "w4a16_device.h"

namespace w4a16_internal {
void set_last_error(const std::string& message);   // w4a16_hip.hip: the message w4a16_last_error() returns
}

namespace w4a16 {

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}

// The maximum over each aligned run of L lanes, in all of them (every lane active).
template <int L>
__device__ __forceinline__ uint32_t lanes_max(uint32_t v) {
    if constexpr (L >= 2) v = dpp_max<0xB1>(v);    // quad_perm [1,0,3,2]
    if constexpr (L >= 4) v = dpp_max<0x4E>(v);    // quad_perm [2,3,0,1]
    if constexpr (L >= 8) v = dpp_max<0x141>(v);   // row_half_mirror
    if constexpr (L >= 16) v = dpp_max<0x140>(v);  // row_mirror
    if constexpr (L >= 32) v = max(v, (uint32_t)__shfl_xor((int)v, 16));
    if constexpr (L >= 64) v = max(v, (uint32_t)__shfl_xor((int)v, 32));
    return v;
}

constexpr int kQuantVectors = 4;   // vectors of 8 weights per lane

struct Vec8 {
    float w[8];
    uint32_t amax;   // bits of the largest |w|: ordered as the values, NaN above infinity
};

__device__ __forceinline__ Vec8 widen(const u32x4& a) {   // 8 fp16 weights
    Vec8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v.w[2 * i] = (float)as_f16x2(a[i]).x;
        v.w[2 * i + 1] = (float)as_f16x2(a[i]).y;
    }
    v.amax = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) v.amax = max(v.amax, __builtin_bit_cast(uint32_t, v.w[i]) & 0x7FFFFFFFu);
    return v;
}

// fl(w / s) rounded half to even. w * rcp(s) is within 3 ulp of the quotient
// (|quotient| <= 7, so within 2e-6); where that leaves the rounding open, and
// for scales whose reciprocal is not a normal number, a correctly rounded
// division decides.
__device__ __forceinline__ int quant_code(float w, float s, float inv, bool plain) {
    const float r = w * inv;
    float n = __builtin_rintf(r);
    if (!(plain && __builtin_fabsf(r - n) < 0.49999f)) n = __builtin_rintf(w / s);
    return n == n ? (int)__builtin_fminf(__builtin_fmaxf(n, -7.0f), 7.0f) : 0;   // NaN: code 0, as torch's cast
}

// Weights of type T (f16 or float), groups of 8 L weights; vecs = N K / 8.
template <typename T, int L>
__global__ void __launch_bounds__(256)
quantize_pack_kernel(const T* __restrict__ w, uint32_t* __restrict__ packed, f16* __restrict__ scales, int64_t vecs) {
    const int64_t base = (int64_t)blockIdx.x * (256 * kQuantVectors) + threadIdx.x;
    constexpr int W = sizeof(T) / 2;   // 16-byte words per vector
    u32x4 raw[kQuantVectors][W];
    const u32x4* src = reinterpret_cast<const u32x4*>(w);
#pragma unroll
    for (int u = 0; u < kQuantVectors; ++u) {
        const int64_t j = min(base + 256 * u, vecs - 1);   // lanes past the end re-read the last vector
#pragma unroll
        for (int i = 0; i < W; ++i) raw[u][i] = load_stream(src + j * W + i);
    }
#pragma unroll
    for (int u = 0; u < kQuantVectors; ++u) {
        const int64_t j = base + 256 * u;
        Vec8 v;
        if constexpr (W == 1) {
            v = widen(raw[u][0]);
        } else {
            v.amax = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t bits = raw[u][i / 4 % W][i & 3];
                v.w[i] = __builtin_bit_cast(float, bits);
                v.amax = max(v.amax, bits & 0x7FFFFFFFu);
            }
        }
        const float amax = __builtin_bit_cast(float, lanes_max<L>(v.amax));
        const float s = amax == 0.0f ? 1.0f : amax / 7.0f;
        const bool plain = s > 1e-30f && s < 1e30f;   // false for NaN
        const float inv = __builtin_amdgcn_rcpf(s);
        uint32_t word = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) word |= ((uint32_t)quant_code(v.w[i], s, inv, plain) & 15u) << (4 * i);
        if (j < vecs) {
            packed[j] = word;
            if ((threadIdx.x & (L - 1)) == 0) scales[j / L] = (f16)s;
        }
    }
}

template <typename T>
bool launch_quantize(int lanes, const void* w, void* packed, void* scales, int64_t vecs, hipStream_t stream) {
    const dim3 grid((unsigned)((vecs + 256 * kQuantVectors - 1) / (256 * kQuantVectors)));
#define QUANT(L)                                                                                              \
    case L:                                                                                                   \
        hipLaunchKernelGGL((quantize_pack_kernel<T, L>), grid, dim3(256), 0, stream, static_cast<const T*>(w), \
                           static_cast<uint32_t*>(packed), static_cast<f16*>(scales), vecs);                  \
        return true;
    switch (lanes) {
        QUANT(2)
        QUANT(4)
        QUANT(8)
        QUANT(16)
        QUANT(32)
        QUANT(64)
    }
#undef QUANT
    return false;
}

}  // namespace w4a16

namespace {
int fail(int code, const std::string& message) {
    w4a16_internal::set_last_error(message);
    return code;
}
}  // namespace

extern "C" int w4a16_quantize_pack(const void* weights, int weight_bytes, uint8_t* packed_weights, void* scales,
                                   int64_t N, int64_t K, int64_t group_size, void* stream) {
    if (weight_bytes != 2 && weight_bytes != 4)
        return fail(W4A16_ERR_CONFIG, "weight_bytes must be 2 (fp16) or 4 (fp32)");
    if (group_size < 16 || group_size > 512 || (group_size & (group_size - 1)) != 0)
        return fail(W4A16_ERR_GROUP_SIZE, "quantize_pack needs group_size to be 16, 32, 64, 128, 256 or 512");
    if (N < 0 || K < 0 || K % group_size != 0)
        return fail(W4A16_ERR_SHAPE, "N and K must be non-negative and K divisible by group_size");
    if (N == 0 || K == 0) return W4A16_OK;
    if (weights == nullptr || packed_weights == nullptr || scales == nullptr)
        return fail(W4A16_ERR_NULL, "weights, packed_weights and scales must be non-NULL");
    if ((reinterpret_cast<uintptr_t>(weights) & 15u) != 0)
        return fail(W4A16_ERR_ALIGNMENT, "weights must be 16-byte aligned");
    if ((reinterpret_cast<uintptr_t>(packed_weights) & 3u) != 0 || (reinterpret_cast<uintptr_t>(scales) & 1u) != 0)
        return fail(W4A16_ERR_ALIGNMENT, "packed_weights must be 4-byte and scales 2-byte aligned");
    if (N > (INT64_MAX >> 4) / K) return fail(W4A16_ERR_TOO_LARGE, "N K too large");
    const int64_t vecs = N * K / 8;
    if ((vecs + 1023) / 1024 > INT32_MAX / 256) return fail(W4A16_ERR_TOO_LARGE, "too many weights for one launch");
    const int lanes = (int)(group_size / 8);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (weight_bytes == 2)
        w4a16::launch_quantize<w4a16::f16>(lanes, weights, packed_weights, scales, vecs, st);
    else
        w4a16::launch_quantize<float>(lanes, weights, packed_weights, scales, vecs, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(W4A16_ERR_LAUNCH, std::string("kernel launch failed: ") + hipGetErrorString(e));
    return W4A16_OK;
}
