// e8t_f32.h -- pieces shared by the kernels on the fp32 matrix instruction: activations of
// any dtype read through bounds-checked buffers, and the 16 x 16 x 4 product itself.
#pragma once

#include "e8t_device.h"
#include "e8t_lut.h"

namespace ojx {

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// n consecutive activations as loaded (fp32: n words, 16-bit: n / 2 words).
template <int DT, int n> struct RawX {
    static constexpr int W = DT == kF32 ? n : n / 2;
    uint32_t w[W];

    // byte offset vo + so (so uniform); kNoRecordOffset (or any offset past the buffer) reads zeros
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, uint32_t vo, int so = 0) {
        if constexpr (W % 4 == 0) {
#pragma unroll
            for (int i = 0; i < W / 4; ++i) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, vo + 16u * i, so, 0);
                w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
            }
        } else {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b, vo, so, 0);
            w[0] = v.x; w[1] = v.y;
        }
    }
    __device__ __forceinline__ void set(const uint32_t (&v)[n]) {  // one value each, as bits
#pragma unroll
        for (int i = 0; i < W; ++i) w[i] = DT == kF32 ? v[i] : v[2 * i % n] | (v[(2 * i + 1) % n] << 16);
    }
    __device__ __forceinline__ float get(int j) const {
        if constexpr (DT == kF32) return __uint_as_float(w[j]);
        const uint32_t h = (w[j / 2] >> (16 * (j & 1))) & 0xFFFFu;
        return DT == kF16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
    }
};

template <int DT> constexpr uint32_t esize() { return DT == kF32 ? 4 : 2; }

// Buffer over `rows` rows of a row-major [M, width] matrix from row m0 (fewer at its end).
template <int DT>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* a, int64_t m0, int64_t M,
                                                              int64_t width, int rows) {
    const int64_t left = M - m0 < rows ? M - m0 : rows;
    return __builtin_amdgcn_make_buffer_rsrc(
        (void*)(static_cast<const char*>(a) + m0 * width * esize<DT>()), (short)0,
        (int)(left * width * esize<DT>()), kRsrcWord3);
}

}  // namespace ojx
