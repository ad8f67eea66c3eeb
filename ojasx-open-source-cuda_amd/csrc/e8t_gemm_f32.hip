// e8t_gemm_f32.hip -- fused E8 linear on the fp32 matrix instruction (gfx950): fp32
// activations, and the bf16 / fp16 shapes the 16-bit MFMA kernels do not take (K or, for
// the backward, N not a multiple of 64).
//
// v_mfma_f32_16x16x4_f32 contracts four k of a 16 x 16 tile in full fp32: lane (g = lane / 16,
// i = lane % 16) supplies A[i][k_g] and B[k_g][i], one value each.  Which four k an
// instruction takes is free as long as A and B agree, so the eight weights of one code serve
// eight instructions without moving between lanes:
//
//   forward   lane (g, n) decodes code 4 b + g of weight row n (k = 32 b + 8 g + j); the
//             instruction of coordinate j contracts the k of the four lanes g, and the
//             matching A values are the lane's own eight consecutive activations;
//   backward  lane (g, c) decodes code c of weight row n0 + g (columns 8 c + j): instruction
//             j contracts the four rows n and belongs to the output columns {8 c + j}, so a
//             wave owns 128 columns and no transpose is needed.
//
// Decoded weights follow the reference's dtype rule (coord * scales.to(dtype), rounded to
// dtype for 2-bit and 1-bit codes); products and sums are fp32.
//
// Bound: the decode (about 30 VALU per code) and 8 matrix instructions of 32 cycles per 512
// weights and 16 activation rows; the loads are small.  Rows are split over the workgroup's
// waves (LDS reduction), the backward's also over workgroups (fp32 partial sums in the
// caller's workspace), since one 16-row tile is a long serial chain of little work.
// Measured against the 64 x 64 SIMT tiles of e8t_gemm_generic.hip (which decode every weight
// separately, from the flat index, and leave most of the chip idle at few rows), ternary in
// fp32: forward M = 1 of 4096 x 4096 (gs 32) 703 -> 15.9 us, M = 16 of 14336 x 4096 (gs 64)
// 773 -> 58 us; backward dX of the latter 3917 -> 38.6 us with its reduction.  Error against
// 64-bit sums 9e-7 -> 3e-7 (2-norm): each wave's chain is a fraction of K.

#include "e8t_device.h"
#include "e8t_internal.h"
#include "e8t_lut.h"
#include "e8t_root.h"

namespace ojx {

namespace {

// Values that lanes outside the matrix read as their activations.
__device__ const float __attribute__((aligned(16))) kZeros8[8] = {0.f, 0.f, 0.f, 0.f,
                                                                 0.f, 0.f, 0.f, 0.f};

// Table of coordinate quads (float4) per format: ternary the 102 four-digit halves of raw =
// 2 * code (81 of them valid), 2-bit the 256 code bytes, 1-bit two quads per code.
template <int FMT> constexpr int quad_entries() {
    return FMT == kFmtTernary ? 102 : FMT == kFmt2Bit ? 256 : 512;
}

template <int FMT>
__device__ __forceinline__ void fill_quads(float4* tab) {
    for (int e = threadIdx.x; e < quad_entries<FMT>(); e += blockDim.x) {
        float4 v;
        if constexpr (FMT == kFmtTernary) {
            v = make_float4((float)(e % 3 - 1), (float)(e / 3 % 3 - 1), (float)(e / 9 % 3 - 1),
                            (float)(e / 27 % 3 - 1));
        } else if constexpr (FMT == kFmt2Bit) {
            v = make_float4((float)(e & 3) - 1.5f, (float)((e >> 2) & 3) - 1.5f,
                            (float)((e >> 4) & 3) - 1.5f, (float)(e >> 6) - 1.5f);
        } else {
            const int8_t* c = &kRootTable.c[e >> 1][4 * (e & 1)];
            v = make_float4((float)c[0], (float)c[1], (float)c[2], (float)c[3]);
        }
        tab[e] = v;
    }
}

// The codes of one weight row: load(t) fetches the two bytes (1-bit: one) that hold code t,
// code() takes its bits out of them.
template <int FMT>
struct CodeRow {
    const uint8_t* p;
    uint32_t odd;  // ternary: the row starts in the middle of a 3-byte pair

    CodeRow() = default;
    __device__ __forceinline__ CodeRow(const uint8_t* packed, int64_t first) {
        odd = FMT == kFmtTernary ? (uint32_t)(first & 1) : 0u;
        p = packed + (FMT == kFmtTernary ? 3 * (first >> 1) : FMT == kFmt2Bit ? 2 * first : first);
    }
    __device__ __forceinline__ uint32_t load(uint32_t t) const {
        if constexpr (FMT == kFmtRoot) return p[t];
        uint16_t v;
        __builtin_memcpy(&v, p + (FMT == kFmtTernary ? (3u * (t + odd)) >> 1 : 2u * t), 2);
        return v;
    }
    // bits of code t as load() returned them
    __device__ __forceinline__ uint32_t code(uint32_t raw, uint32_t t) const {
        return FMT == kFmtTernary ? (raw >> (4u * ((t + odd) & 1u))) & 0xFFFu : raw;
    }
};

template <int FMT, int DT>
__device__ __forceinline__ void decode8(const float4* tab, uint32_t code, float s, float (&w)[8]) {
    uint32_t i0, i1;
    if constexpr (FMT == kFmtTernary) {
        const uint32_t raw = 2u * code;
        i1 = (raw * 25891u) >> 21;  // raw / 81, exact for raw < 8192
        i0 = raw - 81u * i1;
    } else if constexpr (FMT == kFmt2Bit) {
        i0 = code & 255u;
        i1 = code >> 8;
    } else {
        i0 = 2u * code;
        i1 = i0 + 1u;
    }
    const float4 a = tab[i0], b = tab[i1];
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        w[j] = v[j] * s;
        if constexpr (DT != kF32 && FMT != kFmtTernary) {
            if constexpr (DT == kF16) w[j] = f16_bits_to_f32(f32_to_f16_bits(w[j]));
            else w[j] = bf16_bits_to_f32(bf16_bits_hw(w[j]));
        }
    }
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// n consecutive activations as loaded (fp32: n words, 16-bit: n / 2 words).
template <int DT, int n> struct RawX {
    static constexpr int W = DT == kF32 ? n : n / 2;
    uint32_t w[W];

    __device__ __forceinline__ void load(const char* p) {
        if constexpr (W % 4 == 0) {
#pragma unroll
            for (int i = 0; i < W / 4; ++i) {
                const uint4 v = reinterpret_cast<const uint4*>(p)[i];
                w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
            }
        } else {
            const uint2 v = *reinterpret_cast<const uint2*>(p);
            w[0] = v.x; w[1] = v.y;
        }
    }
    __device__ __forceinline__ float get(int j) const {
        if constexpr (DT == kF32) return __uint_as_float(w[j]);
        const uint32_t h = (w[j / 2] >> (16 * (j & 1))) & 0xFFFFu;
        return DT == kF16 ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
    }
};

template <int DT> constexpr int esize() { return DT == kF32 ? 4 : 2; }

}  // namespace

// y[M, N] = x . W^T (+ bias, + adapter).  MT: 16-row activation tiles per wave, R: 16-row
// weight tiles per wave, NW: waves of the workgroup (they split K), U: 32-k blocks fetched
// together, one group of them ahead of the one being contracted.
template <int FMT, int DT, int MT, int R, int NW, int U>
__global__ __launch_bounds__(64 * NW) void gemm_f32_fwd(
    const void* __restrict__ x, const uint8_t* __restrict__ packed,
    const uint16_t* __restrict__ scales, const void* __restrict__ bias, void* __restrict__ y,
    int64_t M, int64_t N, int64_t K, int gs_shift, LoraEp lora) {
    __shared__ float4 tab[quad_entries<FMT>()];
    __shared__ float red[NW * MT * R * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t n0 = (int64_t)blockIdx.x * (16 * R), m0 = (int64_t)blockIdx.y * (16 * MT);
    fill_quads<FMT>(tab);

    const uint32_t codes = (uint32_t)(K >> 3);  // per row
    const uint32_t blocks = (codes + 3) >> 2, per = (blocks + NW - 1) / NW;
    const uint32_t b_begin = wave * per;
    const uint32_t b_end = b_begin + per < blocks ? b_begin + per : blocks;
    const int ss = gs_shift - 3;  // log2 of the codes per scale group

    CodeRow<FMT> row[R];
    const uint16_t* srow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t n = n0 + 16 * r + i16;
        n = n < N ? n : N - 1;  // rows past N repeat the last one, never stored
        row[r] = CodeRow<FMT>(packed, n * codes);
        srow[r] = scales + n * (K >> gs_shift);
    }
    const char* xrow[MT];
    bool xlive[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int64_t m = m0 + 16 * t + i16;
        xlive[t] = m < M;
        xrow[t] = static_cast<const char*>(x) + (m < M ? m : 0) * K * esize<DT>();
    }

    struct Batch {
        uint32_t code[U][R], sc[U][R];
        RawX<DT, 8> xa[U][MT];
    };
    auto load = [&](Batch& f, uint32_t b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t c = 4 * (b + u) + g;
            const bool live = b + u < b_end && c < codes;
            const uint32_t t = live ? c : 0u;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                f.code[u][r] = row[r].load(t);
                f.sc[u][r] = srow[r][t >> ss];
            }
#pragma unroll
            for (int q = 0; q < MT; ++q)
                f.xa[u][q].load(live && xlive[q] ? xrow[q] + (int64_t)t * (8 * esize<DT>())
                                                 : reinterpret_cast<const char*>(kZeros8));
        }
    };
    f32x4 acc[MT][R];
#pragma unroll
    for (int q = 0; q < MT; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[q][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Batch& f, uint32_t b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t c = 4 * (b + u) + g;
            const bool live = b + u < b_end && c < codes;
            const uint32_t t = live ? c : 0u;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float w[8];
                decode8<FMT, DT>(tab, row[r].code(f.code[u][r], t),
                                 live ? scale_for<DT>(f.sc[u][r]) : 0.f, w);
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int q = 0; q < MT; ++q)
                        acc[q][r] = mfma4(f.xa[u][q].get(j), w[j], acc[q][r]);
            }
        }
    };

    Batch f0, f1;
    load(f0, b_begin);
    __syncthreads();  // table ready
    for (uint32_t b = b_begin; b < b_end; b += 2 * U) {
        load(f1, b + U);
        compute(f0, b);
        load(f0, b + 2 * U);
        if (b + U < b_end) compute(f1, b + U);
    }

    // the waves' partial sums, then one store per output
#pragma unroll
    for (int q = 0; q < MT; ++q)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                red[((wave * MT + q) * R + r) * 256 + 64 * e + lane] = acc[q][r][e];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * R * 256; i += 64 * NW) {
        float v = red[i];
#pragma unroll
        for (int k = 1; k < NW; ++k) v += red[k * (MT * R * 256) + i];
        const int tile = i >> 8, q = tile / R, r = tile % R, e = (i >> 6) & 3, l = i & 63;
        const int64_t m = m0 + 16 * q + 4 * (l >> 4) + e, n = n0 + 16 * r + (l & 15);
        if (m < M && n < N) {
            if (bias) v += load_as_f32<DT>(bias, n);
            store_from_f32<DT>(y, m * N + n, v + lora_term<DT>(lora, m, n));
        }
    }
}

// gx[M, K] = gy . W, or (gridDim.z > 1) the fp32 partial sums of row range blockIdx.z in
// part[z][M][K].  VEC: N % 4 == 0 and gy aligned for loads of four values.
template <int FMT, int DT, int MT, int NW, bool VEC>
__global__ __launch_bounds__(64 * NW) void gemm_f32_bwd(
    const void* __restrict__ gy, const uint8_t* __restrict__ packed,
    const uint16_t* __restrict__ scales, void* __restrict__ gx, float* __restrict__ part,
    int64_t M, int64_t N, int64_t K, int gs_shift) {
    __shared__ float4 tab[quad_entries<FMT>()];
    __shared__ f32x4 red[NW / 2][MT * 8][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t m0 = (int64_t)blockIdx.y * (16 * MT);
    fill_quads<FMT>(tab);

    const uint32_t codes = (uint32_t)(K >> 3);
    const uint32_t c = 16 * blockIdx.x + i16;
    const uint32_t cc = c < codes ? c : codes - 1;  // columns past K are never stored
    const uint32_t sidx = cc >> (gs_shift - 3);
    const int64_t sld = K >> gs_shift;
    const int64_t groups = (N + 15) >> 4;  // 16 rows: four instructions' worth per lane group
    const int64_t parts = (int64_t)gridDim.z * NW, p = (int64_t)blockIdx.z * NW + wave;
    const int64_t q_begin = groups * p / parts, q_end = groups * (p + 1) / parts;

    const char* yrow[MT];
    bool ylive[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int64_t m = m0 + 16 * t + i16;
        ylive[t] = m < M;
        yrow[t] = static_cast<const char*>(gy) + (m < M ? m : 0) * N * esize<DT>();
    }
    struct Batch {
        uint32_t code[4], sc[4], odd;
        RawX<DT, 4> ya[MT];
    };
    // rows n = 16 q + 4 g + s, s = 0..3
    auto load = [&](Batch& f, int64_t q) {
        q = q < q_end ? q : q_end - 1;  // a group past the last is loaded again, never used
        const int64_t n0 = 16 * q + 4 * g;
        f.odd = 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t n = n0 + s < N ? n0 + s : N - 1;
            const CodeRow<FMT> row(packed, n * codes);
            f.code[s] = row.load(cc);
            f.odd |= row.odd << s;
            f.sc[s] = scales[n * sld + sidx];
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if constexpr (VEC) {
                f.ya[t].load(ylive[t] && n0 < N ? yrow[t] + n0 * esize<DT>()
                                                : reinterpret_cast<const char*>(kZeros8));
            } else {
                uint32_t v[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const char* a = ylive[t] && n0 + s < N
                                        ? yrow[t] + (n0 + s) * esize<DT>()
                                        : reinterpret_cast<const char*>(kZeros8);
                    if constexpr (DT == kF32) v[s] = *reinterpret_cast<const uint32_t*>(a);
                    else v[s] = *reinterpret_cast<const uint16_t*>(a);
                }
                if constexpr (DT == kF32) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) f.ya[t].w[s] = v[s];
                } else {
                    f.ya[t].w[0] = v[0] | (v[1] << 16);
                    f.ya[t].w[1] = v[2] | (v[3] << 16);
                }
            }
        }
    };
    f32x4 acc[MT][8];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Batch& f, int64_t q) {
        const int64_t n0 = 16 * q + 4 * g;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t code = f.code[s];
            if constexpr (FMT == kFmtTernary)
                code = (code >> (4u * ((cc + ((f.odd >> s) & 1u)) & 1u))) & 0xFFFu;
            float w[8];
            decode8<FMT, DT>(tab, code, n0 + s < N ? scale_for<DT>(f.sc[s]) : 0.f, w);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t][j] = mfma4(f.ya[t].get(s), w[j], acc[t][j]);
        }
    };

    Batch f0, f1;
    if (q_begin < q_end) load(f0, q_begin);
    __syncthreads();  // table ready
    for (int64_t q = q_begin; q < q_end; q += 2) {
        load(f1, q + 1);
        compute(f0, q);
        load(f0, q + 2);
        if (q + 1 < q_end) compute(f1, q + 1);
    }

    // the waves' sums, halving: waves [h, 2h) hand theirs to waves [0, h)
#pragma unroll
    for (int h = NW / 2; h >= 1; h /= 2) {
        if (wave >= h && wave < 2 * h) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int j = 0; j < 8; ++j) red[wave - h][8 * t + j][lane] = acc[t][j];
        }
        __syncthreads();
        if (wave < h) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[t][j] += red[wave][8 * t + j][lane];
        }
        __syncthreads();
    }
    if (wave != 0 || c >= codes) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t m = m0 + 16 * t + 4 * g + e;
            if (m >= M) continue;
            const int64_t at = m * K + 8 * (int64_t)c;
            if (gridDim.z > 1) {
                float* o = part + blockIdx.z * split_stride(M, K) + at;
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = acc[t][j][e];
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) store_from_f32<DT>(gx, at + j, acc[t][j][e]);
            }
        }
    }
}

// ------------------------------------------------------------------ host side

bool gemm_f32_supported(const void* x, const uint8_t* packed, const uint16_t* scales, int64_t M,
                        int64_t N, int64_t K, int64_t gs, int fmt, bool bwd) {
    // rows hold whole codes and whole scale groups of 2^t >= 8 weights (a ternary group is a
    // multiple of 16); the kernels index a row's codes and the grid in 32 bits
    if (gs < 8 || (gs & (gs - 1)) != 0 || gs > (1ll << 30) || K < gs || K % gs != 0) return false;
    if (M < 1 || N < 1 || K >= (1ll << 31) || N >= (1ll << 31) || (M + 15) / 16 > 65535)
        return false;
    // 16-byte loads of eight activations along K (the backward picks its loads by N)
    if (!bwd && ((uintptr_t)x & 15u)) return false;
    if (bwd && ((uintptr_t)x & 3u)) return false;
    return ((uintptr_t)scales & 1u) == 0;
}

// Row splits of the backward over workgroups: towards kF32Waves waves on the chip (two per
// SIMD), while every wave keeps at least four groups of 16 rows.
constexpr int64_t kF32Waves = 2048;
constexpr int kF32BwdWaves = 8;

static int f32_row_tiles(int64_t M) { return M <= 16 ? 1 : M <= 32 ? 2 : 4; }
static int f32_bwd_waves(int mt) { return mt == 4 ? kF32BwdWaves / 2 : kF32BwdWaves; }

int gemm_f32_bwd_splits(int64_t M, int64_t N, int64_t K) {
    const int mt = f32_row_tiles(M), nw = f32_bwd_waves(mt);
    const int64_t wgs = ((K + 127) / 128) * ((M + 16 * mt - 1) / (16 * mt));
    int64_t s = (kF32Waves / nw + wgs - 1) / wgs;
    const int64_t most = ((N + 15) / 16) / (4 * nw);
    if (s > most) s = most;
    if (s > 16) s = 16;
    return s < 1 ? 1 : (int)s;
}

template <int FMT, int DT, int MT, int R, int NW, int U>
static hipError_t launch_f32_fwd_cfg(const void* x, const uint8_t* packed, const uint16_t* scales,
                                     const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                                     int gs_shift, hipStream_t s, const LoraEp& lora) {
    const dim3 grid((unsigned)((N + 16 * R - 1) / (16 * R)),
                    (unsigned)((M + 16 * MT - 1) / (16 * MT)));
    hipLaunchKernelGGL((gemm_f32_fwd<FMT, DT, MT, R, NW, U>), grid, dim3(64 * NW), 0, s, x, packed,
                       scales, bias, y, M, N, K, gs_shift, lora);
    return hipGetLastError();
}

template <int FMT, int DT>
static hipError_t launch_f32_fwd_t(const void* x, const uint8_t* packed, const uint16_t* scales,
                                   const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                                   int sh, hipStream_t s, const LoraEp& lora) {
    const int mt = f32_row_tiles(M);
    const int64_t tiles = (N + 15) / 16;
    if (mt == 1) {
        if (tiles >= 512)
            return launch_f32_fwd_cfg<FMT, DT, 1, 2, 8, 4>(x, packed, scales, bias, y, M, N, K, sh,
                                                           s, lora);
        return launch_f32_fwd_cfg<FMT, DT, 1, 1, 8, 4>(x, packed, scales, bias, y, M, N, K, sh, s,
                                                       lora);
    }
    if (mt == 2)
        return launch_f32_fwd_cfg<FMT, DT, 2, 2, 8, 2>(x, packed, scales, bias, y, M, N, K, sh, s,
                                                       lora);
    if (tiles * ((M + 63) / 64) >= 1024)
        return launch_f32_fwd_cfg<FMT, DT, 4, 4, 4, 1>(x, packed, scales, bias, y, M, N, K, sh, s,
                                                       lora);
    return launch_f32_fwd_cfg<FMT, DT, 4, 2, 8, 1>(x, packed, scales, bias, y, M, N, K, sh, s,
                                                   lora);
}

template <int FMT, int DT, int MT, int NW>
static hipError_t launch_f32_bwd_cfg(const void* gy, const uint8_t* packed,
                                     const uint16_t* scales, void* gx, float* part, int splits,
                                     int64_t M, int64_t N, int64_t K, int sh, hipStream_t s) {
    const dim3 grid((unsigned)((K + 127) / 128), (unsigned)((M + 16 * MT - 1) / (16 * MT)),
                    (unsigned)splits);
    if (N % 4 == 0 && ((uintptr_t)gy & (DT == kF32 ? 15u : 7u)) == 0)
        hipLaunchKernelGGL((gemm_f32_bwd<FMT, DT, MT, NW, true>), grid, dim3(64 * NW), 0, s, gy,
                           packed, scales, gx, part, M, N, K, sh);
    else
        hipLaunchKernelGGL((gemm_f32_bwd<FMT, DT, MT, NW, false>), grid, dim3(64 * NW), 0, s, gy,
                           packed, scales, gx, part, M, N, K, sh);
    const hipError_t e = hipGetLastError();
    if (splits == 1 || e != hipSuccess) return e;
    return launch_split_reduce(part, splits, nullptr, gx, M, K, DT, s, LoraEp{});
}

template <int FMT, int DT>
static hipError_t launch_f32_bwd_t(const void* gy, const uint8_t* packed, const uint16_t* scales,
                                   void* gx, float* part, int splits, int64_t M, int64_t N,
                                   int64_t K, int sh, hipStream_t s) {
    switch (f32_row_tiles(M)) {
    case 1:
        return launch_f32_bwd_cfg<FMT, DT, 1, kF32BwdWaves>(gy, packed, scales, gx, part, splits, M,
                                                            N, K, sh, s);
    case 2:
        return launch_f32_bwd_cfg<FMT, DT, 2, kF32BwdWaves>(gy, packed, scales, gx, part, splits, M,
                                                            N, K, sh, s);
    default:
        return launch_f32_bwd_cfg<FMT, DT, 4, kF32BwdWaves / 2>(gy, packed, scales, gx, part,
                                                                splits, M, N, K, sh, s);
    }
}

static int log2_of(int64_t v) { return 63 - __builtin_clzll((unsigned long long)v); }

template <int FMT>
static hipError_t f32_fwd_fmt(const void* x, const uint8_t* packed, const uint16_t* scales,
                              const void* bias, void* y, int64_t M, int64_t N, int64_t K, int sh,
                              int dt, hipStream_t s, const LoraEp& lora) {
    switch (dt) {
    case kF32:
        return launch_f32_fwd_t<FMT, kF32>(x, packed, scales, bias, y, M, N, K, sh, s, lora);
    case kF16:
        return launch_f32_fwd_t<FMT, kF16>(x, packed, scales, bias, y, M, N, K, sh, s, lora);
    default:
        return launch_f32_fwd_t<FMT, kBF16>(x, packed, scales, bias, y, M, N, K, sh, s, lora);
    }
}

template <int FMT>
static hipError_t f32_bwd_fmt(const void* gy, const uint8_t* packed, const uint16_t* scales,
                              void* gx, float* part, int splits, int64_t M, int64_t N, int64_t K,
                              int sh, int dt, hipStream_t s) {
    switch (dt) {
    case kF32:
        return launch_f32_bwd_t<FMT, kF32>(gy, packed, scales, gx, part, splits, M, N, K, sh, s);
    case kF16:
        return launch_f32_bwd_t<FMT, kF16>(gy, packed, scales, gx, part, splits, M, N, K, sh, s);
    default:
        return launch_f32_bwd_t<FMT, kBF16>(gy, packed, scales, gx, part, splits, M, N, K, sh, s);
    }
}

hipError_t launch_gemm_f32_fwd(const void* x, const uint8_t* packed, const uint16_t* scales,
                               const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                               int64_t gs, int dt, hipStream_t s, int fmt, const LoraEp& lora) {
    const int sh = log2_of(gs);
    if (fmt == kFmtRoot)
        return f32_fwd_fmt<kFmtRoot>(x, packed, scales, bias, y, M, N, K, sh, dt, s, lora);
    if (fmt == kFmt2Bit)
        return f32_fwd_fmt<kFmt2Bit>(x, packed, scales, bias, y, M, N, K, sh, dt, s, lora);
    return f32_fwd_fmt<kFmtTernary>(x, packed, scales, bias, y, M, N, K, sh, dt, s, lora);
}

hipError_t launch_gemm_f32_bwd(const void* gy, const uint8_t* packed, const uint16_t* scales,
                               void* gx, float* part, int splits, int64_t M, int64_t N, int64_t K,
                               int64_t gs, int dt, hipStream_t s, int fmt) {
    const int sh = log2_of(gs);
    if (fmt == kFmtRoot)
        return f32_bwd_fmt<kFmtRoot>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s);
    if (fmt == kFmt2Bit)
        return f32_bwd_fmt<kFmt2Bit>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s);
    return f32_bwd_fmt<kFmtTernary>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s);
}

}  // namespace ojx
