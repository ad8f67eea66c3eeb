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
// Bound: loads' round trips in launches of one or two workgroups per CU (22 to 43% of the wave
// cycles wait), beside the 8 matrix instructions of 32 cycles per 512 weights and 16 activation
// rows (12.5 us for M = 16 of 14336 x 4096, 34 to 37% of the cycles) and the decode's 20-30 VALU
// per code (17%).  The backward also reads its codes 6.5 times: a workgroup's 128 columns take 24
// bytes of each 128-byte line.  Rows are split over the
// workgroup's waves (LDS reduction), the backward's also over workgroups (fp32 partial sums
// in the caller's workspace), since one 16-row tile is a long serial chain of little work.
// Measured against the 64 x 64 SIMT tiles of e8t_gemm_generic.hip (which decode every weight
// separately, from the flat index, and leave most of the chip idle at few rows), ternary
// gs 32 in fp32, us from a graph: forward M = 1 of 4096 x 4096 706 -> 9, M = 16 of 14336 x 4096
// 742 -> 30, M = 64 816 -> 83; backward dX (with its reduction) M = 1 of 4096 x 4096 849 ->
// 14.6, M = 16 of 14336 x 4096 3940 -> 33, M = 64 4595 -> 83.  Error against 64-bit sums
// 9e-7 -> 3e-7 (2-norm): each wave's chain is a fraction of K.

#include "e8t_device.h"
#include "e8t_f32.h"
#include "e8t_internal.h"
#include "e8t_lut.h"
#include "e8t_root.h"

namespace ojx {

namespace {

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

// Code t of a row (rows start on a byte: a ternary row holds whole pairs of codes, K % 16 ==
// 0) lies in the two bytes (1-bit: one) from code_byte(t); code_of takes its bits from them.
template <int FMT> __device__ __forceinline__ uint32_t code_byte(uint32_t t) {
    return FMT == kFmtTernary ? (3u * t) >> 1 : FMT == kFmt2Bit ? 2u * t : t;
}
template <int FMT> __device__ __forceinline__ uint32_t code_of(uint32_t raw, uint32_t t) {
    return FMT == kFmtTernary ? (raw >> (4u * (t & 1u))) & 0xFFFu : raw;
}
template <int FMT> __host__ __device__ constexpr int64_t row_bytes(int64_t codes) {
    return FMT == kFmtTernary ? 3 * codes / 2 : FMT == kFmt2Bit ? 2 * codes : codes;
}

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

}  // namespace

// The waves' partial sums (acc: this wave's tiles, through `red`), then one store per output.
template <int DT, int MT, int R, int NW>
__device__ __forceinline__ void f32_fwd_store(f32x4 (&acc)[MT][R], float* red,
                                              const void* bias, void* y, int64_t M, int64_t N,
                                              int64_t m0, int64_t n0, const LoraEp& lora) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lora.r > 0 && wave == 0)
        lora_add<DT, MT, R>(acc, lora, m0, M, N, lane,
                            [&](int r) { return n0 + 16 * r + (lane & 15); });
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
            store_from_f32<DT>(y, m * N + n, v);
        }
    }
}

// y[M, N] = x . W^T (+ bias, + adapter).  MT: 16-row activation tiles per wave, R: 16-row
// weight tiles per wave, NW: waves of the workgroup (they split K), U: 32-k blocks fetched
// together, one group of them ahead of the one being contracted.  This form reads every code
// and scale on its own, so it takes any row length.
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

    const uint8_t* row[R];
    const uint16_t* srow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t n = n0 + 16 * r + i16;
        n = n < N ? n : N - 1;  // rows past N repeat the last one, never stored
        row[r] = packed + n * row_bytes<FMT>(codes);
        srow[r] = scales + n * (K >> gs_shift);
    }
    // activation rows m0 ..: rows past M lie past the buffer's end and read zeros
    const __amdgpu_buffer_rsrc_t xr = rows_buffer<DT>(x, m0, M, K, 16 * MT);
    uint32_t xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = (uint32_t)(16 * t + i16) * (uint32_t)K * esize<DT>();

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
                f.code[u][r] = 0;
                __builtin_memcpy(&f.code[u][r], row[r] + code_byte<FMT>(t),
                                 FMT == kFmtRoot ? 1 : 2);
                f.sc[u][r] = srow[r][t >> ss];
            }
#pragma unroll
            for (int q = 0; q < MT; ++q)
                f.xa[u][q].load(xr, live ? xrow[q] + t * (8 * esize<DT>()) : kNoRecordOffset);
        }
    };
    // a wave with one tile alternates between two accumulators: back-to-back instructions
    // then never wait for each other's result
    constexpr int NA = MT * R == 1 ? 2 : 1;
    f32x4 acc[NA][MT][R];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int q = 0; q < MT; ++q)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[a][q][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Batch& f, uint32_t b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t c = 4 * (b + u) + g;
            const bool live = b + u < b_end && c < codes;
            const uint32_t t = live ? c : 0u;
            float w[R][8];
#pragma unroll
            for (int r = 0; r < R; ++r)
                decode8<FMT, DT>(tab, code_of<FMT>(f.code[u][r], t),
                                 live ? scale_for<DT>(f.sc[u][r]) : 0.f, w[r]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int q = 0; q < MT; ++q)
                        acc[j % NA][q][r] =
                            mfma4(f.xa[u][q].get(j), w[r][j], acc[j % NA][q][r]);
        }
    };

    // the loads of a batch all go out before the previous batch is contracted (left to
    // itself the scheduler sinks them towards their uses)
    Batch f0, f1;
    load(f0, b_begin);
    __syncthreads();  // table ready
    for (uint32_t b = b_begin; b < b_end; b += 2 * U) {
        load(f1, b + U);
        __builtin_amdgcn_sched_barrier(0);
        compute(f0, b);
        load(f0, b + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        if (b + U < b_end) compute(f1, b + U);
    }
    if constexpr (NA == 2) acc[0][0][0] += acc[NA - 1][0][0];

    f32_fwd_store<DT, MT, R, NW>(acc[0], red, bias, y, M, N, m0, n0, lora);
}

// The same product where rows hold whole 4-byte words of codes and scales (f32_wide_ok): a
// lane loads the eight consecutive codes 8 g .. 8 g + 7 of its row's 256-k chunk, and their
// scales, in one load each, and a 4 x 4 transpose over the lane groups hands it the codes
// 4 u + g, u = 0..7, that its activations belong to (activations are best read four lanes to a
// 128-byte line).  Codes and scales run one chunk ahead, activations XU blocks ahead.
// The two-byte loads and their addresses bound the form above: M = 1 / 16 of 14336 x 4096
// (ternary, gs 32) 45 / 56 us there and 25 / 30 here, M = 512 of 4096 x 4096 195 and 160.
// The transpose: register q of lane group g holds entries (q, q + 4 in the high half) of the
// group's eight; afterwards register q holds entry 4 (2 q + h) + g, h the half.
__device__ __forceinline__ void transpose_groups(uint32_t (&q)[4]) {
    auto s = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false);
    q[0] = s[0]; q[2] = s[1];
    s = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
    q[1] = s[0]; q[3] = s[1];
    s = __builtin_amdgcn_permlane16_swap(q[0], q[1], false, false);
    q[0] = s[0]; q[1] = s[1];
    s = __builtin_amdgcn_permlane16_swap(q[2], q[3], false, false);
    q[2] = s[0]; q[3] = s[1];
}

// A lane's eight codes as loaded, and as 16-bit pairs (t, t + 4).
template <int FMT> struct WideRow {
    static constexpr int W = FMT == kFmtTernary ? 3 : FMT == kFmt2Bit ? 4 : 2;
    static constexpr uint32_t kBytes = 4 * W;  // of eight codes
    uint32_t d[W];

    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, uint32_t vo) {
        if constexpr (W == 3) {
            const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(b, vo, 0, 0);
            d[0] = v.x; d[1] = v.y; d[2] = v.z;
        } else if constexpr (W == 4) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, vo, 0, 0);
            d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
        } else {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b, vo, 0, 0);
            d[0] = v.x; d[1] = v.y;
        }
    }
    __device__ __forceinline__ void pairs(uint32_t (&q)[4]) const {
        if constexpr (FMT == kFmtTernary) {
            const uint32_t c2 = __builtin_amdgcn_alignbit(d[1], d[0], 24) & 0xFFFu;
            const uint32_t c5 = __builtin_amdgcn_alignbit(d[2], d[1], 28) & 0xFFFu;
            q[0] = (d[0] & 0xFFFu) | (d[1] & 0x0FFF0000u);
            q[1] = ((d[0] >> 12) & 0xFFFu) | (c5 << 16);
            q[2] = c2 | ((d[2] << 8) & 0x0FFF0000u);
            q[3] = ((d[1] >> 4) & 0xFFFu) | ((d[2] >> 4) & 0x0FFF0000u);
        } else if constexpr (FMT == kFmt2Bit) {
            q[0] = __builtin_amdgcn_perm(d[2], d[0], 0x05040100u);
            q[1] = __builtin_amdgcn_perm(d[2], d[0], 0x07060302u);
            q[2] = __builtin_amdgcn_perm(d[3], d[1], 0x05040100u);
            q[3] = __builtin_amdgcn_perm(d[3], d[1], 0x07060302u);
        } else {
            q[0] = __builtin_amdgcn_perm(d[1], d[0], 0x0C040C00u);
            q[1] = __builtin_amdgcn_perm(d[1], d[0], 0x0C050C01u);
            q[2] = __builtin_amdgcn_perm(d[1], d[0], 0x0C060C02u);
            q[3] = __builtin_amdgcn_perm(d[1], d[0], 0x0C070C03u);
        }
    }
};

// The scales of a lane's eight codes, GS weights to a scale (64: 64 or more, one scale).
template <int GS> struct WideScale {
    static constexpr int W = GS >= 32 ? 1 : 32 / GS;  // words: 1, 2 (gs 16), 4 (gs 8)
    uint32_t d[W];

    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, uint32_t vo) {
        if constexpr (GS >= 64) {
            d[0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b, vo, 0, 0);
        } else if constexpr (W == 1) {
            d[0] = __builtin_amdgcn_raw_buffer_load_b32(b, vo, 0, 0);
        } else if constexpr (W == 2) {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b, vo, 0, 0);
            d[0] = v.x; d[1] = v.y;
        } else {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, vo, 0, 0);
            d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
        }
    }
    __device__ __forceinline__ void pairs(uint32_t (&q)[4]) const {
        if constexpr (GS >= 64) {
            q[0] = q[1] = q[2] = q[3] = d[0] * 0x10001u;
        } else if constexpr (GS == 32) {  // the scales of codes 0..3 and 4..7
            q[0] = q[1] = q[2] = q[3] = d[0];
        } else if constexpr (GS == 16) {
            q[0] = q[1] = __builtin_amdgcn_perm(d[1], d[0], 0x05040100u);
            q[2] = q[3] = __builtin_amdgcn_perm(d[1], d[0], 0x07060302u);
        } else {
            q[0] = __builtin_amdgcn_perm(d[2], d[0], 0x05040100u);
            q[1] = __builtin_amdgcn_perm(d[2], d[0], 0x07060302u);
            q[2] = __builtin_amdgcn_perm(d[3], d[1], 0x05040100u);
            q[3] = __builtin_amdgcn_perm(d[3], d[1], 0x07060302u);
        }
    }
};

template <int FMT, int DT, int GS, int MT, int R, int NW, int XU>
__global__ __launch_bounds__(64 * NW) void gemm_f32_fwd_wide(
    const void* __restrict__ x, const uint8_t* __restrict__ packed,
    const uint16_t* __restrict__ scales, const void* __restrict__ bias, void* __restrict__ y,
    int64_t M, int64_t N, int64_t K, int gs_shift, LoraEp lora) {
    using Row = WideRow<FMT>;
    __shared__ float4 tab[quad_entries<FMT>()];
    __shared__ float red[NW * MT * R * 256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t n0 = (int64_t)blockIdx.x * (16 * R), m0 = (int64_t)blockIdx.y * (16 * MT);

    const int codes = (int)(K >> 3);  // per row
    const int chunks = (codes + 31) >> 5, per = (chunks + NW - 1) / NW;
    const int c_begin = wave * per;
    const int c_end = c_begin + per < chunks ? c_begin + per : chunks;

    // the workgroup's rows of codes and scales; rows past N lie past the end and read zeros
    const int64_t left = N - n0 < 16 * R ? N - n0 : 16 * R;
    const uint32_t rowbytes = (uint32_t)row_bytes<FMT>(codes);
    const uint32_t srowbytes = (uint32_t)(K >> gs_shift) * 2;
    const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(packed + n0 * rowbytes), (short)0, (int)(left * rowbytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(scales) + n0 * srowbytes), (short)0,
        (int)(left * srowbytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t xr = rows_buffer<DT>(x, m0, M, K, 16 * MT);

    Row cd[R];
    WideScale<GS> sc[R];
    auto load_w = [&](int ch) {  // a chunk past the last reads zeros or a later row, unused
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t row = 16 * r + i16, c = 32 * ch + 8 * g;
            cd[r].load(pr, row * rowbytes + (c >> 3) * Row::kBytes);
            sc[r].load(sr, row * srowbytes + ((c << 3) >> gs_shift) * 2);
        }
    };
    struct XBatch { RawX<DT, 8> a[XU][MT]; };
    auto load_x = [&](XBatch& f, int ch, int u0) {
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int c = 32 * ch + 4 * (u0 + u) + g;
            const bool live = c < codes && ch < c_end;
#pragma unroll
            for (int q = 0; q < MT; ++q)
                f.a[u][q].load(xr, live ? (uint32_t)((16 * q + i16) * codes + c) * (8 * esize<DT>())
                                        : kNoRecordOffset);
        }
    };
    // one tile per wave: two accumulators, so that instructions in a row never wait for each
    // other's result
    constexpr int NA = MT * R == 1 ? 2 : 1;
    f32x4 acc[NA][MT][R];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int q = 0; q < MT; ++q)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[a][q][r] = f32x4{0.f, 0.f, 0.f, 0.f};

    XBatch xb[2];
    load_w(c_begin);
    load_x(xb[0], c_begin, 0);
    fill_quads<FMT>(tab);
    __syncthreads();  // table ready
    for (int ch = c_begin; ch < c_end; ++ch) {
        uint32_t cq[R][4], sq[R][4];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            cd[r].pairs(cq[r]);
            sc[r].pairs(sq[r]);
            transpose_groups(cq[r]);
            transpose_groups(sq[r]);
        }
        load_w(ch + 1);
#pragma unroll
        for (int u0 = 0; u0 < 8; u0 += XU) {
            const XBatch& xc = xb[(u0 / XU) & 1];
            load_x(xb[(u0 / XU + 1) & 1], u0 + XU < 8 ? ch : ch + 1, (u0 + XU) & 7);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out before the contraction
#pragma unroll
            for (int u = 0; u < XU; ++u) {
                const int e = u0 + u;
                const bool live = 32 * ch + 4 * e + g < codes;
                float w[R][8];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t code = e & 1 ? cq[r][e >> 1] >> 16 : cq[r][e >> 1] & 0xFFFFu;
                    const uint32_t s16 = e & 1 ? sq[r][e >> 1] >> 16 : sq[r][e >> 1] & 0xFFFFu;
                    decode8<FMT, DT>(tab, code, live ? scale_for<DT>(s16) : 0.f, w[r]);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int q = 0; q < MT; ++q)
                            acc[j % NA][q][r] =
                                mfma4(xc.a[u][q].get(j), w[r][j], acc[j % NA][q][r]);
            }
        }
    }
    if constexpr (NA == 2) acc[0][0][0] += acc[NA - 1][0][0];
    f32_fwd_store<DT, MT, R, NW>(acc[0], red, bias, y, M, N, m0, n0, lora);
}

// gx[M, K] = gy . W, or (gridDim.z > 1) the fp32 partial sums of row range blockIdx.z in
// part[z][M][K].  VEC: N % 4 == 0 and gy aligned for loads of four values.
template <int FMT, int DT, int MT, int NW, bool VEC>
__global__ __launch_bounds__(64 * NW, 2) void gemm_f32_bwd(
    const void* __restrict__ gy, const uint8_t* __restrict__ packed,
    const uint16_t* __restrict__ scales, void* __restrict__ gx, float* __restrict__ part,
    int64_t M, int64_t N, int64_t K, int gs_shift, LoraEp lora) {
    __shared__ float4 tab[quad_entries<FMT>()];
    __shared__ f32x4 red[NW / 2][MT * 8][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t m0 = (int64_t)blockIdx.y * (16 * MT);

    const uint32_t codes = (uint32_t)(K >> 3);
    const uint32_t c = 16 * blockIdx.x + i16;
    const uint32_t cc = c < codes ? c : codes - 1;  // columns past K are never stored
    const int groups = (int)((N + 15) >> 4);  // 16 rows: four instructions per lane group
    const int parts = gridDim.z * NW, p = blockIdx.z * NW + wave;
    const int q_begin = (int)((int64_t)groups * p / parts);
    const int q_end = (int)((int64_t)groups * (p + 1) / parts);

    // rows past N lie past the buffers' ends: zero codes, zero scales
    const uint32_t rowbytes = (uint32_t)row_bytes<FMT>(codes);
    const uint32_t srowbytes = (uint32_t)(K >> gs_shift) * 2;
    const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)packed, (short)0, (int)(N * rowbytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)scales, (short)0, (int)(N * srowbytes), kRsrcWord3);
    uint32_t vo_code[4], vo_scale[4];  // of row 4 g + s of a group, column code c
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        vo_code[s] = (4 * g + s) * rowbytes + code_byte<FMT>(cc);
        vo_scale[s] = (4 * g + s) * srowbytes + (cc >> (gs_shift - 3)) * 2;
    }

    const __amdgpu_buffer_rsrc_t yr = rows_buffer<DT>(gy, m0, M, N, 16 * MT);
    uint32_t yrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) yrow[t] = (uint32_t)(16 * t + i16) * (uint32_t)N * esize<DT>();
    struct Batch {
        uint32_t code[4], sc[4];
        RawX<DT, 4> ya[MT];
    };
    // rows n = 16 q + 4 g + s, s = 0..3
    auto load = [&](Batch& f, int q) {
        q = q < q_end ? q : q_end - 1;  // a group past the last is loaded again, never used
        const int64_t n0 = 16 * (int64_t)q + 4 * g;
        const int so = uniform_offset(16 * (int64_t)q * rowbytes);
        const int ss = uniform_offset(16 * (int64_t)q * srowbytes);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if constexpr (FMT == kFmtRoot)
                f.code[s] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(pr, vo_code[s], so, 0);
            else
                f.code[s] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(pr, vo_code[s], so, 0);
            f.sc[s] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr, vo_scale[s], ss, 0);
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if constexpr (VEC) {
                f.ya[t].load(yr, n0 < N ? yrow[t] + (uint32_t)n0 * esize<DT>() : kNoRecordOffset);
            } else {
                uint32_t v[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t vo =
                        n0 + s < N ? yrow[t] + (uint32_t)(n0 + s) * esize<DT>() : kNoRecordOffset;
                    if constexpr (DT == kF32) v[s] = __builtin_amdgcn_raw_buffer_load_b32(yr, vo, 0, 0);
                    else v[s] = __builtin_amdgcn_raw_buffer_load_b16(yr, vo, 0, 0);
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
    auto compute = [&](const Batch& f) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            float w[8];
            decode8<FMT, DT>(tab, code_of<FMT>(f.code[s], cc), scale_for<DT>(f.sc[s]), w);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t][j] = mfma4(f.ya[t].get(s), w[j], acc[t][j]);
        }
    };

    Batch f0, f1;
    if (q_begin < q_end) load(f0, q_begin);
    fill_quads<FMT>(tab);
    __syncthreads();  // table ready
    for (int q = q_begin; q < q_end; q += 2) {
        load(f1, q + 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(f0);
        load(f0, q + 2);
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1 < q_end) compute(f1);
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
    if (wave != 0) return;
    if (lora.r > 0)
        lora_add<DT, MT, 8>(acc, lora, m0, M, K, lane, [&](int j) { return 8 * (int64_t)c + j; },
                            blockIdx.z, gridDim.z);
    if (c >= codes) return;
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
    // multiple of 16); 64 activation rows stay below 2^31 bytes (32-bit buffer offsets)
    if (gs < 8 || (gs & (gs - 1)) != 0 || gs > (1ll << 30) || K < gs || K % gs != 0) return false;
    if (M < 1 || N < 1 || K >= (1ll << 23) || N >= (bwd ? 1ll << 23 : 1ll << 31) ||
        (M + 15) / 16 > 65535)
        return false;
    // 16-byte loads of eight activations along K (the backward picks its loads by N)
    if (!bwd && ((uintptr_t)x & 15u)) return false;
    // the backward addresses whole weight buffers in 32 bits, a group of rows past the end
    if (bwd && (N + 16) * (K / 4) >= (1ll << 31)) return false;
    if (bwd && (N + 16) * (K / gs * 2) >= (1ll << 31)) return false;
    if (bwd && ((uintptr_t)x & 3u)) return false;
    return ((uintptr_t)scales & 1u) == 0;
}

// Row splits of the backward over workgroups: towards kF32Waves waves on the chip (four per
// SIMD; with two, M = 1 and 16 of 14336 x 4096 took 33.3 and 34.9 us against 30.1 and 32.7),
// while every wave keeps at least four groups of 16 rows.
constexpr int64_t kF32Waves = 4096;
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

// Rows of whole 4-byte words: codes 12 (ternary), 16 (2-bit) or 8 (1-bit) bytes per 64
// weights, and scales of two bytes (groups of 64 and more are read one scale at a time).
static bool f32_wide_ok(const uint8_t* packed, const uint16_t* scales, int64_t K, int64_t gs,
                        int fmt) {
    const int64_t row16 = K / 16 * (fmt == kFmtTernary ? 3 : fmt == kFmt2Bit ? 4 : 2);
    return K % 16 == 0 && row16 % 4 == 0 && (gs >= 64 || (K / gs) % 2 == 0) &&
           (((uintptr_t)packed | (uintptr_t)scales) & 3u) == 0;
}

template <int FMT, int DT, int MT, int R, int NW>
static hipError_t launch_f32_fwd_cfg(const void* x, const uint8_t* packed, const uint16_t* scales,
                                     const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                                     int sh, hipStream_t s, const LoraEp& lora) {
    constexpr int XU = MT == 4 ? 1 : 2;
    const dim3 grid((unsigned)((N + 16 * R - 1) / (16 * R)),
                    (unsigned)((M + 16 * MT - 1) / (16 * MT)));
#define OJX_LAUNCH(...)                                                                          \
    hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(64 * NW), 0, s, x, packed, scales, bias, y, M,  \
                       N, K, sh, lora)
    if (!f32_wide_ok(packed, scales, K, (int64_t)1 << sh, FMT))
        OJX_LAUNCH(gemm_f32_fwd<FMT, DT, MT, R, NW, XU>);
    else if (sh >= 6)
        OJX_LAUNCH(gemm_f32_fwd_wide<FMT, DT, 64, MT, R, NW, XU>);
    else if (sh == 5)
        OJX_LAUNCH(gemm_f32_fwd_wide<FMT, DT, 32, MT, R, NW, XU>);
    else if (sh == 4)
        OJX_LAUNCH(gemm_f32_fwd_wide<FMT, DT, 16, MT, R, NW, XU>);
    else if constexpr (FMT != kFmtTernary)  // ternary groups are multiples of 16
        OJX_LAUNCH(gemm_f32_fwd_wide<FMT, DT, 8, MT, R, NW, XU>);
#undef OJX_LAUNCH
    return hipGetLastError();
}

template <int FMT, int DT>
static hipError_t launch_f32_fwd_t(const void* x, const uint8_t* packed, const uint16_t* scales,
                                   const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                                   int sh, hipStream_t s, const LoraEp& lora) {
    // Weight tiles per wave: one while that leaves at most two workgroups per CU, then two,
    // which share the activations' loads (M = 16, ternary gs 32: 4096 x 4096 12.5 against
    // 16.3 us, 14336 x 4096 39.8 against 29.7; four tiles 28.4 and 29.7).  Eight waves share
    // a row's K (4 and 16 waves: 10.4 and 9.1 against 9.1 us at M = 1 of 4096 x 4096); at
    // M > 32 a wave's matrix work is long enough for four (M = 512 148.8 against 155.7 us).
    const int mt = f32_row_tiles(M);
    const int64_t wgs = (N + 15) / 16 * ((M + 16 * mt - 1) / (16 * mt));
    auto cfg = mt == 1   ? (wgs >= 512 ? launch_f32_fwd_cfg<FMT, DT, 1, 2, 8>
                                       : launch_f32_fwd_cfg<FMT, DT, 1, 1, 8>)
               : mt == 2 ? (wgs >= 512 ? launch_f32_fwd_cfg<FMT, DT, 2, 2, 8>
                                       : launch_f32_fwd_cfg<FMT, DT, 2, 1, 8>)
                         : (wgs >= 512 ? launch_f32_fwd_cfg<FMT, DT, 4, 2, 4>
                                       : launch_f32_fwd_cfg<FMT, DT, 4, 1, 8>);
    return cfg(x, packed, scales, bias, y, M, N, K, sh, s, lora);
}

template <int FMT, int DT, int MT, int NW>
static hipError_t launch_f32_bwd_cfg(const void* gy, const uint8_t* packed,
                                     const uint16_t* scales, void* gx, float* part, int splits,
                                     int64_t M, int64_t N, int64_t K, int sh, hipStream_t s,
                                     const LoraEp& lora) {
    const dim3 grid((unsigned)((K + 127) / 128), (unsigned)((M + 16 * MT - 1) / (16 * MT)),
                    (unsigned)splits);
    if (N % 4 == 0 && ((uintptr_t)gy & (DT == kF32 ? 15u : 7u)) == 0)
        hipLaunchKernelGGL((gemm_f32_bwd<FMT, DT, MT, NW, true>), grid, dim3(64 * NW), 0, s, gy,
                           packed, scales, gx, part, M, N, K, sh, lora);
    else
        hipLaunchKernelGGL((gemm_f32_bwd<FMT, DT, MT, NW, false>), grid, dim3(64 * NW), 0, s, gy,
                           packed, scales, gx, part, M, N, K, sh, lora);
    const hipError_t e = hipGetLastError();
    if (splits == 1 || e != hipSuccess) return e;
    return launch_split_reduce(part, splits, nullptr, gx, M, K, DT, s);
}

template <int FMT, int DT>
static hipError_t launch_f32_bwd_t(const void* gy, const uint8_t* packed, const uint16_t* scales,
                                   void* gx, float* part, int splits, int64_t M, int64_t N,
                                   int64_t K, int sh, hipStream_t s, const LoraEp& lora) {
    switch (f32_row_tiles(M)) {
    case 1:
        return launch_f32_bwd_cfg<FMT, DT, 1, kF32BwdWaves>(gy, packed, scales, gx, part, splits, M,
                                                            N, K, sh, s, lora);
    case 2:
        return launch_f32_bwd_cfg<FMT, DT, 2, kF32BwdWaves>(gy, packed, scales, gx, part, splits, M,
                                                            N, K, sh, s, lora);
    default:
        return launch_f32_bwd_cfg<FMT, DT, 4, kF32BwdWaves / 2>(gy, packed, scales, gx, part,
                                                                splits, M, N, K, sh, s, lora);
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
                              int sh, int dt, hipStream_t s, const LoraEp& lora) {
    switch (dt) {
    case kF32:
        return launch_f32_bwd_t<FMT, kF32>(gy, packed, scales, gx, part, splits, M, N, K, sh, s, lora);
    case kF16:
        return launch_f32_bwd_t<FMT, kF16>(gy, packed, scales, gx, part, splits, M, N, K, sh, s, lora);
    default:
        return launch_f32_bwd_t<FMT, kBF16>(gy, packed, scales, gx, part, splits, M, N, K, sh, s, lora);
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
                               int64_t gs, int dt, hipStream_t s, int fmt, const LoraEp& lora) {
    const int sh = log2_of(gs);
    if (fmt == kFmtRoot)
        return f32_bwd_fmt<kFmtRoot>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s, lora);
    if (fmt == kFmt2Bit)
        return f32_bwd_fmt<kFmt2Bit>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s, lora);
    return f32_bwd_fmt<kFmtTernary>(gy, packed, scales, gx, part, splits, M, N, K, sh, dt, s, lora);
}

}  // namespace ojx
