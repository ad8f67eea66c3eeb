// e8t_codec.hip -- E8 encoder and decoder kernels for gfx950: ternary 1.5-bit
// (TernaryE8LatticePacker) and 2-bit (E8LatticePacker, at the end of the file).
//
// Encoder: bit-exact restatement of TernaryE8LatticePacker.pack
// (ojasx2/math/lattice.py:338-384) as one fused pass: each weight is read once
// from HBM (2 B for fp16/bf16) and 0.25 B of codes + scale is written.  The
// reference's device route runs ~25 ATen element-wise kernels with int64
// temporaries for the same work.
//
// One lane per flat group: the reference's scale is torch's CPU norm, whose
// summation order is a sequential FMA chain per lane j over w[j], w[j+8], ...
// (8 fp32 lanes), so a group's norm is inherently serial over its 8-vectors.  One
// lane owning the group computes it once (gs/8 + 7 adds per group) and then runs
// the gs/8 nearest-point searches of its 8-vectors; splitting a group across
// lanes would cost a cross-lane exchange per link of the chain.
//
// Decoder: restatement of TernaryE8LatticePacker.unpack (lattice.py:386-419),
// one lane per code pair (3 bytes -> 16 weights), exact for every dtype.

#include "e8t_device.h"
#include "e8t_internal.h"
#include "e8t_root.h"

namespace ojx {

// Correctly rounded quotient w / s from the group's reciprocal y = RN(1/s), by one
// residual correction (Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", IBM J. Res. Dev. 34(1), 1990): q = RN(w*y), r = w - q*s exact
// by fma, RN(q + r*y) == RN(w/s).  The residual is formed on w*2^48 and s*2^48 and
// multiplied back by y*2^-48 (exact power-of-two scalings), so it stays a normal number
// for every finite w, including subnormal ones.  Checked against true division on
// 1.28e8 weights from realistic, tiny, huge, subnormal and random-exponent groups (0
// mismatches); the kernel's results are compared bit for bit with the CPU oracle.
struct GroupRecip {
    float s, y, bs, ys;  // s, RN(1/s), s*2^48, y*2^-48
    bool exact;          // s not finite: fall back to true division
};

__device__ __forceinline__ GroupRecip group_recip(float s) {
    GroupRecip g;
    g.s = s;
    g.y = 1.0f / s;
    g.bs = s * 0x1p48f;
    g.ys = g.y * 0x1p-48f;
    g.exact = !__builtin_isfinite(s);
    return g;
}

__device__ __forceinline__ float div_rn(float w, const GroupRecip& g) {
#pragma clang fp contract(off)
    const float q = w * g.y;
    const float r = __builtin_fmaf(-q, g.bs, w * 0x1p48f);
    return __builtin_fmaf(r, g.ys, q);
}

// The same quotient without the 2^48 scaling, for weights that came from fp16: every
// nonzero fp16 value is at least 2^-24 in magnitude, so the residual is a normal fp32
// number already (checked against true division for every finite fp16 w over 6,000 scales
// from 2^-40 to 2^42: 0 mismatches).  w = -0 gives +0 here, as in div_rn.
__device__ __forceinline__ float div_rn_f16in(float w, const GroupRecip& g) {
#pragma clang fp contract(off)
    const float q = w * g.y;
    const float r = __builtin_fmaf(-q, g.s, w);
    return __builtin_fmaf(r, g.y, q);
}

// Nearest point of one 8-vector of the group with fp32 scale s, as lattice.py:357-373:
//   v = w / s (correctly rounded)
//   q = clamp(rint(v), -1, 1); alt = q == 0 ? (v >= 0 ? 1 : -1) : 0
//   pen = (alt - v)^2 - (q - v)^2 (three rounded ops, never contracted)
//   odd sum(q): q[first argmin pen] = alt;  code = sum (q_i + 1) 3^i / 2.
// All integer-valued quantities are carried in fp32, where they are exact.  This is the
// literal form, used when the group's scale is not finite (true division).
__device__ __forceinline__ uint32_t quantize8_exact(const float* __restrict__ w, float s) {
#pragma clang fp contract(off)
    const float pow3[8] = {1.f, 3.f, 9.f, 27.f, 81.f, 243.f, 729.f, 2187.f};
    float v[8], q[8];
    float qsum = 0.f;
    float raw = 3280.f;  // sum of 3^i: the "+1" of every digit
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = w[i] / s;
        float r = __builtin_rintf(v[i]);
        r = fmaxf(r, -1.f);
        r = fminf(r, 1.f);
        q[i] = r;
        qsum = qsum + r;
        raw = __builtin_fmaf(r, pow3[i], raw);
    }
    float best_pen = 0.f, best_delta = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        float alt = (q[i] == 0.f) ? (v[i] >= 0.f ? 1.f : -1.f) : 0.f;
        float a = alt - v[i];
        float b = q[i] - v[i];
        float a2 = a * a;
        float b2 = b * b;
        float pen = a2 - b2;
        float delta = (alt - q[i]) * pow3[i];
        if (i == 0 || pen < best_pen) {
            best_pen = pen;
            best_delta = delta;
        }
    }
    // sum(q) is an integer in [-8, 8]; odd parity applies the best flip
    int odd = ((int)qsum) & 1;
    raw = odd ? raw + best_delta : raw;
    return ((uint32_t)raw) >> 1;
}

// The same nearest point for a finite scale, in a reduced form with the same results.
// With d = fl(1 - |v|) and t = fl(fl(d * d) - fl(v * v)):
//   * pen == |t| for every finite fp32 v (q == 0 puts both cases' squares in the same two
//     rounded products: alt - v = +-d, q - v = -v; q != 0 swaps them), so the first argmin
//     of pen is the first argmin of |t|;
//   * alt - q == sgn(v) * sgn(t) for every v with |v| < 2^24, where sgn(-0) = +1 (t >= 0
//     exactly when q == 0, and the reference's alt is +1 for v = -0 since -0 >= 0), so the
//     flip adds +-3^i with the sign of (v < 0) XOR t.
// Both identities were checked exhaustively over all 2^32 fp32 bit patterns.  Here
// |v| <= sqrt(gs) * (1 + eps) (the group's norm bounds every weight).  The quotient can be
// -0: the residual division returns +0 for w = -0, but a negative subnormal weight over a
// scale >= 2 rounds to -0, so v's sign is taken by a comparison, not from its sign bit.
// The parity of sum(q) is the parity of the code's base-3 value, since every power of 3
// is odd.  F16IN: the weights came from fp16.
template <bool F16IN>
__device__ __forceinline__ uint32_t quantize8(const float* __restrict__ w, const GroupRecip& g) {
#pragma clang fp contract(off)
    const float pow3[8] = {1.f, 3.f, 9.f, 27.f, 81.f, 243.f, 729.f, 2187.f};
    float raw = 3280.f;  // sum of 3^i: the "+1" of every digit
    float best_t = 0.f, best_v = 0.f, best_p = 0.f;  // t, v and 3^i of the first argmin
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float v = F16IN ? div_rn_f16in(w[i], g) : div_rn(w[i], g);
        float r = __builtin_rintf(v);
        r = fmaxf(r, -1.f);
        r = fminf(r, 1.f);
        raw = __builtin_fmaf(r, pow3[i], raw);
        const float d = 1.f - fabsf(v);
        const float d2 = d * d;
        const float v2 = v * v;
        const float t = d2 - v2;
        if (i == 0 || fabsf(t) < fabsf(best_t)) {
            best_t = t;
            best_v = v;
            best_p = pow3[i];
        }
    }
    const uint32_t sg = (best_v < 0.f ? 0x80000000u : 0u) ^ (__float_as_uint(best_t) & 0x80000000u);
    const int ri = (int)raw;  // exact: 0 .. 6560
    const int fix = (ri & 1) ? (int)__uint_as_float(__float_as_uint(best_p) | sg) : 0;
    return (uint32_t)(ri + fix) >> 1;
}

// Group scale (lattice.py:355-356) with torch's CPU norm order:
// 8 fmaf lanes, lane j over elements j, j+8, ...; lanes summed left to right;
// correctly rounded sqrt; true division by fp32(sqrt(gs)); + fp32(1e-8).
template <int GS>
__device__ __forceinline__ float group_scale(const float* __restrict__ w, float root) {
#pragma clang fp contract(off)
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = w[j] * w[j];
#pragma unroll
    for (int t = 1; t < GS / 8; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = __builtin_fmaf(w[8 * t + j], w[8 * t + j], acc[j]);
    float sum = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) sum = sum + acc[j];
    float nrm = __builtin_sqrtf(sum);
    float s = nrm / root;
    return s + 1e-8f;
}

// Two codes -> 3 bytes (lattice.py:379-383).
__device__ __forceinline__ void pack_pair(uint8_t* b, uint32_t c0, uint32_t c1) {
    b[0] = (uint8_t)(c0 & 0xFFu);
    b[1] = (uint8_t)(((c0 >> 8) & 0x0Fu) | ((c1 & 0x0Fu) << 4));
    b[2] = (uint8_t)((c1 >> 4) & 0xFFu);
}

// Eight weights from a 16-byte aligned, in-range address, as fp32.
template <int WDT>
__device__ __forceinline__ void load8_vec(const void* __restrict__ w, int64_t base, float* out) {
    if constexpr (WDT == kF32) {
        const float4* p = reinterpret_cast<const float4*>((const float*)w + base);
        float4 a = p[0], b = p[1];
        out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
        out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
    } else {
        uint4 a = *reinterpret_cast<const uint4*>((const uint16_t*)w + base);
        uint32_t u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (WDT == kF16) {
                out[2 * i] = f16_bits_to_f32(u[i] & 0xFFFFu);
                out[2 * i + 1] = f16_bits_to_f32(u[i] >> 16);
            } else {
                out[2 * i] = bf16_bits_to_f32(u[i] & 0xFFFFu);
                out[2 * i + 1] = bf16_bits_to_f32(u[i] >> 16);
            }
        }
    }
}

template <int WDT>
__device__ __forceinline__ void load8(const void* __restrict__ w, int64_t base, int64_t numel,
                                      bool vec_ok, float* out) {
    if (vec_ok && base + 8 <= numel) {
        if constexpr (WDT == kF32) {
            const float4* p = reinterpret_cast<const float4*>((const float*)w + base);
            float4 a = p[0], b = p[1];
            out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
            out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
        } else {
            uint4 a = *reinterpret_cast<const uint4*>((const uint16_t*)w + base);
            uint32_t u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (WDT == kF16) {
                    out[2 * i] = f16_bits_to_f32(u[i] & 0xFFFFu);
                    out[2 * i + 1] = f16_bits_to_f32(u[i] >> 16);
                } else {
                    out[2 * i] = bf16_bits_to_f32(u[i] & 0xFFFFu);
                    out[2 * i + 1] = bf16_bits_to_f32(u[i] >> 16);
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            out[i] = (base + i < numel) ? load_as_f32<WDT>(w, base + i) : 0.f;  // F.pad zeros
    }
}

constexpr int kEncThreads = 256;

// GS in {16, 32, 64}: the group stays in registers.
template <int WDT, int GS>
__global__ __launch_bounds__(kEncThreads) void encode_kernel(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, float root, bool vec_ok,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
    constexpr int NV = GS / 8;
    constexpr int BYTES = GS * 3 / 16;
    __shared__ uint8_t stage[kEncThreads * BYTES];
    const int64_t g0 = (int64_t)blockIdx.x * kEncThreads;
    const int64_t g = g0 + threadIdx.x;
    if (g < ngroups) {
        float x[GS];
        if (vec_ok && (g + 1) * GS <= numel) {  // the whole group in range: one address
#pragma unroll
            for (int t = 0; t < NV; ++t) load8_vec<WDT>(w, g * GS + 8 * t, x + 8 * t);
        } else {
#pragma unroll
            for (int t = 0; t < NV; ++t) load8<WDT>(w, g * GS + 8 * t, numel, vec_ok, x + 8 * t);
        }
        const float s = group_scale<GS>(x, root);
        const GroupRecip gr = group_recip(s);
        uint8_t* st = stage + threadIdx.x * BYTES;
        if (!gr.exact) {
#pragma unroll
            for (int p = 0; p < NV / 2; ++p)
                pack_pair(st + 3 * p, quantize8<WDT == kF16>(x + 16 * p, gr),
                          quantize8<WDT == kF16>(x + 16 * p + 8, gr));
        } else {
            for (int p = 0; p < NV / 2; ++p)
                pack_pair(st + 3 * p, quantize8_exact(x + 16 * p, s),
                          quantize8_exact(x + 16 * p + 8, s));
        }
        scales[g] = (uint16_t)f32_to_f16_bits(s);
    }
    __syncthreads();
    // coalesced copy-out of the block's packed bytes
    const int64_t ng = (ngroups - g0) < kEncThreads ? (ngroups - g0) : kEncThreads;
    const int nbytes = (int)ng * BYTES;
    uint8_t* dst = packed + g0 * BYTES;
    if ((((uintptr_t)dst) & 3u) == 0) {
        const int nwords = nbytes >> 2;
        const uint32_t* src32 = reinterpret_cast<const uint32_t*>(stage);
        uint32_t* dst32 = reinterpret_cast<uint32_t*>(dst);
        for (int i = threadIdx.x; i < nwords; i += kEncThreads) dst32[i] = src32[i];
        for (int i = (nwords << 2) + threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    } else {
        for (int i = threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    }
}

// Any GS (multiple of 16): two passes over the group (norm, then codes); the
// second pass re-reads the group through the caches.
template <int WDT>
__global__ __launch_bounds__(kEncThreads) void encode_kernel_any(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, int64_t gs, float root,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
#pragma clang fp contract(off)
    const int64_t g = (int64_t)blockIdx.x * kEncThreads + threadIdx.x;
    if (g >= ngroups) return;
    const int64_t base = g * gs;
    float acc[8];
    for (int t = 0; t < gs / 8; ++t) {
        float x[8];
        load8<WDT>(w, base + 8 * t, numel, false, x);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = (t == 0) ? x[j] * x[j] : __builtin_fmaf(x[j], x[j], acc[j]);
    }
    float sum = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) sum = sum + acc[j];
    float s = __builtin_sqrtf(sum) / root;
    s = s + 1e-8f;
    uint8_t* dst = packed + base * 3 / 16;
    const GroupRecip gr = group_recip(s);
    for (int p = 0; p < gs / 16; ++p) {
        float x[16];
        load8<WDT>(w, base + 16 * p, numel, false, x);
        load8<WDT>(w, base + 16 * p + 8, numel, false, x + 8);
        if (!gr.exact)
            pack_pair(dst + 3 * p, quantize8<WDT == kF16>(x, gr), quantize8<WDT == kF16>(x + 8, gr));
        else pack_pair(dst + 3 * p, quantize8_exact(x, s), quantize8_exact(x + 8, s));
    }
    scales[g] = (uint16_t)f32_to_f16_bits(s);
}

template <int WDT>
static hipError_t launch_encode_t(const void* w, int64_t numel, int64_t gs, uint8_t* packed,
                                  uint16_t* scales, hipStream_t stream) {
    const int64_t padded = numel + (gs - numel % gs) % gs;
    const int64_t ngroups = padded / gs;
    const float root = (float)__builtin_sqrt((double)gs);
    const int64_t blocks = (ngroups + kEncThreads - 1) / kEncThreads;
    const bool vec_ok = (((uintptr_t)w) & 15u) == 0;
    if (gs == 16)
        hipLaunchKernelGGL((encode_kernel<WDT, 16>), dim3((unsigned)blocks), dim3(kEncThreads), 0,
                           stream, w, numel, ngroups, root, vec_ok, packed, scales);
    else if (gs == 32)
        hipLaunchKernelGGL((encode_kernel<WDT, 32>), dim3((unsigned)blocks), dim3(kEncThreads), 0,
                           stream, w, numel, ngroups, root, vec_ok, packed, scales);
    else if (gs == 64)
        hipLaunchKernelGGL((encode_kernel<WDT, 64>), dim3((unsigned)blocks), dim3(kEncThreads), 0,
                           stream, w, numel, ngroups, root, vec_ok, packed, scales);
    else
        hipLaunchKernelGGL((encode_kernel_any<WDT>), dim3((unsigned)blocks), dim3(kEncThreads), 0,
                           stream, w, numel, ngroups, gs, root, packed, scales);
    return hipGetLastError();
}

hipError_t launch_encode(const void* w, int wdt, int64_t numel, int64_t gs, uint8_t* packed,
                         uint16_t* scales, hipStream_t stream) {
    switch (wdt) {
        case kF32: return launch_encode_t<kF32>(w, numel, gs, packed, scales, stream);
        case kF16: return launch_encode_t<kF16>(w, numel, gs, packed, scales, stream);
        default: return launch_encode_t<kBF16>(w, numel, gs, packed, scales, stream);
    }
}

// ---------------------------------------------------------------- decoders
//
// The three packers' unpack (lattice.py:386-419, 252-279, 519-533): coordinate *
// scales.to(dtype), rounded to dtype for 2-bit and 1-bit codes.  Bound by the writes: a
// lane writes 16 bytes (4 fp32 or 8 16-bit weights, half a code or one) of each of its
// pieces, and a wave's store covers 1 KB without a gap.  One lane per 16 weights left 64-byte
// gaps between the lanes of every store, and divided twice by the group size.  us for 14336 x
// 4096, gs 32, to fp32 / fp16 / bf16: ternary 71 / 23.2 / 27.3 -> 36.4 / 20.8 / 20.9, 2-bit 70 /
// 23.1 / 27.4 -> 36.9 / 21.3 / 22.1, 1-bit 86 / 51 / 52 -> 36.0 / 21.9 / 22.2 (fp32: 6.4 TB/s
// written).

constexpr int kDecThreads = 256;

// Bits of v in dtype ODT, rounded once (v kept a rounded fp32 product: -1 * 0 stays -0).
template <int ODT> __device__ __forceinline__ uint32_t out_bits(float v) {
    keep_f32(v);
    if constexpr (ODT == kF32) return __float_as_uint(v);
    else if constexpr (ODT == kF16) return f32_to_f16_bits(v);
    else return f32_to_bf16_bits(v);
}

// FMT's weights e .. e + V - 1 (one code, or one half of it; one scale group) as bits of ODT.
// Ternary and 2-bit weights take one of three or four values per group: each is rounded
// once and selected by digit (digits by 24-bit multiplies; the compiler's division by 3
// multiplies at a quarter of the rate).
template <int FMT, int ODT, int V>
__device__ __forceinline__ void decode_run(const uint8_t* __restrict__ packed, int64_t e,
                                           uint32_t s16, uint32_t (&v)[V]) {
    const float s = scale_for<ODT>(s16);
    if constexpr (FMT == kFmt2Bit) {
        uint32_t bits = packed[e >> 2];
        if constexpr (V == 8) bits |= (uint32_t)packed[(e >> 2) + 1] << 8;
        const uint32_t v0 = out_bits<ODT>(-1.5f * s), v1 = out_bits<ODT>(-0.5f * s),
                       v2 = out_bits<ODT>(0.5f * s), v3 = out_bits<ODT>(1.5f * s);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const uint32_t lo = (bits >> (2 * i)) & 1u ? v1 : v0;
            const uint32_t hi = (bits >> (2 * i)) & 1u ? v3 : v2;
            v[i] = (bits >> (2 * i)) & 2u ? hi : lo;
        }
    } else if constexpr (FMT == kFmtTernary) {
        // code t: 12 bits from bit 12 t, within the two bytes from 3 t / 2 (one load, no branch
        // between even and odd codes)
        const int64_t t = e >> 3;
        uint16_t pair;
        __builtin_memcpy(&pair, packed + ((3 * t) >> 1), 2);
        uint32_t raw = 2u * (((uint32_t)pair >> (4 * (t & 1))) & 0xFFFu);
        if (V == 4 && (e & 4)) raw = (raw * 25891u) >> 21;  // / 81, exact below 8192
        const uint32_t vm = out_bits<ODT>(-1.0f * s), vz = out_bits<ODT>(0.0f * s),
                       vp = out_bits<ODT>(s);
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const uint32_t q = (raw * 43691u) >> 17;  // / 3, exact below 98304 (32-bit product)
            const uint32_t d = raw - 3u * q;
            v[i] = d == 0u ? vm : d == 1u ? vz : vp;
            raw = q;
        }
    } else {
        uint32_t row[V / 4];  // the code's coordinates, one load
        __builtin_memcpy(row, &kRootTable.c[packed[e >> 3]][e & 7], V);
#pragma unroll
        for (int i = 0; i < V; ++i)
            v[i] = out_bits<ODT>((float)(int8_t)(row[i / 4] >> (8 * (i & 3))) * s);
    }
}

// P: pieces per lane; gs_shift: log2 of the group size, or -1 where it is no power of two
template <int FMT, int ODT, int P>
__global__ __launch_bounds__(kDecThreads) void decode_kernel(
    const uint8_t* __restrict__ packed, const uint16_t* __restrict__ scales, int64_t numel,
    int64_t gs, int gs_shift, bool vec_ok, void* __restrict__ out) {
    constexpr int V = ODT == kF32 ? 4 : 8;
    const int64_t first = ((int64_t)blockIdx.x * (P * kDecThreads) + threadIdx.x) * V;
    const int64_t last = (numel - 1) / V * V;  // run that pieces past the end repeat, unstored
    uint32_t v[P][V];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int64_t e0 = first + (int64_t)p * (kDecThreads * V), e = e0 < last ? e0 : last;
        const uint32_t s16 = scales[gs_shift >= 0 ? e >> gs_shift : e / gs];
        decode_run<FMT, ODT, V>(packed, e, s16, v[p]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int64_t e = first + (int64_t)p * (kDecThreads * V);
        if (vec_ok && e + V <= numel) {
            if constexpr (ODT == kF32)
                *reinterpret_cast<uint4*>((uint32_t*)out + e) =
                    make_uint4(v[p][0], v[p][1], v[p][2], v[p][3]);
            else
                *reinterpret_cast<uint4*>((uint16_t*)out + e) =
                    make_uint4(v[p][0] | (v[p][1] << 16), v[p][2] | (v[p][3] << 16),
                               v[p][4] | (v[p][5] << 16), v[p][6] | (v[p][7] << 16));
        } else {
#pragma unroll
            for (int i = 0; i < V; ++i) {
                if (e + i >= numel) continue;
                if constexpr (ODT == kF32) ((uint32_t*)out)[e + i] = v[p][i];
                else ((uint16_t*)out)[e + i] = (uint16_t)v[p][i];
            }
        }
    }
}

// Pieces per lane: one while that fills the chip no more than 32 times over (2M weights to
// fp16, ternary: 3.0 us, with four pieces 3.7), then two, which share a lane's index work and keep
// two loads in flight (1-bit 32M to fp32 24.2 and 22.8), and four for results past the last-level
// cache (256 MB; ternary 256M to bf16 155.8 with two and 147.4).
constexpr int64_t kDecTwoFrom = 8192, kDecFourFrom = 65536;  // blocks of one piece per lane

template <int FMT, int ODT, int P>
static hipError_t launch_decode_p(const uint8_t* packed, const uint16_t* scales, int64_t numel,
                                  int64_t gs, int64_t runs, void* out, hipStream_t stream) {
    const int shift = (gs & (gs - 1)) == 0 ? 63 - __builtin_clzll((unsigned long long)gs) : -1;
    const bool vec = ((uintptr_t)out & 15u) == 0;
    hipLaunchKernelGGL((decode_kernel<FMT, ODT, P>), dim3((unsigned)((runs + P - 1) / P)),
                       dim3(kDecThreads), 0, stream, packed, scales, numel, gs, shift, vec, out);
    return hipGetLastError();
}

template <int FMT, int ODT>
static hipError_t launch_decode_t(const uint8_t* packed, const uint16_t* scales, int64_t numel,
                                  int64_t gs, void* out, hipStream_t stream) {
    constexpr int64_t kPerBlock = kDecThreads * (ODT == kF32 ? 4 : 8);
    const int64_t runs = (numel + kPerBlock - 1) / kPerBlock;
    if (runs < kDecTwoFrom)
        return launch_decode_p<FMT, ODT, 1>(packed, scales, numel, gs, runs, out, stream);
    if (runs < kDecFourFrom)
        return launch_decode_p<FMT, ODT, 2>(packed, scales, numel, gs, runs, out, stream);
    return launch_decode_p<FMT, ODT, 4>(packed, scales, numel, gs, runs, out, stream);
}

template <int FMT>
static hipError_t launch_decode_fmt(const uint8_t* packed, const uint16_t* scales, int64_t numel,
                                    int64_t gs, int odt, void* out, hipStream_t stream) {
    switch (odt) {
        case kF32: return launch_decode_t<FMT, kF32>(packed, scales, numel, gs, out, stream);
        case kF16: return launch_decode_t<FMT, kF16>(packed, scales, numel, gs, out, stream);
        default: return launch_decode_t<FMT, kBF16>(packed, scales, numel, gs, out, stream);
    }
}

hipError_t launch_decode(const uint8_t* packed, const uint16_t* scales, int64_t numel, int64_t gs,
                         int odt, void* out, hipStream_t stream) {
    return launch_decode_fmt<kFmtTernary>(packed, scales, numel, gs, odt, out, stream);
}

hipError_t launch_decode2(const uint8_t* packed, const uint16_t* scales, int64_t numel,
                          int64_t gs, int odt, void* out, hipStream_t stream) {
    return launch_decode_fmt<kFmt2Bit>(packed, scales, numel, gs, odt, out, stream);
}

hipError_t launch_decode1(const uint8_t* codes, const uint16_t* scales, int64_t numel,
                          int64_t gs, int odt, void* out, hipStream_t stream) {
    return launch_decode_fmt<kFmtRoot>(codes, scales, numel, gs, odt, out, stream);
}

// ---------------------------------------------------------------- 2-bit encoder
//
// E8LatticePacker.pack (lattice.py:213-249), bit-exact: the same scale (torch's norm
// order, correctly rounded quotients) and per 8-vector
//   xs = w/s - 0.5; f2 = clamp(rint(xs), -2, 1)
//   alt = xs >= f2 ? clamp(f2 + 1, -2, 1) : clamp(f2 - 1, -2, 1)
//   pen = (alt - xs)^2 - (f2 - xs)^2 (rounded ops, never contracted)
//   odd sum(f2): f2[first argmin pen] = alt;  code_i = f2_i + 2
// A clamped coordinate has alt == f2 and pen 0; as the first minimum its "flip" is a no-op
// and the vector keeps its odd sum, exactly as in the reference.  Returns the 8 codes as
// 16 bits (two packed bytes, code i in bits [2i, 2i+2)).

template <bool EXACT>
__device__ __forceinline__ uint32_t quantize8_2bit(const float* __restrict__ w,
                                                   const GroupRecip& g) {
#pragma clang fp contract(off)
    const float pow4[8] = {1.f, 4.f, 16.f, 64.f, 256.f, 1024.f, 4096.f, 16384.f};
    float xs[8], f2[8];
    float fsum = 0.f;
    float codes = 0.f;  // sum (f2_i + 2) 4^i: exact in fp32
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float v = EXACT ? w[i] / g.s : div_rn(w[i], g);
        xs[i] = v - 0.5f;
        float r = __builtin_rintf(xs[i]);
        r = fmaxf(r, -2.f);
        r = fminf(r, 1.f);
        f2[i] = r;
        fsum = fsum + r;
        codes = __builtin_fmaf(r + 2.f, pow4[i], codes);
    }
    float best_pen = 0.f, best_delta = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float up = fminf(f2[i] + 1.f, 1.f), dn = fmaxf(f2[i] - 1.f, -2.f);
        const float alt = xs[i] >= f2[i] ? up : dn;
        const float a = alt - xs[i];
        const float b = f2[i] - xs[i];
        const float a2 = a * a;
        const float b2 = b * b;
        const float pen = a2 - b2;
        const float delta = (alt - f2[i]) * pow4[i];
        if (i == 0 || pen < best_pen) {
            best_pen = pen;
            best_delta = delta;
        }
    }
    const int odd = ((int)fsum) & 1;  // sum(f2) is an integer in [-16, 8]
    codes = odd ? codes + best_delta : codes;
    return (uint32_t)codes;
}

// GS in {8, 16, 32, 64}: the group stays in registers; bytes staged in LDS and written
// coalesced.
template <int WDT, int GS>
__global__ __launch_bounds__(kEncThreads) void encode2_kernel(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, float root, bool vec_ok,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
    constexpr int NV = GS / 8;
    constexpr int BYTES = GS / 4;
    __shared__ uint8_t stage[kEncThreads * BYTES];
    const int64_t g0 = (int64_t)blockIdx.x * kEncThreads;
    const int64_t g = g0 + threadIdx.x;
    if (g < ngroups) {
        float x[GS];
        if (vec_ok && (g + 1) * GS <= numel) {  // the whole group in range: one address
#pragma unroll
            for (int t = 0; t < NV; ++t) load8_vec<WDT>(w, g * GS + 8 * t, x + 8 * t);
        } else {
#pragma unroll
            for (int t = 0; t < NV; ++t) load8<WDT>(w, g * GS + 8 * t, numel, vec_ok, x + 8 * t);
        }
        const float s = group_scale<GS>(x, root);
        const GroupRecip gr = group_recip(s);
        uint8_t* st = stage + threadIdx.x * BYTES;
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const uint32_t c = gr.exact ? quantize8_2bit<true>(x + 8 * t, gr)
                                        : quantize8_2bit<false>(x + 8 * t, gr);
            st[2 * t] = (uint8_t)(c & 0xFFu);
            st[2 * t + 1] = (uint8_t)(c >> 8);
        }
        scales[g] = (uint16_t)f32_to_f16_bits(s);
    }
    __syncthreads();
    const int64_t ng = (ngroups - g0) < kEncThreads ? (ngroups - g0) : kEncThreads;
    const int nbytes = (int)ng * BYTES;
    uint8_t* dst = packed + g0 * BYTES;
    if ((((uintptr_t)dst) & 3u) == 0) {
        const int nwords = nbytes >> 2;
        const uint32_t* src32 = reinterpret_cast<const uint32_t*>(stage);
        uint32_t* dst32 = reinterpret_cast<uint32_t*>(dst);
        for (int i = threadIdx.x; i < nwords; i += kEncThreads) dst32[i] = src32[i];
        for (int i = (nwords << 2) + threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    } else {
        for (int i = threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    }
}

// Any GS (multiple of 8): norm pass, then the codes, re-reading the group.
template <int WDT>
__global__ __launch_bounds__(kEncThreads) void encode2_kernel_any(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, int64_t gs, float root,
    uint8_t* __restrict__ packed, uint16_t* __restrict__ scales) {
#pragma clang fp contract(off)
    const int64_t g = (int64_t)blockIdx.x * kEncThreads + threadIdx.x;
    if (g >= ngroups) return;
    const int64_t base = g * gs;
    float acc[8];
    for (int t = 0; t < gs / 8; ++t) {
        float x[8];
        load8<WDT>(w, base + 8 * t, numel, false, x);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = (t == 0) ? x[j] * x[j] : __builtin_fmaf(x[j], x[j], acc[j]);
    }
    float sum = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) sum = sum + acc[j];
    float s = __builtin_sqrtf(sum) / root;
    s = s + 1e-8f;
    uint8_t* dst = packed + base / 4;
    const GroupRecip gr = group_recip(s);
    for (int t = 0; t < gs / 8; ++t) {
        float x[8];
        load8<WDT>(w, base + 8 * t, numel, false, x);
        const uint32_t c = gr.exact ? quantize8_2bit<true>(x, gr) : quantize8_2bit<false>(x, gr);
        dst[2 * t] = (uint8_t)(c & 0xFFu);
        dst[2 * t + 1] = (uint8_t)(c >> 8);
    }
    scales[g] = (uint16_t)f32_to_f16_bits(s);
}

template <int WDT>
static hipError_t launch_encode2_t(const void* w, int64_t numel, int64_t gs, uint8_t* packed,
                                   uint16_t* scales, hipStream_t stream) {
    const int64_t padded = numel + (gs - numel % gs) % gs;
    const int64_t ngroups = padded / gs;
    const float root = (float)__builtin_sqrt((double)gs);
    const int64_t blocks = (ngroups + kEncThreads - 1) / kEncThreads;
    const bool vec_ok = (((uintptr_t)w) & 15u) == 0;
    switch (gs) {
        case 8:
            hipLaunchKernelGGL((encode2_kernel<WDT, 8>), dim3((unsigned)blocks), dim3(kEncThreads),
                               0, stream, w, numel, ngroups, root, vec_ok, packed, scales);
            break;
        case 16:
            hipLaunchKernelGGL((encode2_kernel<WDT, 16>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               packed, scales);
            break;
        case 32:
            hipLaunchKernelGGL((encode2_kernel<WDT, 32>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               packed, scales);
            break;
        case 64:
            hipLaunchKernelGGL((encode2_kernel<WDT, 64>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               packed, scales);
            break;
        default:
            hipLaunchKernelGGL((encode2_kernel_any<WDT>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, gs, root, packed,
                               scales);
            break;
    }
    return hipGetLastError();
}

hipError_t launch_encode2(const void* w, int wdt, int64_t numel, int64_t gs, uint8_t* packed,
                          uint16_t* scales, hipStream_t stream) {
    switch (wdt) {
        case kF32: return launch_encode2_t<kF32>(w, numel, gs, packed, scales, stream);
        case kF16: return launch_encode2_t<kF16>(w, numel, gs, packed, scales, stream);
        default: return launch_encode2_t<kBF16>(w, numel, gs, packed, scales, stream);
    }
}

// ---------------------------------------------------------------- 1-bit Root-E8 encoder
//
// RootE8LatticePacker.pack (lattice.py:473-509), per flat group of gs weights:
//   s = torch.norm(w)/sqrt(gs) + 1e-8 (the CPU norm order, as the other packers);
//   v = w / s; code = argmax over the 256 table rows u of v . u/|u| (first maximal index);
//   scale = sum(w * q) / max(sum(q * q), 1e-8) for q = table[code], stored as fp16.
// The code search is root_code (e8t_root.h).  Both sums run in torch's CPU order for a
// contiguous last dim: four
// 8-lane accumulators over the 8-blocks of each 32-block, later 8-blocks into the first
// accumulator, accumulators added in order, then the 8 lanes left to right.

// torch's CPU row-sum order (see above), fed one 8-block at a time.
struct TorchRowSum {
    float acc[4][8];
    int block;
    int main_blocks;  // 8-blocks inside whole 32-blocks
    __device__ __forceinline__ void init(int64_t n) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[a][j] = 0.f;
        block = 0;
        main_blocks = (int)((n / 8) / 4 * 4);
    }
    __device__ __forceinline__ void add8(const float (&x)[8]) {
#pragma clang fp contract(off)
        const int a = block < main_blocks ? (block & 3) : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q == a)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[q][j] = acc[q][j] + x[j];
        ++block;
    }
    __device__ __forceinline__ float result() const {
#pragma clang fp contract(off)
        float lane[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) lane[j] = ((acc[0][j] + acc[1][j]) + acc[2][j]) + acc[3][j];
        float s = lane[0];
#pragma unroll
        for (int j = 1; j < 8; ++j) s = s + lane[j];
        return s;
    }
};

// Codes of one group whose weights are read 8 at a time by `get(t, x)`; accumulates the
// MMSE sums; returns the fp16 scale bits.
// NV: the group's 8-blocks when known at compile time (the loop is then unrolled and a
// register-resident group is indexed statically), else 0 and gs / 8 at run time.
template <int NV = 0, typename Get>
__device__ __forceinline__ uint32_t root_group(const Get& get, int64_t gs, float s,
                                               uint8_t* codes_out) {
#pragma clang fp contract(off)
    const GroupRecip gr = group_recip(s);
    TorchRowSum num, den;
    num.init(gs);
    den.init(gs);
    const int64_t nv = NV > 0 ? NV : gs / 8;
#pragma unroll
    for (int64_t t = 0; t < nv; ++t) {
        float x[8], v[8];
        get(t, x);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = gr.exact ? x[i] / s : div_rn(x[i], gr);
        const uint32_t c = gr.exact ? root_code_full(v) : root_code_fast(v);
        codes_out[t] = (uint8_t)c;
        float wq[8], qq[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float q = (float)kRootTable.c[c][i];
            wq[i] = x[i] * q;
            qq[i] = q * q;
        }
        num.add8(wq);
        den.add8(qq);
    }
    float d = den.result();
    d = d < 1e-8f ? 1e-8f : d;
    return f32_to_f16_bits(num.result() / d);
}

// GS in {8, 16, 32, 64}: the group stays in registers; code bytes staged in LDS and written
// coalesced.
template <int WDT, int GS>
__global__ __launch_bounds__(kEncThreads) void encode1_kernel(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, float root, bool vec_ok,
    uint8_t* __restrict__ codes, uint16_t* __restrict__ scales) {
    constexpr int NV = GS / 8;
    __shared__ uint8_t stage[kEncThreads * NV];
    const int64_t g0 = (int64_t)blockIdx.x * kEncThreads;
    const int64_t g = g0 + threadIdx.x;
    if (g < ngroups) {
        float x[GS];
        if (vec_ok && (g + 1) * GS <= numel) {  // the whole group in range: one address
#pragma unroll
            for (int t = 0; t < NV; ++t) load8_vec<WDT>(w, g * GS + 8 * t, x + 8 * t);
        } else {
#pragma unroll
            for (int t = 0; t < NV; ++t) load8<WDT>(w, g * GS + 8 * t, numel, vec_ok, x + 8 * t);
        }
        const float s = group_scale<GS>(x, root);
        auto get = [&](int64_t t, float (&o)[8]) {
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = x[8 * t + i];
        };
        scales[g] = (uint16_t)root_group<NV>(get, GS, s, stage + threadIdx.x * NV);
    }
    __syncthreads();
    const int64_t ng = (ngroups - g0) < kEncThreads ? (ngroups - g0) : kEncThreads;
    const int nbytes = (int)ng * NV;
    uint8_t* dst = codes + g0 * NV;
    if ((((uintptr_t)dst) & 3u) == 0) {
        const int nwords = nbytes >> 2;
        const uint32_t* src32 = reinterpret_cast<const uint32_t*>(stage);
        uint32_t* dst32 = reinterpret_cast<uint32_t*>(dst);
        for (int i = threadIdx.x; i < nwords; i += kEncThreads) dst32[i] = src32[i];
        for (int i = (nwords << 2) + threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    } else {
        for (int i = threadIdx.x; i < nbytes; i += kEncThreads) dst[i] = stage[i];
    }
}

// Any gs (multiple of 8): norm pass, then the codes, re-reading the group.
template <int WDT>
__global__ __launch_bounds__(kEncThreads) void encode1_kernel_any(
    const void* __restrict__ w, int64_t numel, int64_t ngroups, int64_t gs, float root,
    uint8_t* __restrict__ codes, uint16_t* __restrict__ scales) {
#pragma clang fp contract(off)
    const int64_t g = (int64_t)blockIdx.x * kEncThreads + threadIdx.x;
    if (g >= ngroups) return;
    const int64_t base = g * gs;
    float acc[8];
    for (int t = 0; t < gs / 8; ++t) {
        float x[8];
        load8<WDT>(w, base + 8 * t, numel, false, x);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = (t == 0) ? x[j] * x[j] : __builtin_fmaf(x[j], x[j], acc[j]);
    }
    float sum = acc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) sum = sum + acc[j];
    float s = __builtin_sqrtf(sum) / root;
    s = s + 1e-8f;
    auto get = [&](int64_t t, float (&o)[8]) { load8<WDT>(w, base + 8 * t, numel, false, o); };
    scales[g] = (uint16_t)root_group(get, gs, s, codes + base / 8);
}

template <int WDT>
static hipError_t launch_encode1_t(const void* w, int64_t numel, int64_t gs, uint8_t* codes,
                                   uint16_t* scales, hipStream_t stream) {
    const int64_t padded = numel + (gs - numel % gs) % gs;
    const int64_t ngroups = padded / gs;
    const float root = (float)__builtin_sqrt((double)gs);
    const int64_t blocks = (ngroups + kEncThreads - 1) / kEncThreads;
    const bool vec_ok = (((uintptr_t)w) & 15u) == 0;
    switch (gs) {
        case 8:
            hipLaunchKernelGGL((encode1_kernel<WDT, 8>), dim3((unsigned)blocks), dim3(kEncThreads),
                               0, stream, w, numel, ngroups, root, vec_ok, codes, scales);
            break;
        case 16:
            hipLaunchKernelGGL((encode1_kernel<WDT, 16>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               codes, scales);
            break;
        case 32:
            hipLaunchKernelGGL((encode1_kernel<WDT, 32>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               codes, scales);
            break;
        case 64:
            hipLaunchKernelGGL((encode1_kernel<WDT, 64>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, root, vec_ok,
                               codes, scales);
            break;
        default:
            hipLaunchKernelGGL((encode1_kernel_any<WDT>), dim3((unsigned)blocks),
                               dim3(kEncThreads), 0, stream, w, numel, ngroups, gs, root, codes,
                               scales);
            break;
    }
    return hipGetLastError();
}

hipError_t launch_encode1(const void* w, int wdt, int64_t numel, int64_t gs, uint8_t* codes,
                          uint16_t* scales, hipStream_t stream) {
    switch (wdt) {
        case kF32: return launch_encode1_t<kF32>(w, numel, gs, codes, scales, stream);
        case kF16: return launch_encode1_t<kF16>(w, numel, gs, codes, scales, stream);
        default: return launch_encode1_t<kBF16>(w, numel, gs, codes, scales, stream);
    }
}

}  // namespace ojx
