// e8t_lora.hip -- down-projections and gradients of a LoRA adapter.
//
// E8LatticeLinear.forward adds scaling * ((x @ A) @ B) to the E8 op's output
// (ojasx2/math/lattice.py:839-842; A [in, r], B [r, out]).  The fused forwards of this
// library add u @ B inside their output epilogue (before the one rounding to the activation
// dtype), with u = scaling * (x @ A) in fp32 [M, r] computed here; the backward forms v =
// scaling * (gy @ B^T) with the same kernels, adds v @ A^T in the dX epilogue and computes A's
// and B's gradients from v and u here.
//
// Three forms of the down-projection: lora_row_kernel (a workgroup per row, 16-byte loads; up to
// 512 rows), lora_mul_kernel (tiles of 16 rows on the matrix unit) and lora_down_kernel, the
// general one: any dtype, K and r, one workgroup per activation row, the 256 threads splitting
// K value by value, r partial sums per thread reduced across the wave by shuffles and across
// the waves in LDS.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "e8t_device.h"
#include "e8t_f32.h"
#include "e8t_internal.h"

namespace ojx {

constexpr int kLoraThreads = 256;  // general kernel

template <int DT, int RMAX>
__global__ __launch_bounds__(kLoraThreads) void lora_down_kernel(
    const void* __restrict__ x, const void* __restrict__ a, float* __restrict__ u, int64_t K,
    int r, float scaling, int64_t ldu) {
    __shared__ float red[kLoraThreads / 64][RMAX];
    const int64_t m = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float acc[RMAX];
#pragma unroll
    for (int j = 0; j < RMAX; ++j) acc[j] = 0.f;
    for (int64_t k = tid; k < K; k += kLoraThreads) {
        const float xv = load_as_f32<DT>(x, m * K + k);
#pragma unroll
        for (int j = 0; j < RMAX; ++j)
            if (j < r) acc[j] = __builtin_fmaf(xv, load_as_f32<DT>(a, k * r + j), acc[j]);
    }
#pragma unroll
    for (int j = 0; j < RMAX; ++j) {
        float v = acc[j];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        acc[j] = v;
    }
    if (lane == 0)
#pragma unroll
        for (int j = 0; j < RMAX; ++j) red[wave][j] = acc[j];
    __syncthreads();
    if (tid < r) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kLoraThreads / 64; ++w) v += red[w][tid];
        u[m * ldu + tid] = scaling * v;
    }
}

// Vector form, K % 8 == 0 (16-byte aligned x and factor; r % 8 == 0 where the rank varies
// fastest): one workgroup per (activation row, factor); thread t takes the 8 factor columns
// 8 (t % RS) .. + 7 (RS = r / 8 rounded up to a power of two) of the 8-k chunks t / RS,
// t / RS + 512 / RS, ...: eight values of x and 64 of the factor per chunk in 16-byte loads,
// two chunks in flight per iteration (16-bit), so a decode-sized K (4096: 512 chunks) is one
// round trip.  Partial sums are added across the lanes of equal column slice by shuffles
// and across the 8 waves in LDS.
constexpr int kLoraVecThreads = 512;

// out[m, j] = scaling * sum_k x[m, k] F(k, j), F(k, j) = f[k * sk + j * sj]: x @ A (sk = r,
// sj = 1) or gy @ B^T (sk = 1, sj = N).
struct LoraMul {
    const void* x;
    const void* f;
    float* out;
    int64_t K, sk, sj, r, ldo;
    float scaling;
};
struct LoraMulArgs {
    LoraMul it[kLoraDownItems];
    int64_t M;
};

// Eight consecutive values as loaded.
template <int DT> struct Run8 {
    uint4 v[DT == kF32 ? 2 : 1];

    __device__ __forceinline__ void load(const typename Elem<DT>::T* p) {
#pragma unroll
        for (int i = 0; i < (DT == kF32 ? 2 : 1); ++i) v[i] = reinterpret_cast<const uint4*>(p)[i];
    }
    __device__ __forceinline__ void get(float (&f)[8]) const {
#pragma unroll
        for (int i = 0; i < (DT == kF32 ? 2 : 1); ++i) {
            const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (DT == kF32) {
                    f[4 * i + e] = __uint_as_float(w[e]);
                } else {
                    const uint32_t lo = w[e] & 0xFFFFu, hi = w[e] >> 16;
                    f[2 * e] = DT == kBF16 ? bf16_bits_to_f32(lo) : f16_bits_to_f32(lo);
                    f[2 * e + 1] = DT == kBF16 ? bf16_bits_to_f32(hi) : f16_bits_to_f32(hi);
                }
            }
        }
    }
};

template <int DT, int RS, bool KMAJOR>
__device__ __forceinline__ void lora_row(const LoraMul& it,
                                         float (&red)[kLoraVecThreads / 64][kLoraMaxRank]) {
    using T = typename Elem<DT>::T;
    const int64_t m = blockIdx.x, K = it.K;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = (int)it.r;
    const int sl = tid & (RS - 1);
    constexpr int stride = kLoraVecThreads / RS;
    const int64_t nch = K / 8;
    const bool live = 8 * sl < r;
    const T* xr = static_cast<const T*>(it.x) + m * K;
    const T* f = static_cast<const T*>(it.f) + (KMAJOR ? 8 * sl * K : 8 * sl);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Two workgroups per CU need at most 128 registers: bf16 ranks over 8 take 32-bit offsets (a
    // factor holds under 2^29 values), 118 registers.  With 64-bit ones, 131, 384 rows of K =
    // 4096 at rank 16 took 9.0 us instead of 7.3.  (fp16, 126 registers with 64-bit offsets, is up
    // to 9% slower with 32-bit ones.)
    using Off = std::conditional_t<DT == kBF16 && (RS > 1), uint32_t, int64_t>;
    // run i of chunk c: k = 8 c + i of the 8 columns, or (KMAJOR) column i of the 8 k; columns
    // past r repeat the last one, never stored
    auto load = [&](Run8<DT>& xv, Run8<DT> (&fv)[8], int64_t c) {
        xv.load(xr + 8 * c);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (KMAJOR)
                fv[i].load(f + ((Off)(8 * sl + i < r ? i : r - 1 - 8 * sl) * (Off)K + 8 * (Off)c));
            else fv[i].load(f + (8 * (Off)c + i) * (Off)r);
        }
    };
    auto add = [&](const Run8<DT>& xv, const Run8<DT> (&fv)[8]) {
        float xf[8];
        xv.get(xf);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float ff[8];
            fv[i].get(ff);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (KMAJOR) acc[i] = __builtin_fmaf(xf[e], ff[e], acc[i]);
                else acc[e] = __builtin_fmaf(xf[i], ff[e], acc[e]);
            }
        }
    };
    if constexpr (DT == kF32) {
        if (live)
            for (int64_t c = tid / RS; c < nch; c += stride) {
                Run8<DT> x0, f0[8];
                load(x0, f0, c);
                add(x0, f0);
            }
    } else {
        for (int64_t c = tid / RS; c < nch; c += 2 * stride) {
            const int64_t c1 = c + stride;
            const bool two = c1 < nch;
            Run8<DT> x0, x1, f0[8], f1[8];
            if (live) {
                load(x0, f0, c);
                if (two) load(x1, f1, c1);
            }
            if (live) {
                add(x0, f0);
                if (two) add(x1, f1);
            }
        }
    }
    // lanes of equal slice: lane = sl (mod RS)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        float v = acc[j];
#pragma unroll
        for (int o = 32; o >= RS; o >>= 1) v += __shfl_xor(v, o);
        acc[j] = v;
    }
    if (lane < RS && live)
#pragma unroll
        for (int j = 0; j < 8; ++j) red[wave][8 * lane + j] = acc[j];
    __syncthreads();
    if (tid < r) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kLoraVecThreads / 64; ++w) v += red[w][tid];
        it.out[m * it.ldo + tid] = it.scaling * v;
    }
}

// RS: column slices of 8 (ranks up to 8 RS; every factor of the launch has the same RS)
template <int DT, int RS>
__global__ __launch_bounds__(kLoraVecThreads) void lora_row_kernel(LoraMulArgs args) {
    __shared__ float red[kLoraVecThreads / 64][kLoraMaxRank];
    LoraMul it = args.it[0];
#pragma unroll
    for (int i = 1; i < kLoraDownItems; ++i)
        if ((int)blockIdx.y == i) it = args.it[i];
    if (it.sk == 1) lora_row<DT, RS, true>(it, red);
    else lora_row<DT, RS, false>(it, red);
}

// ------------------------------------------------------------------ on the matrix unit
//
// The products with a factor of rank r <= 64 for many rows, on the matrix unit (any dtype, K
// and r; exact products, fp32 sums).  What bounds them is reading
// x and gy once and, at few rows, the loads' round trips; a row per workgroup re-read the
// whole factor for every row (21.6 us at 2048 x 4096 with rank 8, 19.4 us for 16 fp32 rows).

// A workgroup's waves split K of 16 rows.  Lane (g, i) holds x[i][32 b + 8 g ..] and the
// factor's values of the same eight k for column 16 t + i: eight fp32 instructions per block,
// or one of the 16-bit type's (the same products, exact in fp32, and fp32 sums; with eight
// fp32 instructions on converted values 2048 x 4096 took 10.1 us).
// VEC: rows of x (and of a k-contiguous factor) hold whole aligned groups of eight.
// KMAJOR: the factor is contiguous along k (compile time: a branch around loads would make
// the compiler wait for each of them where the branch ends).
template <int DT> constexpr int lora_waves() { return DT == kF32 ? 8 : 16; }

// Eight values of a row along k: loaded together (VEC) or one by one, kept as loaded (16-bit
// values are put together only where they are used, so that no load is waited for early).
template <int DT, bool VEC> struct Eight {
    uint32_t w[8];

    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, uint32_t vo, int so) {
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < (DT == kF32 ? 2 : 1); ++i) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b, vo + 16u * i, so, 0);
                w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
            }
        }
    }
    __device__ __forceinline__ void one(int e, __amdgpu_buffer_rsrc_t b, uint32_t vo, int so) {
        if constexpr (DT == kF32) w[e] = __builtin_amdgcn_raw_buffer_load_b32(b, vo, so, 0);
        else w[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b, vo, so, 0);
    }
    // fp32: value e; 16-bit: the operand of an instruction that takes all eight
    __device__ __forceinline__ float get(int e) const { return __uint_as_float(w[e]); }
    __device__ __forceinline__ uint4 all() const {
        if constexpr (VEC) return make_uint4(w[0], w[1], w[2], w[3]);
        return make_uint4(w[0] | (w[1] << 16), w[2] | (w[3] << 16), w[4] | (w[5] << 16),
                          w[6] | (w[7] << 16));
    }
};

// 32-k blocks per batch, and (factors whose rank varies fastest) the 16-byte pieces of a batch's
// factor rows, which are contiguous: loaded 64 at a time, they reach the lanes that multiply
// them through the wave's own stretch of LDS.  Loading the values one by one instead bound
// the kernel on the address unit (9 instead of 2 loads per block: 10.9 us at 2048 x 4096, rank
// 8, and 26 for one row of 14336).
template <int DT, int NT> constexpr int lora_batch() { return NT == 1 ? 4 : NT == 2 ? 2 : 1; }
template <int DT, int NT> constexpr int lora_stage_loads() {
    return 32 * lora_batch<DT, NT>() * 16 * NT * (DT == kF32 ? 4 : 2) / 1024;
}

template <int DT, int NT, bool VEC, bool KMAJOR>
__device__ __forceinline__ void lora_mul_tile(const LoraMul& it, int64_t M,
                                              float (&red)[lora_waves<DT>()][NT * 256],
                                              uint4* stage) {
    constexpr uint32_t E = esize<DT>();
    constexpr int U = lora_batch<DT, NT>(), L = lora_stage_loads<DT, NT>();
    constexpr bool kStaged = VEC && !KMAJOR;
    constexpr int NW = lora_waves<DT>();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int64_t m0 = 16 * (int64_t)blockIdx.x;
    const int K = (int)it.K, r = (int)it.r;
    const int blocks = (K + 31) >> 5;
    const int b_begin = (int)((int64_t)blocks * wave / NW);
    const int b_end = (int)((int64_t)blocks * (wave + 1) / NW);
    const __amdgpu_buffer_rsrc_t xr = rows_buffer<DT>(it.x, m0, M, K, 16);
    const __amdgpu_buffer_rsrc_t fr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)it.f, (short)0, (int)(it.K * it.r * E), kRsrcWord3);
    stage += wave * (64 * L);

    struct Batch {
        Eight<DT, VEC> x[U];
        Eight<DT, VEC && KMAJOR> f[kStaged ? 1 : U][kStaged ? 1 : NT];
        u32x4 piece[kStaged ? L : 1];
    };
    // offsets of block 0: rows past M and columns past r lie past the buffers' ends
    const uint32_t xo = ((uint32_t)i16 * (uint32_t)K + 8 * g) * E;
    uint32_t fo[NT];  // staged: this lane's value of its block's first k in the stage
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int j = 16 * t + i16;
        if constexpr (kStaged)  // columns past r repeat the last one, never stored
            fo[t] = (uint32_t)(8 * g * r + (j < r ? j : r - 1)) * E;
        else
            fo[t] = j >= r ? kNoRecordOffset
                           : (KMAJOR ? (uint32_t)j * (uint32_t)K + 8 * g
                                     : (uint32_t)(8 * g * r + j)) * E;
    }
    const uint32_t fstep = KMAJOR ? E : (uint32_t)r * E;
    auto load = [&](Batch& f, int b) {
        if constexpr (kStaged) {
            // the batch's rows: those of blocks past the wave's last read zeros
            const int rows = 32 * (b_end - b < U ? b_end - b : U);
            const int bytes = rows > 0 ? rows * r * (int)E : 0;
#pragma unroll
            for (int l = 0; l < L; ++l) {
                const int o = (64 * l + lane) * 16;
                f.piece[l] = __builtin_amdgcn_raw_buffer_load_b128(
                    fr, o < bytes ? (uint32_t)o : kNoRecordOffset, (int)(32u * b * fstep), 0);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int bu = b + u, k = 32 * bu + 8 * g;
            const bool live = bu < b_end;  // wave-uniform: a block past the last reads zeros
            const int so = (int)(32u * bu * E), sf = (int)(32u * bu * fstep);
            if constexpr (VEC) {
                f.x[u].load(xr, live && k < K ? xo : kNoRecordOffset, so);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    f.x[u].one(e, xr, live && k + e < K ? xo + e * E : kNoRecordOffset, so);
            }
            if constexpr (!kStaged) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint32_t vo = live ? fo[t] : kNoRecordOffset;
                    if constexpr (VEC) {
                        f.f[u][t].load(fr, k < K ? vo : kNoRecordOffset, sf);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)  // k past K: past the end where r is fastest
                            f.f[u][t].one(
                                e, fr, KMAJOR && k + e >= K ? kNoRecordOffset : vo + e * fstep, sf);
                    }
                }
            }
        }
    };
    // two accumulators for a single tile: products in a row never wait for each other
    constexpr int NA = NT == 1 ? 2 : 1;
    f32x4 acc[NA][NT];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Batch& f) {
        if constexpr (kStaged) {
            // a wave's LDS accesses are carried out in order; the empty asms keep the compiler
            // from moving the differently typed reads over the writes
            asm volatile("" ::: "memory");
#pragma unroll
            for (int l = 0; l < L; ++l)
                stage[64 * l + lane] =
                    make_uint4(f.piece[l].x, f.piece[l].y, f.piece[l].z, f.piece[l].w);
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            Eight<DT, VEC && KMAJOR> v[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (kStaged) {
                    const char* p = reinterpret_cast<const char*>(stage) + fo[t];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        v[t].w[e] = *reinterpret_cast<const typename Elem<DT>::Bits*>(
                            p + (uint32_t)(32 * u + e) * fstep);
                } else {
                    v[t] = f.f[u][t];
                }
            }
            if constexpr (DT == kF32) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[e % NA][t] = mfma4(f.x[u].get(e), v[t].get(e), acc[e % NA][t]);
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[u % NA][t] = mfma16<DT>(f.x[u].all(), v[t].all(), acc[u % NA][t]);
            }
        }
    };
    Batch f0, f1;
    load(f0, b_begin);
    for (int b = b_begin; b < b_end; b += 2 * U) {
        load(f1, b + U);
        __builtin_amdgcn_sched_barrier(0);
        compute(f0);
        load(f0, b + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        if (b + U < b_end) compute(f1);
    }
    if constexpr (NA == 2) acc[0][0] += acc[NA - 1][0];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][t * 256 + (4 * g + q) * 16 + i16] = acc[0][t][q];
    __syncthreads();
    for (int i = threadIdx.x; i < NT * 256; i += 64 * NW) {
        float v = red[0][i];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[w][i];
        const int64_t m = m0 + ((i >> 4) & 15);
        const int j = 16 * (i >> 8) + (i & 15);
        if (m < M && j < r) it.out[m * it.ldo + j] = it.scaling * v;
    }
}

template <int DT, int NT, bool VEC>
__global__ __launch_bounds__(64 * lora_waves<DT>()) void lora_mul_kernel(LoraMulArgs args) {
    __shared__ float red[lora_waves<DT>()][NT * 256];
    __shared__ uint4 stage[VEC ? lora_waves<DT>() * 64 * lora_stage_loads<DT, NT>() : 1];
    LoraMul it = args.it[0];
#pragma unroll
    for (int i = 1; i < kLoraDownItems; ++i)
        if ((int)blockIdx.y == i) it = args.it[i];
    if (it.sk == 1) lora_mul_tile<DT, NT, VEC, true>(it, args.M, red, stage);
    else lora_mul_tile<DT, NT, VEC, false>(it, args.M, red, stage);
}

static bool lora_mul_ok(const LoraMul& it, int dt) {
    return it.K >= 1 && it.K < (1ll << 23) && ((uintptr_t)it.x & (dt == kF32 ? 3u : 1u)) == 0 &&
           ((uintptr_t)it.f & (dt == kF32 ? 3u : 1u)) == 0;
}

template <int DT, int NT>
static void launch_lora_mul_nt(const LoraMulArgs& args, int n, bool vec, hipStream_t s) {
    const dim3 grid((unsigned)((args.M + 15) / 16), (unsigned)n), block(64 * lora_waves<DT>());
    if (vec) hipLaunchKernelGGL((lora_mul_kernel<DT, NT, true>), grid, block, 0, s, args);
    else hipLaunchKernelGGL((lora_mul_kernel<DT, NT, false>), grid, block, 0, s, args);
}

template <int DT>
static hipError_t launch_lora_mul_dt(const LoraMulArgs& args, int n, hipStream_t s) {
    bool vec = true;
    int64_t r = 0;
    for (int i = 0; i < n; ++i) {
        const LoraMul& it = args.it[i];
        vec = vec && it.K % 8 == 0 && ((uintptr_t)it.x & 15u) == 0 &&
              ((uintptr_t)it.f & 15u) == 0;
        r = it.r > r ? it.r : r;
    }
    if (r <= 16) launch_lora_mul_nt<DT, 1>(args, n, vec, s);
    else if (r <= 32) launch_lora_mul_nt<DT, 2>(args, n, vec, s);
    else launch_lora_mul_nt<DT, 4>(args, n, vec, s);
    return hipGetLastError();
}

template <int DT>
static hipError_t launch_lora_rows_dt(const LoraMulArgs& args, int n, int rs, hipStream_t s) {
    const dim3 grid((unsigned)args.M, (unsigned)n), block(kLoraVecThreads);
    switch (rs) {
        case 1: hipLaunchKernelGGL((lora_row_kernel<DT, 1>), grid, block, 0, s, args); break;
        case 2: hipLaunchKernelGGL((lora_row_kernel<DT, 2>), grid, block, 0, s, args); break;
        case 4: hipLaunchKernelGGL((lora_row_kernel<DT, 4>), grid, block, 0, s, args); break;
        default: hipLaunchKernelGGL((lora_row_kernel<DT, 8>), grid, block, 0, s, args); break;
    }
    return hipGetLastError();
}

static bool lora_row_ok(const LoraMul& it) {
    return it.K % 8 == 0 && (it.sk == 1 || it.r % 8 == 0) && ((uintptr_t)it.x & 15u) == 0 &&
           ((uintptr_t)it.f & 15u) == 0;
}
static int lora_slices(int64_t r) { return r <= 8 ? 1 : r <= 16 ? 2 : r <= 32 ? 4 : 8; }

// The row form runs for up to 512 rows of one product: two workgroups per CU, all at once.  It
// reads the factor from L2 once per row but has its whole K in flight; tiles of 16 rows read it
// once per tile (us at K = 4096, rows against tiles: bf16 rank 8 512 rows 7.1 and 7.8, 640 rows
// 9.1 and 7.8; rank 64 12.9 and 13.7, 17.5 and 13.7; fp32 rank 8 12.1 and 12.6, 15.9 and 12.6).
// Of several products (a backward pass forms u and v in one launch) for fewer than 512: 300
// rows of 14336 and 4096 with rank 8 in bf16 take 14 us more in tiles, 512 rows of 4096 and
// 4096 with rank 64 21 us less.
static bool lora_row_form(int64_t M, int n) { return M < 512 || (M == 512 && n == 1); }
// Rows below which a factor that cannot be read in 16-byte pieces takes the general kernel.
constexpr int64_t kLoraGeneralBelow = 16;

// Whether the general kernel (a workgroup per row, value by value) is faster than tiles for x @ A:
// few ranks, and rows or factors that the tiles can only read value by value too.  Times in us
// fitted to ranks 1 to 33, 16 to 4096 rows and K = 256 to 14336; its choice is 0.5% from the
// faster form on average.  In us, general against tiles, 64 rows: fp32 rank 3, K = 4096 7.3 and
// 12.0, rank 12 17.6 and 12.0; bf16 rank 3, K = 256 3.1 and 4.0, K = 4096 8.3 and 7.3; bf16 rank 8,
// K = 1001 5.3 and 17.
static bool lora_general_faster(const LoraMul& it, int64_t M, int dt) {
    const bool half = dt != kF32;
    const bool vec = it.K % 8 == 0 && (((uintptr_t)it.x | (uintptr_t)it.f) & 15u) == 0;
    const double r = (double)it.r, k = it.K / 1024.0;
    if (it.r > (vec ? 16 : 32)) return false;
    // a workgroup's sums across its lanes, for as many ranks as its kernel has; and rows past one
    // workgroup per CU: their reads of A overlap, less so where its rows share the same channels
    const double sums = it.r <= 8 ? 3.0 : it.r <= 16 ? 3.6 : 5.2;
    const double more_sums = it.r <= 8 ? 0.45 : it.r <= 16 ? 1.1 : 2.2;
    const double rows = M > 256 ? M / 256.0 - 1.0 : 0.0;
    const double share = it.r % 8 == 0 ? 0.8 : it.r < 8 ? (half ? 0.3 : 0.35) : (half ? 0.4 : 0.6);
    const double per_k = (half ? 0.7 + 0.24 * r : 0.4 + 0.25 * r) * (it.r % 16 == 0 ? 1.7 : 1.0);
    const double general = sums + more_sums * rows + k * (1.0 + share * rows) * per_k;
    double tiles;
    if (half) {
        tiles = !vec ? 10.0 + k * (it.r > 16 ? 4.5 : 7.0)
                     : 5.0 + 0.55 * k > 2.8 + 1.14 * k ? 5.0 + 0.55 * k : 2.8 + 1.14 * k;
    } else {
        tiles = vec ? 4.8 + 2.0 * k : 6.5 + 5.7 * k;
    }
    return general < tiles;
}

// The n products of a launch (n <= kLoraDownItems).
static hipError_t launch_lora_mul(const LoraMulArgs& args, int n, int dt, hipStream_t s) {
    if (lora_row_form(args.M, n)) {
        bool rows = true;
        for (int i = 0; i < n; ++i)
            rows = rows && lora_row_ok(args.it[i]) &&
                   lora_slices(args.it[i].r) == lora_slices(args.it[0].r);
        if (rows) {
            const int rs = lora_slices(args.it[0].r);
            return dt == kF32   ? launch_lora_rows_dt<kF32>(args, n, rs, s)
                   : dt == kF16 ? launch_lora_rows_dt<kF16>(args, n, rs, s)
                                : launch_lora_rows_dt<kBF16>(args, n, rs, s);
        }
    }
    return dt == kF32   ? launch_lora_mul_dt<kF32>(args, n, s)
           : dt == kF16 ? launch_lora_mul_dt<kF16>(args, n, s)
                        : launch_lora_mul_dt<kBF16>(args, n, s);
}

// Gradients of the factors, g(c, j) = sum_m a[m, c] v[m, j] at out[c * oc + j * oj]: A's
// from x and v (oc = r, oj = 1), B's from gy and u (oc = 1, oj = N).
struct LoraGrad {
    const void* a;
    const float* v;
    void* out;
    int64_t C, oc, oj;
    int64_t at;  // first of this gradient's C r values in a split's partial sums
};
struct LoraGradArgs {
    LoraGrad it[2];
    float* part;     // fp32 partial sums of the row splits (gridDim.y > 1)
    int64_t M, total;  // total: values per split
    int r, blocks0;  // blocks0: workgroups of it[0]
};

// A wave owns 128 columns c: lane (g, i) loads a[m0 + g][8 i .. 8 i + 7], eight instructions
// of four rows each (instruction e: columns 8 i + e).  The workgroup's waves and gridDim.y
// split the rows.  VEC: rows of a hold whole aligned groups of eight.
// Every batch of rows is read through a buffer of its own (32-bit offsets, the same for all
// batches), so any M runs with any number of row splits.
constexpr int kLoraGradWaves = 8;

template <int DT, int NT, bool VEC>
__global__ __launch_bounds__(64 * kLoraGradWaves) void lora_grad_kernel(LoraGradArgs args) {
    __shared__ f32x4 red[kLoraGradWaves / 2][8 * NT][64];
    constexpr uint32_t E = esize<DT>();
    constexpr int U = NT == 1 ? 4 : 2;
    const bool second = (int)blockIdx.x >= args.blocks0;
    const LoraGrad it = second ? args.it[1] : args.it[0];
    const int block = (int)blockIdx.x - (second ? args.blocks0 : 0);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    const int r = args.r;
    const int64_t c0 = 128 * (int64_t)block + 8 * i16;  // this lane's columns
    const int64_t groups = (args.M + 3) >> 2;
    const int64_t parts = (int64_t)gridDim.y * kLoraGradWaves;
    const int64_t p = (int64_t)blockIdx.y * kLoraGradWaves + wave;
    const int64_t q_begin = groups * p / parts;
    const int64_t count = groups * (p + 1) / parts - q_begin;
    const int64_t m_begin = 4 * q_begin;
    struct Batch {
        RawX<DT, 8> a[U];
        uint32_t v[U][NT];
    };
    // offsets of a batch's rows; rows past the wave's last lie past the buffers' ends
    // (group u's rows of a: 4 u C values on, in the scalar offset, which the range check covers)
    uint32_t vo_a[VEC ? 1 : 8], vo_v[U][NT];
#pragma unroll
    for (int e = 0; e < (VEC ? 1 : 8); ++e)
        vo_a[e] = c0 + e < it.C ? ((uint32_t)g * (uint32_t)it.C + (uint32_t)(c0 + e)) * E
                                : kNoRecordOffset;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int j = 16 * t + i16;
            vo_v[u][t] = j < r ? (uint32_t)((4 * u + g) * r + j) * 4u : kNoRecordOffset;
        }
    const int so_a = (int)(4 * it.C * E);
    const int64_t m_end = m_begin + 4 * count < args.M ? m_begin + 4 * count : args.M;
    auto load = [&](Batch& f, int64_t q) {  // groups q .. q + U - 1
        const int64_t m = m_begin + 4 * q;
        const int rows = m < m_end ? (int)(m_end - m < 4 * U ? m_end - m : 4 * U) : 0;
        const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(static_cast<const char*>(it.a) + m * it.C * E), (short)0,
            (int)(rows * it.C * E), kRsrcWord3);
        const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(it.v + m * r), (short)0, rows * r * 4, kRsrcWord3);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (VEC) {
                f.a[u].load(ar, vo_a[0], u * so_a);
            } else {
                uint32_t w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if constexpr (DT == kF32)
                        w[e] = __builtin_amdgcn_raw_buffer_load_b32(ar, vo_a[e], u * so_a, 0);
                    else
                        w[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ar, vo_a[e],
                                                                              u * so_a, 0);
                }
                f.a[u].set(w);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
                f.v[u][t] = __builtin_amdgcn_raw_buffer_load_b32(vr, vo_v[u][t], 0, 0);
        }
    };
    f32x4 acc[8][NT];
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[e][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Batch& f) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[e][t] = mfma4(f.a[u].get(e), __uint_as_float(f.v[u][t]), acc[e][t]);
    };
    Batch f0, f1;
    load(f0, 0);
    for (int64_t q = 0; q < count; q += 2 * U) {
        load(f1, q + U);
        __builtin_amdgcn_sched_barrier(0);
        compute(f0);
        load(f0, q + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        if (q + U < count) compute(f1);
    }
#pragma unroll
    for (int h = kLoraGradWaves / 2; h >= 1; h /= 2) {
        if (wave >= h && wave < 2 * h) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int t = 0; t < NT; ++t) red[wave - h][NT * e + t][lane] = acc[e][t];
        }
        __syncthreads();
        if (wave < h) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[e][t] += red[wave][NT * e + t][lane];
        }
        __syncthreads();
    }
    if (wave != 0) return;
    float* part = args.part + (int64_t)blockIdx.y * args.total + it.at;
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t c = 128 * (int64_t)block + 8 * (4 * g + q) + e;
                const int j = 16 * t + i16;
                if (c >= it.C || j >= r) continue;
                const int64_t at = c * it.oc + j * it.oj;
                if (gridDim.y > 1) part[at] = acc[e][t][q];
                else store_from_f32<DT>(it.out, at, acc[e][t][q]);
            }
}

// The row splits' partial sums, rounded once to dtype.
template <int DT>
__global__ __launch_bounds__(256) void lora_grad_reduce_kernel(LoraGradArgs args, int splits,
                                                               int64_t n0) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= args.total) return;
    float v = args.part[i];
    for (int s = 1; s < splits; ++s) v += args.part[s * args.total + i];
    const LoraGrad& it = i < n0 ? args.it[0] : args.it[1];
    store_from_f32<DT>(it.out, i - it.at, v);
}

// Row splits: towards four waves per SIMD over the chip, at least 32 rows per wave.
static int64_t lora_grad_splits(int64_t M, int64_t blocks) {
    int64_t s = 4096 / (blocks * kLoraGradWaves);
    const int64_t most = M / (32 * kLoraGradWaves);
    if (s > most) s = most;
    if (s > 16) s = 16;
    return s < 1 ? 1 : s;
}

static int64_t lora_blocks(int64_t C) { return (C + 127) / 128; }

size_t lora_grads_bytes(int64_t M, int64_t N, int64_t K, int64_t r, bool need_a, bool need_b) {
    const int64_t blocks = (need_a ? lora_blocks(K) : 0) + (need_b ? lora_blocks(N) : 0);
    if (blocks == 0 || M < 1) return 0;
    const int64_t s = lora_grad_splits(M, blocks);
    return s > 1 ? (size_t)s * (size_t)((need_a ? K : 0) + (need_b ? N : 0)) * (size_t)r * 4 : 0;
}

template <int DT, int NT>
static void launch_lora_grad_nt(const LoraGradArgs& args, dim3 grid, bool vec, hipStream_t s) {
    const dim3 block(64 * kLoraGradWaves);
    if (vec) hipLaunchKernelGGL((lora_grad_kernel<DT, NT, true>), grid, block, 0, s, args);
    else hipLaunchKernelGGL((lora_grad_kernel<DT, NT, false>), grid, block, 0, s, args);
}

template <int DT>
static hipError_t launch_lora_grads_dt(const LoraGradArgs& args, int64_t blocks, int64_t splits,
                                       bool vec, int64_t n0, hipStream_t s) {
    const dim3 grid((unsigned)blocks, (unsigned)splits);
    if (args.r <= 16) launch_lora_grad_nt<DT, 1>(args, grid, vec, s);
    else if (args.r <= 32) launch_lora_grad_nt<DT, 2>(args, grid, vec, s);
    else launch_lora_grad_nt<DT, 4>(args, grid, vec, s);
    const hipError_t e = hipGetLastError();
    if (splits == 1 || e != hipSuccess) return e;
    hipLaunchKernelGGL((lora_grad_reduce_kernel<DT>), dim3((unsigned)((args.total + 255) / 256)),
                       dim3(256), 0, s, args, (int)splits, n0);
    return hipGetLastError();
}

hipError_t launch_lora_grads(const void* x, const void* gy, const float* u, const float* v,
                             int64_t M, int64_t N, int64_t K, int64_t r, int dt, void* grad_a,
                             void* grad_b, float* part, size_t part_bytes, hipStream_t stream) {
    if (M < 1 || r < 1 || r > kLoraMaxRank || K >= kLoraGradMaxWidth || N >= kLoraGradMaxWidth)
        return hipErrorInvalidValue;
    const LoraGrad ga{x, v, grad_a, K, r, 1, 0}, gb{gy, u, grad_b, N, 1, N, grad_a ? K * r : 0};
    LoraGradArgs args{};
    int n = 0;
    bool vec = true;
    int64_t blocks = 0;
    for (const LoraGrad* it : {&ga, &gb}) {
        if (!it->out) continue;
        vec = vec && it->C % 8 == 0 && ((uintptr_t)it->a & 15u) == 0;
        blocks += lora_blocks(it->C);
        if (n == 0) args.blocks0 = (int)blocks;
        args.total += it->C * r;
        args.it[n++] = *it;
    }
    if (n == 0) return hipSuccess;
    args.part = part;
    args.M = M;
    args.r = (int)r;
    int64_t splits = lora_grad_splits(M, blocks);
    const int64_t fit = part ? (int64_t)(part_bytes / ((size_t)args.total * 4)) : 0;
    if (splits > fit) splits = fit < 2 ? 1 : fit;
    const int64_t n0 = args.it[0].C * r;
    return dt == kF32   ? launch_lora_grads_dt<kF32>(args, blocks, splits, vec, n0, stream)
           : dt == kF16 ? launch_lora_grads_dt<kF16>(args, blocks, splits, vec, n0, stream)
                        : launch_lora_grads_dt<kBF16>(args, blocks, splits, vec, n0, stream);
}

hipError_t launch_lora_uv(const void* x, const void* gy, const void* a, const void* b,
                          float scaling, int64_t M, int64_t N, int64_t K, int64_t r, int dt,
                          float* u, float* v, hipStream_t stream) {
    LoraMulArgs args{};
    args.M = M;
    int n = 0;
    if (u) args.it[n++] = LoraMul{x, a, u, K, r, 1, r, r, scaling};
    if (v) args.it[n++] = LoraMul{gy, b, v, N, 1, N, r, r, scaling};
    if (n == 0) return hipSuccess;
    for (int i = 0; i < n; ++i)
        if (!lora_mul_ok(args.it[i], dt)) return hipErrorInvalidValue;
    return launch_lora_mul(args, n, dt, stream);
}

template <int DT>
static hipError_t lora_down_dt(const void* x, const void* a, int64_t M, int64_t K, int r,
                               float scaling, float* u, int64_t ldu, hipStream_t s) {
    const dim3 grid((unsigned)M), block(kLoraThreads);
    if (r <= 8) hipLaunchKernelGGL((lora_down_kernel<DT, 8>), grid, block, 0, s, x, a, u, K, r, scaling, ldu);
    else if (r <= 16) hipLaunchKernelGGL((lora_down_kernel<DT, 16>), grid, block, 0, s, x, a, u, K, r, scaling, ldu);
    else if (r <= 32) hipLaunchKernelGGL((lora_down_kernel<DT, 32>), grid, block, 0, s, x, a, u, K, r, scaling, ldu);
    else hipLaunchKernelGGL((lora_down_kernel<DT, 64>), grid, block, 0, s, x, a, u, K, r, scaling, ldu);
    return hipGetLastError();
}

hipError_t launch_lora_down(const void* x, int64_t M, int64_t K, int dt, const LoraDown* items,
                            int n, hipStream_t stream) {
    if (M <= 0 || n <= 0) return hipSuccess;
    if (M > 0x7FFFFFFF) return hipErrorInvalidValue;
    for (int i = 0; i < n; ++i)
        if (items[i].r < 1 || items[i].r > kLoraMaxRank) return hipErrorInvalidValue;
    LoraMulArgs args{};
    args.M = M;
    int k = 0;
    auto flush = [&]() -> hipError_t {
        const int count = k;
        k = 0;
        return count ? launch_lora_mul(args, count, dt, stream) : hipSuccess;
    };
    for (int i = 0; i < n; ++i) {
        const LoraMul it{x, items[i].a, items[i].u, K, items[i].r, 1, items[i].r, items[i].ldu,
                         items[i].scaling};
        // (a single rank of a short K: one chunk per lane is little work, and the general kernel
        // reads it in fewer steps: 64 bf16 rows of 256 3.0 and 3.4 us, of 1024 3.7 and 3.4)
        const bool rows = lora_row_form(M, n) && lora_row_ok(it) && (it.r > 1 || K >= 512);
        if (!lora_mul_ok(it, dt) ||
            (!rows && (M < kLoraGeneralBelow || lora_general_faster(it, M, dt)))) {
            hipError_t e;
            switch (dt) {
                case kF32: e = lora_down_dt<kF32>(x, it.f, M, K, (int)it.r, it.scaling, it.out, it.ldo, stream); break;
                case kF16: e = lora_down_dt<kF16>(x, it.f, M, K, (int)it.r, it.scaling, it.out, it.ldo, stream); break;
                default: e = lora_down_dt<kBF16>(x, it.f, M, K, (int)it.r, it.scaling, it.out, it.ldo, stream); break;
            }
            if (e != hipSuccess) return e;
            continue;
        }
        if (k > 0 && lora_slices(it.r) != lora_slices(args.it[0].r))
            if (hipError_t e = flush()) return e;
        args.it[k++] = it;
        if (k == kLoraDownItems)
            if (hipError_t e = flush()) return e;
    }
    return flush();
}

hipError_t launch_lora_down(const void* x, const void* a, int64_t M, int64_t K, int64_t r,
                            float scaling, int dt, float* u, int64_t ldu, hipStream_t stream) {
    const LoraDown it{a, u, r, ldu, scaling};
    return launch_lora_down(x, M, K, dt, &it, 1, stream);
}

}  // namespace ojx
