// Device helpers shared by the MhcPre kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "mhc_pre.h"
#include "mhc_pre_internal.h"

namespace mhc {
namespace dev {

typedef __bf16 bf16x8_t __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef float f32x4_t __attribute__((__vector_size__(4 * sizeof(float))));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

template <int N>
struct Shape {
    static constexpr int M = N * N + 2 * N;     // mix columns
    static constexpr int NT = (2 * M) / 16;     // [hi | lo] column tiles
    static constexpr int NTHI = (M + 15) / 16;  // tiles holding a hi column
};

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

__device__ __forceinline__ float f16_bits_to_f32(uint32_t h)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// Round-half-even conversions (v_cvt_pk_bf16_f32 / v_cvt_f16_f32).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f)
{
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}

__device__ __forceinline__ uint32_t f32_to_f16_bits(float f)
{
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}

template <bool kBf16>
__device__ __forceinline__ float x_to_f32(uint32_t bits)
{
    return kBf16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
}

template <bool kBf16>
__device__ __forceinline__ uint32_t f32_to_x(float f)
{
    return kBf16 ? f32_to_bf16_bits(f) : f32_to_f16_bits(f);
}

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// Two floats to a packed pair (a in the low half), round-half-even: one
// v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32, where two scalar conversions cost two
// conversions, a shift and an or.
__device__ __forceinline__ uint32_t pack2_bf16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
}

__device__ __forceinline__ uint32_t pack2_f16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, f16x2_t));
}

template <bool kBf16>
__device__ __forceinline__ uint32_t pack2_x(float a, float b)
{
    return kBf16 ? pack2_bf16(a, b) : pack2_f16(a, b);
}

// Packed bf16 hi + lo of two floats: hi = bf16(v), lo = bf16(v - hi), both
// round-half-even (v - hi is exact in fp32).
__device__ __forceinline__ void split2_bf16(float a, float b, uint32_t &hi, uint32_t &lo)
{
    hi = pack2_bf16(a, b);
    lo = pack2_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u));
}

// Unpack 8 16-bit values held in a u32x4 (element e in half e&1 of word e>>1).
template <bool kBf16>
__device__ __forceinline__ void unpack8(const u32x4_t &v, float (&f)[8])
{
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        f[2 * w] = x_to_f32<kBf16>(v[w] & 0xFFFFu);
        f[2 * w + 1] = x_to_f32<kBf16>(v[w] >> 16);
    }
}

__device__ __forceinline__ u32x4_t pack8_bf16(const float (&f)[8])
{
    u32x4_t r;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        r[w] = pack2_bf16(f[2 * w], f[2 * w + 1]);
    }
    return r;
}

// acc + sum of the squares of 8 packed 16-bit values, one fp32 FMA per value
// (unpacking a bf16 pair is one shift and one mask).
template <bool kBf16>
__device__ __forceinline__ float sumsq8(const u32x4_t &v, float acc)
{
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float lo, hi;
        if constexpr (kBf16) {
            lo = __uint_as_float(v[w] << 16);
            hi = __uint_as_float(v[w] & 0xFFFF0000u);
        } else {
            lo = f16_bits_to_f32(v[w] & 0xFFFFu);
            hi = f16_bits_to_f32(v[w] >> 16);
        }
        acc = __builtin_fmaf(lo, lo, acc);
        acc = __builtin_fmaf(hi, hi, acc);
    }
    return acc;
}

// Device-scope (cross-XCD coherent) accesses for data exchanged between
// workgroups inside one launch: global_store / global_load with the sc1
// scope bit.  They write through / read past the per-XCD L2 without the
// whole-cache write-back and invalidate that an agent-scope fence costs.
__device__ __forceinline__ void st_dev(float *p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float ld_dev(const float *p)
{
    return __hip_atomic_load(const_cast<float *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until every memory access this wave issued has completed (stores
// acknowledged at their scope), and keeps the compiler from moving memory
// accesses across the wait.  Placed between the device-scope data stores and
// the atomic that publishes them.
__device__ __forceinline__ void wait_all_memory()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// The value of lane l ^ 8 within each row of 16 lanes (DPP row_ror:8): a VALU
// move, where a shuffle would take an LDS round trip and a wait.
__device__ __forceinline__ float row_swap8(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, false));
}

__device__ __forceinline__ bf16x8_t as_bf16x8(const u32x4_t &v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ f32x4_t mfma16(const u32x4_t &a, const u32x4_t &b, const f32x4_t &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// Cache policies of the buffer instructions below.
constexpr int kCpolNt = 2;    // nontemporal: streamed once
constexpr int kCpolDev = 16;  // sc1: device scope, written through, read past the L1 and L2 of another XCD

constexpr int kPast = 0x40000000;  // an offset past every resource's end: reads zeros, stores nothing

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, bytes, 0x00020000);
}

template <int kCpol>
__device__ __forceinline__ u32x4_t load16(__amdgpu_buffer_rsrc_t r, int off)
{
    return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kCpol));
}

template <int kCpol>
__device__ __forceinline__ void store16(const u32x4_t &v, __amdgpu_buffer_rsrc_t r, int off)
{
    __builtin_amdgcn_raw_buffer_store_b128(
        __builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, v), r, off, 0, kCpol);
}

// Waits until at most `kOut` of this wave's vector-memory loads are still in
// flight (they complete in issue order), without waiting on LDS or exports.
template <int kOut>
__device__ __forceinline__ void wait_vm()
{
    static_assert(kOut >= 0 && kOut < 64, "vmcnt range");
    // s_waitcnt fields: vmcnt [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8].
    constexpr int imm = (kOut & 15) | ((kOut >> 4) << 14) | (7 << 4) | (15 << 8);
    __builtin_amdgcn_s_waitcnt(imm);
}

// Workgroup barrier that orders LDS only (no wait for outstanding global
// accesses, which __syncthreads() would add).
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Calls f(std::integral_constant<int, i>{}) for i = 0 .. kCount-1.
template <typename F, int... kIs>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, kIs...>)
{
    (f(std::integral_constant<int, kIs>{}), ...);
}
template <int kCount, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_seq(f, std::make_integer_sequence<int, kCount>{});
}

// A fragments of k-steps 2q and 2q + 1 from line-layout registers r0 (rows
// 0-7) and r1 (rows 8-15).  In a line register lane l holds row l & 7 and the
// 8 columns at 8(l >> 4) + 32((l >> 3) & 1) of a 64-column line; the A
// fragment wants row l & 15 and columns 8(l >> 4) of its k-step, so lanes
// with bit 3 set take the other register's lane l ^ 8 (DPP row_ror:8 with
// banks 2-3 or 0-1 enabled).
__device__ __forceinline__ void lines_to_frags(const u32x4_t &r0, const u32x4_t &r1, u32x4_t &k0,
                                               u32x4_t &k1)
{
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        k0[w] = (uint32_t)__builtin_amdgcn_update_dpp((int)r0[w], (int)r1[w], 0x128, 0xF, 0xC, false);
        k1[w] = (uint32_t)__builtin_amdgcn_update_dpp((int)r1[w], (int)r0[w], 0x128, 0xF, 0x3, false);
    }
}

// One of the two.
template <int kStep>
__device__ __forceinline__ u32x4_t line_frag(const u32x4_t &r0, const u32x4_t &r1)
{
    u32x4_t k;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        k[w] = kStep == 0 ? (uint32_t)__builtin_amdgcn_update_dpp((int)r0[w], (int)r1[w], 0x128, 0xF, 0xC, false)
                          : (uint32_t)__builtin_amdgcn_update_dpp((int)r1[w], (int)r0[w], 0x128, 0xF, 0x3, false);
    }
    return k;
}

__device__ __forceinline__ f32x4_t mfma16_f16(const u32x4_t &a, const u32x4_t &b, const f32x4_t &c)
{
    typedef _Float16 f16x8_t __attribute__((__vector_size__(8 * sizeof(_Float16))));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// fp16 x -> exact bf16 pair: x = hi + lo (an fp16 significand has 11 bits).
__device__ __forceinline__ void split_f16_to_bf16(const float (&f)[8], u32x4_t &hi, u32x4_t &lo)
{
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t h, l;
        split2_bf16(f[2 * w], f[2 * w + 1], h, l);
        hi[w] = h;
        lo[w] = l;
    }
}

// The kernel's arguments, read again from the kernarg segment.  (Taken from the
// parameter, all of them stay in scalar registers from the start of the kernel
// to their last use, and large kernels spill.)
template <typename Args>
__device__ __forceinline__ const __attribute__((address_space(4))) Args *late_args()
{
    auto *p = (const __attribute__((address_space(4))) Args *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// The epoch of a launch, mixed into every exchange word's tag (LaunchTag).  One
// thread of every workgroup that the launch has (spare ones too, the words stay
// equal) calls replay_load early and launch_epoch once, later.
__device__ __forceinline__ uint32_t replay_load(uint32_t *words, int g)
{
    return words == nullptr
               ? 0u
               : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(make_rsrc(words + g, 4), 0, 0, kCpolDev);
}

template <typename Args>
__device__ __forceinline__ uint32_t launch_epoch(int g, uint32_t loaded)
{
    const auto *a = late_args<Args>();
    uint32_t *words = a->tag.words;
    if (words == nullptr) {
        return a->tag.seed;
    }
    const uint32_t replay = (loaded + 1u) & 0x7FFFFFFFu;
    __builtin_amdgcn_raw_buffer_store_b32(replay, make_rsrc(words + g, 4), 0, 0, kCpolDev);
    return mix32(loaded >= kFilledNumbers ? loaded : a->tag.seed | (replay & ((1u << kReplayBits) - 1u)));
}

// Whether workgroup g is one that gives up its waits at once (Plan::spinEvery).
__device__ __forceinline__ bool hurried(uint32_t every, int g) { return every != 0u && (uint32_t)g % every == 0u; }

// The status word's report of an expired wait whose work was done instead.
__device__ __forceinline__ void st_computed(void *hdr, uint32_t launchId)
{
    typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{kDeviceComputed, launchId}, make_rsrc(hdr, 8), 0, 0, kCpolDev);
}

// Quiet NaN written into the outputs of rows whose exchange wait expired.
__device__ __forceinline__ float poison() { return __uint_as_float(0x7FC00000u); }

// The caller's sticky status word (mhcPreExecutorSetStatusWord), if set: a
// workgroup whose bounded wait expired stores the public timeout status in
// it (a buffer store, device scope); nothing else writes it.
__device__ __forceinline__ void st_status_word(uint32_t *w)
{
    if (w != nullptr) {
        __builtin_amdgcn_raw_buffer_store_b32(
            (uint32_t)MHC_STATUS_DEVICE_TIMEOUT,
            __builtin_amdgcn_make_buffer_rsrc(w, (short)0, 4, 0x00020000), 0, 0, 16 /* sc1 */);
    }
}

// Sigmoid in the reference vector order (code/op_kernel/mhc_pre.cpp:542-555):
// scale, +bias, negate, exp, +1, reciprocal, +eps (only when eps != 0).
__device__ __forceinline__ float ref_sigmoid(float scaled, float bias, float eps)
{
    float v = scaled + bias;
    v = -v;
    v = expf(v);
    v = v + 1.0f;
    v = 1.0f / v;
    if (eps != 0.0f) {
        v = v + eps;
    }
    return v;
}

// invRms = 1 / sqrt(sumsq * invFlatDim + normEps) (code/op_kernel/mhc_pre.cpp:504-519).
__device__ __forceinline__ float ref_inv_rms(float sumsq, float invFlatDim, float normEps)
{
    float v = sumsq * invFlatDim;
    v = v + normEps;
    v = sqrtf(v);
    return 1.0f / v;
}

// The weights of a launch: phi [M][K] and gamma [K] or null, or the prepared
// fragments.
struct WeightsRef {
    const float *phi;
    const float *gamma;
    const u32x4_t *bprep;
    int K;
};

// The lane, opaque: what is derived from it is derived where it is used, not
// kept in registers from the start of the kernel.
__device__ __forceinline__ int lane_here()
{
    int l = (int)(threadIdx.x & 63);
    asm volatile("" : "+v"(l));
    return l;
}

// What a launch whose exchange wait expired computes instead, by any wave alone
// and in the order of the exchange, so that the outputs have the same bits.

// One 64-column strip's sums of a 16-row tile: mix column j (every lane its
// own; 0 from M on), in C fragments, and in lanes 16(r / 4) + r the sum of
// squares of row r.  xr: the tile's valid rows; col0: the strip's first column.
// kApart: hi and lo products in sums of their own, added at the end, and from
// column 16 Q on fp16's x_lo meets both (the strip kernel; the slab kernel adds
// all to one sum and x_lo meets hi only).
template <int N, bool kBf16, bool kApart>
__device__ __forceinline__ void strip_sums(const WeightsRef &wt, __amdgpu_buffer_rsrc_t xr, int D, int col0, int j,
                                           f32x4_t &sum, float &sq)
{
    constexpr int M = Shape<N>::M;
    constexpr int Q = M / 16;
    const int lane = lane_here();
    const int rl = lane & 15;
    const int K = wt.K;
    const bool prep = wt.bprep != nullptr;
    const bool hasGamma = wt.gamma != nullptr;
    const __amdgpu_buffer_rsrc_t pr = make_rsrc(wt.phi, prep ? 0 : M * K * 4);
    const __amdgpu_buffer_rsrc_t gr = make_rsrc(wt.gamma, hasGamma ? K * 4 : 0);
    const __amdgpu_buffer_rsrc_t br = make_rsrc(wt.bprep, prep ? M * K * 4 : 0);
    // hi and lo of the prepared value (k, j): tiles j / 16 and Q + j / 16, or
    // (j >= 16 Q) lanes j % 16 and + 8 of tile 2Q.
    const bool half = j >= 16 * Q;
    const int tile = half ? 2 * Q : j >> 4;
    const int loOff = half ? 8 * 16 : Q * 64 * 16;
    f32x4_t hiSum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t loSum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t gram = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int s = 0; s < N; ++s) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int dc = col0 + 32 * q + 8 * (lane >> 4);
            const int k = s * D + dc;
            const bool live = dc < D;
            const u32x4_t xf = load16<0>(xr, live ? (rl * K + k) * 2 : kPast);
            u32x4_t hi, lo;
            if (prep) {
                const int f = (((k >> 5) * Shape<N>::NT + tile) * 64 + 16 * ((k >> 3) & 3) + (j & 15)) * 16;
                const int off = live && j < M ? f : kPast;
                hi = load16<0>(br, off);
                lo = load16<0>(br, off + loOff);
            } else {
                const int off = live && j < M ? (j * K + k) * 4 : kPast;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const u32x4_t pv = load16<0>(pr, off + 16 * h);
                    const u32x4_t gv = load16<0>(gr, live && hasGamma ? (k + 4 * h) * 4 : kPast);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float a = __uint_as_float(pv[2 * e]);
                        float c = __uint_as_float(pv[2 * e + 1]);
                        if (hasGamma) {
                            a = a * __uint_as_float(gv[2 * e]);
                            c = c * __uint_as_float(gv[2 * e + 1]);
                        }
                        uint32_t hw, lw;
                        split2_bf16(a, c, hw, lw);
                        hi[2 * h + e] = hw;
                        lo[2 * h + e] = lw;
                    }
                }
            }
            u32x4_t xh = xf;
            u32x4_t xl = u32x4_t{0u, 0u, 0u, 0u};
            if constexpr (kBf16) {
                gram = mfma16(xf, xf, gram);
            } else {
                gram = mfma16_f16(xf, xf, gram);
                float f[8];
                unpack8<false>(xf, f);
                split_f16_to_bf16(f, xh, xl);
            }
            hiSum = mfma16(xh, hi, hiSum);
            if constexpr (!kBf16) {
                hiSum = mfma16(xl, hi, hiSum);
            }
            if constexpr (kApart) {
                loSum = mfma16(xh, lo, loSum);
                if constexpr (!kBf16) {
                    const f32x4_t both = mfma16(xl, lo, loSum);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        loSum[e] = half ? both[e] : loSum[e];
                    }
                }
            } else {
                hiSum = mfma16(xh, lo, hiSum);
            }
        }
    }
    sum = kApart ? hiSum + loSum : hiSum;
    const int di = rl & 3;
    sq = di == 0 ? gram[0] : di == 1 ? gram[1] : di == 2 ? gram[2] : gram[3];
}

// The sums of the slices g, g + G, ... of P, each of kStrips strips.
template <int N, bool kBf16, bool kApart, int kStrips>
__device__ __forceinline__ void group_sums(const WeightsRef &wt, __amdgpu_buffer_rsrc_t xr, int D, int P, int j,
                                           int g, int G, f32x4_t &sum, float &sq)
{
    sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    sq = 0.f;
#pragma unroll 1
    for (int p = g; p < P; p += G) {
        f32x4_t slice;
        float sliceSq;
#pragma unroll 1
        for (int st = 0; st < kStrips; ++st) {
            f32x4_t v;
            float u;
            strip_sums<N, kBf16, kApart>(wt, xr, D, 64 * (kStrips * p + st), j, v, u);
            slice = st == 0 ? v : slice + v;
            sliceSq = st == 0 ? u : sliceSq + u;
        }
        sum = sum + slice;
        sq = sq + sliceSq;
    }
}

// The resource of the valid rows of tile rt of x.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const uint16_t *x, int64_t T, int K, int64_t rt)
{
    const int rows = (int)min((int64_t)16, T - 16 * rt);
    return make_rsrc(x + 16 * rt * K, rows * K * 2);
}

// hIn of one wave's 64 columns from col0 of tile rt, with the tile's hPre from
// all of its P slices, added in G groups.
template <int N, bool kBf16, bool kApart, int kStrips>
__device__ __forceinline__ void own_hin(const WeightsRef &wt, const uint16_t *x, uint16_t *hIn, const float *alpha,
                                        const float *bias, int64_t T, int D, int64_t rt, int P, int G, int col0,
                                        float invFlatDim, float normEps, float hcEps)
{
    const int lane = lane_here();
    const int rl = lane & 15;
    const int grp = lane >> 4;
    const __amdgpu_buffer_rsrc_t xr = tile_rsrc(x, T, wt.K, rt);
    f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float sq = 0.f;
#pragma unroll 1
    for (int g = 0; g < G; ++g) {
        f32x4_t v;
        float u;
        group_sums<N, kBf16, kApart, kStrips>(wt, xr, D, P, rl, g, G, v, u);
        sum = sum + v;
        sq = sq + u;
    }
    f32x4_t pre;  // lane (stream, grp): rows 4 grp .. + 3
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float ir = ref_inv_rms(__shfl(sq, 20 * grp + e), invFlatDim, normEps);
        pre[e] = ref_sigmoid(sum[e] * (ir * alpha[0]), bias[rl < N ? rl : 0], hcEps);
    }
    const int rows = (int)min((int64_t)16, T - 16 * rt);
    const __amdgpu_buffer_rsrc_t hr = make_rsrc(hIn + 16 * rt * D, rows * D * 2);
    const int col = col0 + 8 * grp + 32 * ((lane >> 3) & 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = 8 * h + (lane & 7);
        float hv[8];
#pragma unroll
        for (int s = 0; s < N; ++s) {
            // Row `row` of stream s: lane 16 (row / 4) + s, element row % 4.
            float pv = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = __shfl(pre[e], 16 * (row >> 2) + s);
                pv = (row & 3) == e ? v : pv;
            }
            float f[8];
            unpack8<kBf16>(load16<0>(xr, col < D ? (row * wt.K + s * D + col) * 2 : kPast), f);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float prod = pv * f[e];
                hv[e] = s == 0 ? prod : hv[e] + prod;
            }
        }
        u32x4_t out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            out[e] = pack2_x<kBf16>(hv[2 * e], hv[2 * e + 1]);
        }
        store16<0>(out, hr, col < D ? (row * D + col) * 2 : kPast);
    }
}

}  // namespace dev
}  // namespace mhc
