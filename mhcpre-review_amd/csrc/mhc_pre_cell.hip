// Cell kernel for gfx950 (any n, small batches): one launch in place of the
// small-batch GEMM and its epilogue.
//
// What bounds a small batch is not bytes but steps.  Two dependent launches (the
// small-batch GEMM and its epilogue) cost the host about 9 us, and the epilogue
// starts over with partial sums and x that the GEMM had on the chip.  Here
// workgroup (column tile, row tile, slice) holds 64 NS columns of all n streams
// of 16 rows and the weights of 16 mix columns for them, one wave per stream
// and 64-column strip (2 k-steps each).  It writes its sums as one record and
// reads those of the P slices of its row and column tile: one exchange between
// workgroups.  The workgroups of column tile 0 evaluate hPre for themselves and
// write hIn from the x they still hold; the other columns are shared out over
// the slices.
//
// One column tile per workgroup, because building B (about 14 vector
// instructions per pair of weights) and reading phi are what a CU spends its
// time on: with all columns in one workgroup the kernel took 7.2, 10.2 and 7.4
// us at n = 6, D = 256, T = 16, n = 8 the same, and n = 4, D = 2560, T = 16, now
// 5.9, 6.1 and 6.5.  phi is read as whole 128-byte lines and turned into
// fragments by lane swaps (16 bytes per lane of a row each: 8.1 us in the first
// of these).  All that a workgroup needs of the records is read at once: a
// second read for hPost and hRes after hIn cost 2 us.
//
// Measured on MI355X (bf16, gamma, us per call back to back and in a graph of
// calls; before: the two launches): n = 4, D = 256, T = 128 7.1 and 5.5, before
// 10.6 and 7.5; n = 4, D = 7168, T = 16 7.3 and 7.3, before 10.4 and 8.6; n = 6,
// D = 1024, T = 64 7.1 and 7.0, before 10.6 and 8.6; n = 8, D = 1024, T = 32 7.2
// and 7.2, before 11.0 and 10.6.  What is left is the chain of launch, loads,
// record out and records in (an empty launch takes 2.5 to 3 us in a graph); the
// bytes alone take under 1 us.
//
// Every record word is 8 bytes, the fp32 bits and a tag (a hash of the word's
// position XOR the launch's epoch, see launch_epoch), read and written as one
// access at device scope; a word is current exactly when its tag matches, so
// the workspace needs no clearing.  The grid is at most what
// the device holds at once.  Waits are bounded: a workgroup whose wait expires
// (another kernel holds the CUs that the rest needs) computes every slice's
// sums itself, in the order of the exchange, so such a launch is slow and its
// bits are the same.

#include "mhc_pre_device.h"
#include "mhc_pre_internal.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mhc {
namespace {

using namespace dev;

template <int N, int NS>
struct Cell {
    static constexpr int M = Shape<N>::M;
    static constexpr int Q = M / 16;             // whole column tiles
    static constexpr int NT = Shape<N>::NT;      // prepared fragments per k-step
    static constexpr int W = N * NS;             // waves
    static constexpr int kThreads = 64 * W;
    // Record, in 16-byte chunks of two tagged words: chunk 8c + r holds rows 2r
    // and 2r + 1 of column c; column 0 is the sum of squares, c + 1 column c of
    // the workgroup's column tile.
    static constexpr int COLS = 17;
    static constexpr int CHUNKS = COLS * 8;
    static constexpr int WORDS = COLS * 16;
    static constexpr int kPitch = 20;            // floats per column of a wave's sums (distinct LDS banks)
    static constexpr int kMaxLoads = NS == 1 || N == 4 ? 8 : N == 6 ? 6 : 4;  // record loads in flight per thread
    static constexpr int kWavesPerSimd = NS == 1 || N == 4 ? 4 : N;
};

struct CellArgs {
    const uint16_t *x;
    const float *phi;
    const float *gamma;
    const u32x4_t *bprep;  // prepared B fragments [K/32][NT][64] (kPrep only)
    const float *alpha;
    const float *bias;
    uint16_t *hIn;
    float *hPost;
    float *hRes;
    float *hPre;
    uint64_t *recs;  // [column tile][row tile][P] records
    LaunchTag tag;
    char *hdr;  // workspace header: the status word
    uint32_t launchId;
    int T;
    int D;
    int K;
    int P;
    float normEps;
    float hcEps;
    float invFlatDim;
    uint32_t spinLimit;
    uint32_t spinEvery;
};

__device__ __forceinline__ uint32_t rec_tag(uint32_t pos, uint32_t epoch) { return (pos * 0x9E3779B1u) ^ epoch; }

template <int N, int NS, bool kBf16, bool kPrep>
__global__ __launch_bounds__((Cell<N, NS>::kThreads), (Cell<N, NS>::kWavesPerSimd)) void cell_kernel(CellArgs a)
{
    using Z = Cell<N, NS>;
    constexpr int M = Z::M;
    constexpr int Q = Z::Q;
    constexpr int NT = Z::NT;
    constexpr int W = Z::W;
    __shared__ __attribute__((aligned(16))) u32x4_t xsh[N][NS][2][64];  // x, line registers
    __shared__ __attribute__((aligned(16))) float part[W][Z::COLS * Z::kPitch];
    __shared__ __attribute__((aligned(16))) float2 sums[Z::kThreads];  // [slice group][item]
    __shared__ float pre[N][16];
    __shared__ uint32_t epochSh;
    __shared__ uint32_t expiredSh;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int P = a.P;
    // Column tile 0 first: its workgroups' wait is the longest way.
    const int p = blockIdx.x;
    const int tile = blockIdx.y;
    const int ct = blockIdx.z;
    const int group = ct * (int)gridDim.y + tile;
    const uint32_t replays = tid == 0 ? replay_load(a.tag.words, group * P + p) : 0u;
    const bool half = (M & 15) != 0 && ct == Q;  // 8 columns; lanes 8-15 of a row of 16 repeat them
    const int s = w % N;       // the wave's stream
    const int strip = w / N;   // and strip
    const int rl = lane & 15;
    const int grp = lane >> 4;
    const int Ki = a.K;
    const int Di = a.D;
    const int rows = min(16, a.T - 16 * tile);
    const int lineOff = 8 * grp + 32 * ((lane >> 3) & 1);

    // Thread t < count finishes chunk `chunk` of the sums (below), mix column j
    // (8 and up; chunks 0 .. 7 are the sum of squares).  Every workgroup needs
    // the first `crit` chunks.
    const int crit = ct == 0 ? 8 * (N + 1) : 8;
    const int rest = (half ? 72 : Z::CHUNKS) - crit;
    const int count = crit + (rest - p + P - 1) / P;
    const int chunk = tid < crit ? tid : crit + p + P * (tid - crit);
    const int j = 16 * ct + (chunk >> 3) - 1;
    float alpha = 0.f;
    float bias = 0.f;
    if (tid >= 8 && tid < count) {
        alpha = a.alpha[j < N ? 0 : j < 2 * N ? 1 : 2];
        bias = a.bias[j];
    }

    // The sums of slice q over its columns, wave by wave into part[], and its x
    // in xl: a function of the slice alone.
    const auto slice = [&](int q0, u32x4_t (&xl)[2]) {
        const int col0 = (q0 * NS + strip) * 64;
        // Every load goes out before the first use: the weights of the wave's 2
        // k-steps, prepared in fragment order (lane l: k = 32q + 8(l / 16) .. + 7 of
        // the strip, column 16t + l % 16), plain as whole lines (register h, lane l:
        // column 16t + 8h + l % 8, 4 of the k-step's 32 values); columns of x past
        // D read zeros ...
        u32x4_t B[2][2];  // [k-step][hi, lo]
        u32x4_t pv[2][2];
        u32x4_t gv[2];
        const bool hasGamma = a.gamma != nullptr;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if constexpr (kPrep) {
                // Tiles ct and Q + ct, or (the half tile) lanes l % 8 and + 8 of 2Q.
                const __amdgpu_buffer_rsrc_t r = make_rsrc(a.bprep, M * Ki * 4);
                const int dc = col0 + 32 * q + 8 * grp;
                const int k = s * Di + dc;
                const int f =
                    ((k >> 5) * NT * 64 + 16 * ((k >> 3) & 3) + (half ? 128 * Q + (rl & 7) : 64 * ct + rl)) * 16;
                B[q][0] = load16<0>(r, dc < Di ? f : kPast);
                B[q][1] = load16<0>(r, dc < Di ? f + (half ? 128 : 1024 * Q) : kPast);
            } else {
                const __amdgpu_buffer_rsrc_t phiR = make_rsrc(a.phi, M * Ki * 4);
                const __amdgpu_buffer_rsrc_t gamR = make_rsrc(a.gamma, hasGamma ? Ki * 4 : 0);
                const int dc = col0 + 32 * q + 8 * grp + 4 * ((lane >> 3) & 1);
                const int k = s * Di + dc;
                gv[q] = load16<0>(gamR, dc < Di ? k * 4 : kPast);
                pv[q][0] = load16<0>(phiR, dc < Di ? ((16 * ct + (lane & 7)) * Ki + k) * 4 : kPast);
                pv[q][1] = load16<0>(phiR, dc < Di ? ((16 * ct + (half ? 0 : 8) + (lane & 7)) * Ki + k) * 4 : kPast);
            }
        }
        // ... and x as whole lines: register h, lane l: row 8h + l % 8 and the 8
        // columns at lineOff of the strip; rows past T and columns past D are zeros.
        {
            const __amdgpu_buffer_rsrc_t r = make_rsrc(a.x + (int64_t)tile * 16 * Ki, rows * Ki * 2);
            const int col = col0 + lineOff;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                xl[h] = load16<kCpolNt>(r, col < Di ? ((8 * h + (lane & 7)) * Ki + s * Di + col) * 2 : kPast);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!kPrep) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                // gamma phi in line order; then 4 columns 8 (l / 16) .. of the
                // k-step in f[0] and the next 4 in f[1].
                u32x4_t f[2];
                if (hasGamma) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            pv[q][h][e] = __float_as_uint(__uint_as_float(pv[q][h][e]) * __uint_as_float(gv[q][e]));
                        }
                    }
                }
                lines_to_frags(pv[q][0], pv[q][1], f[0], f[1]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t h, l;
                    split2_bf16(__uint_as_float(f[e >> 1][2 * (e & 1)]), __uint_as_float(f[e >> 1][2 * (e & 1) + 1]),
                                h, l);
                    B[q][0][e] = h;
                    B[q][1][e] = l;
                }
            }
        }

        f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
        f32x4_t gram = f32x4_t{0.f, 0.f, 0.f, 0.f};
        {
            u32x4_t kf[2];
            lines_to_frags(xl[0], xl[1], kf[0], kf[1]);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                u32x4_t xh = kf[q];
                if constexpr (kBf16) {
                    gram = mfma16(kf[q], kf[q], gram);
                } else {
                    // fp16 x = hi + lo exactly in bf16; x_lo meets the hi columns
                    // only (x_lo * B_lo is below 2^-16 of the product).
                    gram = mfma16_f16(kf[q], kf[q], gram);
                    u32x4_t xlo;
                    float f[8];
                    unpack8<false>(kf[q], f);
                    split_f16_to_bf16(f, xh, xlo);
                    acc = mfma16(xlo, B[q][0], acc);
                }
                acc = mfma16(xh, B[q][0], acc);
                acc = mfma16(xh, B[q][1], acc);
            }
        }
        // The wave's sums and x into LDS.  C fragment: lane (rl, grp) holds rows 4
        // grp .. + 3 of column rl; Gram diagonal: row r in lane 16(r / 4) + r,
        // register r % 4.
        *reinterpret_cast<f32x4_t *>(&part[w][(rl + 1) * Z::kPitch + 4 * grp]) = acc;
        const int di = rl & 3;
        const float sq = di == 0 ? gram[0] : di == 1 ? gram[1] : di == 2 ? gram[2] : gram[3];
        if ((rl >> 2) == grp) {
            part[w][rl] = sq;
        }
    };
    // Chunk c of the slice: the waves' sums in wave order.
    const auto chunk_sum = [&](int c) {
        const int at = (c >> 3) * Z::kPitch + 2 * (c & 7);
        float2 v = *reinterpret_cast<const float2 *>(&part[0][at]);
#pragma unroll
        for (int i = 1; i < W; ++i) {
            const float2 u = *reinterpret_cast<const float2 *>(&part[i][at]);
            v.x = v.x + u.x;
            v.y = v.y + u.y;
        }
        return v;
    };

    if (tid == 0) {
        expiredSh = 0;
    }
    u32x4_t xl[2];
    slice(p, xl);
    if (ct == 0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            xsh[s][strip][h][lane] = xl[h];
        }
    }
    if (tid == 0) {
        epochSh = launch_epoch<CellArgs>(group * P + p, replays);
    }
    lds_barrier();
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(epochSh);

    // The record.
    const uint32_t tileBase = (uint32_t)(group * P) * (uint32_t)Z::WORDS;
    const __amdgpu_buffer_rsrc_t tr = make_rsrc(a.recs + (size_t)group * P * Z::WORDS, P * Z::WORDS * 8);
    if (tid < Z::CHUNKS) {
        const float2 v = chunk_sum(tid);
        const int word = p * Z::WORDS + 2 * tid;
        u32x4_t wv;
        wv[0] = __float_as_uint(v.x);
        wv[1] = rec_tag(tileBase + (uint32_t)word, epoch);
        wv[2] = __float_as_uint(v.y);
        wv[3] = rec_tag(tileBase + (uint32_t)word + 1u, epoch);
        store16<kCpolDev>(wv, tr, 8 * word);
    }

    // The sums over the tile's slices: the chunks hPre needs and, of the others,
    // every P-th.  Thread t takes item t % most of slice group t / most and
    // adds slices g, g + G, ...; the groups' sums are added in order.  (`most`,
    // the largest count, so that every slice adds in the same order: hPre comes
    // out the same in all of them.)
    const int most = crit + (rest + P - 1) / P;
    bool expired = false;
    int groups = min(P, Z::kThreads / most);
    {
        const int item = tid % most;
        const int g = tid / most;
        const bool act = g < groups && item < count;
        const int word = 2 * (item < crit ? item : crit + p + P * (item - crit));
        const int each = (P + groups - 1) / groups;
        float2 acc2 = make_float2(0.f, 0.f);
        bool need = act;
        for (uint32_t spins = 0;; ++spins) {
            // (A lane that has its sums reads nothing more.  The offsets and tags
            // are worked out anew each time: hoisted, they would spill.)
            int at = word;
            asm volatile("" : "+v"(at));
            uint32_t stale = 0;
            float2 v = make_float2(0.f, 0.f);
            for (int u0 = 0; u0 < each; u0 += Z::kMaxLoads) {
                u32x4_t t[Z::kMaxLoads];
#pragma unroll
                for (int u = 0; u < Z::kMaxLoads; ++u) {
                    const int q = g + groups * (u0 + u);
                    if (u0 + u < each) {  // (the same for the whole workgroup)
                        t[u] = load16<kCpolDev>(tr, need && q < P ? 8 * (q * Z::WORDS + at) : kPast);
                    }
                }
#pragma unroll
                for (int u = 0; u < Z::kMaxLoads; ++u) {
                    const int q = g + groups * (u0 + u);
                    if (u0 + u < each) {
                        const uint32_t pos = tileBase + (uint32_t)(q * Z::WORDS + at);
                        const uint32_t diff = (t[u][1] ^ rec_tag(pos, epoch)) | (t[u][3] ^ rec_tag(pos + 1u, epoch));
                        stale |= q < P ? diff : 0u;
                        v.x = v.x + __uint_as_float(t[u][0]);
                        v.y = v.y + __uint_as_float(t[u][2]);
                    }
                }
            }
            if (need && stale == 0) {
                acc2 = v;
                need = false;
            }
            if (!__any(need)) {
                break;
            }
            if (spins >= a.spinLimit) {
                if (lane == 0) {
                    expiredSh = 1;
                }
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (act) {
            sums[g * most + item] = acc2;
        }
        lds_barrier();
        expired = expiredSh != 0;
    }
    if (expired || hurried(a.spinEvery, group * P + p)) {
        // Every slice's sums once more, added in the same order: the same bits.
        if (tid == 0) {
            const auto *la = late_args<CellArgs>();
            st_computed(la->hdr, la->launchId);
        }
        float2 sum = make_float2(0.f, 0.f);
#pragma unroll 1
        for (int g = 0; g < groups; ++g) {
            float2 v = make_float2(0.f, 0.f);
#pragma unroll 1
            for (int q = g; q < P; q += groups) {
                lds_barrier();  // (part[] and the sums have been read)
                u32x4_t unused[2];
                slice(q, unused);
                lds_barrier();
                if (tid < count) {
                    const float2 u = chunk_sum(chunk);
                    v.x = v.x + u.x;
                    v.y = v.y + u.y;
                }
            }
            sum.x = g == 0 ? v.x : sum.x + v.x;
            sum.y = g == 0 ? v.y : sum.y + v.y;
        }
        if (tid < count) {
            sums[tid] = sum;
        }
        groups = 1;
        lds_barrier();
    }
    if (tid >= 8 && tid < count) {
        const auto total = [&](int item) {
            float2 v = sums[item];
            for (int g = 1; g < groups; ++g) {
                const float2 u = sums[g * most + item];
                v.x = v.x + u.x;
                v.y = v.y + u.y;
            }
            return v;
        };
        const float2 mix = total(tid);
        const float2 ss = total(chunk & 7);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int r = 2 * (chunk & 7) + e;
            const int64_t row = (int64_t)tile * 16 + r;
            const float iv = ref_inv_rms(e == 0 ? ss.x : ss.y, a.invFlatDim, a.normEps);
            const float scaled = (e == 0 ? mix.x : mix.y) * (iv * alpha);
            if (j < 2 * N) {
                const float v = ref_sigmoid(scaled, bias, j < N ? a.hcEps : 0.0f);
                if (j < N) {
                    pre[j][r] = v;
                    if (a.hPre != nullptr && p == 0 && r < rows) {
                        a.hPre[row * N + j] = v;
                    }
                } else if (r < rows) {
                    a.hPost[row * N + (j - N)] = v * 2.0f;
                }
            } else if (r < rows) {
                a.hRes[row * (N * N) + (j - 2 * N)] = scaled + bias;
            }
        }
    }

    // hIn of this slice's columns: one line register's 8 columns per thread.
    if (ct == 0) {
        lds_barrier();
    }
    if (ct == 0 && tid < 128 * NS) {
        const int c = tid >> 7;
        const int h = (tid >> 6) & 1;
        const int row = 8 * h + (lane & 7);
        const int col = (p * NS + c) * 64 + lineOff;
        float hv[8];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float f[8];
            unpack8<kBf16>(xsh[i][c][h][lane], f);
            const float pv8 = pre[i][row];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float prod = pv8 * f[e];
                hv[e] = i == 0 ? prod : hv[e] + prod;
            }
        }
        u32x4_t out;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            out[e] = pack2_x<kBf16>(hv[2 * e], hv[2 * e + 1]);
        }
        store16<kCpolNt>(out, make_rsrc(a.hIn + (int64_t)tile * 16 * Di, rows * Di * 2),
                         col < Di ? (row * Di + col) * 2 : kPast);
    }
}

template <int N, int NS, bool kBf16, bool kPrep>
struct Instance {
    static int coresident(int numCUs)
    {
        int perCU = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &perCU, reinterpret_cast<const void *>(&cell_kernel<N, NS, kBf16, kPrep>), Cell<N, NS>::kThreads, 0) !=
            hipSuccess) {
            return -1;
        }
        return perCU * numCUs;
    }
    static hipError_t launch(const Plan &p, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream)
    {
        char *ws = static_cast<char *>(workspace);
        CellArgs a;
        a.x = static_cast<const uint16_t *>(p.x);
        a.phi = p.phi;
        a.gamma = p.hasGamma ? p.gamma : nullptr;
        a.bprep = static_cast<const u32x4_t *>(p.bprep);
        a.alpha = p.alpha;
        a.bias = p.bias;
        a.hIn = static_cast<uint16_t *>(p.hIn);
        a.hPost = p.hPost;
        a.hRes = p.hRes;
        a.hPre = p.hasHPre ? p.hPre : nullptr;
        a.recs = reinterpret_cast<uint64_t *>(ws + p.wsCellRecs);
        a.tag = tag;
        a.hdr = ws;
        a.launchId = launchId;
        a.T = (int)p.T;
        a.D = (int)p.D;
        a.K = (int)p.K;
        a.P = p.cellP;
        a.normEps = p.normEps;
        a.hcEps = p.hcEps;
        a.invFlatDim = p.invFlatDim;
        a.spinLimit = p.cellSpinLimit();
        a.spinEvery = p.spinEvery;
        const unsigned tiles = (unsigned)((p.T + 15) / 16);
        const dim3 grid((unsigned)p.cellP, tiles, (unsigned)(p.cellGrid / (p.cellP * tiles)));
        const dim3 block(Cell<N, NS>::kThreads);
        if (!p.fusedCooperative) {
            hipLaunchKernelGGL((cell_kernel<N, NS, kBf16, kPrep>), grid, block, 0, stream, a);
            return hipGetLastError();
        }
        void *args[] = {&a};
        return hipLaunchCooperativeKernel(reinterpret_cast<const void *>(&cell_kernel<N, NS, kBf16, kPrep>), grid, block,
                                          args, 0, stream);
    }
};

// Calls f(Instance<...>{}) for the plan's instance.
template <int N, typename F>
auto with_instance_n(const Plan &p, F &&f)
{
    const auto prep = [&](auto ns, auto bf16) {
        constexpr int NS = decltype(ns)::value;
        constexpr bool kBf16 = decltype(bf16)::value;
        return p.bprep != nullptr ? f(Instance<N, NS, kBf16, true>{}) : f(Instance<N, NS, kBf16, false>{});
    };
    const auto type = [&](auto ns) { return p.isBf16 ? prep(ns, std::true_type{}) : prep(ns, std::false_type{}); };
    return p.cellStrips == 2 ? type(std::integral_constant<int, 2>{}) : type(std::integral_constant<int, 1>{});
}
template <typename F>
auto with_instance(const Plan &p, F &&f)
{
    return p.n == 4 ? with_instance_n<4>(p, f) : p.n == 6 ? with_instance_n<6>(p, f) : with_instance_n<8>(p, f);
}

}  // namespace

size_t cell_record_bytes() { return 17 * 16 * 8; }

int cell_max_coresident(const Plan &p, int numCUs)
{
    return with_instance(p, [&](auto i) { return decltype(i)::coresident(numCUs); });
}

hipError_t launch_cell(const Plan &p, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream)
{
    return with_instance(p, [&](auto i) { return decltype(i)::launch(p, workspace, tag, launchId, stream); });
}

}  // namespace mhc
