// Slab kernel for gfx950 (n = 6): x is read from HBM once and held in VGPRs
// until its hIn is written, while the sums of a row's K-slices meet through
// exchange rings in memory.  The idea is the strip kernel's (n = 4); the shape
// is another because B = gamma * phi (bf16 hi + lo) takes twice the bytes per
// value of K and a record twice the columns.
//
// What bounds it: at n = 6, D = 4096, T = 4096 (bf16, prepared weights) a tile
// takes a team of 32 slices 1.6 us, 3.8 TB/s of x and hIn; the CUs' own chains
// (MFMA 1 us, the strips' meeting 0.7, hIn and the loads 1.4 per own step) and
// the reducers bound it, not HBM (the same accesses without arithmetic: 5.7
// TB/s).  Measured against the rows path's GEMM and second read of x: 96.9 ->
// 70.6 us; D = 1024, T = 2048 26.0 -> 21.4 us (split path before).
//
// Slice workgroup: 128 columns of each of the 6 streams (768 values of K),
// whose B (144 KB) stays in LDS for the whole launch.  8 waves: wave w holds
// strip w % 2 (64 columns of every stream) and belongs to group w / 2; group g
// takes the team steps g, g + 4, ... (its own steps jj), so that four tiles
// are in different phases on a CU and one group's exchange runs in the shadow
// of the others' loads.  A wave keeps a ring of four tiles (16 rows x 6
// streams x 64 columns, 48 VGPRs each).  Own step jj of a wave:
//   1. the poll for the hPre of own tile jj - 2;
//   2. the MFMAs of own tile jj (x in line registers, a DPP exchange to A
//      fragments, B from LDS) and a Gram MFMA whose diagonal is the sum of
//      squares;
//   3. the two strips of the group meet in LDS: strip 0 takes column tile 0
//      and the sum of squares of both, strip 1 tiles 1 and 2, and each writes
//      its part of the slice's record from registers, as tagged words;
//   4. hIn of own tile jj - 2, and the loads of own tile jj + 2 into its
//      registers.
// So a tile's loads have an own step (four tiles' time) to arrive, and its
// exchange has two.
//
// Team.  P = ceil(D / 128) slice workgroups and R reducer workgroups; team t
// takes the 16-row tiles t, t + numTeams, ...; its k-th tile is step k.  Teams
// live inside one XCD (workgroup g runs on XCD g mod X; the exchange then
// stays in that XCD's L2) or across the device (exchange words stored through
// to memory).  Placement affects speed only.
//
// Exchange words.  What the hPre of a tile waits for (its sum of squares and
// hPre columns) and every flag is an 8-byte word: the fp32 bits and a tag (a
// hash of the word's position XOR the launch's epoch), read and written as one
// access; a word is current exactly when its tag matches, so nothing is
// counted, reset or cleared.  The epoch is launch_epoch's: no other launch has
// it.  The hPost and hRes columns, five sixths of a record, are plain values:
// a wave stores its flag for step m an own step later, when a counter wait has
// shown that its stores of m are done, and readers look at the flag first.
//
// Reducers.  The waves of a team's reducer workgroups work alone, one tile at
// a time, without barriers: a tile's reduction is a chain of memory round
// trips (2 us and more while x streams), so many tiles have to be in work at
// once.  They add over the slices in slice order.  The first CC waves take the
// sum of squares and the hPre columns, of the steps k = class mod CC: they
// evaluate invRms and hPre and publish the broadcast block.  The others take
// one of three blocks of 14 hPost / hRes columns, of the steps k = class mod
// CR, and store the step they have finished reading in their "done" word; a
// broadcast of step u is published only when the done words say that the
// records of step u - 16 and before have all been read.
//
// Ring slots.  Step m uses slot m mod S, S = 28.  A wave writes its part of
// record m after the hIn of its own step jj - 3, step m - 12, so it has seen
// that step's broadcast.  Hence the hPost / hRes columns of step m - 28 and
// before have been read, and CC divides 16, so the wave that published step m
// - 12 has finished step m - 28, the slot's previous one.  Broadcast m is
// written only after every wave has written its part of record m, hence after
// each has used the broadcasts up to m - 12 of its group, and m - 28 is the
// same group's.
//
// Every wait on another workgroup is bounded.  A wave whose wait expires
// (another kernel holds the CUs the rest of the grid needs) computes what it
// was waiting for itself, from x and the weights in the order of the exchange,
// and goes on alone: such a launch is slow (6.3 ms at n = 6, D = 4096, T = 4096
// with every wait expired) and its bits are the same.  From then on a slice's
// wave writes nothing into the rings, whose slots are free only in the order
// above.

#include "mhc_pre_device.h"
#include "mhc_pre_internal.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mhc {
namespace {

using namespace dev;

constexpr int kStrips = 2;                 // 64-column strips per slice
constexpr int kGroups = 4;                 // wave groups, each on its own tiles
constexpr int kWaves = kStrips * kGroups;  // two per SIMD
constexpr int kThreads = kWaves * 64;
constexpr int kCols = 64 * kStrips;        // x columns of every stream per slice
constexpr int kRing = 4;                   // x tiles of a wave: in use, two waiting for hPre, loading
constexpr int kLag = 2;                    // hIn of own tile jj at own step jj + 2
constexpr int kRingSlots = 28;             // exchange ring slots (see above)
constexpr int kDoneLag = 16;               // steps a broadcast runs ahead of the other columns' reads
constexpr int kMaxSlices = 64;             // slices of a team
constexpr int kRestBlocks = 3;             // blocks of 14 hPost / hRes columns
constexpr int kRestCols = 14;
constexpr int kMaxRest = 48;               // waves that take them
static_assert(kRingSlots == kGroups * (kLag + 1) + kDoneLag, "ring slots");
constexpr int kXccIdReg = (3 << 11) | 20;  // s_getreg operand: HW_REG_XCC_ID, bits [3:0]

template <int N>
struct Geo {
    static constexpr int M = N * N + 2 * N;
    static constexpr int Q = M / 16;  // column tiles
    static constexpr int NT = 2 * Q;  // hi tiles, then lo tiles
    static constexpr int KS = 2 * N;  // 32-column k-steps of a strip
    static_assert(N == 6, "B of a slice fits LDS, and three column tiles split 1 : 2 over the strips");
    // Record of one (tile, slice), in 16-byte chunks, in the order in which the
    // slice's lanes hold them, so that every store instruction writes whole
    // 128-byte lines (a store of half lines costs masked writes):
    //   tagged, rows 2r and 2r + 1 of mix column j < 8: (r % 2) * 32 + 8(r / 2) + j;
    //   tagged, rows 2r and 2r + 1 of the sum of squares: kSqChunk + r;
    //   plain, rows 4q .. 4q + 3 of mix column j: kPlain + 64(j / 16) + 16q + j % 16.
    static constexpr int kSqChunk = 64;
    static constexpr int kPlain = kSqChunk + 8;
    static constexpr int CHUNKS = kPlain + 64 * Q;
    static constexpr int WORDS = 2 * CHUNKS;  // in 8-byte words
    __device__ static int crit_chunk(int j, int r) { return (r & 1) * 32 + 8 * (r >> 1) + j; }
    __device__ static int plain_chunk(int j, int q) { return kPlain + 64 * (j >> 4) + 16 * q + (j & 15); }
    static constexpr int BWORDS = N * 16;  // broadcast block: hPre, [stream][row]
};

struct SlabArgs {
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
    uint64_t *recs;   // [team][S][P] records
    uint64_t *flags;  // [team][S][P][2] words: strip 0 and 1 of the slice have stored their plain columns
    uint64_t *bcast;  // [team][S] broadcast blocks
    uint64_t *done;   // [team][kMaxRest] words: the latest step a wave has finished reading
    LaunchTag tag;
    char *hdr;        // workspace header: the status word
    uint32_t launchId;
    int64_t T;
    int64_t D;
    int64_t K;
    int RT;        // 16-row tiles
    int P;         // slices per team
    int R;         // reducer workgroups per team
    int CC;        // reducer waves of the hPre columns (1, 2, 4 or 8)
    int CR;        // reducer waves of each block of the others
    int nGroups;   // XCDs, or 1: teams across the device
    int perGroup;  // teams per group
    float normEps;
    float hcEps;
    float invFlatDim;
    uint32_t spinLimit;
    uint32_t spinEvery;
};

// (Each phase of the kernel loads the arguments that it uses.)
typedef const __attribute__((address_space(4))) SlabArgs *ArgsPtr;
__device__ __forceinline__ ArgsPtr phase_args() { return late_args<SlabArgs>(); }

__device__ __forceinline__ WeightsRef weights_of(ArgsPtr p) { return {p->phi, p->gamma, p->bprep, (int)p->K}; }

__device__ __forceinline__ uint32_t rec_tag(uint32_t pos, uint32_t epoch) { return (pos * 0x9E3779B1u) ^ epoch; }
__device__ __forceinline__ uint32_t bcast_tag(uint32_t pos, uint32_t epoch)
{
    return (pos * 0x85EBCA77u) ^ epoch ^ 0xC2B2AE3Du;
}
__device__ __forceinline__ uint32_t flag_tag(uint32_t pos, uint32_t epoch)
{
    return (pos * 0x165667B1u) ^ epoch ^ 0x9E3779B9u;
}
__device__ __forceinline__ uint32_t done_tag(uint32_t pos, uint32_t epoch)
{
    return (pos * 0xC2B2AE35u) ^ epoch ^ 0x27D4EB2Fu;
}

__device__ __forceinline__ void store_exchange(const u32x4_t &v, __amdgpu_buffer_rsrc_t r, int off, bool local)
{
    if (local) {
        store16<0>(v, r, off);
    } else {
        store16<kCpolDev>(v, r, off);
    }
}

// ---------------------------------------------------------------------------
// Reducer waves.  U: record loads in flight per lane (of a sum over the
// slices).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint2 load_word(__amdgpu_buffer_rsrc_t r, int off)
{
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kCpolDev));
}
template <int kCpol>
__device__ __forceinline__ void store_word(const uint2 &v, __amdgpu_buffer_rsrc_t r, int off)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned int, v), r,
                                          off, 0, kCpol);
}

// What the reducer waves of a team share.
template <int N>
struct Team {
    int team, ntiles, P, numTeams;
    bool local;
    uint32_t epoch, spinLimit;
    uint64_t *recs;
    __amdgpu_buffer_rsrc_t flags, done;
    uint32_t donePos;
    float invFlatDim, normEps;
    int64_t T;
    __device__ __forceinline__ Team(ArgsPtr ap, int t, int n, bool l, uint32_t e)
        : team(t), ntiles(n), P(ap->P), numTeams(ap->nGroups * ap->perGroup), local(l), epoch(e),
          spinLimit(hurried(ap->spinEvery, blockIdx.x) ? 0u : ap->spinLimit),
          recs(ap->recs + (size_t)t * kRingSlots * ap->P * Geo<N>::WORDS),
          flags(make_rsrc(ap->flags + (size_t)t * kRingSlots * ap->P * 2, kRingSlots * ap->P * 16)),
          done(make_rsrc(ap->done + (size_t)t * kMaxRest, kMaxRest * 8)), donePos((uint32_t)(t * kMaxRest)),
          invFlatDim(ap->invFlatDim), normEps(ap->normEps), T(ap->T)
    {
    }
    __device__ __forceinline__ int tile(int k) const { return team + numTeams * k; }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t records(int k) const
    {
        return make_rsrc(recs + (size_t)(k % kRingSlots) * P * Geo<N>::WORDS, P * Geo<N>::WORDS * 8);
    }
    // Word position of the tile's records.
    __device__ __forceinline__ uint32_t base(int k) const
    {
        return (uint32_t)tile(k) * (uint32_t)P * (uint32_t)Geo<N>::WORDS;
    }
};

// The sum of squares and the hPre columns of the steps k = cls mod CC: lane l
// takes rows 2(l / 8) and + 1 of column l % 8 - 1 (0: the sum of squares).
template <int N, bool kBf16, int U>
__device__ __forceinline__ void crit_wave(ArgsPtr ap, const Team<N> &tm, int cls, int CC, int CR)
{
    using Z = Geo<N>;
    const int lane = threadIdx.x & 63;
    const int ic = lane & 7;
    const int rp = lane >> 3;
    const bool act = ic <= N;
    const int word = 2 * (ic == 0 ? Z::kSqChunk + rp : Z::crit_chunk(ic - 1, rp));
    const bool out = ic > 0 && act;  // this lane has mix column ic - 1
    const float alpha = ap->alpha[0];
    const float bias = out ? ap->bias[ic - 1] : 0.f;
    const float hcEps = ap->hcEps;
    float *const hPre = ap->hPre;
    uint64_t *const bcast = ap->bcast + (size_t)tm.team * kRingSlots * Z::BWORDS;
    const bool watch = lane < kRestBlocks * CR;  // this lane watches a done word
    // The word of each slice that its wave stores last.
    const int hint = 2 * Z::crit_chunk(7, 7);
    bool expired = false;  // a wait of this wave has expired: no more waiting, no more broadcasts

    for (int k = cls; k < tm.ntiles; k += CC) {
        const int rt = tm.tile(k);
        const __amdgpu_buffer_rsrc_t tr = tm.records(k);
        const uint32_t base = tm.base(k);
        // The latest step of the watched wave's class up to k - kDoneLag.
        const int due = k - kDoneLag - (k - kDoneLag - lane / kRestBlocks + 64 * CR) % CR;
        float2 acc;
        bool got = false;
        for (uint32_t spins = 0;; ++spins) {
            // First one word of each slice: waves that polled whole records
            // kept the CU's memory queue full, and every round trip through
            // it long.
            const uint2 hw = load_word(tr, lane < tm.P ? 8 * (lane * Z::WORDS + hint) : kPast);
            const uint2 dw = load_word(tm.done, watch ? 8 * lane : kPast);
            bool ok = lane >= tm.P || hw.y == rec_tag(base + (uint32_t)(lane * Z::WORDS + hint), tm.epoch);
            ok = ok && (!watch || due < 0 ||
                        (dw.y == done_tag(tm.donePos + (uint32_t)lane, tm.epoch) && (int)dw.x >= due));
            if (__all(ok)) {
                acc = make_float2(0.f, 0.f);
                for (int q0 = 0; q0 < tm.P; q0 += U) {
                    u32x4_t t[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        t[u] = load16<kCpolDev>(tr, act && q0 + u < tm.P ? 8 * ((q0 + u) * Z::WORDS + word) : kPast);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const uint32_t pos = base + (uint32_t)((q0 + u) * Z::WORDS + word);
                        ok = ok && (!act || q0 + u >= tm.P ||
                                    (t[u][1] == rec_tag(pos, tm.epoch) && t[u][3] == rec_tag(pos + 1u, tm.epoch)));
                        acc.x = acc.x + __uint_as_float(t[u][0]);
                        acc.y = acc.y + __uint_as_float(t[u][2]);
                    }
                }
                if (__all(ok)) {
                    got = true;
                    break;
                }
            }
            if (expired || spins >= tm.spinLimit) {
                if (!expired && lane == 0) {
                    st_computed(ap->hdr, ap->launchId);
                }
                expired = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        float2 sq;
        if (got) {
            sq.x = __shfl(acc.x, lane & 56);
            sq.y = __shfl(acc.y, lane & 56);
        } else {
            f32x4_t v;  // lane (column, q): rows 4q .. + 3
            float u;
            group_sums<N, kBf16, false, kStrips>(weights_of(ap), tile_rsrc(ap->x, tm.T, (int)ap->K, rt), (int)ap->D,
                                                 tm.P, lane & 15, 0, 1, v, u);
            const int from = 16 * (rp >> 1) + (ic > 0 ? ic - 1 : 0);
            const f32x4_t r4 = {__shfl(v[0], from), __shfl(v[1], from), __shfl(v[2], from), __shfl(v[3], from)};
            acc = (rp & 1) ? make_float2(r4[2], r4[3]) : make_float2(r4[0], r4[1]);
            sq.x = __shfl(u, 16 * (rp >> 1) + 2 * rp);
            sq.y = __shfl(u, 16 * (rp >> 1) + 2 * rp + 1);
        }
        if (out) {
            u32x4_t wv;
            const int idx = (ic - 1) * 16 + 2 * rp;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float ir = ref_inv_rms(e == 0 ? sq.x : sq.y, tm.invFlatDim, tm.normEps);
                const float v = ref_sigmoid((e == 0 ? acc.x : acc.y) * (ir * alpha), bias, hcEps);
                wv[2 * e] = __float_as_uint(v);
                wv[2 * e + 1] = bcast_tag((uint32_t)rt * (uint32_t)Z::BWORDS + (uint32_t)(idx + e), tm.epoch);
                const int64_t row = (int64_t)rt * 16 + 2 * rp + e;
                if (hPre != nullptr && row < tm.T) {
                    hPre[row * N + ic - 1] = v;
                }
            }
            if (got) {
                store_exchange(wv, make_rsrc(bcast + (size_t)(k % kRingSlots) * Z::BWORDS, Z::BWORDS * 8), idx * 8,
                               tm.local);
            }
        }
    }
}

// hPost / hRes columns N + 14 b .. + 13 of the steps k = cls mod CR, done word
// `ru`: lane l < 56 takes rows 4(l / 14) .. + 3 of column l % 14 of them, the
// last 8 lanes the sum of squares.
template <int N, bool kBf16, int U>
__device__ __forceinline__ void rest_wave(ArgsPtr ap, const Team<N> &tm, int ru, int CR)
{
    using Z = Geo<N>;
    static_assert(kRestBlocks * kRestCols == Z::M - N && 4 * kRestCols == 56, "columns of a reducer wave");
    const int lane = threadIdx.x & 63;
    const int first = N + kRestCols * (ru % kRestBlocks);
    const int cls = ru / kRestBlocks;
    const bool out = lane < 56;
    const int quad = lane / kRestCols;
    const int j = first + lane % kRestCols;
    const int word = 2 * (out ? Z::plain_chunk(j, quad) : Z::kSqChunk + (lane & 7));
    const float alpha = ap->alpha[j < 2 * N ? 1 : 2];
    const float bias = out ? ap->bias[j] : 0.f;
    float *const hPost = ap->hPost;
    float *const hRes = ap->hRes;
    bool expired = false;  // a wait of this wave has expired: no more waiting

    for (int k = cls; k < tm.ntiles; k += CR) {
        const int rt = tm.tile(k);
        const __amdgpu_buffer_rsrc_t tr = tm.records(k);
        const uint32_t base = tm.base(k);
        f32x4_t acc;
        bool got = false;
        for (uint32_t spins = 0;; ++spins) {
            // Both strips' flags of slice `lane`; the values are read after.
            const int fw = 2 * ((k % kRingSlots) * tm.P + lane);
            const u32x4_t f = load16<kCpolDev>(tm.flags, lane < tm.P ? 8 * fw : kPast);
            const uint32_t fpos = 2u * ((uint32_t)rt * (uint32_t)tm.P + (uint32_t)lane);
            bool ok = lane >= tm.P ||
                      (f[1] == flag_tag(fpos, tm.epoch) && f[3] == flag_tag(fpos + 1u, tm.epoch));
            if (__all(ok)) {
                acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
                for (int q0 = 0; q0 < tm.P; q0 += U) {
                    u32x4_t t[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        t[u] = load16<kCpolDev>(tr, q0 + u < tm.P ? 8 * ((q0 + u) * Z::WORDS + word) : kPast);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const uint32_t pos = base + (uint32_t)((q0 + u) * Z::WORDS + word);
                        ok = ok && (out || q0 + u >= tm.P ||
                                    (t[u][1] == rec_tag(pos, tm.epoch) && t[u][3] == rec_tag(pos + 1u, tm.epoch)));
                        acc = acc + __builtin_bit_cast(f32x4_t, t[u]);
                    }
                }
                if (__all(ok)) {
                    got = true;
                    break;
                }
            }
            if (expired || spins >= tm.spinLimit) {
                if (!expired && lane == 0) {
                    st_computed(ap->hdr, ap->launchId);
                }
                expired = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (lane == 0) {
            store_word<kCpolDev>(make_uint2((uint32_t)k, done_tag(tm.donePos + (uint32_t)ru, tm.epoch)), tm.done,
                                 8 * ru);
        }
        float sq[4];
        if (got) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sq[e] = __shfl(acc[2 * (e & 1)], 56 + 2 * (quad & 3) + (e >> 1));
            }
        } else {
            f32x4_t v;  // lane (column - first, q): rows 4q .. + 3
            float u;
            group_sums<N, kBf16, false, kStrips>(weights_of(ap), tile_rsrc(ap->x, tm.T, (int)ap->K, rt), (int)ap->D,
                                                 tm.P, first + (lane & 15), 0, 1, v, u);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[e] = __shfl(v[e], 16 * (quad & 3) + lane % kRestCols);
                sq[e] = __shfl(u, 20 * (quad & 3) + e);
            }
        }
        if (out) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float ir = ref_inv_rms(sq[e], tm.invFlatDim, tm.normEps);
                const float scaled = acc[e] * (ir * alpha);
                const int64_t row = (int64_t)rt * 16 + 4 * quad + e;
                if (row < tm.T) {
                    if (j < 2 * N) {
                        hPost[row * N + (j - N)] = ref_sigmoid(scaled, bias, 0.0f) * 2.0f;
                    } else {
                        hRes[row * (N * N) + (j - 2 * N)] = scaled + bias;
                    }
                }
            }
        }
    }
}

// Reducer wave `unit` of a team.
template <int N, bool kBf16, int U>
__device__ __forceinline__ void reducer_wave(ArgsPtr ap, int team, int ntiles, int unit, bool local, uint32_t epoch)
{
    const int CC = ap->CC;
    const int CR = ap->CR;
    const Team<N> tm(ap, team, ntiles, local, epoch);
    if (unit < CC) {
        crit_wave<N, kBf16, U>(ap, tm, unit, CC, CR);
    } else if (unit - CC < kRestBlocks * CR) {
        rest_wave<N, kBf16, U>(ap, tm, unit - CC, CR);
    }
}

// ---------------------------------------------------------------------------
// The kernel.
// ---------------------------------------------------------------------------
template <int N, bool kBf16, bool kPrep>
__global__ __launch_bounds__(kThreads) void slab_kernel(SlabArgs a)
{
    using Z = Geo<N>;
    constexpr int M = Z::M;
    constexpr int Q = Z::Q;
    constexpr int NT = Z::NT;
    constexpr int KS = Z::KS;
    constexpr int L = kRing;
    __shared__ __attribute__((aligned(16))) u32x4_t bsh[kStrips][KS][NT][64];
    // The strips' sums on their way to the other strip of the group: column
    // tile 0 and the sum of squares of strip 1, tiles 1 and 2 of strip 0.
    __shared__ __attribute__((aligned(16))) f32x4_t xch[kGroups][Q][64];
    __shared__ float xchSq[kGroups][16];
    __shared__ uint32_t arrived[kGroups];  // sums written, 2 per own step
    __shared__ uint32_t taken[kGroups];    // sums read, 2 per own step
    __shared__ uint32_t epochSh;

    const int tid = threadIdx.x;
    const int g = blockIdx.x;
    const uint32_t replays = tid == 0 ? replay_load(a.tag.words, g) : 0u;
    const int xcd = g % a.nGroups;
    const int jg = g / a.nGroups;
    const int teamSize = a.P + a.R;
    const int tj = jg / teamSize;
    const int team = xcd + a.nGroups * tj;
    const int numTeams = a.nGroups * a.perGroup;
    const int ntiles = tj < a.perGroup && team < a.RT ? (a.RT - team + numTeams - 1) / numTeams : 0;
    if (tid == 0) {
        epochSh = launch_epoch<SlabArgs>(g, replays);
    }
    if (tid < kGroups) {
        arrived[tid] = 0;
        taken[tid] = 0;
    }
    if (ntiles == 0) {
        return;  // a spare workgroup, or a team without tiles
    }
    const int role = jg % teamSize;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool local = a.nGroups > 1 && (int)(__builtin_amdgcn_s_getreg(kXccIdReg) & 15) == xcd;

    if (role >= a.P) {
        lds_barrier();
        const uint32_t epoch = __builtin_amdgcn_readfirstlane(epochSh);
        // (an instance whose loads cover the team and little more: all of
        // them are issued in every round of a poll)
        const int unit = (role - a.P) * kWaves + w;
        if (a.P <= 8) {
            reducer_wave<N, kBf16, 8>(phase_args(), team, ntiles, unit, local, epoch);
        } else if (a.P <= 16) {
            reducer_wave<N, kBf16, 16>(phase_args(), team, ntiles, unit, local, epoch);
        } else {
            reducer_wave<N, kBf16, 32>(phase_args(), team, ntiles, unit, local, epoch);
        }
        return;
    }

    // ---- slice workgroup ----
    const ArgsPtr wa = phase_args();
    const int Ki = (int)wa->K;
    const int Di = (int)wa->D;
    const int strip = w & 1;
    const int grp4 = w >> 1;  // the wave's group
    const int rl = lane & 15;
    const int q4 = lane >> 4;
    const int lineOff = 8 * q4 + 32 * ((lane >> 3) & 1);  // columns of this lane in a 64-column line
    const int col0 = role * kCols + 64 * strip;           // the strip's first column
    const int col = col0 + lineOff;                       // this lane's 8 columns
    const bool colLive = col < Di;  // past D: loads zeros, stores nothing

    // B of the slice into LDS, fragments (strip, ks = 2s + q, t): lane l holds
    // k = 32q + 8(l / 16) + e of stream s and the strip, of column 16t + l % 16
    // (hi for t < Q, lo of the same columns for t >= Q); 0 past D.  Wave w
    // builds the three k-steps f = 3w .. 3w + 2 of the 24; every load goes out
    // before the first use.
    constexpr int KW = kStrips * KS / kWaves;
    static_assert(KW * kWaves == kStrips * KS, "whole k-steps per wave");
    const auto unit_k = [&](int i, int &k) {  // the k of this lane in unit i; false past D
        const int f = KW * w + i;
        const int ks = f % KS;
        const int dc = role * kCols + 64 * (f / KS) + 32 * (ks & 1) + 8 * q4;
        k = (ks >> 1) * Di + dc;
        return dc < Di;
    };
    u32x4_t bw[KW][NT];
    if constexpr (kPrep) {
#pragma unroll
        for (int i = 0; i < KW; ++i) {
            int k;
            const bool live = unit_k(i, k);
            const int64_t f = (int64_t)(k >> 5) * NT * 64 + 16 * ((k >> 3) & 3) + rl;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                bw[i][t] = live ? wa->bprep[f + 64 * t] : u32x4_t{0u, 0u, 0u, 0u};
            }
        }
    }
    u32x4_t gv[kPrep ? 1 : KW][2];
    const bool hasGamma = wa->gamma != nullptr;
    if constexpr (!kPrep) {
        const __amdgpu_buffer_rsrc_t phiR = make_rsrc(wa->phi, M * Ki * 4);
        const __amdgpu_buffer_rsrc_t gamR = make_rsrc(wa->gamma, hasGamma ? Ki * 4 : 0);
#pragma unroll
        for (int i = 0; i < KW; ++i) {
            int k;
            const bool live = unit_k(i, k);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                gv[i][h] = load16<0>(gamR, live ? (k + 4 * h) * 4 : kPast);
#pragma unroll
                for (int t = 0; t < Q; ++t) {
                    bw[i][Q * h + t] = load16<0>(phiR, live ? ((16 * t + rl) * Ki + k + 4 * h) * 4 : kPast);
                }
            }
        }
    }
    // Every wave's weight loads are in the CU's memory queue before any x load
    // (a wave stalls at a load while the queue is full, and the B build is
    // what everything waits for).
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    const ArgsPtr la = phase_args();
    const int T32 = (int)la->T;
    const uint32_t xTileBytes = 16u * (uint32_t)Ki * 2u;
    const uint32_t hTileBytes = 16u * (uint32_t)Di * 2u;
    const char *xBase = reinterpret_cast<const char *>(la->x);
    char *hBase = reinterpret_cast<char *>(la->hIn);
    uint64_t *recsBase = la->recs + (size_t)team * kRingSlots * la->P * Z::WORDS;
    uint64_t *flagsBase = la->flags + (size_t)team * kRingSlots * la->P * 2;
    const int P32 = la->P;
    const int spinLimit = (int)min(hurried(la->spinEvery, g) ? 0u : la->spinLimit, 0x7FFFFFFFu);
    const __amdgpu_buffer_rsrc_t bcastAll =
        make_rsrc(la->bcast + (size_t)team * kRingSlots * Z::BWORDS, kRingSlots * Z::BWORDS * 8);
    const int nmine = (ntiles - grp4 + kGroups - 1) / kGroups;  // own steps (0 if none)
    const auto tile_of = [&](int jj) { return team + numTeams * (kGroups * jj + grp4); };
    const auto rows_of = [&](int jj) { return (jj >= 0 && jj < nmine) ? min(16, T32 - tile_of(jj) * 16) : 0; };
    const auto slot_of = [&](int jj) { return (kGroups * jj + grp4) % kRingSlots; };

    // x of a tile: line register (s, h) holds, in lane l, row 8h + (l & 7) and
    // the 8 columns at col of stream s.  The buffer resource is based at the
    // tile's first row and sized to its valid rows: rows past T, steps past
    // the last tile and columns past D read zeros without a memory access.
    u32x4_t xb[L][N][2];
    const int xLane = colLive ? ((lane & 7) * Ki + col) * 2 : kPast;
    const int hLane = colLive ? ((lane & 7) * Di + col) * 2 : kPast;
    // Half h of a tile's lines.  The stream's offset is in the resource's base:
    // as part of the lanes' offsets it would take 12 registers.
    const auto load_half = [&](int jj, u32x4_t(&d)[N][2], auto hc) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        const char *base = xBase + (uint64_t)(uint32_t)tile_of(jj) * xTileBytes;
        const int rows = rows_of(jj);
#pragma unroll
        for (int s = 0; s < N; ++s) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc(base + 2 * s * Di, max(0, 2 * (rows * Ki - s * Di)));
            d[s][h] = load16<kCpolNt>(r, xLane + 16 * h * Ki);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    // The first tile's loads go out before the B build, the second's after.
    load_half(0, xb[0], H0{});
    load_half(0, xb[0], H1{});
#pragma unroll
    for (int i = 0; i < KW; ++i) {
        const int f = KW * w + i;
        u32x4_t(*dst)[64] = bsh[f / KS][f % KS];
        if constexpr (!kPrep) {
#pragma unroll
            for (int t = 0; t < Q; ++t) {
                float b[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    b[e] = __uint_as_float(bw[i][Q * (e >> 2) + t][e & 3]);
                    if (hasGamma) {
                        b[e] = b[e] * __uint_as_float(gv[i][e >> 2][e & 3]);
                    }
                }
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    uint32_t hi, lo;
                    split2_bf16(b[2 * p], b[2 * p + 1], hi, lo);
                    bw[i][t][p] = hi;
                    bw[i][Q + t][p] = lo;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            dst[t][lane] = bw[i][t];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_half(1, xb[1], H0{});
    load_half(1, xb[1], H1{});
#pragma unroll
    for (int s = 0; s < N; ++s) {
        xb[2][s][0] = xb[2][s][1] = xb[3][s][0] = xb[3][s][1] = u32x4_t{0u, 0u, 0u, 0u};
    }
    lds_barrier();
    const uint32_t epoch = __builtin_amdgcn_readfirstlane(epochSh);

    // The lane, opaque: what is derived from it in a step is derived there,
    // not kept in a register for the whole loop (there is none to spare).
    const auto lane_here = [&]() __attribute__((always_inline)) {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    // Polls of the broadcast block: lane l (< 8N) reads the words of stream l
    // / 8, rows l % 8 and 8 + l % 8.
    bool dead = false;  // this wave's wait has expired: no more hIn from it
    int failFrom = 0;   // ... from this own tile on
    uint2 pw[2];
    const auto poll = [&](int jj) __attribute__((always_inline)) {
        const int l = lane_here();
        const int off = l < 8 * N ? (slot_of(jj) * Z::BWORDS + 16 * (l >> 3) + (l & 7)) * 8 : kPast;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            pw[h] = load_word(bcastAll, off + 64 * h);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // This wave's flag of own step jj.  Its stores of that step must be done.
    const auto put_flag = [&](int jj) __attribute__((always_inline)) {
        const uint32_t fpos = 2u * ((uint32_t)tile_of(jj) * (uint32_t)P32 + (uint32_t)role) + (uint32_t)strip;
        const __amdgpu_buffer_rsrc_t fr = make_rsrc(flagsBase + 2 * ((size_t)slot_of(jj) * P32 + role),
                                                    jj >= 0 && !dead ? 16 : 0);
        const uint2 wv = make_uint2(0u, flag_tag(fpos, epoch));
        const int off = lane_here() == 0 ? 8 * strip : kPast;
        if (local) {
            store_word<0>(wv, fr, off);
        } else {
            store_word<kCpolDev>(wv, fr, off);
        }
    };
    // hIn of own tile jj from ring registers d, with hPre from the last poll.
    const auto hin_part = [&](int jj, u32x4_t(&d)[N][2], auto after) __attribute__((always_inline)) {
        const int rt = tile_of(jj);
        const bool live = jj >= 0 && jj < nmine;
        const int l = lane_here();
        const auto there = [&]() __attribute__((always_inline)) {
            const uint32_t pos = (uint32_t)rt * (uint32_t)Z::BWORDS + (uint32_t)(16 * (l >> 3) + (l & 7));
            return __all(l >= 8 * N ||
                         (pw[0].y == bcast_tag(pos, epoch) && pw[1].y == bcast_tag(pos + 8u, epoch)));
        };
        if (live && !dead && !there()) {
            for (int spins = 0;; ++spins) {
                __builtin_amdgcn_s_sleep(1);
                poll(jj);
                if (there()) {
                    break;
                }
                if (spins >= spinLimit) {
                    dead = true;
                    failFrom = jj;
                    break;
                }
            }
        }
        const __amdgpu_buffer_rsrc_t hr =
            make_rsrc(hBase + (uint64_t)(uint32_t)rt * hTileBytes, live && !dead ? rows_of(jj) * Di * 2 : 0);
        static_for<2>([&](auto hc) __attribute__((always_inline)) {
            constexpr int h = decltype(hc)::value;
            float hv[8];
#pragma unroll
            for (int s = 0; s < N; ++s) {
                const float pre = __shfl(__uint_as_float(pw[h].x), 8 * s + (l & 7));
                float f[8];
                unpack8<kBf16>(d[s][h], f);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float prod = pre * f[e];
                    hv[e] = s == 0 ? prod : hv[e] + prod;
                }
            }
            u32x4_t out;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                out[p] = pack2_x<kBf16>(hv[2 * p], hv[2 * p + 1]);
            }
            store16<kCpolNt>(out, hr, hLane + 8 * h * Di * 2);
            __builtin_amdgcn_sched_barrier(0);
            after(hc);
        });
    };

    const auto step = [&](int j0, auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value;
        // An opaque copy: the addresses are derived in each step, not held
        // for every unrolled one.
        int jj = __builtin_amdgcn_readfirstlane(j0 + b);
        asm volatile("" : "+s"(jj));
        poll(jj >= kLag ? jj - kLag : 0);
        const int lane = lane_here();

        f32x4_t acc[Q];
        f32x4_t gram = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < Q; ++t) {
            acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        // B of the next half k-step (hi tiles, then lo tiles) is read from LDS
        // while this half's MFMAs run.
        u32x4_t bn[2][Q];
#pragma unroll
        for (int t = 0; t < Q; ++t) {
            bn[0][t] = bsh[strip][0][t][lane];
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            // (one k-step of a line pair at a time: registers)
            const u32x4_t xf = ks % 2 == 0 ? line_frag<0>(xb[b][ks / 2][0], xb[b][ks / 2][1])
                                           : line_frag<1>(xb[b][ks / 2][0], xb[b][ks / 2][1]);
#pragma unroll
            for (int t = 0; t < Q; ++t) {
                bn[1][t] = bsh[strip][ks][Q + t][lane];
            }
            u32x4_t xh = xf, xl = xf;
            if constexpr (!kBf16) {
                // fp16 x = hi + lo exactly in bf16; x_lo meets the hi columns
                // only (x_lo * B_lo is below 2^-16 of the product).
                gram = mfma16_f16(xf, xf, gram);
                float f[8];
                unpack8<false>(xf, f);
                split_f16_to_bf16(f, xh, xl);
            } else {
                gram = mfma16(xf, xf, gram);
            }
#pragma unroll
            for (int t = 0; t < Q; ++t) {
                acc[t] = mfma16(xh, bn[0][t], acc[t]);
            }
            if constexpr (!kBf16) {
#pragma unroll
                for (int t = 0; t < Q; ++t) {
                    acc[t] = mfma16(xl, bn[0][t], acc[t]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (ks + 1 < KS) {
#pragma unroll
                for (int t = 0; t < Q; ++t) {
                    bn[0][t] = bsh[strip][ks + 1][t][lane];
                }
            }
#pragma unroll
            for (int t = 0; t < Q; ++t) {
                acc[t] = mfma16(xh, bn[1][t], acc[t]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const int le = lane_here();
        const int rl = le & 15;
        const int q4 = le >> 4;
        // Gram diagonal: row r sits in lane 16(r / 4) + r, register r % 4.
        const int di = rl & 3;
        float sq = di == 0 ? gram[0] : di == 1 ? gram[1] : di == 2 ? gram[2] : gram[3];
        const bool diag = (rl >> 2) == q4;

        // The strips meet.  A wave writes its sums once the other has taken
        // those of the step before, counts itself in and waits for the other;
        // the wait also holds a group that is a step ahead of another one (the
        // SIMDs favour the older waves; a group left to run ahead leaves the
        // others the last steps alone).  Every count waited for is reached:
        // the waves of this workgroup run all their steps.
        const auto count = [](uint32_t *c) {
            return __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        while (count(&taken[grp4]) < 2u * (uint32_t)jj) {
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (strip == 0) {
#pragma unroll
            for (int t = 1; t < Q; ++t) {
                xch[grp4][t][le] = acc[t];
            }
        } else {
            xch[grp4][0][le] = acc[0];
            if (diag) {
                xchSq[grp4][rl] = sq;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (le == 0) {
            __hip_atomic_fetch_add(&arrived[grp4], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        for (;;) {
            bool met = count(&arrived[grp4]) >= 2u * (uint32_t)(jj + 1);
#pragma unroll
            for (int o = 0; o < kGroups; ++o) {
                const int theirs = (ntiles - o + kGroups - 1) / kGroups;
                met = met && count(&arrived[o]) >= 2u * (uint32_t)min(jj, theirs);
            }
            if (met) {
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");

        // This wave's part of the slice's record (strip 0's sums plus strip
        // 1's), column 16t + rl, rows 4 q4 .. + 3.
        {
            const uint32_t base =
                ((uint32_t)tile_of(jj) * (uint32_t)P32 + (uint32_t)role) * (uint32_t)Z::WORDS;
            const __amdgpu_buffer_rsrc_t rr = make_rsrc(recsBase + ((size_t)slot_of(jj) * P32 + role) * Z::WORDS,
                                                        dead ? 0 : Z::WORDS * 8);
            const auto put = [&](int t, const f32x4_t &v) __attribute__((always_inline)) {
                store_exchange(__builtin_bit_cast(u32x4_t, v), rr, 16 * (Z::kPlain + 64 * t + le), local);
            };
            if (strip == 0) {
                const float otherSq = xchSq[grp4][rl];
                const f32x4_t sum = acc[0] + xch[grp4][0][le];
                put(0, sum);
                const uint32_t sqWord = (uint32_t)(2 * Z::kSqChunk + rl);
                const uint2 wv = make_uint2(__float_as_uint(sq + otherSq), rec_tag(base + sqWord, epoch));
                if (local) {
                    store_word<0>(wv, rr, diag ? 8 * (int)sqWord : kPast);
                } else {
                    store_word<kCpolDev>(wv, rr, diag ? 8 * (int)sqWord : kPast);
                }
                // Columns 0 .. 7 as tagged words (6 and 7 fill the lines).
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    const int word = 2 * Z::crit_chunk(rl & 7, 2 * q4 + e / 2);
                    const uint32_t pos = base + (uint32_t)word;
                    u32x4_t cv;
                    cv[0] = __float_as_uint(sum[e]);
                    cv[1] = rec_tag(pos, epoch);
                    cv[2] = __float_as_uint(sum[e + 1]);
                    cv[3] = rec_tag(pos + 1u, epoch);
                    store_exchange(cv, rr, rl < 8 ? 8 * word : kPast, local);
                }
            } else {
#pragma unroll
                for (int t = 1; t < Q; ++t) {
                    put(t, xch[grp4][t][le] + acc[t]);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            if (le == 0) {
                __hip_atomic_fetch_add(&taken[grp4], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        __builtin_amdgcn_sched_barrier(0);

        // The flag of the step before: its record stores are older than this
        // step's poll, and this step's record stores, the only accesses issued
        // since (4 by strip 0, 2 by strip 1; counters count in issue order),
        // are all that may be outstanding.
        if (strip == 0) {
            wait_vm<4>();
        } else {
            wait_vm<2>();
        }
        __builtin_amdgcn_sched_barrier(0);
        put_flag(jj - 1);
        __builtin_amdgcn_sched_barrier(0);

        // hIn of own tile jj - 2; its registers take own tile jj + 2.
        constexpr int hb = (b + L - kLag) % L;
        hin_part(jj - kLag, xb[hb], [&](auto hc) __attribute__((always_inline)) { load_half(jj + L - kLag, xb[hb], hc); });
    };
    static_assert(L == 4 && kLag == 2, "tiles 0 and 1 load before the first step, jj + 2 in step jj");
    int j0 = 0;
    for (; j0 + L <= nmine; j0 += L) {
        static_for<L>([&](auto bc) __attribute__((always_inline)) { step(j0, bc); });
    }
    // The last tiles' hIn: own tiles jj - 2 of the steps nmine and nmine + 1,
    // in a copy of the loop's body for the last, partial round.
    const auto finish = [&]() __attribute__((always_inline)) {  // the last step's flag
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_sched_barrier(0);
        put_flag(nmine - 1);
    };
    static_for<L + kLag - 1>([&](auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value;
        if (nmine > 0 && j0 + b == nmine) {
            finish();
        }
        if (j0 + b < nmine) {
            if constexpr (b < L) {
                step(j0, bc);
            }
        } else if (j0 + b < nmine + kLag && j0 + b >= kLag) {
            poll(j0 + b - kLag);
            hin_part(j0 + b - kLag, xb[(b + L - kLag) % L], [](auto) {});
        }
    });
    if (dead) {
        // A wait expired: this wave's hIn from that tile on, alone.
        const ArgsPtr ca = phase_args();
        if (lane == 0) {
            st_computed(ca->hdr, ca->launchId);
        }
#pragma unroll 1
        for (int i = failFrom; i < nmine; ++i) {
            own_hin<N, kBf16, false, kStrips>(weights_of(ca), ca->x, ca->hIn, ca->alpha, ca->bias, ca->T, Di,
                                              tile_of(i), ca->P, 1, col0, ca->invFlatDim, ca->normEps, ca->hcEps);
        }
    }
}

template <int N, bool kBf16, bool kPrep>
int slab_coresident_t(int numCUs)
{
    int perCU = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &perCU, reinterpret_cast<const void *>(&slab_kernel<N, kBf16, kPrep>), kThreads, 0) !=
        hipSuccess) {
        return -1;
    }
    return perCU * numCUs;
}

template <int N, bool kBf16, bool kPrep>
hipError_t launch_slab_t(const Plan &p, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream)
{
    char *ws = static_cast<char *>(workspace);
    SlabArgs a;
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
    a.recs = reinterpret_cast<uint64_t *>(ws + p.wsSlabRecs);
    a.bcast = reinterpret_cast<uint64_t *>(ws + p.wsSlabBcast);
    a.flags = reinterpret_cast<uint64_t *>(ws + p.wsSlabFlags);
    a.done = reinterpret_cast<uint64_t *>(ws + p.wsSlabDone);
    a.tag = tag;
    a.hdr = ws;
    a.launchId = launchId;
    a.T = p.T;
    a.D = p.D;
    a.K = p.K;
    a.RT = (int)p.fusedTiles;
    a.P = p.slab.P;
    a.R = p.slab.R;
    a.CC = p.slab.CC;
    a.CR = p.slab.CR;
    a.nGroups = p.slab.groups;
    a.perGroup = p.slab.teams;
    a.normEps = p.normEps;
    a.hcEps = p.hcEps;
    a.invFlatDim = p.invFlatDim;
    a.spinLimit = p.ownSpinLimit();
    a.spinEvery = p.spinEvery;
    if (!p.fusedCooperative) {
        hipLaunchKernelGGL((slab_kernel<N, kBf16, kPrep>), dim3((unsigned)p.slab.grid), dim3(kThreads), 0,
                           stream, a);
        return hipGetLastError();
    }
    void *args[] = {&a};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void *>(&slab_kernel<N, kBf16, kPrep>),
                                      dim3((unsigned)p.slab.grid), dim3(kThreads), args, 0, stream);
}

}  // namespace

int slab_columns() { return kCols; }
int slab_max_slices() { return kMaxSlices; }
int slab_done_words() { return kMaxRest; }
int slab_groups() { return kGroups; }
int slab_strips() { return kStrips; }
int slab_ring_slots() { return kRingSlots; }
int slab_record_words() { return Geo<6>::WORDS; }
int slab_bcast_words() { return Geo<6>::BWORDS; }

int slab_max_coresident(const Plan &p, int numCUs)
{
    if (p.n != 6) {
        return -1;
    }
    if (p.bprep != nullptr) {
        return p.isBf16 ? slab_coresident_t<6, true, true>(numCUs) : slab_coresident_t<6, false, true>(numCUs);
    }
    return p.isBf16 ? slab_coresident_t<6, true, false>(numCUs) : slab_coresident_t<6, false, false>(numCUs);
}

hipError_t launch_slab(const Plan &p, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream)
{
    if (p.n != 6) {
        return hipErrorNotSupported;
    }
    if (p.bprep != nullptr) {
        return p.isBf16 ? launch_slab_t<6, true, true>(p, workspace, tag, launchId, stream)
                        : launch_slab_t<6, false, true>(p, workspace, tag, launchId, stream);
    }
    return p.isBf16 ? launch_slab_t<6, true, false>(p, workspace, tag, launchId, stream)
                    : launch_slab_t<6, false, false>(p, workspace, tag, launchId, stream);
}

}  // namespace mhc
