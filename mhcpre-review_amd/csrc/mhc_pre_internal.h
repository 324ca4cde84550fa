// Internal launch plan shared by the host library and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace mhc {

// The path a shape belongs to: the kernels it runs, unless the cell, slab or
// strip kernel runs in place of them (Plan::cellP, slab, stripInstead).
enum class Path : int {
    kSplit = 0,   // prep B, split-K MFMA GEMM + sumsq partials, epilogue + hIn (x read twice)
    kFused = 1,   // one persistent kernel: x read once, kept in registers
    kStrip = 2,   // one persistent kernel: XCD-local teams, B in LDS, x in a register ring
    kRows = 3,    // prep B, split-K GEMM over 256-row blocks (B through an LDS ring), epilogue + hIn
};

// Device status word (first 8 bytes of the workspace): the low half holds a
// code, the high half the host launch id of the launch that wrote it.  The
// strip and fused kernels write (launch id, kDeviceTimeout) only when a wait
// runs out, those that then compute what they waited for (launch id,
// kDeviceComputed); the split path's first kernel writes kDeviceOk into the low
// half.
constexpr uint32_t kDeviceOk = 0u;
constexpr uint32_t kDeviceTimeout = 0x7107u;
constexpr uint32_t kDeviceComputed = 0x7108u;  // an expired wait's work was done instead: the outputs are right

// Bytes reserved at the head of the workspace: the status word at 0, and words
// that only launches captured when the library's own were used up need
// (mhc_pre_replay.hip).
constexpr size_t kWsReplayOff = 256;  // uint32 [kMaxExchangeGrid]
constexpr int kMaxExchangeGrid = 2048;  // largest grid of a kernel whose workgroups exchange words
constexpr size_t kWsHeaderBytes = kWsReplayOff + 4 * kMaxExchangeGrid;

// What the kernels whose workgroups exchange words (cell, slab, strip, fused)
// mix into every tag, so that no word of another launch is taken for one of
// this launch's, whatever the workspace held before: the hash (mix32, a
// bijection) of a number that no other launch of the process has.  An eager
// launch: its own number, 31 bits of it (`seed`, hashed; `words` null).  The
// replays of a captured launch share their arguments: it has a number among the
// captured ones (`seed`, its upper 21 bits, 10 the highest two) and one word per
// workgroup, equal in all of them, to which each replay adds one; the lower 11
// bits are that count's, for a replay finds at its own places what the one
// before it left there.  Without such words of its own, a node before the
// launch sets words of the workspace to a whole number (11 the highest bits).
struct LaunchTag {
    uint32_t seed = 0;
    uint32_t *words = nullptr;
};
constexpr uint32_t kCapturedNumbers = 0x80000000u;
constexpr int kReplayBits = 11;
constexpr uint32_t kFilledNumbers = 0xC0000000u;

// The finalizer of MurmurHash3: neighbouring numbers' hashes differ in half
// their bits.
__host__ __device__ inline uint32_t mix32(uint32_t v)
{
    v ^= v >> 16;
    v *= 0x85EBCA6Bu;
    v ^= v >> 13;
    v *= 0xC2B2AE35u;
    return v ^ (v >> 16);
}

// The tag of launch `launchId` with `grid` workgroups, on the current device
// `device` (mhc_pre_replay.hip).
hipError_t make_launch_tag(uint32_t launchId, int device, int grid, void *workspace, hipStream_t stream,
                           LaunchTag &tag);
// The current device's array of replay words (looked up once per device).
hipError_t replay_words_address(int device, uint32_t **ptr);

// The most that a wave may have to compute (Plan::ownStrips, about a second)
// where the slab or strip kernel runs in place of kernels that wait for nobody.
constexpr int64_t kMaxOwnStrips = int64_t{1} << 17;

// Work distribution of the slab kernel (mhc_pre_slab.hip).
struct SlabGeometry {
    int P = 0;       // slice workgroups per team
    int groups = 0;  // XCDs (teams inside an XCD), or 1 (teams across the device)
    int teams = 0;   // teams per group
    int R = 0;       // reducer workgroups per team
    int CC = 0;      // reducer waves of the hPre columns (1, 2, 4 or 8)
    int CR = 0;      // reducer waves of each block of the other columns (up to 8)
    int grid = 0;    // workgroups: one per CU
    int xcds = 0;    // XCDs of the device it was planned for
};

struct Plan {
    Path path = Path::kSplit;

    // Problem shape.
    int n = 0;        // streams
    int M = 0;        // n*n + 2n
    int NT = 0;       // 16-wide column tiles of the [hi | lo] B operand: 2M / 16
    int64_t T = 0;    // rows (tokens)
    int64_t D = 0;    // per-stream width
    int64_t K = 0;    // n * D
    bool isBf16 = true;
    bool hasGamma = false;
    bool hasHPre = false;
    // Strip and fused path launch.  By default a plain launch of a grid sized
    // to the device's co-residency limit: every workgroup is resident as long
    // as no other kernel occupies the device, and the kernels' bounded waits
    // turn any other case into a reported timeout rather than a hang.
    // MHCPRE_LAUNCH=cooperative selects a cooperative launch, which
    // guarantees co-residency next to concurrent work at the cost of a
    // slower dispatch (about 20 us per launch on MI355X).
    bool fusedCooperative = false;
    // Polls of a strip or fused wait before it records kDeviceTimeout and
    // gives up (about a second).  MHCPRE_SPIN_LIMIT at phase 1 overrides it,
    // for tests of the timeout path.
    uint32_t spinLimit = 1u << 20;
    // Test knob (MHCPRE_SPIN_EVERY=k): in kernels whose expired waits are
    // computed, every k-th workgroup gives up at its first poll (in the cell
    // kernel also where that finds its data); 0: none.
    uint32_t spinEvery = 0;
    // The same for kernels whose expired waits are computed instead: about as
    // long as that takes, so that such a launch takes at most about twice as
    // long as it had to (two launches that hold half of each other's CUs would
    // stand still otherwise).  Measured on MI355X with every wait expired: the
    // cell kernel 2 to 4 us per slice (n = 4, D = 1024, T = 512 38 us, n = 4, D =
    // 7168, T = 16 126); a wave of the slab and strip kernels 6 to 10 us per
    // 64-column strip of a tile's rows, over all of K (n = 6, D = 1024, T = 2048
    // 0.36 ms, D = 4096, T = 4096 6.3 ms; n = 4, D = 7056, T = 2048 5.9 ms).  A
    // poll takes about 0.7 us.  (At least 2^12 there: a first tile's hPre is
    // waited for more than 64 polls in an undisturbed launch.)
    uint32_t cellSpinLimit() const { return spinLimit < 64u + 4u * cellP ? spinLimit : 64u + 4u * cellP; }
    uint32_t ownSpinLimit() const
    {
        const uint32_t polls = ownStrips < (1 << 9) ? 1u << 12 : 8u * (uint32_t)ownStrips;
        return spinLimit < polls ? spinLimit : polls;
    }
    int ownStrips = 0;  // strips that a wave of the slab or strip kernel computes if its first wait expires
    float normEps = 1e-6f;
    float hcEps = 1e-6f;
    float invFlatDim = 0.f;  // fl(1.0f / K), as code/op_host/mhc_pre.cpp:154

    // Split path: K-slices of the GEMM and k-steps (32 wide) per slice.
    int splitS = 1;
    int ksPerSlice = 0;

    // Fused path parameters (fusedGrid / fusedTeams are filled per launch
    // from the device's co-residency limit).
    int fusedDw = 0;          // x columns per slice (32 * k-steps)
    int fusedP = 0;           // slices per row tile = D / fusedDw
    int fusedGrid = 0;        // workgroups in the cooperative grid
    int fusedTeams = 0;       // teams of fusedP workgroups
    int64_t fusedTiles = 0;   // 16-row tiles

    // Strip path (n = 4, from D = 192): P = ceil(D / 256) slice
    // workgroups of 256 columns and R reducer workgroups per team, teams
    // formed inside one XCD or across the device.  stripR, stripXcds,
    // stripTeamsPerXcd and stripGrid are filled per launch from the device.
    int stripP = 0;
    bool stripInstead = false;  // the strip kernel runs in place of the split path's (which stays
                                // the fallback, its layout in the workspace)
    int stripMaxTeams = 0;  // teams the workspace's exchange rings are sized for (those of the
                            // device phase 1 planned for)
    int stripR = 0;
    int stripXcds = 0;
    int stripTeamsPerXcd = 0;
    int stripGrid = 0;

    // Slab kernel (n = 6; slab.P == 0: not taken): one launch that runs in place of
    // the rows or split path's kernels, whose layout the workspace also holds
    // (the fallback on a device that cannot co-schedule its grid).
    SlabGeometry slab;

    // Cell kernel (small batches; cellP == 0: not taken): one launch that runs
    // in place of the path's own kernels, which stay the fallback.
    int cellP = 0;       // slices of 64 cellStrips columns
    int cellStrips = 1;  // 1 or 2
    int cellGrid = 0;    // workgroups: cellP per 16-row and 16-column tile

    // Rows path (K % 128 == 0): rowsS K-ranges (contiguous runs of
    // rows_stage_ksteps()-k-step stages) over rowsBlocks blocks of
    // rows_block_rows() rows.
    int rowsS = 0;
    int rowsBlocks = 0;
    // The block GEMM builds B from phi and gamma itself (no prep launch);
    // otherwise a prep kernel writes B fragments to the workspace first.
    bool rowsBFromPhi = false;
    // Small batches (T <= rows_small_rows(n, false), or up to twice that with
    // K >= 16384): one GEMM workgroup per K-range of rows_small_ksteps()
    // k-steps, B built from phi by the workgroup itself, no prep launch.
    bool rowsSmall = false;
    // Partial sums stored row-major, [T][rowsS][M+1] (each row's sums
    // contiguous for its epilogue), instead of [rowsS][T][M+1].
    bool rowsRowMajor = false;

    // Workspace layout (byte offsets).  The paths' regions overlap: a
    // workspace holds one launch at a time.
    size_t wsBsplit = 0;      // split: B fragments
    size_t wsPartial = 0;     // split: [S][T][M+1] partials
    size_t wsFinal = 0;       // fused: per-tile hPre / invRms blocks (tagged words)
    size_t wsFusedPartial = 0;// fused: per-(tile, slice) exchange records (tagged words)
    size_t wsFusedEnd = 0;    // fused: end of its layout (0: no fused layout)
    size_t wsSplitEnd = 0;    // split: end of its layout
    size_t wsStripBcast = 0;  // strip: per-team rings of broadcast blocks (tagged words)
    size_t wsStripRecs = 0;   // strip: per-team rings of P exchange records (tagged words)
    size_t wsRowsB = 0;       // rows (prep launch): B fragments [K/32][NT][64 lanes] x 16 bytes
    size_t wsRowsPartial = 0; // rows: partials, [rowsS][T][M+1] or [T][rowsS][M+1]
    size_t wsSlabBcast = 0;   // slab: per-team rings of broadcast blocks
    size_t wsSlabFlags = 0;   // slab: per-team rings of the slices' flags
    size_t wsSlabDone = 0;    // slab: the reducer waves' done words
    size_t wsSlabRecs = 0;    // slab: per-team rings of P exchange records
    size_t wsCellRecs = 0;    // cell: [tile][cellP] records
    size_t wsTotal = 0;

    // Bound device pointers (caller memory).
    uint32_t *statusWord = nullptr;  // strip / fused launches: the caller's sticky status word
    const void *x = nullptr;
    const float *phi = nullptr;
    const float *alpha = nullptr;
    const float *bias = nullptr;
    const float *gamma = nullptr;
    void *hIn = nullptr;
    float *hPost = nullptr;
    float *hRes = nullptr;
    float *hPre = nullptr;
    // Prepared B operand (mhcPrePrepareWeights), or null: the kernels then
    // build B from phi and gamma.  Layout of launch_prepare_b.
    const void *bprep = nullptr;
};

// Built-in workspace of mhcPreNoAlloc (mhc_pre_noalloc.hip): kScratchBytes
// per device, in the library's device code object.  scratch_address gives the
// current device's copy (the caller makes `device` current).
constexpr size_t kScratchBytes = size_t{64} << 20;
hipError_t scratch_address(int device, void **ptr);

// Kernel launchers (mhc_pre_kernels.hip).  Each returns the first HIP error.
hipError_t launch_split(const Plan &plan, void *workspace, hipStream_t stream);
// launchId: host-side id of the launch, written with kDeviceTimeout into the
// status word when a bounded wait expires (the exchange epoch itself comes
// from the workspace header).
hipError_t launch_fused(const Plan &plan, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream);

hipError_t launch_strip(const Plan &plan, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream);

// Cell kernel (mhc_pre_cell.hip).
hipError_t launch_cell(const Plan &plan, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream);
int cell_max_coresident(const Plan &plan, int numCUs);
size_t cell_record_bytes();

// Slab kernel (mhc_pre_slab.hip): one launch, x read once.
hipError_t launch_slab(const Plan &plan, void *workspace, const LaunchTag &tag, uint32_t launchId, hipStream_t stream);
int slab_max_coresident(const Plan &plan, int numCUs);
int slab_columns();                          // x columns per slice
int slab_max_slices();                       // largest P
int slab_done_words();                       // words of a team's done array
int slab_groups();                           // wave groups of a slice workgroup
int slab_strips();                           // 64-column strips of a slice
int slab_ring_slots();                       // exchange ring slots per team
int slab_record_words();                     // tagged 8-byte words of a record
int slab_bcast_words();                      // ... and of a broadcast block

// Prepared B operand (mhc_pre_rows.hip): B = gamma (.) phi (gamma may be
// null) split into bf16 hi + lo MFMA fragments, [K/32 k-steps][2M/16 column
// tiles][64 lanes] x 16 bytes.  Lane l of fragment (ks, t) holds k = 32 ks +
// 8 (l / 16) .. + 7 of one column: tile t < Q = M/16 the hi half of column
// 16 t + l % 16, tile Q + t the lo half of the same column; when M % 16 == 8
// tile 2Q holds column 16 Q + l % 8, hi in lanes l % 16 < 8 and lo in the
// others.  The strip and fused kernels keep B in LDS in this same column
// order, and the rows path's GEMM reads it as it is.
hipError_t launch_prepare_b(int n, const float *phi, const float *gamma, void *bfrag, int64_t K,
                            hipStream_t stream);

// Rows path (mhc_pre_rows.hip); nXcd: XCDs of the device (work placement
// only).
hipError_t launch_rows(const Plan &plan, void *workspace, int nXcd, hipStream_t stream);
// Row blocks up to which the block GEMM builds B from phi itself (see
// mhc_pre_rows.hip); above it a prep launch writes B fragments first.
constexpr int64_t kRowsPhiMaxBlocks = 16;
// Whether the rows-path epilogue of `rows` rows over S K-ranges runs its
// 1024-thread variant (mhc_pre_rows.hip).
bool rows_epilogue_wide(int n, int S, int64_t rows);
// Rows per work item, k-steps per stage and work-items per workgroup of the
// rows-path GEMM.
int rows_block_rows();
int rows_stage_ksteps();
int rows_gemm_threads();
// Largest batch of the small-batch GEMM and k-steps per workgroup there.
// Rows the small-batch GEMM holds (the wide variant: twice as many).
int rows_small_rows(int n, bool wide);
int rows_small_ksteps();

// Stream probe (mhc_pre_stream.hip): reads readBytes (a multiple of 4096) from
// src and writes writeBytes (a multiple of 1024) to dst in the best-served
// access pattern, with `workgroups` workgroups of 512 threads.
hipError_t launch_stream_probe(const void *src, int64_t readBytes, void *dst, int64_t writeBytes,
                               int workgroups, hipStream_t stream);

// Workgroups of the strip kernel that can be resident per CU (x numCUs), or
// -1 if the plan has no strip kernel.
int strip_max_coresident(const Plan &plan, int numCUs);

// Wave groups of a slice workgroup of the strip kernel, and 64-column strips of
// a slice.
int strip_groups();
int strip_strips();
// Exchange ring slots per team of the strip kernel, and the tagged 8-byte
// words of one exchange record (per slice) and of one broadcast block.
int strip_ring_slots();
int strip_record_words();
int strip_bcast_words();
// Teams of P slices (plus their reducers) that cusPerXcd CUs of one XCD
// hold; 0 when not even one fits.
int strip_teams_per_xcd(int P, int cusPerXcd);
// Largest number of slice workgroups per team the strip kernel supports.
int strip_max_slices();
// Reducer workgroups per team the strip kernel uses when `available` (>= 1)
// workgroups per team are left over after the slices (1, 2 or 4; the ring
// size depends on it).
int strip_reducers(int available);

// Rows per launch of the one-workgroup-per-row epilogue kernels (rows and
// split paths): a grid's work-items must stay below 2^32, so larger batches
// take several launches.
constexpr int64_t kEpilogueRowsPerLaunch = int64_t{1} << 20;

// Largest number of fused-path workgroups that can be co-resident on a device
// with numCUs compute units, or -1 if the plan has no fused kernel.
int fused_max_coresident(const Plan &plan, int numCUs);

// Fused-path workspace geometry for n streams, in 8-byte tagged words: one
// exchange record of M + 1 columns x 16 rows per (row tile, slice), and one
// broadcast block of n + 1 columns x 16 rows per row tile.
inline int fused_record_words(int n) { return (n * n + 2 * n + 1) * 16; }
inline int fused_bcast_words(int n) { return (n + 1) * 16; }

}  // namespace mhc
