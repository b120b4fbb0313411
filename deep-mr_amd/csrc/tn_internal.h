// Internal types shared by the tilenufft HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "tilenufft.h"
#include "tn_worklist.h"

namespace tn {

constexpr int kBlock = 256;        // threads per workgroup (4 wave64)
constexpr int kWave = 64;
constexpr int kMaxWidth = 16;      // largest kernel width supported per axis
constexpr int kStagedMaxWidth = 8; // widest kernel of the staged interpolation and the tile gridding
                                   // variants; wider kernels gather and grid through the matrix
// launch "kind" of a table: ndim * kKindStride + widest kernel width
constexpr int kKindStride = 32;
constexpr int kind_ndim(int kind) { return kind / kKindStride; }
constexpr int kind_width(int kind) { return kind % kKindStride; }
constexpr int kInterpBlockPts = 256;  // samples per interpolation work item
constexpr size_t kGridLdsBudget = 80 * 1024;  // LDS per gridding workgroup (two per CU)
constexpr size_t kInterpLdsBudget = 64 * 1024;  // LDS per staged-interpolation workgroup
// samples per lane in the staged interpolation: 1 in 2D, 2 in 3D (each
// measured fastest on its workload; both appear in one table only alone)
constexpr int staged_ept(int ndim) { return ndim == 3 ? 2 : 1; }
constexpr int kLoadBatch = 4;  // global loads per lane issued before their LDS writes in staging loops
// default coils per region load of the staged interpolation, below what the
// LDS budget allows so that more workgroups fit on a CU (measured fastest:
// 2D 16x16 tiles, 8 coils 0.125 ms vs 16 coils 0.189 ms; 3D 8x8x16 tiles,
// 2 coils 1.33 ms vs 3 coils 1.61 ms)
constexpr int kInterpChunk2d = 8;
constexpr int kInterpChunk3d = 2;
// Default staged-interpolation tiles (measured fastest with the chunks above).
constexpr int staged_tile(int ndim, int axis) {  // axis: 0 x, 1 y, 2 z
    return axis == 0 ? 16 : axis == 1 ? (ndim == 3 ? 8 : 16) : ndim == 3 ? 8 : 1;
}
// Most coils per chunk, taps and cells per region (rows rounded up to pairs)
// of the staged interpolation's register-addressed loads: the default chunks
// and the regions of the default tiles, in steps of a pair per lane.
constexpr int staged_coils(int ndim) { return ndim == 3 ? kInterpChunk3d : kInterpChunk2d; }
constexpr int staged_width(int ndim) { return ndim == 3 ? 5 : 6; }
constexpr int staged_cells(int ndim, int wc) {
    const int pairs = (staged_tile(ndim, 0) + wc) / 2 * (staged_tile(ndim, 1) + wc - 1) *
                      (ndim == 3 ? staged_tile(ndim, 2) + wc - 1 : 1);
    return (pairs + kBlock - 1) / kBlock * kBlock * 2;
}
// Where those loads are used. They hold more registers than the row-by-row
// load (2D, 4 taps: 84 for 66, five waves per SIMD for seven; single cells 100;
// 3D, 4 taps: 167 for 110), which costs nothing while a launch's workgroups are
// all resident, up to kStagedFew of them (four per CU), and has to be made up
// by fewer instructions per plane beyond. Fewest planes of an item for which
// it is, measured against row by row: pairs of cells in 2D with one to three
// taps from the first plane on (0.95 to 1.02 of the time), four and six taps
// from three (one plane 1.06, three 0.97; eight 0.81), five, where the waves
// drop from six to four, from six (three 1.05, six 0.98, eight 0.88); single
// cells only with six taps from three (three 0.98; four taps 1.19 with one
// plane and 1.07 with eight); 3D from three (one 1.18, two 1.04 to 1.10, three
// 0.93 to 1.02, eight 0.84). 0: at no number.
constexpr int64_t kStagedFew = 1024;
constexpr int staged_planes(int ndim, int wc, int vec) {
    if (ndim == 3) return 3;
    if (vec == 1) return wc == 6 ? 3 : 0;
    return wc <= 3 ? 1 : wc == 5 ? 6 : 3;
}
constexpr int interp_segment(int ndim) { return 256 * staged_ept(ndim); }  // samples per staged work item
constexpr int kGridSplitDefault = 2048;  // max tile entries per gridding workgroup
constexpr int kGridBatch = 256;  // tile entries staged in LDS per gridding batch
constexpr int kGridPad = 4;      // accumulator row padding (floats)

// Gridding variants: one LDS atomic per tap and sample over entries spread
// across footprint origins, or per-lane register runs over origin-sorted
// entries (for at most kRunsMaxTaps taps per sample).
// Matrix: per-cell sums over the plan's sparse gridding matrix (CSR by grid
// cell), one lane per cell. Tiles (2D and 3D): one wave per small tile, whose
// cells' sums the matrix cores form over the tile's entries in sample order with
// per-sample taps from a plan table (tn_tiles.hip).
enum GridMode { kGridAuto = 0, kGridSpread = 1, kGridRuns = 2, kGridMatrix = 3, kGridTiles = 4 };
// Tile gridding (matrix cores): a tile is four patches of 4x4 cells, the z
// planes of a 4x4x4 tile in 3D and the quadrants of an 8x8 tile in 2D.
__host__ __device__ constexpr int tiles_dim(int ndim, int axis) {  // axis: 0 x, 1 y, 2 z
    return ndim == 3 ? 4 : axis < 2 ? 8 : 1;
}
constexpr int kTilesMaxWidth = 6;  // most taps per axis
constexpr int kTilesBlocks = 4;    // most blocks of 8 coils per item
constexpr int kTilesCopyCoils = 8; // coils per workgroup of the coil-minor copy
// Most entries of a tile that one wave takes by default; larger tiles go to a
// workgroup's four waves. Short chains keep the sums as exact as the matrix
// rows (61x101x84 kooshball, error against 64 bits: 7.9e-7 at 96, 8.7e-7 at
// 192, 1.2e-6 at 384; the matrix 7.9e-7) and small problems balanced
// (CG-SENSE, 195 k entries: 1.95 ms a solve at 64-96, 2.02 at 160, 2.16 at
// 256); the large kooshball (27 M entries) takes 4% longer than at 384.
constexpr int kTilesWave = 96;
// Samples of a table (bytes) from which the gridding reads a coil-minor copy: in
// place, the records of an entry's coils lie in different rows and a wave's
// loads touch four times the cache lines, which the L2s serve while they hold
// the samples. In 2D the copy costs 5 us (16 coils, 31 MiB: 50 us in place, 56
// with it); in 3D it gains 5% already at 8 MiB and 10% from 40 MiB on (8 coils
// of 256^3, 39 MiB: 624 and 573 us; 312 MiB: 1494 and 1350). The line is a
// compromise of the two: radials of 75 and 150 MiB would be faster in place (92
// and 179 us for 118 and 203).
constexpr int64_t kTilesCopyBytes = 48ll << 20;
// Tap record of a sample: the taps of each axis, padded with zeros to wpad
// words (16-byte aligned).
__host__ __device__ constexpr int tiles_pad(int wmax) { return wmax <= 4 ? 4 : 8; }
__host__ __device__ constexpr int tiles_tap_stride(int ndim, int wpad) { return ndim * wpad; }
constexpr int kMatrixLongRow = 128;  // default (2D): rows with more entries get a whole workgroup
constexpr int kMatrixLongRow3d = 256;  // default (3D): kooshball 128^3 at osf 2: 3.74 ms against 4.33 (128), 4.30 (512)
constexpr int kMatrixChunk = 16;     // default coils per item (record width of the coil-minor copy)
constexpr uint64_t kMatrixAutoBytes = 4ull << 30;  // largest gridding matrix the automatic mode builds
constexpr int kMatrixPasses = 4;     // cell passes per item of the coil-minor matrix gridding
constexpr int kLongGroups = 32;      // lane groups summing one long row of the coil-minor matrix gridding
constexpr int64_t kStaticScratchFloats = 8ll << 20;  // fixed gridding workspace: 32 MiB per device
constexpr int kMaxDevices = 64;
constexpr int kXcds = 8;          // accelerator complex dies (each with its own L2)
constexpr int kRunsMaxTaps = 36;  // register budget of the run sums of one z plane (W <= 6)
constexpr int kRunsBatch = 256;                 // entries per staged batch (= kBlock)
constexpr int kRunsMaxCoils = 64;               // coils per item: 4 waves x up to 16 lanes per group

// 32-bit words per staged entry of the register-run gridding: origin key,
// (tile-local tap-0 offset, wrap tap) per axis, W weights per axis.
__host__ __device__ constexpr int runs_record_words(int ndim, int wc) { return 1 + 2 * ndim + ndim * wc; }

// Dynamic LDS bytes of the gridding kernel for `ncoil` coils of a tile.
inline size_t grid_lds_bytes(int ncoil, int64_t plane, int wc, int mode = kGridSpread, int ndim = 3) {
    if (mode == kGridRuns)  // interleaved accumulators, entry records, sample values
        return sizeof(float) * (2 * (size_t)ncoil * plane + 4 + (size_t)runs_record_words(ndim, wc) * kRunsBatch +
                                2 * (size_t)(ncoil + 1) * kRunsBatch);
    return sizeof(float) * (2 * (size_t)ncoil * plane + 4 * (size_t)kGridBatch +
                            3 * (size_t)wc * kGridBatch + 2 * (size_t)ncoil * kGridBatch);
}

// Interpolation variants.
enum InterpMode { kInterpAuto = 0, kInterpGather = 1, kInterpStaged = 2 };

// One trajectory (frame) bound to its data placement for a launch. All
// per-axis arrays are (x, y, z) so that axis d matches coordinate column d.
struct alignas(16) Job {
    int32_t G[3];       // oversampled grid (x, y, z); z = 1 in 2D
    int32_t W[3];       // kernel width; 1 = Cartesian axis
    int32_t shift[3];   // output index = (tap + shift) mod G
    int32_t T[3];       // gridding tile
    int32_t NT[3];      // tiles per axis
    int32_t IT[3];      // staged-interpolation tile
    int32_t INT_[3];    // staged-interpolation tiles per axis
    int32_t tchunk;     // tile gridding: coils per chunk of the coil-minor copy
    int32_t pad1;
    float beta[3];
    float inv_scale;
    int32_t ndim;
    int32_t nbatch;     // coils (batch) of this job
    int32_t mlong;      // matrix gridding: rows with more entries are summed by a whole workgroup
    int64_t npts;
    const float *coord;       // (npts, ndim) grid units
    const float4 *entries;    // (x, y, z, bits(sample)) sorted by tile
    const int32_t *bin_off;   // (ntiles + 1) offsets into entries
    const float4 *pentries;   // each sample once, sorted by the interpolation
                              // tile holding its footprint origin (3D: then
                              // by the origin cell)
    const int32_t *pbin_off;  // (interp tiles + 1) offsets into pentries
    const int32_t *mrow;      // matrix gridding: (cells + 1) row offsets of this frame
    const int2 *mnz;          // matrix gridding: (sample, weight bits) per entry
    int64_t grid_off;         // complex elements from the grid base
    int64_t grid_bstride;     // complex elements between coils
    int64_t samp_off;
    int64_t samp_bstride;
    int64_t w_off;            // offset into the weight base (-1: no weight)
    int64_t st_off;           // matrix / tile gridding: this job's coil-minor sample copy in the table's buffer
    const int2 *tent;         // tile gridding: (sample, tile-local footprint origin x, y, z + 16 in bytes 0-2),
                              // sorted by tile, samples ascending; bin_off holds the offsets
    const int2 *rows;         // tile gridding: this frame's row ranges (tn_plan::d_rows)
    const float *taps;        // tile gridding: tap records of this frame's samples
};

// Low-rank subspace arguments of a launch (ncoeff == 0: plain transform).
// Interpolation: coef = basis_adjoint (nframes, ncoeff). Gridding: coef =
// basis (ncoeff, nframes). The plan holds all frames as one trajectory of
// nframes * frame_npts samples.
struct LowRank {
    const float2 *coef = nullptr;
    int32_t ncoeff = 0;
    int32_t nframes = 1;
    int32_t frame_npts = 1;
};

struct LaunchTables {
    Job *d_jobs = nullptr;
    Item *d_interp = nullptr;
    Item *d_grid = nullptr;
    Item *d_fold = nullptr;
    int64_t *d_slot_base = nullptr;  // float offset of each fold slot in d_scratch
    float *d_scratch = nullptr;      // partial tiles of split gridding tiles
    int64_t n_interp = 0;
    int64_t n_grid = 0;
    int64_t n_fold = 0;
    int64_t scratch_floats = 0;
    int grid_coils = 1;        // coils per gridding workgroup (LDS bound)
    size_t grid_lds = 0;       // dynamic LDS bytes for the gridding kernel
    int kind_interp = 0;       // kernel variant selector
    int kind_grid = 0;
    int interp_mode = kInterpGather;
    size_t interp_lds = 0;     // dynamic LDS bytes for the staged interpolation
    int interp_coils = 1;      // coils per LDS region load (staged interpolation)
    int grid_mode = kGridSpread;  // gridding variant (matches the plans' entry order)
    // matrix and tile gridding over a coil-minor copy of the samples: chunks of
    // st_cw coils, [chunk][sample][st_cw] per job, built by the copy items
    Item *d_tr = nullptr;
    int64_t n_tr = 0;
    float2 *d_st = nullptr;  // of the tile gridding only for launches that bring none
    int64_t st_elems = 0;
    int st_cw = 0;  // 0: the samples are read in place
    bool st_wide = false;  // tile gridding: offsets of samples read in place would pass 32 bits
    int wpad = 0;   // tile gridding: words per axis of the tap records
    int interp_vec = 0;  // staged interpolation: cells per load the regions allow (2, 1), 0: row by row only
    int interp_planes = 0;  // planes per sample, the average over the jobs
    int st_cpl = 1; // coils per lane of the matrix kernel over the copy (1 or 2)
    int64_t device_bytes = 0;  // bytes of the device allocations above
};

// Line transforms of one axis: N pixels <-> L grid points, by a kernel of
// length L (M = 0), by radices at run time (M = 0, radices.n > 0), or as chirp
// transforms by convolutions of length M (see tn_chirp.hip).
struct ChirpTable {  // one direction
    const float2 *in = nullptr;   // factors of the inputs
    const float2 *out = nullptr;  // factors of the outputs
    const float2 *b = nullptr;    // transform of the chirp, divided by M
};
// Radices of a length with small factors (see tn_smooth.hip).
constexpr int kSmoothPasses = 6;
struct SmoothRadices {
    int n = 0;  // passes, 0: not such an axis
    int r[kSmoothPasses] = {};
    int pitch = 0;  // LDS float2 per column
};
struct FftAxis {
    int N = 1, L = 1, M = 0;
    SmoothRadices radices;
    const float2 *tw = nullptr;  // exp(-2 pi i m / L), or / M
    ChirpTable fwd, inv;
};

}  // namespace tn

struct tn_plan {
    int device = 0;
    tn_plan_params p{};        // (z, y, x) as given; apod pointers cleared
    int32_t tile[3] = {1, 1, 1};   // (z, y, x)
    int32_t ntiles[3] = {1, 1, 1};
    int64_t ntiles_total = 1;
    int32_t itile[3] = {1, 1, 1};  // staged-interpolation tile (z, y, x)
    int32_t nitiles[3] = {1, 1, 1};
    int64_t nitiles_total = 1;
    float4 *d_pentries = nullptr;
    int32_t *d_pbin_off = nullptr;
    std::vector<int32_t> h_pbin_off;  // host copies (work-list construction)
    std::vector<int32_t> h_bin_off;
    std::vector<int32_t> h_mrow;      // host copy of d_mrow (work-list construction)
    // matrix-gridding runs per frame, keyed by the cells-per-item limit
    // (built once per plan; launch tables of any coil count reuse them; the
    // long-row threshold is the plan's grid_split, fixed for its lifetime)
    mutable std::map<int, std::vector<std::vector<tn::MatrixRun>>> mruns;
    float *d_coord = nullptr;
    float4 *d_entries = nullptr;
    int32_t *d_bin_off = nullptr;
    float *d_apod[3] = {nullptr, nullptr, nullptr};
    int64_t nentries = 0;
    int64_t footprint = -1;
    int grid_mode = tn::kGridSpread;  // effective gridding variant (entry order)
    int mix_mode = tn::kGridSpread;   // the variant asked for, or the automatic one without the tiles (batch_modes_mix)
    int32_t *d_mrow = nullptr;  // matrix gridding: row offsets, (nframes * cells + 1)
    int2 *d_mnz = nullptr;      // matrix gridding: (sample, weight bits) sorted by (frame, cell)
    tn::FftAxis axis[3];        // line transforms of the FFT stages, (x, y, z)
    float2 *d_fft = nullptr;    // their tables; null: no FFT stages
    bool stages_only = false;   // made by tn_stages_create: no samples, bins or tables
    bool fft_direct = false;    // every axis has a kernel of its own length (the pruned stages)
    int64_t fft_bytes = 0;
    int64_t mnnz = 0;
    int2 *d_tent = nullptr;     // tile gridding entries
    // tile gridding: per frame and (z, y) row of tiles, the signed x range
    // [lo, hi) of its tiles that footprints reach (x - G for the upper half of
    // the grid, so that a range around the centre of k-space is one piece)
    int2 *d_rows = nullptr;
    float *d_taps = nullptr;    // tile gridding: tap records, tiles_tap_stride words per sample
    int wpad = 0;
    std::map<int64_t, tn::LaunchTables> cache;
    std::map<int64_t, tn::LaunchTables> cache_gather;  // gather-mode tables (low-rank interpolation)
    std::map<int64_t, tn::LaunchTables> cache_lowrank; // tables of the low-rank gridding (no coil-minor copy)
};

struct tn_batch {
    int device = 0;
    std::vector<tn::LaunchTables> tables;  // one per gridding variant among the plans
    std::vector<tn_plan *> plans;
};

namespace tn {

// Error reporting (thread-local message + return code).
int fail(int code, const char *fmt, ...);
void clear_error();

// Fills job records for every frame of `plan` with the given placement.
void make_jobs(const tn_plan *plan, int64_t nbatch, int64_t grid_off,
               int64_t samp_off, int64_t w_off, std::vector<Job> &jobs);
void free_tables(LaunchTables &t);

// Kernel launchers (defined in the kernel translation units).
int launch_interp(const LaunchTables &t, const float2 *grid, float2 *samp,
                  const float *weight, hipStream_t stream);
int launch_grid(const LaunchTables &t, const float2 *samp, float2 *grid,
                const float *weight, hipStream_t stream, LowRank lr = LowRank{},
                float *scratch = nullptr, bool ranged = false, float2 *copy = nullptr);
// (ranged: cells beyond the row ranges may be left unwritten; copy: room for the
// sample copy of the tile gridding, null: the table's own, or none)
// Device address of the fixed gridding workspace on `device` (looked up once
// per device with hipGetSymbolAddress; no allocation).
int static_scratch(int device, float **out);
int launch_interp_lowrank(const LaunchTables &t, const float2 *grid, float2 *samp,
                          const float *weight, hipStream_t stream, LowRank lr);
// Sums the partial tiles of split gridding tiles (nothing when none are split).
int launch_fold(const LaunchTables &t, float2 *grid, const float *scratch, hipStream_t stream);
int launch_apod_pad(const tn_plan *plan, const float2 *image, float2 *grid,
                    int64_t nimg, hipStream_t stream);
int launch_crop_apod(const tn_plan *plan, const float2 *grid, float2 *image,
                     int64_t nimg, hipStream_t stream);
int build_bins(tn_plan *plan, hipStream_t stream);
// Whether an explicit grid_mode 4 is accepted: 3D, at most 4 taps per axis,
// grids of whole 8x8x4 blocks with at least two per axis. (The automatic mode
// uses the tile gridding beyond that, where tiles_serve says so.)
inline bool tiles_fit(const tn_plan_params &p) {
    if (p.ndim != 3) return false;
    const int block[3] = {4, 8, 8};  // params are (z, y, x)
    for (int d = 0; d < 3; ++d)
        if (p.width[d] > 4 || p.grid[d] % block[d] != 0 || p.grid[d] < 2 * block[d]) return false;
    return true;
}
bool tiles_serve(const tn_plan_params &p);
// Entries of a tile plan (coordinates uploaded): below 2^31 - 1 an upper bound, else exact.
int tile_entries(const tn_plan *plan, hipStream_t stream, int64_t &n);
int launch_tiles(const LaunchTables &t, const float2 *samp, float2 *grid, const float *weight, hipStream_t stream,
                 const LowRank &lr, float *scratch, bool ranged, float2 *st);
int build_matrix(tn_plan *plan, hipStream_t stream);
// Pruned, fused oversampled-grid FFT stages (2D and 3D plans).
int build_fft(tn_plan *plan, hipStream_t stream);
int launch_fft_forward(const tn_plan *plan, const float2 *image, float2 *grid, int64_t nimg, hipStream_t stream,
                       bool ranged = false);
int launch_fft_adjoint(const tn_plan *plan, float2 *grid, float2 *image, int64_t nimg, hipStream_t stream,
                       bool ranged = false);
int launch_fft_z_forward(const tn_plan *plan, const float2 *image, float2 *zout, int64_t nimg, hipStream_t stream);
int launch_fft_z_adjoint(const tn_plan *plan, const float2 *zin, float2 *image, int64_t nimg, hipStream_t stream);
int launch_convolve(const tn_plan *plan, const float2 *image, const float2 *kern, int64_t nkern, float2 *out,
                    float2 *work0, float2 *work1, int64_t nimg, hipStream_t stream);
// Whether the plan's whole transforms leave out the grid cells that no
// footprint reaches (3D, row ranges, and a kernel of its own length along x).
bool rows_ranged(const tn_plan *plan, int64_t nbatch);
// Lengths with factors up to 17 (tn_smooth.hip).
bool smooth_radices(int L, SmoothRadices &f);
int smooth_prepare(const FftAxis &a);
int smooth_rows(const FftAxis &a, bool inverse, float2 *data, int64_t nlines, hipStream_t stream);
int smooth_product(const FftAxis &a, float2 *data, int64_t nlines, const float2 *kern, int64_t nk, hipStream_t stream);
int smooth_cols(const FftAxis &a, bool inverse, const float2 *src, float2 *dst, int64_t nimg, int cols, int pitch,
                int hx, const float *apx, const float *apy, float scale, hipStream_t stream);
// Chirp transforms (tn_chirp.hip) of axes with a chirp_length: their tables in
// float2 (appended to `host`; chirp_bind sets the pointers for a table that
// starts at `base`), and the stages.
void chirp_tables(const FftAxis &a, std::vector<float2> &host);
void chirp_bind(FftAxis &a, const float2 *base);
int chirp_prepare(const FftAxis &a);
int chirp_rows(const FftAxis &a, bool inverse, float2 *data, int64_t nlines, hipStream_t stream);
int chirp_product(const FftAxis &a, float2 *data, int64_t nlines, const float2 *kern, int64_t nk, hipStream_t stream);
int chirp_cols(const FftAxis &a, bool inverse, const float2 *src, float2 *dst, int64_t nimg, int cols, int pitch,
               int hx, const float *apx, const float *apy, float scale, hipStream_t stream);
int count_footprint(tn_plan *plan, hipStream_t stream);

// Variant selection shared by the table builder and the launchers.
int interp_kind(const std::vector<Job> &jobs);

}  // namespace tn

#define TN_HIP(call)                                                          \
    do {                                                                      \
        hipError_t e_ = (call);                                               \
        if (e_ != hipSuccess)                                                 \
            return ::tn::fail(TN_E_HIP, "%s failed: %s (%s:%d)", #call,       \
                              hipGetErrorString(e_), __FILE__, __LINE__);     \
    } while (0)
