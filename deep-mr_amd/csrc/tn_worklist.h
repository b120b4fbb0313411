// Work items of the gridding and interpolation launches, and the host-side
// construction of the sparse-matrix gridding items. Plain C++ (no HIP
// types), so the construction can be checked by a host-only program.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#ifdef __HIPCC__
#define TN_HOST_DEVICE __host__ __device__
#else
#define TN_HOST_DEVICE
#endif

namespace tn {

// Pieces of a kernel footprint along one axis for the tile gridding: the
// cells base .. base + W - 1 (mod G, W <= G, 0 <= base < G) as (tile, local
// origin) pairs: cell c of a tile is tap c - local of the footprint where that
// lies in [0, W). Cells before the wrap give the tiles they meet the origin
// base - t T, wrapped cells base - G - t T; a tile can hold both a first and a
// wrapped piece (grids shorter than T + W - 1), whose cells are disjoint.
// local is in [-(W - 1), T - 1]. Returns the number of pieces, at most
// kMaxPieces for W <= 8 and T >= 4.
constexpr int kMaxPieces = 6;
TN_HOST_DEVICE inline int axis_pieces(int base, int W, int G, int T, int (&tile)[kMaxPieces],
                                      int (&local)[kMaxPieces]) {
    int n = 0;
    const int end = base + W;
    const int stop = end < G ? end : G;
    for (int t = base / T; t * T < stop && n < kMaxPieces; ++t) {
        tile[n] = t;
        local[n++] = base - t * T;
    }
    for (int t = 0; t * T < end - G && n < kMaxPieces; ++t) {
        tile[n] = t;
        local[n++] = base - G - t * T;
    }
    return n;
}

// Convolution length of an axis of N pixels and L grid points done as a chirp
// transform, 0: none. Lengths at most a half apart, from 96 on a third, so that
// padding costs little; unit axes (1D data as one row) keep the separate kernels.
constexpr int kChirpLengths[] = {32,  48,  64,  96,  128, 160, 192, 240,  256,
                                 320, 384, 480, 512, 640, 768, 1024, 1280, 1536};
inline int chirp_length(int N, int L) {
    if (L < 2) return 0;
    for (int M : kChirpLengths)
        if (M >= (int64_t)N + L - 1) return M;
    return 0;
}

// Most pieces of a footprint of W taps along an axis of tiles of T cells: the
// tiles it can meet, one more for a wrap.
constexpr int most_pieces(int W, int T) { return (W + T - 2) / T + 2; }

// Planes per sample of a launch, the rounded average over its jobs: a small job
// of few planes does not choose the others' loads (the staged interpolation).
template <class Jobs>
int mean_planes(const Jobs &jobs) {
    int64_t samples = 0, planes = 0;
    for (const auto &j : jobs) {
        samples += j.npts;
        planes += j.npts * j.nbatch;
    }
    return samples == 0 ? 0 : (int)((planes + samples / 2) / samples);
}

constexpr int kMatrixCoils = 16;   // widest record of the matrix gridding (coils per item)
constexpr int kMatrixStage = 1024; // entries of a run of cells staged in LDS (also the longest short row), 3D
constexpr int kMatrixStage2d = 512; // the same in 2D: a smaller stage leaves LDS for more workgroups per CU
                                    // (spiral 8x16: 0.175 against 0.181 ms; in 3D 512 measured slower)
constexpr int kMatrixPart = 2048;  // entries per workgroup of a long row; longer rows are summed
                                   // in parts (kMatrixCoils-wide partial records, folded in order)

// LDS-staged entries per matrix-gridding item for plans of `ndim` dimensions.
inline int matrix_stage(int ndim) { return ndim == 3 ? kMatrixStage : kMatrixStage2d; }

// Work item. Gathering interpolation: unit = sample block. Staged
// interpolation: unit = tile, [e0, e1) = slice of its entries. Gridding:
// unit = tile, [e0, e1) = slice of its entries; part / slot >= 0 when the
// tile is split (partial `part` of fold slot `slot`), slot = -1 otherwise.
// Tile fold items: unit = tile, e0 = slot, e1 = number of parts, elements
// [part, slot) of the partial tile. Matrix gridding items: see matrix_items.
struct alignas(16) Item {
    int32_t job, unit, c0, c1;
    int32_t e0, e1, part, slot;
};

constexpr int kFoldChunks = 32;      // most workgroups per tile fold item
constexpr int kFoldChainParts = 16;  // parts per element chain above which a tile fold is spread wider

// Fold items of one split gridding tile (coils c0 .. c1 - 1, `nparts`
// partial tiles of `elems` elements in fold slot `slot`): one workgroup of
// `block` lanes walks a tile of at most kFoldChainParts parts; a tile of more
// parts (a longer dependent chain per element) spreads its elements over
// ceil(parts / kFoldChainParts) contiguous ranges, at most kFoldChunks and at
// most one per `block` elements (one element per lane at the limit).
inline void tile_fold_items(int job, int tile, int c0, int c1, int slot, int nparts, int64_t elems, int block,
                            std::vector<Item> &fold) {
    const int64_t nsub = std::max<int64_t>(
        1, std::min<int64_t>({(int64_t)kFoldChunks, (elems + block - 1) / block,
                              ((int64_t)nparts + kFoldChainParts - 1) / kFoldChainParts}));
    const int64_t per = (elems + nsub - 1) / nsub;
    for (int64_t k = 0; k < nsub && k * per < elems; ++k)
        fold.push_back(Item{job, tile, c0, c1, slot, nparts, (int32_t)(k * per),
                            (int32_t)std::min(elems, (k + 1) * per)});
}

constexpr int kTilesGroup = 4;  // tile-gridding items (waves) per workgroup
constexpr int kDealXcds = 8;    // XCDs the hardware deals workgroups to in turn
constexpr int kTilesBase = 24;  // a tile's own cost in entries, for the balance over the XCDs
constexpr int32_t kTilesJoin = 1 << 30;  // flag of an item's unit: the workgroup's four items share the tile

constexpr int32_t kTilesFill = -2;       // slot of an item that zeroes a run of e1 tiles without entries
constexpr int kTilesFillCells = 64;      // most cells of such a run: 512-byte rows

// Runs of tiles without entries along the rows of a frame: at a run's first
// tile its length (at most `longest`), 0 at every other tile.
inline std::vector<int32_t> empty_runs(const int32_t *off, const int32_t (&nt)[3], int longest) {
    std::vector<int32_t> run((size_t)nt[0] * nt[1] * nt[2], 0);
    for (size_t row = 0; row < run.size(); row += nt[0])
        for (int x = 0, first = -1; x < nt[0]; ++x) {
            const size_t t = row + x;
            if (off[t] != off[t + 1]) {
                first = -1;
                continue;
            }
            if (first < 0 || run[row + first] == longest) first = x;
            ++run[row + first];
        }
    return run;
}

// Cost of an item in entries, for the balance: a tile's own cost is mostly its
// stores, which a run of empty tiles makes in longer rows.
inline int64_t tiles_cost(const Item &it) {
    return it.slot == kTilesFill ? (int64_t)kTilesBase / 2 * it.e1 : kTilesBase + (it.e1 - it.e0);
}

// Tiles of a frame in bricks (x fastest inside and over the bricks), so that
// neighbours along every axis are near each other in the work list.
inline std::vector<int32_t> brick_order(const int32_t (&nt)[3], int ndim) {
    const int b[3] = {8, ndim == 3 ? 4 : 8, ndim == 3 ? 4 : 1};  // x, y, z
    std::vector<int32_t> order;
    order.reserve((size_t)nt[0] * nt[1] * nt[2]);
    for (int z0 = 0; z0 < nt[2]; z0 += b[2])
        for (int y0 = 0; y0 < nt[1]; y0 += b[1])
            for (int x0 = 0; x0 < nt[0]; x0 += b[0])
                for (int z = z0; z < std::min(nt[2], z0 + b[2]); ++z)
                    for (int y = y0; y < std::min(nt[1], y0 + b[1]); ++y)
                        for (int x = x0; x < std::min(nt[0], x0 + b[0]); ++x)
                            order.push_back((z * nt[1] + y) * nt[0] + x);
    return order;
}

// Work list of the tile gridding, four items per workgroup: first the
// workgroups that share a tile (`joined`), as listed (the hardware deals
// workgroups to the XCDs in turn, which spreads a hot tile's parts over all of
// them), then the other tiles (`grid`, which becomes the whole list) in one
// contiguous range per XCD, so that neighbouring tiles, which read many of the
// same samples, share an L2. The ranges hold equal work (entries, plus
// kTilesBase for a tile's own cost), not equal numbers of tiles: on a kooshball
// the XCDs of the dense centre otherwise worked 1.7 times as long as the
// average one. Shorter ranges are filled up with empty items (job -1).
inline void tiles_deal(std::vector<Item> &joined, std::vector<Item> &grid) {
    constexpr int64_t per = kTilesGroup, kXcds = kDealXcds;
    const Item none{-1, 0, 0, 0, 0, 0, 0, -1};
    std::vector<Item> rest;
    rest.swap(grid);
    grid.swap(joined);
    if (rest.empty()) return;
    while (grid.size() % (per * kXcds)) grid.push_back(none);
    const int64_t wg = ((int64_t)rest.size() + per - 1) / per;
    double total = 0;
    for (const Item &it : rest) total += tiles_cost(it);
    int64_t first[kXcds + 1] = {0}, longest = 0;  // workgroup ranges
    double sum = 0;
    int x = 0;
    for (int64_t w = 0; w < wg; ++w) {
        while (x + 1 < kXcds && sum >= total * (x + 1) / kXcds) first[++x] = w;
        for (int64_t q = w * per; q < std::min<int64_t>((w + 1) * per, (int64_t)rest.size()); ++q)
            sum += tiles_cost(rest[q]);
    }
    while (x < kXcds) first[++x] = wg;
    for (x = 0; x < kXcds; ++x) longest = std::max(longest, first[x + 1] - first[x]);
    grid.reserve(grid.size() + longest * kXcds * per);
    for (int64_t w = 0; w < longest; ++w)
        for (x = 0; x < kXcds; ++x)
            for (int64_t q = 0; q < per; ++q) {
                const int64_t from = (first[x] + w) * per + q;
                grid.push_back(first[x] + w < first[x + 1] && from < (int64_t)rest.size() ? rest[from] : none);
            }
}

// Matrix-gridding work of one frame, independent of the coils: a run of
// ncells consecutive cells from `cell` whose entries are [e0, e0 + ne), or,
// with ncells < 0, a long row `cell` summed in -ncells parts.
struct MatrixRun {
    int32_t cell, ncells, e0, ne;
};

// Runs of one frame from its CSR row offsets row[0 .. ncell]: consecutive
// cells with at most cpi cells and at most `stage` entries per run, so that
// a run's entries (contiguous in the CSR order) fit the kernel's LDS stage;
// a row longer than mlong (<= stage) ends the run and becomes a long-row run
// of ceil(len / kMatrixPart) parts. Long rows are listed first.
inline void matrix_runs_of(const int32_t *row, int64_t ncell, int cpi, int mlong, std::vector<MatrixRun> &out,
                           int stage = kMatrixStage) {
    std::vector<MatrixRun> shorts;
    int64_t start = 0;
    int ncells = 0, nent = 0;
    auto close = [&]() {
        if (ncells > 0) shorts.push_back(MatrixRun{(int32_t)start, ncells, row[start], row[start + ncells] - row[start]});
        ncells = 0;
        nent = 0;
    };
    for (int64_t c = 0; c < ncell; ++c) {
        const int len = row[c + 1] - row[c];
        if (len > mlong) {
            close();
            out.push_back(MatrixRun{(int32_t)c, -((len + kMatrixPart - 1) / kMatrixPart), row[c], len});
            continue;
        }
        if (ncells == cpi || nent + len > stage) close();
        if (ncells == 0) start = c;
        ++ncells;
        nent += len;
    }
    close();
    out.insert(out.end(), shorts.begin(), shorts.end());
}

// Gridding items of one job (frame, `nbatch` coils in records of mc coils)
// from its runs. A run of cells: unit = first cell, e1 = cell count | entry
// count << 16, slot = first entry, e0 = coil record, part = 0. A long row:
// one item per part (unit = cell, e1 = part, part = 1, e0 = coil record);
// with several parts, slot = first partial record (kMatrixCoils complex
// values each, 2 * kMatrixCoils floats of scratch) and one fold item (e1 =
// number of parts, part = 0, slot = first record) sums them in part order;
// slot = -1 for a single part. Appends to grid / fold, advances scratch
// (floats).
inline void matrix_items(int job, const std::vector<MatrixRun> &runs, int nbatch, int mc, std::vector<Item> &grid,
                         std::vector<Item> &fold, int64_t &scratch) {
    for (const MatrixRun &r : runs) {
        for (int c0 = 0; c0 < nbatch; c0 += mc) {
            const int c1 = std::min(nbatch, c0 + mc);
            if (r.ncells > 0) {
                grid.push_back(Item{job, r.cell, c0, c1, c0 / mc, r.ncells | (r.ne << 16), 0, r.e0});
                continue;
            }
            const int nparts = -r.ncells;
            if (nparts == 1) {
                grid.push_back(Item{job, r.cell, c0, c1, c0 / mc, 0, 1, -1});
                continue;
            }
            const int32_t rec = (int32_t)(scratch / (2 * kMatrixCoils));
            scratch += (int64_t)nparts * 2 * kMatrixCoils;
            for (int k = 0; k < nparts; ++k) grid.push_back(Item{job, r.cell, c0, c1, c0 / mc, k, 1, rec});
            fold.push_back(Item{job, r.cell, c0, c1, c0 / mc, nparts, 0, rec});
        }
    }
}

}  // namespace tn
