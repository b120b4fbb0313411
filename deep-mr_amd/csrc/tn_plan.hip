// Plan construction on the device: tile binning of every sample.
//
// Each sample is entered into every gridding tile its kernel footprint
// touches (owner-computes: a tile later accumulates only the taps that fall
// inside it, so every tile is written exactly once without global atomics).
// Entries are keyed by (frame, tile) and sorted with a stable radix sort, so
// inside a tile the samples keep ascending sample order: the gridding
// accumulation order is fixed and the adjoint is deterministic.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "tn_internal.h"
#include "tn_kb.h"

namespace tn {
namespace {

struct AxisGeom {
    int G, W, shift, T;
};

struct BinGeom {
    float beta[3];       // Kaiser-Bessel beta (x, y, z)
    int ndim;
    int64_t npts;
    int nframes;
    AxisGeom ax[3];      // (x, y, z)
    int NT[3];           // tiles per axis (x, y, z)
    int64_t ntiles;      // product of NT
};

// Distinct tiles touched along one axis by a footprint starting at `base`.
// A footprint that wraps around the grid edge can come back into a tile it
// already touched (when the last tile is narrower than W - 1), so the check
// is against every tile collected so far, not only the previous one.
__device__ __forceinline__ int axis_tiles(const AxisGeom &a, int base, int (&tl)[kMaxWidth]) {
    int n = 0;
    for (int k = 0; k < a.W; ++k) {
        const int t = wrap_add(base, k, a.G) / a.T;
        bool seen = false;
        for (int j = 0; j < n; ++j) seen |= (tl[j] == t);
        if (!seen) tl[n++] = t;
    }
    return n;
}

__device__ __forceinline__ float beta_of(const BinGeom &g, int d) { return g.beta[d]; }

__device__ __forceinline__ int axis_base(const AxisGeom &a, float g) {
    if (a.W == 1) return wrap_mod((int)g + a.shift, a.G);
    const float x0 = ceilf(g - 0.5f * (float)a.W);
    return wrap_mod((int)x0 + a.shift, a.G);
}

__global__ void bin_count_kernel(BinGeom geo, const float *__restrict__ coord,
                                 int32_t *__restrict__ counts) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        int c = 1;
        for (int d = 0; d < geo.ndim; ++d) {
            int tl[kMaxWidth];
            const int base = axis_base(geo.ax[d], coord[i * geo.ndim + d]);
            c *= axis_tiles(geo.ax[d], base, tl);
        }
        counts[i] = c;
    }
}

// Primary bins: every sample once, keyed by the tile holding its footprint
// origin (the staged interpolation loads that tile plus a W-1 halo).
__global__ void bin_primary_kernel(BinGeom geo, const float *__restrict__ coord,
                                   uint32_t *__restrict__ keys, int32_t *__restrict__ vals) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t frame = i / geo.npts;
        int t[3] = {0, 0, 0};
        for (int d = 0; d < geo.ndim; ++d)
            t[d] = axis_base(geo.ax[d], coord[i * geo.ndim + d]) / geo.ax[d].T;
        const int64_t tile = ((int64_t)t[2] * geo.NT[1] + t[1]) * geo.NT[0] + t[0];
        keys[i] = (uint32_t)(frame * geo.ntiles + tile);
        vals[i] = (int32_t)(i - frame * geo.npts);
    }
}

__global__ void bin_emit_kernel(BinGeom geo, const float *__restrict__ coord,
                                const int32_t *__restrict__ offsets,
                                uint32_t *__restrict__ keys, int32_t *__restrict__ vals) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t frame = i / geo.npts;
        const int32_t pt = (int32_t)(i - frame * geo.npts);
        int tl[3][kMaxWidth];
        int nt[3] = {1, 1, 1};
        for (int d = 0; d < 3; ++d) tl[d][0] = 0;
        for (int d = 0; d < geo.ndim; ++d) {
            const int base = axis_base(geo.ax[d], coord[i * geo.ndim + d]);
            nt[d] = axis_tiles(geo.ax[d], base, tl[d]);
        }
        int32_t pos = offsets[i];
        for (int a = 0; a < nt[2]; ++a)
            for (int b = 0; b < nt[1]; ++b)
                for (int c = 0; c < nt[0]; ++c) {
                    const int64_t tile =
                        ((int64_t)tl[2][a] * geo.NT[1] + tl[1][b]) * geo.NT[0] + tl[0][c];
                    keys[pos] = (uint32_t)(frame * geo.ntiles + tile);
                    vals[pos] = pt;
                    ++pos;
                }
    }
}

// bin_off[k] = first entry whose key >= k, for k in [0, nbins]; e == n
// stands for a virtual key nbins.
__global__ void bin_offsets_kernel(const uint32_t *__restrict__ keys, int64_t n, int64_t nbins,
                                   int32_t *__restrict__ bin_off) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e <= n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = e < n ? (int64_t)keys[e] : nbins;
        const int64_t kp = e > 0 ? (int64_t)keys[e - 1] : -1;
        for (int64_t b = kp + 1; b <= k; ++b) bin_off[b] = (int32_t)e;
    }
}

// Gridding matrix entries of every sample, in (sample, tap) order, tap x
// fastest: key = frame * cells + output cell, value = (sample within its
// frame, weight bits) packed low/high in 64 bits. The weight is the product
// of the per-axis Kaiser-Bessel taps (z * y first, then x), the same taps
// the other gridding variants evaluate.
__global__ void matrix_emit_kernel(BinGeom geo, const float *__restrict__ coord, int taps,
                                   uint32_t *__restrict__ keys, uint64_t *__restrict__ vals) {
    const int64_t total = geo.npts * geo.nframes;
    const int64_t ncell = (int64_t)geo.ax[0].G * geo.ax[1].G * geo.ax[2].G;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t frame = i / geo.npts;
        const int64_t p = i - frame * geo.npts;
        int base[3] = {0, 0, 0};
        float w[3][kMaxWidth];
        for (int d = 0; d < 3; ++d) {
            if (d < geo.ndim) {
                axis_taps<kMaxWidth>(coord[i * geo.ndim + d], geo.ax[d].W, geo.ax[d].G, geo.ax[d].shift, beta_of(geo, d),
                             base[d], w[d]);
            } else {
                w[d][0] = 1.0f;
            }
        }
        const int Wx = geo.ax[0].W, Wy = geo.ax[1].W;
        const int64_t e0 = i * taps;
        for (int t = 0; t < taps; ++t) {
            const int kx = t % Wx, ky = (t / Wx) % Wy, kz = t / (Wx * Wy);
            const int64_t cell = ((int64_t)wrap_add(base[2], kz, geo.ax[2].G) * geo.ax[1].G +
                                  wrap_add(base[1], ky, geo.ax[1].G)) * geo.ax[0].G +
                                 wrap_add(base[0], kx, geo.ax[0].G);
            const float wt = (w[2][kz] * w[1][ky]) * w[0][kx];
            keys[e0 + t] = (uint32_t)(frame * ncell + cell);
            vals[e0 + t] = ((uint64_t)(uint32_t)__float_as_int(wt) << 32) | (uint64_t)(uint32_t)p;
        }
    }
}

// Tile gridding: the pieces of sample i's footprint per axis (unused axes:
// tile 0, origin 0); returns their product, the sample's entry count.
__device__ __forceinline__ int tile_pieces(const BinGeom &geo, const float *c, int (&nt)[3],
                                           int (&tile)[3][kMaxPieces], int (&local)[3][kMaxPieces]) {
    int n = 1;
    for (int d = 0; d < 3; ++d) {
        nt[d] = 1;
        tile[d][0] = local[d][0] = 0;
        if (d < geo.ndim)
            nt[d] = axis_pieces(axis_base(geo.ax[d], c[d]), geo.ax[d].W, geo.ax[d].G, geo.ax[d].T, tile[d], local[d]);
        n *= nt[d];
    }
    return n;
}

// Tile entries of all samples, in 64 bits (the offsets are 32-bit): pieces of
// the tile gridding's footprints, or distinct tiles.
template <bool PIECES>
__global__ void entry_total_kernel(BinGeom geo, const float *__restrict__ coord, unsigned long long *__restrict__ sum) {
    const int64_t total = geo.npts * geo.nframes;
    unsigned long long n = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        int c = 1;
        if (PIECES) {
            int nt[3], tile[3][kMaxPieces], local[3][kMaxPieces];
            c = tile_pieces(geo, coord + i * geo.ndim, nt, tile, local);
        } else {
            for (int d = 0; d < geo.ndim; ++d) {
                int tl[kMaxWidth];
                c *= axis_tiles(geo.ax[d], axis_base(geo.ax[d], coord[i * geo.ndim + d]), tl);
            }
        }
        n += (unsigned long long)c;
    }
    if (n > 0) atomicAdd(sum, n);
}

__global__ void tiles_count_kernel(BinGeom geo, const float *__restrict__ coord, int32_t *__restrict__ counts) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        int nt[3], tile[3][kMaxPieces], local[3][kMaxPieces];
        counts[i] = tile_pieces(geo, coord + i * geo.ndim, nt, tile, local);
    }
}

// Tile gridding entries of every sample, keyed by (frame, tile): value =
// (sample within its frame, tile-local origin + 16 per axis in bytes).
__global__ void tiles_emit_kernel(BinGeom geo, const float *__restrict__ coord, const int32_t *__restrict__ offsets,
                                  uint32_t *__restrict__ keys, uint64_t *__restrict__ vals) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t frame = i / geo.npts;
        const uint32_t p = (uint32_t)(i - frame * geo.npts);
        int nt[3], tile[3][kMaxPieces], local[3][kMaxPieces];
        tile_pieces(geo, coord + i * geo.ndim, nt, tile, local);
        int32_t pos = offsets[i];
        for (int a = 0; a < nt[2]; ++a)
            for (int b = 0; b < nt[1]; ++b)
                for (int c = 0; c < nt[0]; ++c) {
                    const int64_t t = ((int64_t)tile[2][a] * geo.NT[1] + tile[1][b]) * geo.NT[0] + tile[0][c];
                    const uint32_t loc = (uint32_t)(local[0][c] + 16) | (uint32_t)(local[1][b] + 16) << 8 |
                                         (uint32_t)(local[2][a] + 16) << 16;
                    keys[pos] = (uint32_t)(frame * geo.ntiles + t);
                    vals[pos] = ((uint64_t)loc << 32) | p;
                    ++pos;
                }
    }
}

// Row ranges (tn_plan::d_rows) from the tile offsets: one lane per row of tiles.
__global__ void tiles_rows_kernel(BinGeom geo, const int32_t *__restrict__ bin_off, int64_t nrows,
                                  int2 *__restrict__ rows) {
    const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const AxisGeom a = geo.ax[0];
    const int64_t t0 = r * geo.NT[0];
    int lo = 0, hi = 0;
    for (int t = 0; t < geo.NT[0]; ++t) {
        if (bin_off[t0 + t] == bin_off[t0 + t + 1]) continue;
        for (int x = t * a.T; x < min((t + 1) * a.T, a.G); ++x) {
            const int u = signed_x(x, a.G);
            const bool first = lo == hi;
            lo = first ? u : min(lo, u);
            hi = first ? u + 1 : max(hi, u + 1);
        }
    }
    rows[r] = make_int2(lo, hi);
}

// Tap records of the tile gridding (tiles_tap_stride): the taps
// the other gridding variants evaluate, padded with zeros.
template <int WP>
__global__ void tiles_taps_kernel(BinGeom geo, const float *__restrict__ coord, float *__restrict__ taps) {
    const int64_t total = geo.npts * geo.nframes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        float *t = taps + i * tiles_tap_stride(geo.ndim, WP);
        for (int d = 0; d < geo.ndim; ++d) {
            int base;
            float w[WP];
            axis_taps<WP>(coord[i * geo.ndim + d], geo.ax[d].W, geo.ax[d].G, geo.ax[d].shift, beta_of(geo, d), base, w);
            for (int k = 0; k < WP; ++k) t[d * WP + k] = w[k];
        }
    }
}

__global__ void bin_gather_kernel(BinGeom geo, const float *__restrict__ coord,
                                  const uint32_t *__restrict__ keys,
                                  const int32_t *__restrict__ vals, int64_t n,
                                  float4 *__restrict__ entries) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t frame = keys[e] / geo.ntiles;
        const int32_t pt = vals[e];
        const float *c = coord + (frame * geo.npts + pt) * geo.ndim;
        float4 v;
        v.x = c[0];
        v.y = geo.ndim > 1 ? c[1] : 0.0f;
        v.z = geo.ndim > 2 ? c[2] : 0.0f;
        v.w = __int_as_float(pt);
        entries[e] = v;
    }
}

// Reordering of gridding bins: inside each bin, entries are ordered by
// (rank of the sample among the bin's samples with the same footprint
// origin, origin, sample). Consecutive entries then mostly have distinct
// origins, so the lanes of one LDS atomic in the gridding kernel update
// distinct cells. The order is a pure function of the trajectory.
__device__ __forceinline__ uint32_t entry_origin(const BinGeom &geo, const float4 &en) {
    const float c[3] = {en.x, en.y, en.z};
    int b[3] = {0, 0, 0};
    for (int d = 0; d < geo.ndim; ++d) b[d] = axis_base(geo.ax[d], c[d]);
    const uint32_t gy = geo.ndim > 1 ? geo.ax[1].G : 1;
    return ((uint32_t)b[2] * gy + (uint32_t)b[1]) * (uint32_t)geo.ax[0].G + (uint32_t)b[0];
}

__global__ void origin_key_kernel(BinGeom geo, const uint32_t *__restrict__ bin_keys,
                                  const float4 *__restrict__ entries, int64_t n,
                                  uint64_t *__restrict__ key, int32_t *__restrict__ val) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        key[e] = ((uint64_t)bin_keys[e] << 32) | entry_origin(geo, entries[e]);
        val[e] = (int32_t)e;
    }
}

__global__ void group_head_kernel(const uint64_t *__restrict__ key, int64_t n, int32_t *__restrict__ head) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        head[e] = (e == 0 || key[e] != key[e - 1]) ? (int32_t)e : 0;
}

__global__ void rank_key_kernel(const uint64_t *__restrict__ key, const int32_t *__restrict__ start,
                                int64_t n, uint64_t *__restrict__ key2) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        key2[e] = (key[e] >> 32 << 32) | (uint32_t)(e - start[e]);
}

__global__ void permute_entries_kernel(const float4 *__restrict__ src, const int32_t *__restrict__ idx,
                                       int64_t n, float4 *__restrict__ dst) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        dst[e] = src[idx[e]];
}

struct MaxOp {
    __device__ __forceinline__ int32_t operator()(int32_t a, int32_t b) const { return a > b ? a : b; }
};

// Marks every grid cell touched by a footprint (one frame).
__global__ void footprint_mark_kernel(BinGeom geo, const float *__restrict__ coord,
                                      uint8_t *__restrict__ mask) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < geo.npts;
         i += (int64_t)gridDim.x * blockDim.x) {
        int base[3] = {0, 0, 0};
        int w[3] = {1, 1, 1};
        for (int d = 0; d < geo.ndim; ++d) {
            base[d] = axis_base(geo.ax[d], coord[i * geo.ndim + d]);
            w[d] = geo.ax[d].W;
        }
        const int Gx = geo.ax[0].G, Gy = geo.ndim > 1 ? geo.ax[1].G : 1;
        const int Gz = geo.ndim > 2 ? geo.ax[2].G : 1;
        for (int a = 0; a < w[2]; ++a) {
            const int z = geo.ndim > 2 ? wrap_add(base[2], a, Gz) : 0;
            for (int b = 0; b < w[1]; ++b) {
                const int y = geo.ndim > 1 ? wrap_add(base[1], b, Gy) : 0;
                for (int c = 0; c < w[0]; ++c) {
                    const int x = wrap_add(base[0], c, Gx);
                    mask[((int64_t)z * Gy + y) * Gx + x] = 1;
                }
            }
        }
    }
}

__global__ void count_mask_kernel(const uint8_t *__restrict__ mask, int64_t n,
                                  unsigned long long *__restrict__ out) {
    unsigned long long local = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        local += mask[i];
    __shared__ unsigned long long red[kBlock];
    red[threadIdx.x] = local;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(out, red[0]);
}

BinGeom make_geom(const tn_plan *plan, bool primary = false) {
    BinGeom g{};
    g.ndim = plan->p.ndim;
    g.npts = plan->p.npts;
    g.nframes = plan->p.nframes;
    for (int d = 0; d < 3; ++d) {
        const int zyx = 2 - d;
        g.ax[d].G = plan->p.grid[zyx];
        g.ax[d].W = plan->p.width[zyx];
        g.ax[d].shift = plan->p.shift[zyx];
        g.beta[d] = plan->p.beta[zyx];
        g.ax[d].T = primary ? plan->itile[zyx] : plan->tile[zyx];
        g.NT[d] = primary ? plan->nitiles[zyx] : plan->ntiles[zyx];
    }
    g.ntiles = primary ? plan->nitiles_total : plan->ntiles_total;
    return g;
}

unsigned grid_blocks(int64_t n) {
    const int64_t b = (n + kBlock - 1) / kBlock;
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>(b, 65536));
}

// RAII holder for temporaries of the plan build.
struct DevBuf {
    void *p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
};

}  // namespace

namespace {

// Stable radix sort of (key, sample) pairs, then per-bin offsets and the
// sorted entry records (coordinates + sample index).
int order_by_origin(const BinGeom &geo, const uint32_t *bin_keys, int64_t n, float4 *entries,
                    bool spread, hipStream_t stream);

// Entry order inside each bin: sample order, footprint-origin order (runs
// of equal origin, gridding by register runs) or round-robin over origins
// (gridding by per-sample LDS atomics).
enum EntryOrder { kOrderSample = 0, kOrderOrigin = 1, kOrderSpread = 2 };

int sort_entries(const BinGeom &geo, const float *coord, void *keys, void *vals, int64_t n,
                 int32_t *bin_off, float4 **entries, hipStream_t stream, int order = kOrderSample) {
    const int64_t nbins = geo.nframes * geo.ntiles;
    DevBuf keys_sorted, vals_sorted, sort_tmp;
    TN_HIP(hipMalloc(&keys_sorted.p, sizeof(uint32_t) * n));
    TN_HIP(hipMalloc(&vals_sorted.p, sizeof(int32_t) * n));
    int end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) < (uint64_t)nbins) ++end_bit;
    size_t sort_bytes = 0;
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (uint32_t *)keys,
                                              (uint32_t *)keys_sorted.p, (int32_t *)vals,
                                              (int32_t *)vals_sorted.p, (int)n, 0, end_bit,
                                              stream));
    TN_HIP(hipMalloc(&sort_tmp.p, sort_bytes));
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(sort_tmp.p, sort_bytes, (uint32_t *)keys,
                                              (uint32_t *)keys_sorted.p, (int32_t *)vals,
                                              (int32_t *)vals_sorted.p, (int)n, 0, end_bit,
                                              stream));
    hipLaunchKernelGGL(bin_offsets_kernel, dim3(grid_blocks(n + 1)), dim3(kBlock), 0, stream,
                       (const uint32_t *)keys_sorted.p, n, nbins, bin_off);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMalloc(entries, sizeof(float4) * std::max<int64_t>(n, 1)));
    hipLaunchKernelGGL(bin_gather_kernel, dim3(grid_blocks(n)), dim3(kBlock), 0, stream, geo,
                       coord, (const uint32_t *)keys_sorted.p, (const int32_t *)vals_sorted.p, n,
                       *entries);
    TN_HIP(hipGetLastError());
    if (order != kOrderSample) {
        int rc = order_by_origin(geo, (const uint32_t *)keys_sorted.p, n, *entries, order == kOrderSpread,
                                 stream);
        if (rc) return rc;
    }
    TN_HIP(hipStreamSynchronize(stream));  // temporaries are freed on scope exit
    return TN_OK;
}

int order_by_origin(const BinGeom &geo, const uint32_t *bin_keys, int64_t n, float4 *entries,
                    bool spread, hipStream_t stream) {
    DevBuf k1, v1, k1s, v1s, head, start, k2, v2s, tmp, copy;
    TN_HIP(hipMalloc(&k1.p, sizeof(uint64_t) * n));
    TN_HIP(hipMalloc(&v1.p, sizeof(int32_t) * n));
    TN_HIP(hipMalloc(&k1s.p, sizeof(uint64_t) * n));
    TN_HIP(hipMalloc(&v1s.p, sizeof(int32_t) * n));
    TN_HIP(hipMalloc(&head.p, sizeof(int32_t) * n));
    TN_HIP(hipMalloc(&start.p, sizeof(int32_t) * n));
    TN_HIP(hipMalloc(&k2.p, sizeof(uint64_t) * n));
    TN_HIP(hipMalloc(&v2s.p, sizeof(int32_t) * n));
    TN_HIP(hipMalloc(&copy.p, sizeof(float4) * n));
    const unsigned nb = grid_blocks(n);
    hipLaunchKernelGGL(origin_key_kernel, dim3(nb), dim3(kBlock), 0, stream, geo, bin_keys, entries, n,
                       (uint64_t *)k1.p, (int32_t *)v1.p);
    TN_HIP(hipGetLastError());
    size_t bytes = 0, b2 = 0, b3 = 0;
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (uint64_t *)k1.p, (uint64_t *)k1s.p,
                                              (int32_t *)v1.p, (int32_t *)v1s.p, (int)n, 0, 64, stream));
    TN_HIP(hipcub::DeviceScan::InclusiveScan(nullptr, b2, (int32_t *)head.p, (int32_t *)start.p, MaxOp(),
                                             (int)n, stream));
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, b3, (uint64_t *)k2.p, (uint64_t *)k1s.p,
                                              (int32_t *)v1s.p, (int32_t *)v2s.p, (int)n, 0, 64, stream));
    TN_HIP(hipMalloc(&tmp.p, std::max(bytes, std::max(b2, b3))));
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, (uint64_t *)k1.p, (uint64_t *)k1s.p,
                                              (int32_t *)v1.p, (int32_t *)v1s.p, (int)n, 0, 64, stream));
    if (!spread) {  // (bin, origin, sample) order
        TN_HIP(hipMemcpyAsync(copy.p, entries, sizeof(float4) * n, hipMemcpyDeviceToDevice, stream));
        hipLaunchKernelGGL(permute_entries_kernel, dim3(nb), dim3(kBlock), 0, stream, (const float4 *)copy.p,
                           (const int32_t *)v1s.p, n, entries);
        TN_HIP(hipGetLastError());
        TN_HIP(hipStreamSynchronize(stream));
        return TN_OK;
    }
    hipLaunchKernelGGL(group_head_kernel, dim3(nb), dim3(kBlock), 0, stream, (const uint64_t *)k1s.p, n,
                       (int32_t *)head.p);
    TN_HIP(hipGetLastError());
    TN_HIP(hipcub::DeviceScan::InclusiveScan(tmp.p, b2, (int32_t *)head.p, (int32_t *)start.p, MaxOp(),
                                             (int)n, stream));
    hipLaunchKernelGGL(rank_key_kernel, dim3(nb), dim3(kBlock), 0, stream, (const uint64_t *)k1s.p,
                       (const int32_t *)start.p, n, (uint64_t *)k2.p);
    TN_HIP(hipGetLastError());
    // stable: equal (bin, rank) keep the (bin, origin, sample) order
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, b3, (uint64_t *)k2.p, (uint64_t *)k1s.p,
                                              (int32_t *)v1s.p, (int32_t *)v2s.p, (int)n, 0, 64, stream));
    TN_HIP(hipMemcpyAsync(copy.p, entries, sizeof(float4) * n, hipMemcpyDeviceToDevice, stream));
    hipLaunchKernelGGL(permute_entries_kernel, dim3(nb), dim3(kBlock), 0, stream, (const float4 *)copy.p,
                       (const int32_t *)v2s.p, n, entries);
    TN_HIP(hipGetLastError());
    TN_HIP(hipStreamSynchronize(stream));
    return TN_OK;
}

// Tile entries of all samples. Exact (a pass over the samples) only where their
// largest possible number passes the 32 bits of the offsets, else that number.
int entry_total(const BinGeom &geo, const float *coord, bool pieces, hipStream_t stream, int64_t &n) {
    const uint64_t total = (uint64_t)geo.npts * (uint64_t)geo.nframes;
    uint64_t most = total;
    for (int d = 0; d < geo.ndim; ++d) most *= most_pieces(geo.ax[d].W, geo.ax[d].T);
    n = (int64_t)most;
    if (most < (uint64_t)INT32_MAX) return TN_OK;
    DevBuf sum;
    unsigned long long exact = 0;
    TN_HIP(hipMalloc(&sum.p, sizeof(exact)));
    TN_HIP(hipMemsetAsync(sum.p, 0, sizeof(exact), stream));
    hipLaunchKernelGGL(pieces ? entry_total_kernel<true> : entry_total_kernel<false>,
                       dim3(std::min(grid_blocks((int64_t)total), 2048u)), dim3(kBlock), 0, stream, geo, coord,
                       (unsigned long long *)sum.p);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(&exact, sum.p, sizeof(exact), hipMemcpyDeviceToHost, stream));
    TN_HIP(hipStreamSynchronize(stream));
    n = (int64_t)exact;
    return TN_OK;
}

// Entries (sorted by (frame, tile), each tile's samples ascending: the sums'
// fixed order) and tap records of the tile gridding, for plans of fewer than
// 2^31 - 1 entries (tile_entries).
int build_tiles(tn_plan *plan, const BinGeom &geo, int64_t nbins, hipStream_t stream) {
    const int64_t total = geo.npts * geo.nframes;
    DevBuf counts, offsets, tmp;
    TN_HIP(hipMalloc(&counts.p, sizeof(int32_t) * total));
    TN_HIP(hipMalloc(&offsets.p, sizeof(int32_t) * total));
    hipLaunchKernelGGL(tiles_count_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream, geo, plan->d_coord,
                       (int32_t *)counts.p);
    TN_HIP(hipGetLastError());
    size_t scan_bytes = 0, sort_bytes = 0;
    TN_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (int32_t *)counts.p, (int32_t *)offsets.p, (int)total,
                                            stream));
    TN_HIP(hipMalloc(&tmp.p, scan_bytes));
    TN_HIP(hipcub::DeviceScan::ExclusiveSum(tmp.p, scan_bytes, (int32_t *)counts.p, (int32_t *)offsets.p, (int)total,
                                            stream));
    int32_t last[2] = {0, 0};
    TN_HIP(hipMemcpyAsync(&last[0], (int32_t *)offsets.p + (total - 1), sizeof(int32_t), hipMemcpyDeviceToHost, stream));
    TN_HIP(hipMemcpyAsync(&last[1], (int32_t *)counts.p + (total - 1), sizeof(int32_t), hipMemcpyDeviceToHost, stream));
    TN_HIP(hipStreamSynchronize(stream));
    const int64_t n = (int64_t)last[0] + last[1];
    plan->nentries = n;
    int end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) < (uint64_t)nbins) ++end_bit;
    DevBuf keys, vals, keys_sorted, sort_tmp;
    TN_HIP(hipMalloc(&keys.p, sizeof(uint32_t) * n));
    TN_HIP(hipMalloc(&vals.p, sizeof(uint64_t) * n));
    TN_HIP(hipMalloc(&keys_sorted.p, sizeof(uint32_t) * n));
    TN_HIP(hipMalloc(&plan->d_tent, sizeof(int2) * n));
    hipLaunchKernelGGL(tiles_emit_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream, geo, plan->d_coord,
                       (const int32_t *)offsets.p, (uint32_t *)keys.p, (uint64_t *)vals.p);
    TN_HIP(hipGetLastError());
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (uint32_t *)keys.p, (uint32_t *)keys_sorted.p,
                                              (uint64_t *)vals.p, (uint64_t *)plan->d_tent, (int)n, 0, end_bit, stream));
    TN_HIP(hipMalloc(&sort_tmp.p, sort_bytes));
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(sort_tmp.p, sort_bytes, (uint32_t *)keys.p, (uint32_t *)keys_sorted.p,
                                              (uint64_t *)vals.p, (uint64_t *)plan->d_tent, (int)n, 0, end_bit, stream));
    hipLaunchKernelGGL(bin_offsets_kernel, dim3(grid_blocks(n + 1)), dim3(kBlock), 0, stream,
                       (const uint32_t *)keys_sorted.p, n, nbins, plan->d_bin_off);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMalloc(&plan->d_taps, sizeof(float) * tiles_tap_stride(geo.ndim, plan->wpad) * total));
    hipLaunchKernelGGL(plan->wpad == 4 ? tiles_taps_kernel<4> : tiles_taps_kernel<8>, dim3(grid_blocks(total)),
                       dim3(kBlock), 0, stream, geo, plan->d_coord, plan->d_taps);
    TN_HIP(hipGetLastError());
    TN_HIP(hipMemcpyAsync(plan->h_bin_off.data(), plan->d_bin_off, sizeof(int32_t) * (nbins + 1), hipMemcpyDeviceToHost,
                          stream));
    TN_HIP(hipStreamSynchronize(stream));  // temporaries are freed on scope exit
    return TN_OK;
}

}  // namespace

// The automatic mode grids through the tiles where the kernel has at most
// kTilesMaxWidth taps per axis and the entries (8 bytes each, at most the
// product of the pieces a footprint can have) and tap records fit the budget
// and 32-bit offsets.
bool tiles_serve(const tn_plan_params &p) {
    uint64_t pieces = 1;
    int wmax = 1;
    for (int d = 3 - p.ndim; d < 3; ++d) {
        const int T = tiles_dim(p.ndim, 2 - d);
        wmax = std::max(wmax, p.width[d]);
        pieces *= most_pieces(p.width[d], T);
    }
    const uint64_t total = (uint64_t)p.nframes * (uint64_t)p.npts;
    uint64_t tiles = p.nframes;
    for (int d = 0; d < 3; ++d) {
        const int T = tiles_dim(p.ndim, 2 - d);
        tiles *= (p.grid[d] + T - 1) / T;
    }
    return wmax <= kTilesMaxWidth && total * pieces < (uint64_t)INT32_MAX && tiles < (uint64_t)INT32_MAX / 2 &&
           total * 4 * tiles_tap_stride(p.ndim, tiles_pad(wmax)) + total * pieces * 8 <= 4 * kMatrixAutoBytes;
}

int tile_entries(const tn_plan *plan, hipStream_t stream, int64_t &n) {
    return entry_total(make_geom(plan), plan->d_coord, true, stream, n);
}

int build_bins(tn_plan *plan, hipStream_t stream) {
    const BinGeom geo = make_geom(plan);
    const BinGeom pgeo = make_geom(plan, true);
    const int64_t total = geo.npts * geo.nframes;
    const int64_t nbins = geo.nframes * geo.ntiles;
    const int64_t npbins = pgeo.nframes * pgeo.ntiles;
    if (nbins >= (int64_t)UINT32_MAX || npbins >= (int64_t)UINT32_MAX)
        return fail(TN_E_RANGE, "too many tiles (%lld)", (long long)std::max(nbins, npbins));

    TN_HIP(hipMalloc(&plan->d_bin_off, sizeof(int32_t) * (nbins + 1)));
    TN_HIP(hipMalloc(&plan->d_pbin_off, sizeof(int32_t) * (npbins + 1)));
    plan->h_pbin_off.assign(npbins + 1, 0);
    plan->h_bin_off.assign(nbins + 1, 0);
    if (total == 0) {
        TN_HIP(hipMemsetAsync(plan->d_bin_off, 0, sizeof(int32_t) * (nbins + 1), stream));
        TN_HIP(hipMemsetAsync(plan->d_pbin_off, 0, sizeof(int32_t) * (npbins + 1), stream));
        TN_HIP(hipStreamSynchronize(stream));
        plan->nentries = 0;
        // an empty gridding matrix: all-zero row offsets, so every cell is
        // written as zero
        if (plan->grid_mode == kGridMatrix) return build_matrix(plan, stream);
        return TN_OK;
    }

    // ---- gridding bins: every tile a footprint touches --------------------
    if (plan->grid_mode == kGridTiles) {
        int rc = build_tiles(plan, geo, nbins, stream);
        if (rc) return rc;
        if (plan->p.ndim == 3) {
            const int64_t nrows = nbins / geo.NT[0];
            TN_HIP(hipMalloc(&plan->d_rows, sizeof(int2) * nrows));
            hipLaunchKernelGGL(tiles_rows_kernel, dim3((unsigned)((nrows + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                               geo, plan->d_bin_off, nrows, plan->d_rows);
            TN_HIP(hipGetLastError());
        }
    } else if (plan->grid_mode == kGridMatrix) {  // gridding reads the matrix instead
        TN_HIP(hipMemsetAsync(plan->d_bin_off, 0, sizeof(int32_t) * (nbins + 1), stream));
        plan->nentries = 0;
        int rc = build_matrix(plan, stream);
        if (rc) return rc;
    } else {
        int64_t n = 0;
        int rc = entry_total(geo, plan->d_coord, false, stream, n);
        if (rc) return rc;
        if (n >= INT32_MAX) return fail(TN_E_RANGE, "too many tile entries (%lld)", (long long)n);
        DevBuf counts, offsets, scan_tmp;
        TN_HIP(hipMalloc(&counts.p, sizeof(int32_t) * total));
        TN_HIP(hipMalloc(&offsets.p, sizeof(int32_t) * (total + 1)));
        hipLaunchKernelGGL(bin_count_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream, geo,
                           plan->d_coord, (int32_t *)counts.p);
        TN_HIP(hipGetLastError());
        size_t tmp_bytes = 0;
        TN_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, (int32_t *)counts.p,
                                                (int32_t *)offsets.p, (int)total, stream));
        TN_HIP(hipMalloc(&scan_tmp.p, tmp_bytes));
        TN_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.p, tmp_bytes, (int32_t *)counts.p,
                                                (int32_t *)offsets.p, (int)total, stream));
        int32_t last_off = 0, last_cnt = 0;
        TN_HIP(hipMemcpyAsync(&last_off, (int32_t *)offsets.p + (total - 1), sizeof(int32_t),
                              hipMemcpyDeviceToHost, stream));
        TN_HIP(hipMemcpyAsync(&last_cnt, (int32_t *)counts.p + (total - 1), sizeof(int32_t),
                              hipMemcpyDeviceToHost, stream));
        TN_HIP(hipStreamSynchronize(stream));
        n = (int64_t)last_off + last_cnt;
        plan->nentries = n;
        DevBuf keys, vals;
        TN_HIP(hipMalloc(&keys.p, sizeof(uint32_t) * n));
        TN_HIP(hipMalloc(&vals.p, sizeof(int32_t) * n));
        hipLaunchKernelGGL(bin_emit_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream, geo,
                           plan->d_coord, (const int32_t *)offsets.p, (uint32_t *)keys.p,
                           (int32_t *)vals.p);
        TN_HIP(hipGetLastError());
        rc = sort_entries(geo, plan->d_coord, keys.p, vals.p, n, plan->d_bin_off, &plan->d_entries, stream,
                          plan->grid_mode == kGridRuns ? kOrderOrigin : kOrderSpread);
        if (rc) return rc;
        plan->h_bin_off.assign(nbins + 1, 0);
        TN_HIP(hipMemcpyAsync(plan->h_bin_off.data(), plan->d_bin_off, sizeof(int32_t) * (nbins + 1),
                              hipMemcpyDeviceToHost, stream));
        TN_HIP(hipStreamSynchronize(stream));
    }
    // ---- interpolation bins: every sample once -----------------------------
    {
        DevBuf keys, vals;
        TN_HIP(hipMalloc(&keys.p, sizeof(uint32_t) * total));
        TN_HIP(hipMalloc(&vals.p, sizeof(int32_t) * total));
        hipLaunchKernelGGL(bin_primary_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream,
                           pgeo, plan->d_coord, (uint32_t *)keys.p, (int32_t *)vals.p);
        TN_HIP(hipGetLastError());
        // 3D: footprint-origin order inside each tile, so that the lanes of
        // a wave read neighbouring cells of the staged region (fewer LDS bank
        // conflicts; every sample's sum is the same whichever lane forms it);
        // 2D measures the same either way and keeps sample order
        int rc = sort_entries(pgeo, plan->d_coord, keys.p, vals.p, total, plan->d_pbin_off,
                              &plan->d_pentries, stream, pgeo.ndim == 3 ? kOrderOrigin : kOrderSample);
        if (rc) return rc;
        TN_HIP(hipMemcpyAsync(plan->h_pbin_off.data(), plan->d_pbin_off, sizeof(int32_t) * (npbins + 1),
                              hipMemcpyDeviceToHost, stream));
        TN_HIP(hipStreamSynchronize(stream));
    }
    return TN_OK;
}

// Sparse gridding matrix of every frame, CSR by output cell: the entries of
// every sample are sorted by (frame, cell) with a stable radix sort, so the
// samples of one cell stay in ascending order (a fixed summation order).
int build_matrix(tn_plan *plan, hipStream_t stream) {
    const BinGeom geo = make_geom(plan);
    const int64_t total = geo.npts * geo.nframes;
    const int64_t ncell = (int64_t)plan->p.grid[0] * plan->p.grid[1] * plan->p.grid[2];
    const int64_t nrows = ncell * geo.nframes;
    const int taps = plan->p.width[0] * plan->p.width[1] * plan->p.width[2];
    const int64_t n = total * taps;
    if (nrows >= (int64_t)UINT32_MAX) return fail(TN_E_RANGE, "gridding matrix: too many rows (%lld)", (long long)nrows);
    if (n >= INT32_MAX) return fail(TN_E_RANGE, "gridding matrix: too many entries (%lld)", (long long)n);
    if (geo.npts > ((int64_t)1 << 28)) return fail(TN_E_RANGE, "gridding matrix: too many samples per frame");
    TN_HIP(hipMalloc(&plan->d_mrow, sizeof(int32_t) * (nrows + 1)));
    TN_HIP(hipMalloc(&plan->d_mnz, sizeof(int2) * std::max<int64_t>(n, 1)));
    plan->mnnz = n;
    if (n == 0) {
        TN_HIP(hipMemsetAsync(plan->d_mrow, 0, sizeof(int32_t) * (nrows + 1), stream));
        TN_HIP(hipStreamSynchronize(stream));
        plan->h_mrow.assign(nrows + 1, 0);
        return TN_OK;
    }
    DevBuf keys, vals, keys_sorted, tmp;
    TN_HIP(hipMalloc(&keys.p, sizeof(uint32_t) * n));
    TN_HIP(hipMalloc(&vals.p, sizeof(uint64_t) * n));
    TN_HIP(hipMalloc(&keys_sorted.p, sizeof(uint32_t) * n));
    hipLaunchKernelGGL(matrix_emit_kernel, dim3(grid_blocks(total)), dim3(kBlock), 0, stream, geo, plan->d_coord,
                       taps, (uint32_t *)keys.p, (uint64_t *)vals.p);
    TN_HIP(hipGetLastError());
    int end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) < (uint64_t)nrows) ++end_bit;
    size_t bytes = 0;
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (uint32_t *)keys.p, (uint32_t *)keys_sorted.p,
                                              (uint64_t *)vals.p, (uint64_t *)plan->d_mnz, (int)n, 0, end_bit,
                                              stream));
    TN_HIP(hipMalloc(&tmp.p, bytes));
    TN_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, (uint32_t *)keys.p, (uint32_t *)keys_sorted.p,
                                              (uint64_t *)vals.p, (uint64_t *)plan->d_mnz, (int)n, 0, end_bit,
                                              stream));
    hipLaunchKernelGGL(bin_offsets_kernel, dim3(grid_blocks(n + 1)), dim3(kBlock), 0, stream,
                       (const uint32_t *)keys_sorted.p, n, nrows, plan->d_mrow);
    TN_HIP(hipGetLastError());
    plan->h_mrow.resize(nrows + 1);
    TN_HIP(hipMemcpyAsync(plan->h_mrow.data(), plan->d_mrow, sizeof(int32_t) * (nrows + 1), hipMemcpyDeviceToHost,
                          stream));
    TN_HIP(hipStreamSynchronize(stream));  // temporaries are freed on scope exit
    return TN_OK;
}

int count_footprint(tn_plan *plan, hipStream_t stream) {
    const BinGeom geo = make_geom(plan);
    const int64_t gvol = (int64_t)plan->p.grid[0] * plan->p.grid[1] * plan->p.grid[2];
    DevBuf mask, counter;
    TN_HIP(hipMalloc(&mask.p, gvol));
    TN_HIP(hipMalloc(&counter.p, sizeof(unsigned long long)));
    TN_HIP(hipMemsetAsync(counter.p, 0, sizeof(unsigned long long), stream));
    for (int f = 0; f < geo.nframes; ++f) {
        TN_HIP(hipMemsetAsync(mask.p, 0, gvol, stream));
        hipLaunchKernelGGL(footprint_mark_kernel, dim3(grid_blocks(geo.npts)), dim3(kBlock), 0,
                           stream, geo, plan->d_coord + (int64_t)f * geo.npts * geo.ndim,
                           (uint8_t *)mask.p);
        TN_HIP(hipGetLastError());
        hipLaunchKernelGGL(count_mask_kernel, dim3(grid_blocks(gvol)), dim3(kBlock), 0, stream,
                           (const uint8_t *)mask.p, gvol, (unsigned long long *)counter.p);
        TN_HIP(hipGetLastError());
    }
    unsigned long long cells = 0;
    TN_HIP(hipMemcpyAsync(&cells, counter.p, sizeof(cells), hipMemcpyDeviceToHost, stream));
    TN_HIP(hipStreamSynchronize(stream));
    plan->footprint = (int64_t)cells;
    return TN_OK;
}

}  // namespace tn
