// Tile gridding on the matrix cores (samples -> grid) for gfx950.
//
// One wave owns one item: a gridding tile (4x4x4 cells in 3D, 8x8 in 2D) of
// one frame, up to NC blocks of 8 coils, and a range of the tile's entries
// (the samples whose footprints meet it, ascending). Entry by entry the tile
// receives weight(cell) * value(coil): over four entries that is the product
// of a (coil values x 4) and a (4 x cells) matrix, so the sums are formed by
// v_mfma_f32_16x16x4_f32 -- 16 rows are the real and imaginary parts of 8
// coils, 16 columns a 4x4 patch of cells, and the tile is four such patches
// (the z planes in 3D, the quadrants in 2D). The instruction adds the four
// products in ascending order, each with one rounding (measured: bitwise a
// chain of fused multiply-adds), and taps outside the footprint enter with
// weight zero, so a cell's sum is the one a loop over its samples in
// ascending order gives.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tn_internal.h"
#include "tn_kb.h"

namespace tn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(8))) Pair2 {  // two complex values, 8-byte aligned
    float v[4];
};

// Coil-minor copy of the samples: coils it.e1 .. of record p of chunk it.e0
// receive coils c0 .. c1 - 1 of sample p, scaled by inv_scale and the density
// weight, and zeros up to the record's end or the item's eight coils. One
// workgroup takes kBlock samples: coalesced reads along each coil, then one
// 64-byte piece of a record per eight lanes.
__global__ __launch_bounds__(kBlock) void tiles_copy_kernel(const Job *__restrict__ jobs,
                                                            const Item *__restrict__ items,
                                                            const float2 *__restrict__ samp,
                                                            const float *__restrict__ weight,
                                                            float2 *__restrict__ st, int rec) {
    __shared__ float2 tile[kBlock * (kTilesCopyCoils + 1)];
    const Item it = items[blockIdx.x];
    const Job &J = jobs[it.job];
    const int t = threadIdx.x, nc = it.c1 - it.c0, nw = min(kTilesCopyCoils, rec - it.e1);
    const int64_t p0 = (int64_t)it.unit * kBlock, p = p0 + t, npts = J.npts;
    if (p < npts) {
        float sc = J.inv_scale;
        if (weight != nullptr && J.w_off >= 0) sc *= weight[J.w_off + p];
        const float2 *s = samp + J.samp_off + (int64_t)it.c0 * J.samp_bstride + p;
        const int64_t bs = J.samp_bstride;
        float2 a[kTilesCopyCoils];
#pragma unroll
        for (int j = 0; j < kTilesCopyCoils; ++j)
            if (j < nc) a[j] = s[j * bs];
#pragma unroll
        for (int j = 0; j < kTilesCopyCoils; ++j)
            if (j < nw)
                tile[t * (kTilesCopyCoils + 1) + j] =
                    j < nc ? make_float2(a[j].x * sc, a[j].y * sc) : make_float2(0.0f, 0.0f);
    }
    __syncthreads();
    float2 *dst = st + J.st_off + ((int64_t)it.e0 * npts + p0) * rec + it.e1;
    const int np = (int)min((int64_t)kBlock, npts - p0);
    int lcw = 0;  // lanes per record: the coils rounded up to a power of two
    while (1 << lcw < nw) ++lcw;
    const int j = t & ((1 << lcw) - 1);
    if (j < nw)
        for (int r = t >> lcw; r < np; r += kBlock >> lcw)
            dst[(int64_t)r * rec + j] = tile[r * (kTilesCopyCoils + 1) + j];
}

// Where an item's sample values come from: the samples themselves, their
// coil-minor copy, or the samples times the basis (low rank: accumulator coils
// are (coil, coefficient) pairs).
enum TileFrom { kInPlace = 0, kCopy = 1, kLowRank = 2 };
struct TileSrc {
    const float2 *samp;
    const float *weight;
    const float2 *st;
    int rec;  // coils per record of the copy (even)
    LowRank lr;
    uint32_t div_mul;  // s / lr.frame_npts = (umulhi(div_mul, s) + s) >> div_shift
    int32_t div_shift;
    bool ranged;  // cells outside the row ranges need not be written
};

// Taps d .. d + 3 of an axis, zeros outside [0, WP): a barrel shift of the taps
// between zeros.
template <int WP>
__device__ __forceinline__ float4 tap_window(const float (&t)[WP], int d) {
    const int s = min(max(d, -4), WP) + 4;
    float a[WP + 8];
#pragma unroll
    for (int j = 0; j < WP + 8; ++j) a[j] = j >= 4 && j < WP + 4 ? t[j - 4] : 0.0f;
#pragma unroll
    for (int sh = 8; sh > 0; sh >>= 1) {
        const bool on = (s & sh) != 0;
#pragma unroll
        for (int j = 0; j < WP + 8; ++j)
            if (j < 3 + sh) a[j] = on ? (j + sh < WP + 8 ? a[j + sh] : 0.0f) : a[j];
    }
    return make_float4(a[0], a[1], a[2], a[3]);
}

// Orders this wave's LDS traffic for the compiler: lanes read words that other
// lanes of the wave stored, and store words that others have read, which the
// hardware keeps in program order but a lane's own addresses do not show. No
// instruction.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Zeros for a run of it.e1 tiles without entries, in rows of up to
// kTilesFillCells cells, two per lane and two rows per store (ranged: where
// the transform reads). A tile by itself is stored in 32-byte pieces, which
// the memory takes at 1.7 TB/s once the grids pass the caches: 500 spokes x
// 256 samples, 8 coils of 256^3, 73% of the tiles empty: 650 us, 447 in runs
// (the gridding matrix 488); their first adjoint, which builds the work list,
// 8.0 -> 4.7 ms.
template <int NDIM>
__device__ __forceinline__ void fill_tiles(const Job &J, const Item &it, bool ranged, float2 *__restrict__ grid,
                                           int lane) {
    constexpr int TX = tiles_dim(NDIM, 0), TY = tiles_dim(NDIM, 1), TZ = tiles_dim(NDIM, 2);
    constexpr int PAIRS = kTilesFillCells / 2;
    const int Gx = J.G[0], Gy = J.G[1], Gz = J.G[2], row = it.unit / J.NT[0];
    const int x0 = it.unit % J.NT[0] * TX, y0 = row % J.NT[1] * TY, z0 = row / J.NT[1] * TZ;
    const int x = x0 + 2 * (lane % PAIRS), end = min(x0 + it.e1 * TX, Gx);
    bool read = x < end;
    if (ranged) {
        const int2 range = J.rows[row];
        const int a = signed_x(x, Gx), b = signed_x(x + 1, Gx);
        read = read && ((a >= range.x && a < range.y) || (x + 1 < end && b >= range.x && b < range.y));
        if (!__any(read)) return;
    }
    const Pair2 zeros = {{0.0f, 0.0f, 0.0f, 0.0f}};
    const int rows = (it.c1 - it.c0) * TY * TZ;
    float2 *const g = grid + J.grid_off + it.c0 * J.grid_bstride + x;
#pragma unroll 4
    for (int r = lane / PAIRS; r < rows; r += kWave / PAIRS) {
        const int y = y0 + r % TY, z = z0 + r / TY % TZ;
        if (!read || y >= Gy || z >= Gz) continue;
        float2 *p = g + r / (TY * TZ) * J.grid_bstride + ((int64_t)z * Gy + y) * Gx;
        if (x + 1 < end)
            *(Pair2 *)p = zeros;
        else
            *p = make_float2(0.0f, 0.0f);
    }
}

// Tile gridding. The entries are taken sixteen at a time. Loading: four lanes
// per entry, lane r taking 16 bytes of its tap record and of its sample record
// (one load instruction for the sixteen entries each), turning the taps into
// the weights of the tile's cells along one axis (3D: axis r, four cells; 2D:
// axis r / 2, half r & 1 of the eight cells) and storing both in the wave's
// LDS. Summing: the matrix core's operands are read from there, lane (k, i)
// holding word i of the coil values and the weight of cell i for entry k of a
// group of four. The next sixteen entries' records are in flight meanwhile;
// a wave uses only its own part of the LDS, whose operations complete in
// order, so there are no barriers.
//
// What bounds it. 3D (kooshball 128^3, 8 coils, osf 2: 27 M entries): issue; the
// vector units work 53% of their cycles and the matrix cores 33%. Copy, kernel
// and fold take 0.12 + 1.19 + 0.02 ms with every cell written and 0.11 + 1.00 +
// 0.02 in the whole adjoint, against 3.37 ms for the gridding matrix, whose
// gathers of one record per tap were bound by their rate. 2D (8 x 16 spirals on
// 512^2): latency, 22% and 14% at 12 waves per CU; 0.032 + 0.121 + 0.009 ms
// against 0.028 + 0.147. The dense product spends most of its terms on zeros,
// hence small tiles, and the patches that none of a group's four entries reaches
// are left out (when that was added: 1.02 -> 0.94 ms in 3D, 52 -> 38 us in 2D).
// The patches are the outer loop: with the groups outside, the compiler copied
// every sum at every branch (1.8 ms). Each lane loading its
// own operands from memory took 2.4 ms: the texture addresser was busy 80% of
// the time, 18 cycles for each of 21 load instructions per sixteen entries.
template <int NDIM, int WP, int NC, int FROM>
__global__ __launch_bounds__(kBlock, NC <= 2 ? 4 : 2) void grid_tiles_kernel(
    const Job *__restrict__ jobs, const Item *__restrict__ items, int64_t nitems, TileSrc src,
    float2 *__restrict__ grid, float *__restrict__ scratch, const int64_t *__restrict__ slot_base) {
    constexpr int TX = tiles_dim(NDIM, 0), TY = tiles_dim(NDIM, 1), TZ = tiles_dim(NDIM, 2);
    constexpr int TS = tiles_tap_stride(NDIM, WP);
    constexpr int B = 16;  // entries per step
    // a wave's LDS: the weights [entry][axis][cell] and values [block][entry]
    // [coil part] of a step, and after the last one the sums of a block on
    // their way out, [coil][cell] with a pitch of CP cells
    constexpr int CP = TX * TY * TZ + 2;
    constexpr int words = B * 4 * (1 + NC) > 4 * CP ? B * 4 * (1 + NC) : 4 * CP;  // float4
    __shared__ float4 lds[kBlock / kWave][words];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t idx = (int64_t)blockIdx.x * (kBlock / kWave) + wave;
    if (idx >= nitems) return;
    const Item it = items[idx];
    if (it.job < 0) return;  // filler
    const Job &J = jobs[it.job];
    if (it.slot == kTilesFill) {
        fill_tiles<NDIM>(J, it, src.ranged, grid, threadIdx.x % kWave);
        return;
    }
    const int lane = threadIdx.x % kWave, k = lane >> 4, i = lane & 15, cx = i & 3, cy = i >> 2;
    const int nc = it.c1 - it.c0;
    float4 *const swt = lds[wave], *const sval = swt + B * 4;
    const int2 *const ent = J.tent;
    const float *const taps = J.taps;
    f32x4 acc[4][NC];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int n = 0; n < NC; ++n) acc[p][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // loading lane (j, r): 16 bytes (two coils) r of each block of entry j
    const int j = lane >> 2, r = lane & 3;
    const int axis = NDIM == 3 ? min(r, 2) : r >> 1, half = NDIM == 3 ? 0 : 4 * (r & 1);
    // coils past the item's last repeat it: their sums are not stored
    const float *const wt = FROM != kCopy && src.weight != nullptr && J.w_off >= 0 ? src.weight + J.w_off : nullptr;
    const float inv_scale = J.inv_scale;
    const float2 *const samp = src.samp + J.samp_off;
    const float2 *const st =
        FROM == kCopy ? src.st + J.st_off + (int64_t)(it.c0 / max(J.tchunk, 1)) * J.npts * src.rec : nullptr;
    uint32_t off[NC][2], coef[NC][2];  // in place: element offsets of the coil rows (below 2^29); basis rows
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = it.c0 + min(8 * n + 2 * r + h, nc - 1), b = FROM == kLowRank ? c / src.lr.ncoeff : c;
            off[n][h] = FROM == kInPlace ? (uint32_t)(b * J.samp_bstride) : b;
            coef[n][h] = FROM == kLowRank ? (uint32_t)((c - b * src.lr.ncoeff) * src.lr.nframes) : 0u;
        }
    auto values = [&](int s, float4 (&v)[NC]) {
        if (FROM == kCopy) {
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                const int c = 8 * n + 2 * r;
                v[n] = c < nc ? *(const float4 *)(st + (int64_t)s * src.rec + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            return;
        }
        float sc = inv_scale;
        if (wt != nullptr) sc *= wt[s];
        const uint32_t f = FROM == kLowRank ? (__umulhi(src.div_mul, (uint32_t)s) + (uint32_t)s) >> src.div_shift : 0u;
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            float2 a[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (FROM == kLowRank) {
                    const float2 x = samp[off[n][h] * J.samp_bstride + s], q = src.lr.coef[coef[n][h] + f];
                    a[h] = make_float2(q.x * x.x - q.y * x.y, q.x * x.y + q.y * x.x);
                } else {
                    a[h] = samp[off[n][h] + (uint32_t)s];
                }
            }
            v[n] = make_float4(a[0].x * sc, a[0].y * sc, a[1].x * sc, a[1].y * sc);
        }
    };
    auto axis_taps_of = [&](int s, float (&t)[WP]) {
        const float4 *p = (const float4 *)(taps + (int64_t)s * TS + axis * WP);
#pragma unroll
        for (int h = 0; h < WP / 4; ++h) {
            const float4 q = p[h];
            t[4 * h] = q.x;
            t[4 * h + 1] = q.y;
            t[4 * h + 2] = q.z;
            t[4 * h + 3] = q.w;
        }
    };
    const int elast = it.e1 - 1;
    bool odd = false;  // a value that is not finite: zero weights would spread it
    if (it.e0 < it.e1) {
        int2 en = ent[min(it.e0 + j, elast)], next = ent[min(it.e0 + B + j, elast)];
        float t[WP];
        float4 v[NC];
        axis_taps_of(en.x, t);
        values(en.x, v);
        for (int e = it.e0; e < it.e1; e += B) {
            const bool live = e + j < it.e1;
            float4 w = tap_window<WP>(t, half - (((en.y >> (8 * axis)) & 255) - 16));
            if (!live) w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (NDIM < 3 || r < 3) swt[4 * j + r] = w;
            // which patches each group of four entries reaches (16 bits of a
            // mask per group): the z planes, or the x and y halves, with a
            // weight other than zero
            uint64_t reach[4];
            if (NDIM == 3) {
                reach[0] = __ballot(r == 2 && w.x != 0.0f);
                reach[1] = __ballot(r == 2 && w.y != 0.0f);
                reach[2] = __ballot(r == 2 && w.z != 0.0f);
                reach[3] = __ballot(r == 2 && w.w != 0.0f);
            } else {
                const uint64_t any = __ballot(w.x != 0.0f || w.y != 0.0f || w.z != 0.0f || w.w != 0.0f);
#pragma unroll
                for (int p = 0; p < 4; ++p) reach[p] = (any >> (p & 1)) & (any >> (2 + (p >> 1))) & 0x1111111111111111ull;
            }
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                if (!live) v[n] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                odd |= !(__builtin_isfinite(v[n].x) && __builtin_isfinite(v[n].y) && __builtin_isfinite(v[n].z) &&
                         __builtin_isfinite(v[n].w));
                sval[n * B * 4 + 4 * j + r] = v[n];
            }
            wave_lds_order();  // the step's words stored
            en = next;
            if (e + B < it.e1) {  // the next sixteen
                axis_taps_of(en.x, t);
                values(en.x, v);
                next = ent[min(e + 2 * B + j, elast)];
            }
            // operands of the four groups: values, and what the weights are formed from
            float a[B / 4][NC], wx[B / 4][2], wy[B / 4][2], wz[B / 4][4];
#pragma unroll
            for (int u = 0; u < B / 4; ++u) {
                const float *ws = (const float *)(swt + 4 * (4 * u + k));
#pragma unroll
                for (int n = 0; n < NC; ++n) a[u][n] = ((const float *)(sval + n * B * 4 + 4 * (4 * u + k)))[i];
                wx[u][0] = ws[cx];
                if (NDIM == 3) {
                    wy[u][0] = ws[4 + cy];
                    const float4 z = *(const float4 *)(ws + 8);
                    wz[u][0] = z.x;
                    wz[u][1] = z.y;
                    wz[u][2] = z.z;
                    wz[u][3] = z.w;
                } else {
                    wx[u][1] = ws[4 + cx];
                    wy[u][0] = ws[8 + cy];
                    wy[u][1] = ws[12 + cy];
                }
            }
            wave_lds_order();  // and read
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int u = 0; u < B / 4; ++u) {
                    if (((reach[p] >> (16 * u)) & 0xffff) == 0) continue;  // adds nothing
                    // (wz wy) wx, as in the other variants
                    const float w = NDIM == 3 ? (wz[u][p] * wy[u][0]) * wx[u][0] : wy[u][p >> 1] * wx[u][p & 1];
#pragma unroll
                    for (int n = 0; n < NC; ++n)
                        acc[p][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][n], w, acc[p][n], 0, 0, 0);
                }
        }
    }
    if (__any(odd)) {  // again, each lane adding to its cells inside the footprints only
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int n = 0; n < NC; ++n) acc[p][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int e = it.e0; e < it.e1; ++e) {
            const int2 en = ent[e];
            const int lx = (en.y & 255) - 16, ly = ((en.y >> 8) & 255) - 16, lz = ((en.y >> 16) & 255) - 16;
            const float *t = taps + (int64_t)en.x * TS;
            float4 v[NC];
            values(en.x, v);
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                // coils 2 k and 2 k + 1 of the block, from the lane that loads them
                const float a[4] = {__shfl(v[n].x, k, kWave), __shfl(v[n].y, k, kWave), __shfl(v[n].z, k, kWave),
                                    __shfl(v[n].w, k, kWave)};
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int kx = (NDIM == 3 ? cx : cx + 4 * (p & 1)) - lx;
                    const int ky = (NDIM == 3 ? cy : cy + 4 * (p >> 1)) - ly, kz = p - lz;
                    if ((unsigned)kx < (unsigned)J.W[0] && (unsigned)ky < (unsigned)J.W[1] &&
                        (NDIM < 3 || (unsigned)kz < (unsigned)J.W[2])) {
                        const float w = NDIM == 3 ? (t[2 * WP + kz] * t[WP + ky]) * t[kx] : t[WP + ky] * t[kx];
#pragma unroll
                        for (int q = 0; q < 4; ++q) acc[p][n][q] += w * a[q];
                    }
                }
            }
        }
    }

    // lane (k, i) holds cell i of each patch for coils 2 k and 2 k + 1 of each
    // block; through the LDS the lanes store two cells of a row each (16 bytes;
    // straight from the lanes, in 32-byte pieces of 16 rows, the stores kept the
    // texture addresser busy for most of the 2D kernel's time)
    const int Gx = J.G[0], Gy = J.G[1], Gz = J.G[2];
    const int64_t bs = J.grid_bstride;
    const bool joined = (it.unit & kTilesJoin) != 0;  // the workgroup's waves share the tile
    const int tile = it.unit & ~kTilesJoin, NTx = J.NT[0], NTy = J.NT[1];
    const int x0 = (tile % NTx) * TX, y0 = ((tile / NTx) % NTy) * TY, z0 = tile / (NTx * NTy) * TZ;
    const bool inside = x0 + TX <= Gx && y0 + TY <= Gy && z0 + TZ <= Gz;
    const int64_t origin = J.grid_off + it.c0 * bs + ((int64_t)z0 * Gy + y0) * Gx + x0;
    float2 *const part =
        it.slot >= 0 ? (float2 *)(scratch + slot_base[it.slot]) + (int64_t)it.part * nc * (TX * TY * TZ) : nullptr;
    float2 *const out = (float2 *)lds[wave];
    constexpr int PAIRS = TX * TY * TZ / 2, CPI = kWave / PAIRS;  // cell pairs per coil, coils per store
    static_assert(8 / CPI == kBlock / kWave, "a joined workgroup's waves take one store of a block each");
    const int pair = lane % PAIRS, px = 2 * (pair % (TX / 2)), py = (pair / (TX / 2)) % TY, pz = pair / (TX / 2 * TY);
    const int64_t poff = ((int64_t)pz * Gy + py) * Gx + px;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        if (joined && n > 0)
            __syncthreads();  // the previous block's sums read
        else
            wave_lds_order();
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int x = NDIM == 3 ? cx : cx + 4 * (p & 1), y = NDIM == 3 ? cy : cy + 4 * (p >> 1);
            const int cell = ((NDIM == 3 ? p : 0) * TY + y) * TX + x;
            out[2 * k * CP + cell] = make_float2(acc[p][n][0], acc[p][n][1]);
            out[(2 * k + 1) * CP + cell] = make_float2(acc[p][n][2], acc[p][n][3]);
        }
        if (joined)
            __syncthreads();
        else
            wave_lds_order();
#pragma unroll
        for (int q = 0; q < 8 / CPI; ++q) {
            const int c = q * CPI + lane / PAIRS;
            if (8 * n + c >= nc || (joined && q != wave)) continue;
            const int at = c * CP + 2 * pair;
            float2 a, b;
            if (joined) {  // the waves' sums, added in pairs
                float2 u[kBlock / kWave][2];
#pragma unroll
                for (int g = 0; g < kBlock / kWave; ++g)
#pragma unroll
                    for (int h = 0; h < 2; ++h) u[g][h] = ((const float2 *)lds[g])[at + h];
                static_assert(kBlock / kWave == 4, "four waves");
                a = make_float2((u[0][0].x + u[1][0].x) + (u[2][0].x + u[3][0].x),
                                (u[0][0].y + u[1][0].y) + (u[2][0].y + u[3][0].y));
                b = make_float2((u[0][1].x + u[1][1].x) + (u[2][1].x + u[3][1].x),
                                (u[0][1].y + u[1][1].y) + (u[2][1].y + u[3][1].y));
            } else {
                a = out[at];
                b = out[at + 1];
            }
            const Pair2 v = {{a.x, a.y, b.x, b.y}};
            if (part != nullptr) {  // partial of a split tile, in fold_kernel's (coil, z, y, x) order
                *(Pair2 *)(part + (int64_t)(8 * n + c) * (TX * TY * TZ) + 2 * pair) = v;
            } else {
                float2 *g = grid + origin + (8 * n + c) * bs + poff;
                if (inside) {
                    *(Pair2 *)g = v;
                } else if (y0 + py < Gy && z0 + pz < Gz) {
                    if (x0 + px < Gx) g[0] = a;
                    if (x0 + px + 1 < Gx) g[1] = b;
                }
            }
        }
    }
}

using TilesFn = void (*)(const Job *, const Item *, int64_t, TileSrc, float2 *, float *, const int64_t *);

template <int NDIM, int WP, int FROM>
TilesFn pick_blocks(int blocks) {
    switch (blocks) {
        case 1: return grid_tiles_kernel<NDIM, WP, 1, FROM>;
        case 2: return grid_tiles_kernel<NDIM, WP, 2, FROM>;
        case 3: return grid_tiles_kernel<NDIM, WP, 3, FROM>;
        case 4: return grid_tiles_kernel<NDIM, WP, 4, FROM>;
        default: return nullptr;
    }
}

template <int FROM>
TilesFn pick_tiles(int ndim, int wpad, int blocks) {
    if (ndim == 2) return wpad == 4 ? pick_blocks<2, 4, FROM>(blocks) : pick_blocks<2, 8, FROM>(blocks);
    return wpad == 4 ? pick_blocks<3, 4, FROM>(blocks) : pick_blocks<3, 8, FROM>(blocks);
}

}  // namespace

int launch_tiles(const LaunchTables &t, const float2 *samp, float2 *grid, const float *weight, hipStream_t stream,
                 const LowRank &lr, float *scratch, bool ranged, float2 *st) {
    const int ndim = kind_ndim(t.kind_grid);
    const int blocks = (t.grid_coils + 7) / 8;
    if ((ndim != 2 && ndim != 3) || kind_width(t.kind_grid) > kTilesMaxWidth || blocks < 1 || blocks > kTilesBlocks)
        return fail(TN_E_ARG, "tile gridding: %dD, width %d, %d coils per item", ndim, kind_width(t.kind_grid),
                    t.grid_coils);
    if (st == nullptr) st = t.d_st;
    // without room for the copy the samples are read in place: the same bits,
    // where their offsets fit
    const bool copy = lr.ncoeff == 0 && t.st_cw > 0 && st != nullptr;
    if (lr.ncoeff == 0 && t.st_wide && !copy) return fail(TN_E_ARG, "tile gridding: no room for the sample copy");
    TileSrc src{samp, weight, st, t.st_cw, lr, 0u, 0, ranged};
    if (lr.ncoeff > 0) {
        // division of a sample index (< 2^31) by frame_npts: l = ceil(log2 d),
        // m = floor(2^32 (2^l - d) / d) + 1
        const uint64_t d = (uint64_t)lr.frame_npts;
        int l = 0;
        while (((uint64_t)1 << l) < d) ++l;
        src.div_mul = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - d)) / d + 1);
        src.div_shift = l;
    }
    if (copy) {
        hipLaunchKernelGGL(tiles_copy_kernel, dim3((unsigned)t.n_tr), dim3(kBlock), 0, stream, t.d_jobs, t.d_tr, samp,
                           weight, st, t.st_cw);
        TN_HIP(hipGetLastError());
    }
    const TilesFn fn = lr.ncoeff > 0 ? pick_tiles<kLowRank>(ndim, t.wpad, blocks)
                       : copy        ? pick_tiles<kCopy>(ndim, t.wpad, blocks)
                                     : pick_tiles<kInPlace>(ndim, t.wpad, blocks);
    const int64_t groups = (t.n_grid + kBlock / kWave - 1) / (kBlock / kWave);
    hipLaunchKernelGGL(fn, dim3((unsigned)groups), dim3(kBlock), 0, stream, t.d_jobs, t.d_grid, t.n_grid, src, grid,
                       scratch, t.d_slot_base);
    TN_HIP(hipGetLastError());
    return launch_fold(t, grid, scratch, stream);
}

}  // namespace tn
