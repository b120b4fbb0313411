// Oversampled-grid FFT stages of the 2D NUFFT for gfx950, pruned to the
// lines that carry data and fused with the zero padding, the apodization
// and the crop (src/deepmr/fft/nufft.py:499-505 forward: apodize, resize,
// fft with norm=None; :587-593 adjoint: ifft, resize, apodize).
//
// Index maps: image pixel m of an axis sits at grid index (m - N/2) mod G
// (the centring shifts folded into the placement, as in the other stages),
// so a grid line along y holds data only at the Ny rows with
// (y + Ny/2) mod Gy < Ny until the y transform has run, and likewise along x.
//
//   forward  columns: image columns -> apodize -> DFT along y -> grid columns
//                     (only the Nx columns that carry data)
//            rows:    DFT along x of every grid row, reading only its Nx
//                     data columns
//   adjoint  rows:    inverse DFT along x of every grid row, writing only
//                     the Nx columns the crop keeps
//            columns: inverse DFT along y of those columns, keeping the Ny
//                     image rows, scaled by 1 / (Gx Gy), apodized
//
// Each line transform is a mixed-radix Stockham FFT (fft_radix_at) run by
// one wave: the radix-R butterflies of a pass are evaluated in registers
// with twiddles from a table computed in double precision on the host, and
// the passes exchange data through that wave's LDS line. All reads of a pass
// are issued before its writes, and a wave's LDS operations complete in
// order, so a line is transformed in place without barriers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "tn_fft.h"
#include "tn_kb.h"

namespace tn {
namespace {

// Which cells of a grid row hold values: line -> frame, tile row -> signed x
// range (tn_plan::d_rows); r null: every cell. At most 2^31 lines.
struct RowRanges {
    const int2 *r = nullptr;
    int ny = 1, ty = 1, nty = 1, nz = 1, tz = 1, ntz = 1, frames = 1;
    bool d3 = false;  // rows of a 3D plan
};

// Row transforms along x, in place, rows_per_wave(L) grid rows (length
// L = Gx) per wave. Forward: reads only the Nx data columns (the others are
// zeros). Inverse: writes only the Nx columns the crop keeps. Bound by memory
// in 3D: with ranges, cells that no footprint reaches are not written
// (forward) or not read and taken as zeros (inverse), and rows without any are
// skipped. A kooshball leaves half of the grid (8 coils of 256^3, whole calls:
// forward 1.36 -> 1.29 ms, adjoint, whose gridding leaves them too, 1.88 -> 1.70).
// RANGES: the rows of 3D plans, whether they have ranges or not (one kernel, so
// that both give the same bits).
template <int L, bool INV, bool RANGES>
__global__ __launch_bounds__(kBlock) void fft_rows_kernel(float2 *__restrict__ data, int64_t nlines, int Nx,
                                                          const float2 *__restrict__ tw, RowRanges g) {
    constexpr int RL = rows_per_wave(L);
    __shared__ float2 lds[kBlock / kWave * RL][fft_line(L)];
    __shared__ int2 span[RANGES ? kBlock / kWave : 1][RL];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * RL;
    if (line0 >= nlines) return;  // no barriers below
    // a row past the last one reads the last and writes nothing
    auto row = [&](int l) { return data + min(line0 + l, nlines - 1) * L; };
    if constexpr (RANGES) {
        int2 s = make_int2(0, 0);
        if (lane < RL) {
            s = make_int2(-L, L);
            if (g.r != nullptr) {
                const int line = (int)min(line0 + lane, nlines - 1), plane = line / g.ny, image = plane / g.nz;
                const int y = line - plane * g.ny, z = plane - image * g.nz;
                s = g.r[((int64_t)(image % g.frames) * g.ntz + z / g.tz) * g.nty + y / g.ty];
            }
            span[wave][lane] = s;
        }
        if (__ballot(s.x < s.y) == 0) {
            if (INV)
                for (int l = 0; l < RL && line0 + l < nlines; ++l)
                    for (int i = lane; i < L; i += kWave)
                        if (kept(i, Nx, L)) row(l)[i] = make_float2(0.0f, 0.0f);
            return;
        }
        __asm__ __volatile__("" ::: "memory");  // one wave: its LDS operations complete in order
    }
    auto held = [&](int l, int i) {
        if (!RANGES) return true;
        const int2 s = span[wave][l];
        const int u = signed_x(i, L);
        return u >= s.x && u < s.y;
    };
    float2 *buf = lds[wave * RL];
    if (!INV) {
        fft_lines<L, RL, false>(
            lane, tw, buf, fft_line(L), [&](int l, int i) { return kept(i, Nx, L) ? row(l)[i] : make_float2(0.0f, 0.0f); },
            [&](int l, int i, float2 v) {
                if (line0 + l < nlines && held(l, i)) row(l)[i] = v;
            });
    } else {
        fft_lines<L, RL, true>(
            lane, tw, buf, fft_line(L), [&](int l, int i) { return held(l, i) ? row(l)[i] : make_float2(0.0f, 0.0f); },
            [&](int l, int i, float2 v) {
                if (line0 + l < nlines && kept(i, Nx, L)) row(l)[i] = v;
            });
    }
}

// A row's whole share of a convolution, in place on rows of the N data columns:
// padded to L, transformed, times the row's kernel values (rows repeat after
// nk), transformed back and cropped, without leaving the wave's LDS lines.
template <int L>
__global__ __launch_bounds__(kBlock) void fft_product_kernel(float2 *__restrict__ data, int64_t nlines, int N,
                                                             const float2 *__restrict__ kern, int64_t nk,
                                                             const float2 *__restrict__ tw) {
    constexpr int RL = rows_per_wave(L), pitch = fft_line(L);
    __shared__ float2 lds[kBlock / kWave * RL][pitch];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * RL;
    if (line0 >= nlines) return;  // no barriers below
    // a row past the last one reads the last and writes nothing
    auto line = [&](int l) { return min(line0 + l, nlines - 1); };
    auto pixel = [&](int i) { return i + N / 2 < L ? i + N / 2 : i + N / 2 - L; };  // < N: data
    const int64_t k0 = line0 % nk;
    auto krow = [&](int l) { return kern + (k0 + l < nk ? k0 + l : (line0 + l) % nk) * L; };
    float2 *buf = lds[wave * RL];
    fft_lines<L, RL, false>(
        lane, tw, buf, pitch,
        [&](int l, int i) {
            const int m = pixel(i);
            return m < N ? data[line(l) * N + m] : make_float2(0.0f, 0.0f);
        },
        [&](int l, int i, float2 v) { buf[l * pitch + lds_at<L>(i)] = v; });
    __asm__ __volatile__("" ::: "memory");  // other lanes' elements below: keep the reads behind the writes
    fft_lines<L, RL, true>(
        lane, tw, buf, pitch, [&](int l, int i) { return cmul(buf[l * pitch + lds_at<L>(i)], krow(l)[i]); },
        [&](int l, int i, float2 v) {
            const int m = pixel(i);
            if (m < N && line0 + l < nlines) data[(line0 + l) * N + m] = v;
        });
}

// Forward column stage: image columns mx0 .. mx0 + C - 1 of image b are
// apodized (x then y, as the separate pre-pass does), placed at their grid
// rows in LDS, transformed along y (length L = Gy; rows without data are
// zeros) and written to grid columns (mx - hx) mod Gx (hx = Nx/2 for the x
// axis of a grid; 0 where the columns are a flattened (y, x) plane that a
// later stage places).
template <int L, int C>
__global__ __launch_bounds__(kBlock) void fft_cols_fwd_kernel(const float2 *__restrict__ img,
                                                              float2 *__restrict__ grid, int64_t nimg, int Nx,
                                                              int Ny, int Gx, int hx, const float *__restrict__ apx,
                                                              const float *__restrict__ apy,
                                                              const float2 *__restrict__ tw) {
    constexpr int LP = fft_line(L) + fft_pad(C);
    extern __shared__ float2 lds[];  // C * LP
    int64_t b;
    int mx0;
    if (!column_block(nimg, Nx, C, b, mx0)) return;
    const int hy = Ny / 2;
    for (int i0 = threadIdx.x; i0 < Ny * C; i0 += kLoadBatch * kBlock) {  // loads first, then the LDS writes
        float2 v[kLoadBatch];
        float ax[kLoadBatch], ay[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int my = i / C, mx = mx0 + i % C;
            v[u] = make_float2(0.0f, 0.0f);
            ax[u] = ay[u] = 1.0f;
            if (i < Ny * C && mx < Nx) {
                v[u] = img[(b * Ny + my) * (int64_t)Nx + mx];
                if (apx) ax[u] = apx[mx];
                if (apy) ay[u] = apy[my];
            }
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            if (i >= Ny * C) continue;
            const int my = i / C, c = i % C;
            const float2 w = cscale(cscale(v[u], ax[u]), ay[u]);  // x then y, as the separate pre-pass
            int y = my - hy;
            if (y < 0) y += L;
            lds[c * LP + y] = w;
        }
    }
    __syncthreads();
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    {   // wave w transforms columns w, w + 4, ... together
        constexpr int NL = C / (kBlock / kWave);
        constexpr int pitch = kBlock / kWave * LP;
        float2 *col = lds + wave * LP;
        fft_lines<L, NL, false>(
            lane, tw, col, pitch, [&](int l, int i) { return kept(i, Ny, L) ? col[l * pitch + i] : make_float2(0.0f, 0.0f); },
            [&](int l, int i, float2 v) { col[l * pitch + i] = v; });
    }
    __syncthreads();
    for (int i = threadIdx.x; i < L * C; i += kBlock) {
        const int y = i / C, c = i % C;
        const int mx = mx0 + c;
        if (mx < Nx) {
            int x = mx - hx;
            if (x < 0) x += Gx;
            grid[(b * L + y) * (int64_t)Gx + x] = lds[c * LP + y];
        }
    }
}

// Adjoint column stage: grid columns (mx - hx) mod Gx for image columns
// mx0 .. mx0 + C - 1, inverse-transformed along y (L = Gy); the Ny image rows
// are scaled by 1 / (Gx Gy), apodized (x then y) and written to the image.
template <int L, int C>
__global__ __launch_bounds__(kBlock) void fft_cols_inv_kernel(const float2 *__restrict__ grid,
                                                              float2 *__restrict__ img, int64_t nimg, int Nx,
                                                              int Ny, int Gx, int hx, const float *__restrict__ apx,
                                                              const float *__restrict__ apy,
                                                              const float2 *__restrict__ tw, float scale) {
    constexpr int LP = fft_line(L) + fft_pad(C);
    extern __shared__ float2 lds[];  // C * LP
    int64_t b;
    int mx0;
    if (!column_block(nimg, Nx, C, b, mx0)) return;
    const int hy = Ny / 2;
    for (int i0 = threadIdx.x; i0 < L * C; i0 += kLoadBatch * kBlock) {  // loads first, then the LDS writes
        float2 v[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int y = i / C, mx = mx0 + i % C;
            v[u] = make_float2(0.0f, 0.0f);
            if (i < L * C && mx < Nx) {
                int x = mx - hx;
                if (x < 0) x += Gx;
                v[u] = grid[(b * L + y) * (int64_t)Gx + x];
            }
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            if (i < L * C) lds[(i % C) * LP + i / C] = v[u];
        }
    }
    __syncthreads();
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    {   // wave w transforms columns w, w + 4, ... together
        constexpr int NL = C / (kBlock / kWave);
        constexpr int pitch = kBlock / kWave * LP;
        float2 *col = lds + wave * LP;
        fft_lines<L, NL, true>(
            lane, tw, col, pitch, [&](int l, int i) { return col[l * pitch + i]; },
            [&](int l, int i, float2 v) { col[l * pitch + i] = v; });
    }
    __syncthreads();
    for (int i0 = threadIdx.x; i0 < Ny * C; i0 += kLoadBatch * kBlock) {  // apodization loads first
        float ax[kLoadBatch], ay[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int my = i / C, mx = mx0 + i % C;
            ax[u] = ay[u] = 1.0f;
            if (i < Ny * C && mx < Nx) {
                if (apx) ax[u] = apx[mx];
                if (apy) ay[u] = apy[my];
            }
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int my = i / C, c = i % C, mx = mx0 + c;
            if (i < Ny * C && mx < Nx) {
                int y = my - hy;
                if (y < 0) y += L;
                const float2 v = cscale(cscale(cscale(lds[c * LP + y], scale), ax[u]), ay[u]);
                img[(b * Ny + my) * (int64_t)Nx + mx] = v;
            }
        }
    }
}

using RowFn = void (*)(float2 *, int64_t, int, const float2 *, RowRanges);
using ProductFn = void (*)(float2 *, int64_t, int, const float2 *, int64_t, const float2 *);
using ColFwdFn = void (*)(const float2 *, float2 *, int64_t, int, int, int, int, const float *, const float *,
                          const float2 *);
using ColInvFn = void (*)(const float2 *, float2 *, int64_t, int, int, int, int, const float *, const float *,
                          const float2 *, float);

struct FftFns {
    int L = 0;
    RowFn row_fwd[2] = {}, row_inv[2] = {};  // 2D plans, 3D plans
    ProductFn product = nullptr;
    ColFwdFn col_fwd = nullptr;
    ColInvFn col_inv = nullptr;
    int C = 0;
    size_t lds = 0;  // dynamic LDS bytes of the column kernels
};

template <int L>
FftFns fns_for() {
    FftFns f;
    f.L = L;
    f.C = col_group(L);
    f.row_fwd[0] = fft_rows_kernel<L, false, false>;
    f.row_fwd[1] = fft_rows_kernel<L, false, true>;
    f.row_inv[0] = fft_rows_kernel<L, true, false>;
    f.row_inv[1] = fft_rows_kernel<L, true, true>;
    f.product = fft_product_kernel<L>;
    f.col_fwd = fft_cols_fwd_kernel<L, col_group(L)>;
    f.col_inv = fft_cols_inv_kernel<L, col_group(L)>;
    f.lds = col_lds_bytes(L);
    return f;
}

// Transform lengths with kernels: the oversampled sizes ceil(osf N) of
// N = 64, 128, 192, 256, 320, 384, 512 at osf 1.25, 1.5 and 2 (all of the
// form 2^a 3^b 5^c), 64 .. 1024, and the short lengths 16 .. 48 of small
// grids and of Cartesian slice axes (osf 1).
FftFns fft_fns(int L) {
    switch (L) {
        case 16: return fns_for<16>();
        case 24: return fns_for<24>();
        case 32: return fns_for<32>();
        case 40: return fns_for<40>();
        case 48: return fns_for<48>();
        case 64: return fns_for<64>();
        case 80: return fns_for<80>();
        case 96: return fns_for<96>();
        case 128: return fns_for<128>();
        case 160: return fns_for<160>();
        case 192: return fns_for<192>();
        case 240: return fns_for<240>();
        case 256: return fns_for<256>();
        case 288: return fns_for<288>();
        case 320: return fns_for<320>();
        case 384: return fns_for<384>();
        case 400: return fns_for<400>();
        case 480: return fns_for<480>();
        case 512: return fns_for<512>();
        case 576: return fns_for<576>();
        case 640: return fns_for<640>();
        case 768: return fns_for<768>();
        case 1024: return fns_for<1024>();
        default: return FftFns{};
    }
}

int launch_rows(const FftAxis &a, bool inverse, float2 *data, int64_t nlines, hipStream_t stream,
                const RowRanges &ranges) {
    if (a.M) return chirp_rows(a, inverse, data, nlines, stream);
    if (a.radices.n) return smooth_rows(a, inverse, data, nlines, stream);
    const FftFns f = fft_fns(a.L);
    hipLaunchKernelGGL(inverse ? f.row_inv[ranges.d3] : f.row_fwd[ranges.d3], dim3(row_blocks(nlines, a.L)), dim3(kBlock), 0, stream, data,
                       nlines, a.N, a.tw, ranges);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int launch_product(const FftAxis &a, float2 *data, int64_t nlines, const float2 *kern, int64_t nk, hipStream_t stream) {
    if (a.M) return chirp_product(a, data, nlines, kern, nk, stream);
    if (a.radices.n) return smooth_product(a, data, nlines, kern, nk, stream);
    hipLaunchKernelGGL(fft_fns(a.L).product, dim3(row_blocks(nlines, a.L)), dim3(kBlock), 0, stream, data, nlines, a.N,
                       kern, nk, a.tw);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

// Columns `cols` of nimg images, placed at x = (mx - hx) mod pitch of the grid.
int launch_cols(const FftAxis &a, bool inverse, const float2 *src, float2 *dst, int64_t nimg, int cols, int pitch,
                int hx, const float *apx, const float *apy, hipStream_t stream, float scale = 1.0f) {
    if (a.M) return chirp_cols(a, inverse, src, dst, nimg, cols, pitch, hx, apx, apy, scale, stream);
    if (a.radices.n) return smooth_cols(a, inverse, src, dst, nimg, cols, pitch, hx, apx, apy, scale, stream);
    const FftFns f = fft_fns(a.L);
    const dim3 blocks(col_blocks(nimg, cols, f.C));
    if (inverse)
        hipLaunchKernelGGL(f.col_inv, blocks, dim3(kBlock), f.lds, stream, src, dst, nimg, cols, a.N, pitch, hx, apx,
                           apy, a.tw, scale);
    else
        hipLaunchKernelGGL(f.col_fwd, blocks, dim3(kBlock), f.lds, stream, src, dst, nimg, cols, a.N, pitch, hx, apx,
                           apy, a.tw);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

}  // namespace

// 2D and 3D plans: each axis by a kernel of its grid length where there is
// one, else by radices at run time where its factors allow, else as a chirp
// transform; no stages where an axis has none of them.
int build_fft(tn_plan *plan, hipStream_t stream) {
    const int ndim = plan->p.ndim;
    std::vector<float2> host;
    size_t at[3] = {};
    bool direct = true;
    for (int a = 0; a < ndim; ++a) {  // 0: x (grid[2]), 1: y (grid[1]), 2: z (grid[0])
        FftAxis &ax = plan->axis[a];
        ax.N = plan->p.shape[2 - a];
        ax.L = plan->p.grid[2 - a];
        const FftFns f = fft_fns(ax.L);
        if (f.L == 0 && !smooth_radices(ax.L, ax.radices) && (ax.M = chirp_length(ax.N, ax.L)) == 0) return TN_OK;
        direct = direct && f.L != 0;
        at[a] = host.size();
        if (f.L == 0) {
            const int rc = ax.M ? chirp_prepare(ax) : smooth_prepare(ax);
            if (rc) return rc;
        }
        if (ax.M) {
            chirp_tables(ax, host);
            continue;
        }
        if (a > 0 && f.L != 0) {  // dynamic LDS of the column tiles (up to 64 KiB with these column counts)
            TN_HIP(hipFuncSetAttribute((const void *)f.col_fwd, hipFuncAttributeMaxDynamicSharedMemorySize, (int)f.lds));
            TN_HIP(hipFuncSetAttribute((const void *)f.col_inv, hipFuncAttributeMaxDynamicSharedMemorySize, (int)f.lds));
        }
        const double pi = 3.14159265358979323846;
        for (int m = 0; m < ax.L; ++m) {
            const double ang = -2.0 * pi * (double)m / (double)ax.L;
            host.push_back(make_float2((float)std::cos(ang), (float)std::sin(ang)));
        }
    }
    plan->fft_bytes = (int64_t)(sizeof(float2) * host.size());
    TN_HIP(hipMalloc(&plan->d_fft, plan->fft_bytes));
    TN_HIP(hipMemcpyAsync(plan->d_fft, host.data(), plan->fft_bytes, hipMemcpyHostToDevice, stream));
    TN_HIP(hipStreamSynchronize(stream));  // before the host table goes out of scope
    for (int a = 0; a < ndim; ++a) {
        if (plan->axis[a].M)
            chirp_bind(plan->axis[a], plan->d_fft + at[a]);
        else
            plan->axis[a].tw = plan->d_fft + at[a];
    }
    plan->fft_direct = direct;
    return TN_OK;
}

// 3D only: the grids of 2D plans mostly stay in the caches, and the range of a
// row is one more dependent load before its data (20 frames of 240^2 94 ->
// 103 us, unrolled CG-SENSE 1.95 -> 2.04 ms; the checks alone 97 us, 1.98 ms).
bool rows_ranged(const tn_plan *plan, int64_t nbatch) {
    const int64_t lines = nbatch * plan->p.nframes * plan->p.grid[0] * plan->p.grid[1];
    return plan->p.ndim == 3 && plan->d_rows && plan->d_fft && plan->axis[0].M == 0 && plan->axis[0].radices.n == 0 &&
           lines < INT32_MAX;
}

static RowRanges row_ranges(const tn_plan *plan, bool ranged) {
    RowRanges g;
    g.d3 = plan->p.ndim == 3;
    if (!ranged) return g;
    return RowRanges{plan->d_rows,    plan->p.grid[1], plan->tile[1],   plan->ntiles[1], plan->p.grid[0],
                     plan->tile[0],   plan->ntiles[0], plan->p.nframes, g.d3};
}

int launch_fft_forward(const tn_plan *plan, const float2 *image, float2 *grid, int64_t nimg, hipStream_t stream,
                       bool ranged) {
    if (nimg == 0) return TN_OK;
    const FftAxis &x = plan->axis[0], &y = plan->axis[1];
    const int rc = launch_cols(y, false, image, grid, nimg, x.N, x.L, x.N / 2, plan->d_apod[2], plan->d_apod[1], stream);
    return rc ? rc : launch_rows(x, false, grid, nimg * y.L, stream, row_ranges(plan, ranged));
}

int launch_fft_adjoint(const tn_plan *plan, float2 *grid, float2 *image, int64_t nimg, hipStream_t stream,
                       bool ranged) {
    if (nimg == 0) return TN_OK;
    const FftAxis &x = plan->axis[0], &y = plan->axis[1];
    const int rc = launch_rows(x, true, grid, nimg * y.L, stream, row_ranges(plan, ranged));
    const float scale = (float)(1.0 / ((double)x.L * (double)y.L));
    return rc ? rc
              : launch_cols(y, true, grid, image, nimg, x.N, x.L, x.N / 2, plan->d_apod[2], plan->d_apod[1], stream,
                            scale);
}

// z stage of the 3D plans: each image volume (Nz, Ny, Nx) is a 2D image of
// Nz rows and Ny*Nx columns; the column kernels transform it along z (length
// Gz) with the z apodization, the z placement (mz - Nz/2) mod Gz (forward) or
// crop (adjoint) and, in the adjoint, the 1/Gz scale; the columns keep their
// flattened (y, x) order (hx = 0) for the plane stages.
int launch_fft_z_forward(const tn_plan *plan, const float2 *image, float2 *zout, int64_t nimg, hipStream_t stream) {
    if (nimg == 0) return TN_OK;
    const int cols = plan->p.shape[1] * plan->p.shape[2];
    return launch_cols(plan->axis[2], false, image, zout, nimg, cols, cols, 0, nullptr, plan->d_apod[0], stream);
}

int launch_fft_z_adjoint(const tn_plan *plan, const float2 *zin, float2 *image, int64_t nimg, hipStream_t stream) {
    if (nimg == 0) return TN_OK;
    const int cols = plan->p.shape[1] * plan->p.shape[2];
    return launch_cols(plan->axis[2], true, zin, image, nimg, cols, cols, 0, nullptr, plan->d_apod[0], stream,
                       (float)(1.0 / (double)plan->p.grid[0]));
}

// Convolution of nimg images with `kern` (nkern kernels of the grid's size in
// FFT order, image i taking kernel i mod nkern): pad, DFT, product, inverse DFT,
// crop. The placement cancels: the columns stay in image order. work0 (3D):
// nimg * Gz * Ny * Nx, work1: nimg * (Gz) * Gy * Nx complex values.
int launch_convolve(const tn_plan *plan, const float2 *image, const float2 *kern, int64_t nkern, float2 *out,
                    float2 *work0, float2 *work1, int64_t nimg, hipStream_t stream) {
    if (nimg == 0) return TN_OK;
    const FftAxis &x = plan->axis[0], &y = plan->axis[1], &z = plan->axis[2];
    const bool d3 = plan->p.ndim == 3;
    const int plane = x.N * y.N;
    const int64_t nplanes = d3 ? nimg * z.L : nimg;
    const double cells = (double)x.L * y.L * (d3 ? z.L : 1);
    int rc = TN_OK;
    if (d3) rc = launch_cols(z, false, image, work0, nimg, plane, plane, 0, nullptr, nullptr, stream);
    if (!rc) rc = launch_cols(y, false, d3 ? work0 : image, work1, nplanes, x.N, x.N, 0, nullptr, nullptr, stream);
    if (!rc) rc = launch_product(x, work1, nplanes * y.L, kern, nkern * (d3 ? z.L : 1) * y.L, stream);
    if (!rc)
        rc = launch_cols(y, true, work1, d3 ? work0 : out, nplanes, x.N, x.N, 0, nullptr, nullptr, stream,
                         (float)(1.0 / cells));
    if (!rc && d3) rc = launch_cols(z, true, work0, out, nimg, plane, plane, 0, nullptr, nullptr, stream);
    return rc;
}

}  // namespace tn
