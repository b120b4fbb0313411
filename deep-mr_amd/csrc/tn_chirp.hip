// FFT stages of grid lengths without a kernel of their own (any length L >= 2
// whose convolution fits): chirp (Bluestein) line transforms for gfx950.
//
// With nk = (n^2 + k^2 - (k - n)^2) / 2 a line transform of N pixels onto L
// grid points (or back) is a convolution with a chirp: inputs times in[], a
// cyclic convolution of length M >= N + L - 1 with b, outputs times out[]. A
// wave holds its lines in LDS through both length-M transforms (the Stockham
// passes of tn_fft.h), so a stage moves the bytes the direct one does: the
// zero padding, apodization, placement and crop are fused the same way.
//
// The alternative is the library's transform of the whole padded grid between
// the separate pad and crop kernels, which reads and writes the zeros, and
// takes passes and transposes of its own for lengths with large factors. It is
// slower up to the longest convolution (1018^2 grids, N + G - 1 = 1526: one
// image 46 us for 94, 32 images 815 for 1240; 127^3, 4 images 190 for 418).
// Two transforms round twice: outputs move both ways against the library's
// (whole calls with such lengths: error against 64 bits 0.8 to 1.07 of the
// former).
#include <cmath>
#include <complex>
#include <vector>

#include "tn_fft.h"

namespace tn {
namespace {

template <int M, int NL, class Src, class Dst>
__device__ __forceinline__ void chirp_lines(int lane, const float2 *__restrict__ tw, const float2 *__restrict__ b,
                                            float2 *buf, int pitch, Src src, Dst dst) {
    fft_lines<M, NL, false>(lane, tw, buf, pitch, src,
                            [&](int l, int i, float2 v) { buf[l * pitch + lds_at<M>(i)] = v; });
    __asm__ __volatile__("" ::: "memory");  // other lanes' elements below: keep the reads behind the writes
    fft_lines<M, NL, true>(
        lane, tw, buf, pitch, [&](int l, int i) { return cmul(buf[l * pitch + lds_at<M>(i)], b[i]); }, dst);
}

// Row transforms in place, nin inputs to nout outputs of rows of L; element i
// of either sits at x = (i - h) mod L.
template <int M>
__global__ __launch_bounds__(kBlock) void chirp_rows_kernel(float2 *__restrict__ data, int64_t nlines, int L, int nin,
                                                            int hin, int nout, int hout, ChirpTable t,
                                                            const float2 *__restrict__ tw) {
    constexpr int RL = rows_per_wave(M);
    __shared__ float2 lds[kBlock / kWave * RL][fft_line(M)];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * RL;
    if (line0 >= nlines) return;  // no barriers below
    // a row past the last one reads the last and writes nothing
    auto row = [&](int l) { return data + min(line0 + l, nlines - 1) * L; };
    auto at = [&](int i, int h) { return i < h ? i - h + L : i - h; };
    chirp_lines<M, RL>(
        lane, tw, t.b, lds[wave * RL], fft_line(M),
        [&](int l, int i) { return i < nin ? cmul(row(l)[at(i, hin)], t.in[i]) : make_float2(0.0f, 0.0f); },
        [&](int l, int i, float2 v) {
            if (line0 + l < nlines && i < nout) row(l)[at(i, hout)] = cmul(v, t.out[i]);
        });
}

// The product rows (see fft_product_kernel): the chirp factors of the grid
// points cancel between the two transforms.
template <int M>
__global__ __launch_bounds__(kBlock) void chirp_product_kernel(float2 *__restrict__ data, int64_t nlines, int L, int N,
                                                               ChirpTable f, ChirpTable b,
                                                               const float2 *__restrict__ tw,
                                                               const float2 *__restrict__ kern, int64_t nk) {
    constexpr int RL = rows_per_wave(M), pitch = fft_line(M);
    __shared__ float2 lds[kBlock / kWave * RL][pitch];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * RL;
    if (line0 >= nlines) return;  // no barriers below
    // a row past the last one reads the last and writes nothing
    auto row = [&](int l) { return data + min(line0 + l, nlines - 1) * N; };
    const int64_t k0 = line0 % nk;
    auto krow = [&](int l) { return kern + (k0 + l < nk ? k0 + l : (line0 + l) % nk) * L; };
    const float2 zero = make_float2(0.0f, 0.0f);
    float2 *buf = lds[wave * RL];
    chirp_lines<M, RL>(
        lane, tw, f.b, buf, pitch, [&](int l, int i) { return i < N ? cmul(row(l)[i], f.in[i]) : zero; },
        [&](int l, int i, float2 v) { buf[l * pitch + lds_at<M>(i)] = v; });
    __asm__ __volatile__("" ::: "memory");
    chirp_lines<M, RL>(
        lane, tw, b.b, buf, pitch,
        [&](int l, int i) { return i < L ? cmul(buf[l * pitch + lds_at<M>(i)], krow(l)[i]) : zero; },
        [&](int l, int i, float2 v) {
            if (line0 + l < nlines && i < N) row(l)[i] = cmul(v, b.out[i]);
        });
}

// Column stages, as the direct ones: image columns mx0 .. mx0 + C - 1 of
// image b <-> grid columns (mx - hx) mod Gx. INV: grid -> image.
template <int M, int C, bool INV>
__global__ __launch_bounds__(kBlock) void chirp_cols_kernel(const float2 *__restrict__ src, float2 *__restrict__ dst,
                                                            int64_t nimg, int Nx, int Ny, int L, int Gx, int hx,
                                                            const float *__restrict__ apx,
                                                            const float *__restrict__ apy, ChirpTable t,
                                                            const float2 *__restrict__ tw, float scale) {
    constexpr int LP = fft_line(M) + fft_pad(C);
    extern __shared__ float2 lds[];  // C * LP
    int64_t b;
    int mx0;
    if (!column_block(nimg, Nx, C, b, mx0)) return;
    const int nin = INV ? L : Ny, nout = INV ? Ny : L;
    auto grid_x = [&](int mx) { return mx < hx ? mx - hx + Gx : mx - hx; };
    for (int i0 = threadIdx.x; i0 < nin * C; i0 += kLoadBatch * kBlock) {  // loads first, then the LDS writes
        float2 v[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int y = i / C, mx = mx0 + i % C;
            v[u] = make_float2(0.0f, 0.0f);
            if (i < nin * C && mx < Nx)
                v[u] = INV ? src[(b * L + y) * (int64_t)Gx + grid_x(mx)] : src[(b * Ny + y) * (int64_t)Nx + mx];
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            if (i >= nin * C) continue;
            const int y = i / C, c = i % C, mx = mx0 + c;
            float2 w = v[u];
            if (!INV && mx < Nx) {  // x then y, as the separate pre-pass
                if (apx) w = cscale(w, apx[mx]);
                if (apy) w = cscale(w, apy[y]);
            }
            lds[c * LP + y] = cmul(w, t.in[y]);
        }
    }
    __syncthreads();
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    {   // wave w transforms columns w, w + 4, ... together
        constexpr int NL = C / (kBlock / kWave);
        constexpr int pitch = kBlock / kWave * LP;
        float2 *col = lds + wave * LP;
        chirp_lines<M, NL>(
            lane, tw, t.b, col, pitch,
            [&](int l, int i) { return i < nin ? col[l * pitch + i] : make_float2(0.0f, 0.0f); },
            [&](int l, int i, float2 v) {
                if (i < nout) col[l * pitch + i] = v;
            });
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nout * C; i += kBlock) {
        const int y = i / C, c = i % C, mx = mx0 + c;
        if (mx >= Nx) continue;
        float2 v = cmul(lds[c * LP + y], t.out[y]);
        if (!INV) {
            dst[(b * L + y) * (int64_t)Gx + grid_x(mx)] = v;
        } else {
            v = cscale(v, scale);
            if (apx) v = cscale(v, apx[mx]);
            if (apy) v = cscale(v, apy[y]);
            dst[(b * Ny + y) * (int64_t)Nx + mx] = v;
        }
    }
}

using RowFn = void (*)(float2 *, int64_t, int, int, int, int, int, ChirpTable, const float2 *);
using ProductFn = void (*)(float2 *, int64_t, int, int, ChirpTable, ChirpTable, const float2 *, const float2 *, int64_t);
using ColFn = void (*)(const float2 *, float2 *, int64_t, int, int, int, int, int, const float *, const float *,
                       ChirpTable, const float2 *, float);
struct Fns {
    RowFn rows = nullptr;
    ProductFn product = nullptr;
    ColFn cols[2] = {nullptr, nullptr};  // forward, inverse
    int C = 0;
    size_t lds = 0;
};

template <int M>
Fns fns_for() {
    Fns f;
    f.C = col_group(M);
    f.rows = chirp_rows_kernel<M>;
    f.product = chirp_product_kernel<M>;
    f.cols[0] = chirp_cols_kernel<M, col_group(M), false>;
    f.cols[1] = chirp_cols_kernel<M, col_group(M), true>;
    f.lds = col_lds_bytes(M);
    return f;
}

Fns fns(int M) {
    switch (M) {
        case 32: return fns_for<32>();
        case 48: return fns_for<48>();
        case 64: return fns_for<64>();
        case 96: return fns_for<96>();
        case 128: return fns_for<128>();
        case 160: return fns_for<160>();
        case 192: return fns_for<192>();
        case 240: return fns_for<240>();
        case 256: return fns_for<256>();
        case 320: return fns_for<320>();
        case 384: return fns_for<384>();
        case 480: return fns_for<480>();
        case 512: return fns_for<512>();
        case 640: return fns_for<640>();
        case 768: return fns_for<768>();
        case 1024: return fns_for<1024>();
        case 1280: return fns_for<1280>();
        case 1536: return fns_for<1536>();
        default: return Fns{};
    }
}

using Cd = std::complex<double>;

Cd unit(int64_t num, int64_t den) {  // exp(i pi num / den)
    const double ang = 3.14159265358979323846 * (double)(num % (2 * den)) / (double)den;
    return Cd(std::cos(ang), std::sin(ang));
}

// Mixed-radix DFT of in[0], in[stride], ... (n values) in double precision;
// root[k] = exp(-2 pi i k / M), rs = M / n.
void host_dft(const Cd *in, int stride, Cd *out, int n, const std::vector<Cd> &root, int rs) {
    if (n == 1) {
        out[0] = in[0];
        return;
    }
    int p = 2;
    while (n % p != 0) ++p;
    const int m = n / p, M = (int)root.size();
    for (int q = 0; q < p; ++q) host_dft(in + (size_t)q * stride, stride * p, out + q * m, m, root, rs * p);
    std::vector<Cd> v(p);
    for (int k = 0; k < m; ++k) {
        for (int q = 0; q < p; ++q) v[q] = out[q * m + k] * root[(int64_t)q * k * rs % M];
        for (int r = 0; r < p; ++r) {
            Cd s = v[0];
            for (int q = 1; q < p; ++q) s += v[q] * root[(int64_t)q * r * m * rs % M];
            out[k + r * m] = s;
        }
    }
}

}  // namespace

// tw[M], then per direction (forward, inverse) in, out and b. Signed pixel
// n = m - N / 2; c(n) = exp(-i pi n^2 / L).
void chirp_tables(const FftAxis &a, std::vector<float2> &host) {
    const int N = a.N, L = a.L, M = a.M, h = N / 2;
    auto put = [&](Cd v) { host.push_back(make_float2((float)v.real(), (float)v.imag())); };
    auto c = [&](int64_t n) { return unit(-(n * n % (2 * L)), L); };
    std::vector<Cd> root(M), line(M), out(M);
    for (int k = 0; k < M; ++k) put(root[k] = unit(-2 * k, M));
    for (int inv = 0; inv < 2; ++inv) {
        auto pixel = [&](int m) { return inv ? std::conj(c(m - h)) : c(m - h); };
        auto point = [&](int k) { return inv ? std::conj(c(k)) : c(k); };
        const int nin = inv ? L : N, nout = inv ? N : L;
        for (int i = 0; i < nin; ++i) put(inv ? point(i) : pixel(i));
        for (int i = 0; i < nout; ++i) put(inv ? pixel(i) : point(i));
        // the chirp at out - in = j: grid point - pixel (forward) or pixel - grid point
        std::fill(line.begin(), line.end(), Cd(0.0, 0.0));
        for (int j = -(nin - 1); j < nout; ++j) line[(j + M) % M] = inv ? c(j - h) : std::conj(c(j + h));
        host_dft(line.data(), 1, out.data(), M, root, 1);
        for (int k = 0; k < M; ++k) put(out[k] / (double)M);
    }
}

void chirp_bind(FftAxis &a, const float2 *base) {
    a.tw = base;
    base += a.M;
    for (int inv = 0; inv < 2; ++inv) {
        ChirpTable &t = inv ? a.inv : a.fwd;
        t.in = base;
        t.out = base + (inv ? a.L : a.N);
        t.b = base + a.N + a.L;
        base += a.N + a.L + a.M;
    }
}

int chirp_prepare(const FftAxis &a) {
    const Fns f = fns(a.M);
    for (ColFn fn : f.cols)
        TN_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)f.lds));
    return TN_OK;
}

int chirp_rows(const FftAxis &a, bool inverse, float2 *data, int64_t nlines, hipStream_t stream) {
    const int h = a.N / 2;
    hipLaunchKernelGGL(fns(a.M).rows, dim3(row_blocks(nlines, a.M)), dim3(kBlock), 0, stream, data, nlines, a.L,
                       inverse ? a.L : a.N, inverse ? 0 : h, inverse ? a.N : a.L, inverse ? h : 0,
                       inverse ? a.inv : a.fwd, a.tw);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int chirp_product(const FftAxis &a, float2 *data, int64_t nlines, const float2 *kern, int64_t nk, hipStream_t stream) {
    hipLaunchKernelGGL(fns(a.M).product, dim3(row_blocks(nlines, a.M)), dim3(kBlock), 0, stream, data, nlines, a.L, a.N,
                       a.fwd, a.inv, a.tw, kern, nk);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int chirp_cols(const FftAxis &a, bool inverse, const float2 *src, float2 *dst, int64_t nimg, int cols, int pitch,
               int hx, const float *apx, const float *apy, float scale, hipStream_t stream) {
    const Fns f = fns(a.M);
    hipLaunchKernelGGL(f.cols[inverse], dim3(col_blocks(nimg, cols, f.C)), dim3(kBlock), f.lds, stream, src, dst, nimg,
                       cols, a.N, a.L, pitch, hx, apx, apy, inverse ? a.inv : a.fwd, a.tw, scale);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

}  // namespace tn
