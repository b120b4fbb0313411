// FFT stages of grid lengths with factors up to 17 that have no kernel of
// their own: one kernel for every such length, the radices at run time.
//
// Fusion and tiles as in the direct stages (tn_fft.hip): rows in place, or
// columns of an image, held in LDS by one wave through all passes. A pass
// reads one buffer and writes the other (at run time the butterflies of a pass
// cannot all sit in registers between its reads and writes), and its
// butterflies are dealt to the lanes over all lines of the wave. The inverse
// is the forward transform of (im, re) pairs, swapped back on the way out.
//
// A chirp transform (tn_chirp.hip) would serve these lengths too, at twice the
// passes on nearly twice the points, and with more rounding: 2D grids of 330
// points, two coils, eight CG steps gave 3.7e-6 against 64 bits for 3.1e-6.
#include <algorithm>

#include "tn_fft.h"

namespace tn {
namespace {

// cos or sin of 2 pi i / R, 1 <= i <= R / 2
template <int R>
constexpr float prime_root(int i, bool sine) {
    if (R == 7) {
        constexpr float c[] = {0.62348980185873359f, -0.22252093395631434f, -0.90096886790241903f};
        constexpr float s[] = {0.78183148246802980f, 0.97492791218182362f, 0.43388373911755823f};
        return sine ? s[i - 1] : c[i - 1];
    }
    if (R == 11) {
        constexpr float c[] = {0.84125353283118121f, 0.41541501300188644f, -0.14231483827328500f,
                              -0.65486073394528499f, -0.95949297361449737f};
        constexpr float s[] = {0.54064081745559756f, 0.90963199535451833f, 0.98982144188093280f,
                              0.75574957435425827f, 0.28173255684142967f};
        return sine ? s[i - 1] : c[i - 1];
    }
    if (R == 13) {
        constexpr float c[] = {0.88545602565320991f, 0.56806474673115592f, 0.12053668025532301f,
                              -0.35460488704253545f, -0.74851074817110119f, -0.97094181742605201f};
        constexpr float s[] = {0.46472317204376851f, 0.82298386589365635f, 0.99270887409805397f,
                              0.93501624268541483f, 0.66312265824079519f, 0.23931566428755768f};
        return sine ? s[i - 1] : c[i - 1];
    }
    if (R == 17) {
        constexpr float c[] = {0.93247222940435581f, 0.73900891722065909f, 0.44573835577653831f,
                              0.09226835946330202f, -0.27366299007208289f, -0.60263463637925629f,
                              -0.85021713572961399f, -0.98297309968390179f};
        constexpr float s[] = {0.36124166618715292f, 0.67369564364655721f, 0.89516329135506234f,
                              0.99573417629503447f, 0.96182564317281904f, 0.79801722728023960f,
                              0.52643216287735606f, 0.18374951781657037f};
        return sine ? s[i - 1] : c[i - 1];
    }
    return 0.0f;
}

// DFT of an odd prime length from the sums and differences of mirrored inputs.
template <int R>
__device__ __forceinline__ void dft_prime(float2 (&v)[R]) {
    constexpr int H = R / 2;
    float2 a[H], b[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
        a[k] = cadd(v[k + 1], v[R - 1 - k]);
        b[k] = csub(v[k + 1], v[R - 1 - k]);
    }
    const float2 v0 = v[0];
#pragma unroll
    for (int k = 0; k < H; ++k) v[0] = cadd(v[0], a[k]);
#pragma unroll
    for (int j = 1; j <= H; ++j) {
        float2 m = v0, n = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            const int i = j * k % R;
            const float c = prime_root<R>(i <= H ? i : R - i, false);
            const float s = i <= H ? prime_root<R>(i, true) : -prime_root<R>(R - i, true);
            m.x += c * a[k - 1].x;
            m.y += c * a[k - 1].y;
            n.x += s * b[k - 1].x;
            n.y += s * b[k - 1].y;
        }
        v[j] = make_float2(m.x + n.y, m.y - n.x);
        v[R - j] = make_float2(m.x - n.y, m.y + n.x);
    }
}

__device__ __forceinline__ int pad8(int a) { return a + (a >> 3); }

// One pass of radix R over nl lines, as fft_passes: ns = product of the
// earlier radices.
template <int R>
__device__ __forceinline__ void smooth_pass(int lane, int L, int ns, int nl, int pitch, const float2 *in, float2 *out,
                                            const float2 *__restrict__ tw) {
    const int M = L / R, ts = M / ns;
    const float im = 1.0f / (float)M, is = 1.0f / (float)ns;  // t < 2^14: the quotients below are exact
    for (int t = lane; t < nl * M; t += kWave) {
        const int l = (int)(((float)t + 0.5f) * im), j = t - l * M;
        const int q = (int)(((float)j + 0.5f) * is), k = j - q * ns;
        const float2 *src = in + l * pitch;
        float2 *dst = out + l * pitch;
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = src[pad8(j + r * M)];
        if (ns > 1) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmul(v[r], tw[r * k * ts]);
        }
        if constexpr (R == 7 || R > 10)
            dft_prime<R>(v);
        else
            dft<R, false>(v);
        const int d = q * ns * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) dst[pad8(d + r * ns)] = v[r];
    }
}

// All passes over nl lines of pitch float2 from `a`, with `b` as the other
// buffer; returns the buffer of the result.
__device__ __forceinline__ float2 *smooth_lines(int lane, const SmoothRadices &f, int L, int nl, int pitch, float2 *a,
                                                float2 *b, const float2 *__restrict__ tw) {
    int ns = 1;
    for (int p = 0; p < f.n; ++p) {
        __asm__ __volatile__("" ::: "memory");  // other lanes' elements: reads stay behind the last pass's writes
        switch (f.r[p]) {
            case 2: smooth_pass<2>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 3: smooth_pass<3>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 4: smooth_pass<4>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 5: smooth_pass<5>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 6: smooth_pass<6>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 7: smooth_pass<7>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 8: smooth_pass<8>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 10: smooth_pass<10>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 11: smooth_pass<11>(lane, L, ns, nl, pitch, a, b, tw); break;
            case 13: smooth_pass<13>(lane, L, ns, nl, pitch, a, b, tw); break;
            default: smooth_pass<17>(lane, L, ns, nl, pitch, a, b, tw); break;
        }
        ns *= f.r[p];
        float2 *t = a;
        a = b;
        b = t;
    }
    __asm__ __volatile__("" ::: "memory");
    return a;
}

template <bool INV>
__device__ __forceinline__ float2 swapped(float2 v) {
    return INV ? make_float2(v.y, v.x) : v;
}

// Row transforms in place of rows of L: forward reads the N data columns (x =
// (m - N/2) mod L), inverse writes them. nl rows per wave.
template <bool INV>
__global__ __launch_bounds__(kBlock) void smooth_rows_kernel(float2 *__restrict__ data, int64_t nlines, int L, int N,
                                                             SmoothRadices f, const float2 *__restrict__ tw, int nl) {
    extern __shared__ float2 lds[];  // per wave: two buffers of nl lines
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * nl;
    if (line0 >= nlines) return;  // no barriers below
    const int pitch = fft_line(L);
    float2 *a = lds + wave * 2 * nl * pitch, *b = a + nl * pitch;
    nl = (int)min((int64_t)nl, nlines - line0);
    float2 *row = data + line0 * L;
    const float il = 1.0f / (float)L;  // the quotients below are exact (t < 2^14)
    const int total = nl * L;
    for (int t0 = lane; t0 < total; t0 += kLoadBatch * kWave) {  // loads first, then the LDS writes
        float2 v[kLoadBatch];
        int to[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int t = t0 + u * kWave;
            const int l = (int)(((float)t + 0.5f) * il), i = t - l * L;
            to[u] = l * pitch + pad8(i);
            v[u] = make_float2(0.0f, 0.0f);
            if (t < total && (INV || kept(i, N, L))) v[u] = row[t];
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u)
            if (t0 + u * kWave < total) a[to[u]] = swapped<INV>(v[u]);
    }
    const float2 *res = smooth_lines(lane, f, L, nl, pitch, a, b, tw);
#pragma unroll 4
    for (int t = lane; t < total; t += kWave) {
        const int l = (int)(((float)t + 0.5f) * il), i = t - l * L;
        if (!INV || kept(i, N, L)) row[t] = swapped<INV>(res[l * pitch + pad8(i)]);
    }
}

// The product rows (see fft_product_kernel), nl rows of N per wave.
__global__ __launch_bounds__(kBlock) void smooth_product_kernel(float2 *__restrict__ data, int64_t nlines, int L, int N,
                                                                SmoothRadices f, const float2 *__restrict__ tw, int nl,
                                                                const float2 *__restrict__ kern, int64_t nk) {
    extern __shared__ float2 lds[];  // per wave: two buffers of nl lines
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t line0 = ((int64_t)blockIdx.x * (kBlock / kWave) + wave) * nl;
    if (line0 >= nlines) return;  // no barriers below
    const int pitch = fft_line(L);
    float2 *a = lds + wave * 2 * nl * pitch, *b = a + nl * pitch;
    nl = (int)min((int64_t)nl, nlines - line0);
    const float il = 1.0f / (float)L;  // the quotients below are exact (t < 2^14)
    const int total = nl * L;
    auto pixel = [&](int i) { return i + N / 2 < L ? i + N / 2 : i + N / 2 - L; };  // < N: data
#pragma unroll 4
    for (int t = lane; t < total; t += kWave) {
        const int l = (int)(((float)t + 0.5f) * il), i = t - l * L, m = pixel(i);
        a[l * pitch + pad8(i)] = m < N ? data[(line0 + l) * N + m] : make_float2(0.0f, 0.0f);
    }
    float2 *res = smooth_lines(lane, f, L, nl, pitch, a, b, tw);
    const int64_t k0 = line0 % nk;
#pragma unroll 4
    for (int t = lane; t < total; t += kWave) {  // swapped for the inverse
        const int l = (int)(((float)t + 0.5f) * il), i = t - l * L;
        const int64_t kr = k0 + l < nk ? k0 + l : (line0 + l) % nk;
        float2 *v = res + l * pitch + pad8(i);
        *v = swapped<true>(cmul(*v, kern[kr * L + i]));
    }
    res = smooth_lines(lane, f, L, nl, pitch, res, res == a ? b : a, tw);
#pragma unroll 4
    for (int t = lane; t < total; t += kWave) {
        const int l = (int)(((float)t + 0.5f) * il), i = t - l * L, m = pixel(i);
        if (m < N) data[(line0 + l) * N + m] = swapped<true>(res[l * pitch + pad8(i)]);
    }
}

// Column stages (see tn_fft.hip), C = 2^lc columns per workgroup, C / 4 per wave.
template <bool INV>
__global__ __launch_bounds__(kBlock) void smooth_cols_kernel(const float2 *__restrict__ src, float2 *__restrict__ dst,
                                                             int64_t nimg, int Nx, int Ny, int L, int Gx, int hx,
                                                             const float *__restrict__ apx,
                                                             const float *__restrict__ apy, SmoothRadices f,
                                                             const float2 *__restrict__ tw, float scale, int lc) {
    extern __shared__ float2 lds[];  // two buffers of C lines
    const int C = 1 << lc, pitch = f.pitch;
    int64_t b;
    int mx0;
    if (!column_block(nimg, Nx, C, b, mx0)) return;
    const int hy = Ny / 2;
    auto grid_x = [&](int mx) { return mx < hx ? mx - hx + Gx : mx - hx; };
    float2 *a = lds, *o = lds + C * pitch;
    // loads first, then the LDS writes; forward: the image rows, and zeros for the others
    const int rows = INV ? L : Ny;
    for (int i0 = threadIdx.x; i0 < rows << lc; i0 += kLoadBatch * kBlock) {
        float2 v[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int y = i >> lc, mx = mx0 + (i & (C - 1));
            v[u] = make_float2(0.0f, 0.0f);
            if (y < rows && mx < Nx)
                v[u] = INV ? src[(b * L + y) * (int64_t)Gx + grid_x(mx)] : src[(b * Ny + y) * (int64_t)Nx + mx];
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int i = i0 + u * kBlock;
            const int y = i >> lc, c = i & (C - 1), mx = mx0 + c;
            if (y >= rows) continue;
            float2 w = v[u];
            if (!INV && mx < Nx) {  // x then y, as the separate pre-pass
                if (apx) w = cscale(w, apx[mx]);
                if (apy) w = cscale(w, apy[y]);
            }
            a[c * pitch + pad8(INV ? y : y < hy ? y - hy + L : y - hy)] = swapped<INV>(w);
        }
    }
    if (!INV)
        for (int i = threadIdx.x; i < (L - Ny) << lc; i += kBlock)
            a[(i & (C - 1)) * pitch + pad8(Ny - hy + (i >> lc))] = make_float2(0.0f, 0.0f);
    __syncthreads();
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, nl = C / (kBlock / kWave);
    // wave w holds columns w * nl .. (contiguous lines); every wave ends in the same buffer
    const float2 *mine = smooth_lines(lane, f, L, nl, pitch, a + wave * nl * pitch, o + wave * nl * pitch, tw);
    const float2 *res = mine - wave * nl * pitch;
    __syncthreads();
    const int outs = INV ? Ny : L;
    for (int i = threadIdx.x; i < outs << lc; i += kBlock) {
        const int y = i >> lc, c = i & (C - 1), mx = mx0 + c;
        if (mx >= Nx) continue;
        if (!INV) {
            dst[(b * L + y) * (int64_t)Gx + grid_x(mx)] = res[c * pitch + pad8(y)];
        } else {
            float2 v = cscale(swapped<INV>(res[c * pitch + pad8(y < hy ? y - hy + L : y - hy)]), scale);
            if (apx) v = cscale(v, apx[mx]);
            if (apy) v = cscale(v, apy[y]);
            dst[(b * Ny + y) * (int64_t)Nx + mx] = v;
        }
    }
}

// Fewest passes for n from the radices below (larger first); returns the
// number of passes, or 99.
int factor(int n, int *r) {
    if (n == 1) return 0;
    for (int p : {17, 13, 11, 7})
        if (n % p == 0) {
            r[0] = p;
            return 1 + factor(n / p, r + 1);
        }
    int best = 99;
    for (int p : {10, 8, 6, 5, 4, 3, 2}) {
        if (n % p != 0) continue;
        int rest[kSmoothPasses + 1];
        const int c = 1 + factor(n / p, rest);
        if (c < best && c <= kSmoothPasses) {
            best = c;
            r[0] = p;
            std::copy(rest, rest + c - 1, r + 1);
        }
    }
    return best;
}

// Padded float2 per line; the columns of a tile start pitch * 2 words apart,
// odd multiples of which spread a row's C columns over the banks.
int col_pitch(int L) { return fft_line(L) | 1; }

// Columns per workgroup: 16 (a 128-byte line per row) while two buffers fit
// 48 KiB of LDS and the launch has four workgroups per CU, at least 4 (one
// per wave).
int col_log2(int L, int64_t cols) {
    int lc = 4;
    while (lc > 2 && ((size_t)16 * col_pitch(L) << lc > 48 * 1024 || cols >> lc < 1024)) --lc;
    return lc;
}

size_t col_lds(int L, int lc) { return sizeof(float2) * 2 * col_pitch(L) << lc; }

// Rows per wave: lanes filled by several lines, at most 512 elements (two
// buffers of 1024 left two waves per SIMD: 39116 rows of 105 44 us for 29), while
// the launch has sixteen waves per CU.
int row_lines(int L, int64_t nlines) {
    return (int)std::max<int64_t>(1, std::min<int64_t>({8, 512 / fft_line(L), nlines / 4096}));
}

size_t row_lds(int L, int nl) { return sizeof(float2) * (kBlock / kWave) * 2 * nl * fft_line(L); }

}  // namespace

bool smooth_radices(int L, SmoothRadices &f) {
    if (L < 2 || L > 1024) return false;
    int rest = L;
    for (int p : {2, 3, 5, 7, 11, 13, 17})
        while (rest % p == 0) rest /= p;
    if (rest != 1) return false;
    int r[kSmoothPasses + 8];
    f.n = factor(L, r);
    if (f.n > kSmoothPasses) return false;
    std::copy(r, r + f.n, f.r);
    f.pitch = col_pitch(L);
    return true;
}

int smooth_prepare(const FftAxis &a) {
    for (auto fn : {smooth_rows_kernel<false>, smooth_rows_kernel<true>})
        TN_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)row_lds(1024, 1)));
    TN_HIP(hipFuncSetAttribute((const void *)smooth_product_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)row_lds(1024, 1)));
    for (auto fn : {smooth_cols_kernel<false>, smooth_cols_kernel<true>})
        TN_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)col_lds(1024, 2)));
    return TN_OK;
}

int smooth_rows(const FftAxis &a, bool inverse, float2 *data, int64_t nlines, hipStream_t stream) {
    const int nl = row_lines(a.L, nlines);
    const int64_t rpb = (int64_t)nl * (kBlock / kWave);
    hipLaunchKernelGGL(inverse ? smooth_rows_kernel<true> : smooth_rows_kernel<false>,
                       dim3((unsigned)((nlines + rpb - 1) / rpb)), dim3(kBlock), row_lds(a.L, nl), stream, data, nlines,
                       a.L, a.N, a.radices, a.tw, nl);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int smooth_product(const FftAxis &a, float2 *data, int64_t nlines, const float2 *kern, int64_t nk, hipStream_t stream) {
    const int nl = row_lines(a.L, nlines);
    const int64_t rpb = (int64_t)nl * (kBlock / kWave);
    hipLaunchKernelGGL(smooth_product_kernel, dim3((unsigned)((nlines + rpb - 1) / rpb)), dim3(kBlock),
                       row_lds(a.L, nl), stream, data, nlines, a.L, a.N, a.radices, a.tw, nl, kern, nk);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

int smooth_cols(const FftAxis &a, bool inverse, const float2 *src, float2 *dst, int64_t nimg, int cols, int pitch,
                int hx, const float *apx, const float *apy, float scale, hipStream_t stream) {
    const int lc = col_log2(a.L, nimg * cols);
    hipLaunchKernelGGL(inverse ? smooth_cols_kernel<true> : smooth_cols_kernel<false>,
                       dim3(col_blocks(nimg, cols, 1 << lc)), dim3(kBlock), col_lds(a.L, lc), stream, src, dst, nimg, cols,
                       a.N, a.L, pitch, hx, apx, apy, a.radices, a.tw, scale, lc);
    TN_HIP(hipGetLastError());
    return TN_OK;
}

}  // namespace tn
