// Device building blocks of the line transforms (included by the FFT
// translation units): in-register DFTs, the Stockham passes of one wave, the
// tile shapes and the per-axis tables of a plan.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "tn_internal.h"

namespace tn {
namespace {

// LDS column padding of a C-column tile, in float2: a column stride of
// 64 / C mod 16 float2 puts the 64 lanes of a row-major tile load (C columns
// x 64 / C rows) on 16 distinct bank pairs, four lanes each.
constexpr int fft_pad(int C) { return 64 / C; }

// Radices of a length-L transform: the fewest passes from 10, 8, 6, 5, 4, 3 and
// 2, with the smallest largest radix that reaches that count (register use,
// full waves), larger radices first; radix 16 where that saves a fourth pass
// (768 = 16 8 6, 1024 = 16 8 8). A pass is an exchange through LDS: 240 = 8 6 5
// and 400 = 10 8 5 take three passes where 8, 4, 2, 3, 5 alone take four. Two
// passes instead of three by radix 16 (256 = 16 16) cost the occupancy more
// than the exchange gives: 8 coils of 256^3 inverse 1.94 ms for 1.89 ms.
template <int L, int CAP>
constexpr int fft_min_pass() {
    if constexpr (L == 1) {
        return 0;
    } else {
        int best = 99;
        auto use = [&](auto r) {
            constexpr int R = decltype(r)::value;
            if constexpr (R <= CAP && L % R == 0) {
                const int n = 1 + fft_min_pass<L / R, CAP>();
                best = n < best ? n : best;
            }
        };
        use(std::integral_constant<int, 16>{});
        use(std::integral_constant<int, 10>{});
        use(std::integral_constant<int, 8>{});
        use(std::integral_constant<int, 6>{});
        use(std::integral_constant<int, 5>{});
        use(std::integral_constant<int, 4>{});
        use(std::integral_constant<int, 3>{});
        use(std::integral_constant<int, 2>{});
        return best;
    }
}
template <int L>
constexpr int fft_cap() {
    constexpr int p8 = fft_min_pass<L, 8>(), p10 = fft_min_pass<L, 10>(), p16 = fft_min_pass<L, 16>();
    return p10 > 3 && p16 < p10 ? 16 : p10 < p8 ? 10 : 8;
}
template <int L>
constexpr int fft_npass() {
    return fft_min_pass<L, fft_cap<L>()>();
}
// Radix of the first pass with radices up to CAP, and of pass P.
template <int L, int CAP>
constexpr int fft_first() {
    int r = 0;
    auto use = [&](auto c) {
        constexpr int R = decltype(c)::value;
        if constexpr (R <= CAP && L % R == 0)
            if (r == 0 && fft_min_pass<L / R, CAP>() + 1 == fft_min_pass<L, CAP>()) r = R;
    };
    use(std::integral_constant<int, 16>{});
    use(std::integral_constant<int, 10>{});
    use(std::integral_constant<int, 8>{});
    use(std::integral_constant<int, 6>{});
    use(std::integral_constant<int, 5>{});
    use(std::integral_constant<int, 4>{});
    use(std::integral_constant<int, 3>{});
    use(std::integral_constant<int, 2>{});
    return r;
}
template <int L, int P, int CAP>
constexpr int fft_radix_from() {
    if constexpr (P == 0)
        return fft_first<L, CAP>();
    else
        return fft_radix_from<L / fft_first<L, CAP>(), P - 1, CAP>();
}
template <int L, int P>
constexpr int fft_radix_at() {
    return fft_radix_from<L, P, fft_cap<L>()>();
}

// The Stockham passes keep a line in LDS with one float2 of padding after
// every 8 (16 where the first radix is 16): the scattered writes of the first
// pass (lane j at R j + r) then fall on distinct banks instead of 8 or 16
// lanes per bank. A line of L elements takes fft_line(L) float2.
constexpr int fft_line(int L) { return L + L / 8; }
template <int L>
__device__ __forceinline__ int lds_at(int a) {
    return a + (a >> (fft_radix_at<L, 0>() == 16 ? 4 : 3));
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// a * (s i) with s = -1 (forward) or +1 (inverse)
template <bool INV>
__device__ __forceinline__ float2 mul_j(float2 a) {
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// In-register DFTs of length R (sign -1 forward, +1 inverse).
template <bool INV>
__device__ __forceinline__ void dft4(float2 &a0, float2 &a1, float2 &a2, float2 &a3) {
    const float2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = mul_j<INV>(csub(a1, a3));
    a0 = cadd(t0, t2);
    a1 = cadd(t1, t3);
    a2 = csub(t0, t2);
    a3 = csub(t1, t3);
}

template <bool INV>
__device__ __forceinline__ void dft3(float2 &a0, float2 &a1, float2 &a2) {
    const float c = -0.5f, sn = 0.86602540378443865f;
    const float2 t1 = cadd(a1, a2), t2 = cscale(mul_j<INV>(csub(a1, a2)), sn);
    const float2 m = cadd(a0, cscale(t1, c));
    a0 = cadd(a0, t1);
    a1 = cadd(m, t2);
    a2 = csub(m, t2);
}

template <bool INV>
__device__ __forceinline__ void dft5(float2 &a0, float2 &a1, float2 &a2, float2 &a3, float2 &a4) {
    const float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
    const float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
    const float2 t1 = cadd(a1, a4), t2 = cadd(a2, a3);
    const float2 t3 = csub(a1, a4), t4 = csub(a2, a3);
    const float2 m1 = cadd(a0, cadd(cscale(t1, c1), cscale(t2, c2)));
    const float2 m2 = cadd(a0, cadd(cscale(t1, c2), cscale(t2, c1)));
    const float2 n1 = mul_j<INV>(cadd(cscale(t3, s1), cscale(t4, s2)));
    const float2 n2 = mul_j<INV>(csub(cscale(t3, s2), cscale(t4, s1)));
    a0 = cadd(a0, cadd(t1, t2));
    a1 = cadd(m1, n1);
    a4 = csub(m1, n1);
    a2 = cadd(m2, n2);
    a3 = csub(m2, n2);
}

template <bool INV>
__device__ __forceinline__ void dft2(float2 &a0, float2 &a1) {
    const float2 t = a0;
    a0 = cadd(t, a1);
    a1 = csub(t, a1);
}

// a * exp(s i pi n / 8) for the constants (c, sn) = (cos, sin)(pi n / 8)
template <bool INV>
__device__ __forceinline__ float2 rot(float2 a, float c, float sn) {
    return cmul(a, make_float2(c, INV ? sn : -sn));
}

template <int R, bool INV>
__device__ __forceinline__ void dft(float2 (&v)[R]) {
    if constexpr (R == 2) {
        dft2<INV>(v[0], v[1]);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
        float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
        dft4<INV>(e0, e1, e2, e3);
        dft4<INV>(o0, o1, o2, o3);
        const float h = 0.70710678118654752f;
        const float2 w1 = cscale(cadd(o1, mul_j<INV>(o1)), h);   // exp(s i pi/4) o1
        const float2 w2 = mul_j<INV>(o2);                        // exp(s i pi/2) o2
        const float2 w3 = cscale(csub(mul_j<INV>(o3), o3), h);   // exp(s 3i pi/4) o3
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, w1);
        v[5] = csub(e1, w1);
        v[2] = cadd(e2, w2);
        v[6] = csub(e2, w2);
        v[3] = cadd(e3, w3);
        v[7] = csub(e3, w3);
    } else if constexpr (R == 3) {
        dft3<INV>(v[0], v[1], v[2]);
    } else if constexpr (R == 5) {
        dft5<INV>(v[0], v[1], v[2], v[3], v[4]);
    } else if constexpr (R == 6) {  // 2 x 3 without twiddles: n = 3 a + 2 b, k = 3 a + 4 b (mod 6)
        float2 e0 = v[0], e1 = v[2], e2 = v[4], o0 = v[3], o1 = v[5], o2 = v[1];
        dft3<INV>(e0, e1, e2);
        dft3<INV>(o0, o1, o2);
        v[0] = cadd(e0, o0);
        v[3] = csub(e0, o0);
        v[4] = cadd(e1, o1);
        v[1] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[5] = csub(e2, o2);
    } else if constexpr (R == 10) {  // 2 x 5 without twiddles: n = 5 a + 2 b, k = 5 a + 6 b (mod 10)
        float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], e4 = v[8];
        float2 o0 = v[5], o1 = v[7], o2 = v[9], o3 = v[1], o4 = v[3];
        dft5<INV>(e0, e1, e2, e3, e4);
        dft5<INV>(o0, o1, o2, o3, o4);
        v[0] = cadd(e0, o0);
        v[5] = csub(e0, o0);
        v[6] = cadd(e1, o1);
        v[1] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[7] = csub(e2, o2);
        v[8] = cadd(e3, o3);
        v[3] = csub(e3, o3);
        v[4] = cadd(e4, o4);
        v[9] = csub(e4, o4);
    } else if constexpr (R == 16) {  // 4 x 4: n = 4 a + b, k = c + 4 d
        const float c1 = 0.92387953251128674f, s1 = 0.38268343236508977f, h = 0.70710678118654752f;
#pragma unroll
        for (int b = 0; b < 4; ++b) dft4<INV>(v[b], v[4 + b], v[8 + b], v[12 + b]);  // v[4 c + b]
        v[5] = rot<INV>(v[5], c1, s1);
        v[6] = rot<INV>(v[6], h, h);
        v[7] = rot<INV>(v[7], s1, c1);
        v[9] = rot<INV>(v[9], h, h);
        v[10] = mul_j<INV>(v[10]);
        v[11] = rot<INV>(v[11], -h, h);
        v[13] = rot<INV>(v[13], s1, c1);
        v[14] = rot<INV>(v[14], -h, h);
        v[15] = rot<INV>(v[15], -c1, -s1);
#pragma unroll
        for (int c = 0; c < 4; ++c) dft4<INV>(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);  // v[4 c + d]
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int d = c + 1; d < 4; ++d) {  // to v[c + 4 d]
                const float2 t = v[4 * c + d];
                v[4 * c + d] = v[4 * d + c];
                v[4 * d + c] = t;
            }
    }
}

// Stockham passes P.. of NL length-L lines held by one wave. Pass P, radix R,
// NS = product of the earlier radices: butterfly j < L/R of a line reads
// elements j + r L/R, multiplies element r by W_{NS R}^{r (j mod NS)}, runs the
// R-point DFT and stores element r at (j / NS) NS R + (j mod NS) + r NS. Pass 0
// reads line l through src(l, i), the last pass writes through dst(l, i, v),
// the others use buf + l * pitch (the wave's LDS lines of fft_line(L) float2,
// addressed through lds_at; src / dst may address them too, unpadded).
// Passes of at most 32 butterflies a line take several lines side by side, S
// lanes each (one line alone leaves 32 of 64 lanes idle at L = 256, radix 8):
// a lane has the same butterfly in every line, so its twiddles are shared.
// (Dealing the butterflies of all lines to the lanes without gaps, with its
// divisions and twiddles per item, was slower: 240 and 320 by 8%.)
template <int L, int NL, int P, int NS, bool INV, class Src, class Dst>
__device__ __forceinline__ void fft_passes(int lane, const float2 *__restrict__ tw, float2 *buf, int pitch, Src &src,
                                           Dst &dst) {
    constexpr int NP = fft_npass<L>();
    constexpr int R = fft_radix_at<L, P>();
    constexpr int M = L / R;
    constexpr int S = M > 32 ? kWave : M > 16 ? 32 : M > 8 ? 16 : M > 4 ? 8 : M > 2 ? 4 : M;
    constexpr int G = kWave / S;                 // lines side by side
    constexpr int QJ = (M + kWave - 1) / kWave;  // steps per line (G = 1)
    constexpr int Q = G > 1 ? (NL + G - 1) / G : NL * QJ;
    constexpr int TS = L / (NS * R);  // twiddle table stride
    float2 v[Q][R];
    auto line_of = [&](int q) { return G > 1 ? lane / S + q * G : q / QJ; };
    auto fly_of = [&](int q) { return G > 1 ? lane % S : lane + q % QJ * kWave; };
    auto idle = [&](int q) {
        return (M % S != 0 && fly_of(q) >= M) || (G > 1 && NL % G != 0 && line_of(q) >= NL);
    };
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (idle(q)) continue;
        const int l = line_of(q), j = fly_of(q);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (P == 0)
                v[q][r] = src(l, j + r * M);
            else
                v[q][r] = buf[l * pitch + lds_at<L>(j + r * M)];
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (idle(q)) continue;
        if constexpr (NS > 1) {
            const int k = fly_of(q) % NS;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                float2 w = tw[r * k * TS];
                if (INV) w.y = -w.y;
                v[q][r] = cmul(v[q][r], w);
            }
        }
        dft<R, INV>(v[q]);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (idle(q)) continue;
        const int l = line_of(q), j = fly_of(q);
        const int k = j % NS;
        const int d = (j / NS) * NS * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (P == NP - 1)
                dst(l, d + r * NS, v[q][r]);
            else
                buf[l * pitch + lds_at<L>(d + r * NS)] = v[q][r];
        }
    }
    if constexpr (P + 1 < NP) fft_passes<L, NL, P + 1, NS * R, INV>(lane, tw, buf, pitch, src, dst);
}

template <int L, int NL, bool INV, class Src, class Dst>
__device__ __forceinline__ void fft_lines(int lane, const float2 *__restrict__ tw, float2 *buf, int pitch, Src src,
                                          Dst dst) {
    fft_passes<L, NL, 0, 1, INV>(lane, tw, buf, pitch, src, dst);
}

// data index of pixel-space position i of an axis: kept iff (i + N/2) mod L < N
__device__ __forceinline__ bool kept(int i, int N, int L) {
    int m = i + N / 2;
    if (m >= L) m -= L;
    return m < N;
}

// Rows per wave, transformed together (independent loads in flight, shared
// twiddles): four up to L = 256, two up to 512, one above, where the LDS lines
// would cost occupancy (on 256^3 and 192^3 grids four rows cut the 3D stages by
// 3-5%, while four rows of 512 or eight of 256 were slower).
constexpr int rows_per_wave(int L) { return L <= 256 ? 4 : L <= 512 ? 2 : 1; }

// Block of C adjacent image columns of one image, dealt to the XCDs in
// contiguous ranges (neighbouring column groups share cache lines).
__device__ __forceinline__ bool column_block(int64_t nimg, int Nx, int C, int64_t &b, int &mx0) {
    const int ngrp = (Nx + C - 1) / C;
    const int64_t nblk = nimg * ngrp;
    const int64_t per = (nblk + kXcds - 1) / kXcds;
    const int64_t blk = (int64_t)(blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (blk >= nblk) return false;
    b = blk / ngrp;
    mx0 = (int)(blk - b * ngrp) * C;
    return true;
}

// Columns per column-stage workgroup. The strided row segments, not the
// transform, bound these stages; still, wider tiles (16 columns at L = 512,
// 66 KiB of LDS, two workgroups per CU) measured slower than 8 columns at
// four workgroups per CU.
constexpr int col_group(int L) { return L <= 256 ? 16 : L <= 512 ? 8 : 4; }
constexpr size_t col_lds_bytes(int L) {
    return sizeof(float2) * (size_t)col_group(L) * (fft_line(L) + fft_pad(col_group(L)));
}

inline unsigned col_blocks(int64_t nimg, int Nx, int C) {
    const int64_t n = nimg * ((Nx + C - 1) / C);
    return (unsigned)((n + kXcds - 1) / kXcds * kXcds);
}

inline unsigned row_blocks(int64_t nlines, int L) {
    const int64_t rpb = (int64_t)rows_per_wave(L) * (kBlock / kWave);
    return (unsigned)((nlines + rpb - 1) / rpb);
}

}  // namespace
}  // namespace tn
