// The advection term's x-part (advection3d, operators.F:9-276) for any x grid of 2, 3 and 5: the
// three inverse transforms, the six products and the six forward transforms of every (y, z) line
// in one kernel, with no physical field in memory (fourx with fill, fourier.F:1-115; mult.F;
// pack_fftw with 1/mgalx).
//
// What bounds it: the nine fields of M modes per line cross HBM once, 9 x 16 B x M per line, and
// everything else happens in registers and LDS.
//
// Two neighbouring lines share a complex transform, for each of u, v, w and each product, so a line costs 1.5
// inverse and 3 forward complex transforms of X points.  (Sharing it between u and v of a line, and between uu
// and vv, leaves the rounding of the larger in the smaller: at 384 x 128 x 257^2 the v and w components of a
// duct flow's advection were 7.9e-15 and 6.4e-15 off, now 5.3e-15 and 5.4e-15; with rocFFT's transforms of one
// real line each 5.6e-15 and 5.5e-15.  A value that is not finite spreads to both lines.)  A transform is a
// Stockham sequence of passes of radix 2, 3, 4, 5 or 8 through one LDS image per line: a workgroup reads all
// its butterflies into registers, waits, and writes them back, so one image is enough.  The inverse's last
// pass and the forward's first have the same radix R (4, 6 or 10): a butterfly's outputs x = j + i X/R of the
// one are its inputs of the other, so the physical values u, v, w and their products never leave the registers
// of the thread that owns butterfly j of a pair of lines.
//
// A workgroup owns T consecutive lines (of the plane's m^2, y fastest): for each mode a run of
// 16 T bytes, read and written by consecutive lanes.  Lines are padded by one complex value in
// eight, which keeps the strided writes of radix 4 and 8 off each other's banks; the line stride
// is odd.  Consecutive workgroups of one XCD own neighbouring tiles, so the cache lines that two
// tiles share are fetched into one L2.
//
// Measured (the 9 fields' bytes over the launch): 615 us at 384 points x 128 modes x 257^2 lines
// (2.0 TB/s; rocFFT's batched transforms with pad, multiply and pack kernels, which this replaces,
// took 5690 us), 44 us at 120 x 40 x 97^2 (257 us), 72 us at 144 x 48 x 129^2 (the dense transform
// of k_xprod: 129 us).  Counters at 384 points: the vector units issue a third of the time, LDS is
// busy a third; the rest is waits at the barriers between passes.  The roots of unity are read from
// LDS, not from memory: gathers of 16 bytes per lane through the L1 cost 1.2 times as much.
#include <algorithm>
#include <cmath>
#include <functional>

#include "advect.h"

namespace duct {

namespace {

__device__ __forceinline__ d2v cmul(d2v a, d2v b) { return d2v{a[0] * b[0] - a[1] * b[1], a[0] * b[1] + a[1] * b[0]}; }
// times e^(+i phi) (inverse) or e^(-i phi) (forward), w = (cos phi, sin phi)
template <bool INV>
__device__ __forceinline__ d2v twid(d2v a, d2v w)
{
    return INV ? cmul(a, w) : d2v{a[0] * w[0] + a[1] * w[1], a[1] * w[0] - a[0] * w[1]};
}
// times +i (inverse) or -i (forward)
template <bool INV>
__device__ __forceinline__ d2v rot(d2v a) { return INV ? d2v{-a[1], a[0]} : d2v{a[1], -a[0]}; }

template <bool INV>
__device__ __forceinline__ void dft3(d2v& a, d2v& b, d2v& c)
{
    constexpr double s = 0.86602540378443864676;
    const d2v t1 = b + c, t2 = a - 0.5 * t1, t3 = s * rot<INV>(b - c);
    a = a + t1;
    b = t2 + t3;
    c = t2 - t3;
}

template <bool INV>
__device__ __forceinline__ void dft4(d2v& a, d2v& b, d2v& c, d2v& d)
{
    const d2v t0 = a + c, t1 = a - c, t2 = b + d, t3 = rot<INV>(b - d);
    a = t0 + t2;
    b = t1 + t3;
    c = t0 - t2;
    d = t1 - t3;
}

template <bool INV>
__device__ __forceinline__ void dft5(d2v& a, d2v& b, d2v& c, d2v& d, d2v& e)
{
    constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    const d2v p1 = b + e, p2 = c + d, m1 = rot<INV>(b - e), m2 = rot<INV>(c - d);
    const d2v x1 = a + c1 * p1 + c2 * p2, x2 = a + c2 * p1 + c1 * p2;
    const d2v y1 = s1 * m1 + s2 * m2, y2 = s2 * m1 - s1 * m2;
    a = a + p1 + p2;
    b = x1 + y1;
    e = x1 - y1;
    c = x2 + y2;
    d = x2 - y2;
}

// v[k] <- sum_i v[i] e^(+-2 pi i k / R), natural order
template <int R, bool INV>
__device__ __forceinline__ void dft(d2v (&v)[R])
{
    if constexpr (R == 2) {
        const d2v t = v[0] - v[1];
        v[0] = v[0] + v[1];
        v[1] = t;
    } else if constexpr (R == 3) {
        dft3<INV>(v[0], v[1], v[2]);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 5) {
        dft5<INV>(v[0], v[1], v[2], v[3], v[4]);
    } else {   // even R: the transforms of the even and odd inputs, joined with the R-th roots
        constexpr int H = R / 2;
        d2v e[H], o[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            e[i] = v[2 * i];
            o[i] = v[2 * i + 1];
        }
        dft<H, INV>(e);
        dft<H, INV>(o);
        if constexpr (R == 6) {
            constexpr double s = 0.86602540378443864676;
            o[1] = twid<INV>(o[1], d2v{0.5, s});
            o[2] = twid<INV>(o[2], d2v{-0.5, s});
        } else if constexpr (R == 8) {
            constexpr double s = 0.70710678118654752440;
            o[1] = s * (o[1] + rot<INV>(o[1]));
            o[2] = rot<INV>(o[2]);
            o[3] = s * (rot<INV>(o[3]) - o[3]);
        } else {
            static_assert(R == 10, "radix");
            constexpr double c1 = 0.80901699437494742410, s1 = 0.58778525229247312917;
            constexpr double c2 = 0.30901699437494742410, s2 = 0.95105651629515357212;
            o[1] = twid<INV>(o[1], d2v{c1, s1});
            o[2] = twid<INV>(o[2], d2v{c2, s2});
            o[3] = twid<INV>(o[3], d2v{-c2, s2});
            o[4] = twid<INV>(o[4], d2v{-c1, s1});
        }
#pragma unroll
        for (int i = 0; i < H; ++i) {
            v[i] = e[i] + o[i];
            v[i + H] = e[i] - o[i];
        }
    }
}

__device__ __forceinline__ int pad8(int x) { return x + (x >> 3); }
// e / d for 0 <= e < 2^13 and inv = 1 / d (exact: the quotient's distance to an integer is >= 1 / (2 d))
__device__ __forceinline__ int div_by(int e, float inv) { return (int)(((float)e + 0.5f) * inv); }

// One Stockham pass of radix r over nl lines, in place.
template <int PT, int r, bool INV>
__device__ __forceinline__ void pass_r(d2v* Z, const XfftPass& p, const d2v* tw, int nl, int ld, int tid,
                                       int nth)
{
    constexpr int MB = (PT + r - 1) / r;   // butterflies per thread
    const int total = nl * p.nb;
    asm volatile("" : "+v"(tid));   // keeps this pass's addresses out of the registers of the others
    d2v v[MB][r];
    int dst[MB];
#pragma unroll
    for (int s = 0; s < MB; ++s) {
        const int e = tid + s * nth;
        if (e < total) {
            const int l = div_by(e, p.inv_nb), j = e - l * p.nb;
            const int k = j - p.ns * div_by(j, p.inv_ns), t = k * p.tw;
            const d2v* src = Z + l * ld;
#pragma unroll
            for (int i = 0; i < r; ++i) v[s][i] = src[pad8(j + i * p.nb)];
            if (p.ns > 1) {
#pragma unroll
                for (int i = 1; i < r; ++i) v[s][i] = twid<INV>(v[s][i], tw[pad8(t * i)]);
            }
            dft<r, INV>(v[s]);
            dst[s] = (j - k) * r + k;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < MB; ++s) {
        const int e = tid + s * nth;
        if (e < total) {
            d2v* out = Z + div_by(e, p.inv_nb) * ld;
#pragma unroll
            for (int i = 0; i < r; ++i) out[pad8(dst[s] + i * p.ns)] = v[s][i];
        }
    }
    lds_barrier();
}

template <int PT, bool INV>
__device__ __forceinline__ void run_pass(d2v* Z, const XfftPass& p, const d2v* tw, int nl, int ld, int tid,
                                         int nth)
{
    switch (p.r) {
        case 2: pass_r<PT, 2, INV>(Z, p, tw, nl, ld, tid, nth); break;
        case 3: pass_r<PT, 3, INV>(Z, p, tw, nl, ld, tid, nth); break;
        case 4: pass_r<PT, 4, INV>(Z, p, tw, nl, ld, tid, nth); break;
        case 5: pass_r<PT, 5, INV>(Z, p, tw, nl, ld, tid, nth); break;
        default: pass_r<PT, 8, INV>(Z, p, tw, nl, ld, tid, nth); break;
    }
}

}  // namespace

template <int R>
__global__ __launch_bounds__(kXfftMaxThreads, R == 4 ? 3 : 2) void k_xprod_fft(XprodFftArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    d2v* Z = (d2v*)smem_raw;                   // T lines of stride ld, then the X roots of unity
    d2v* tw = Z + a.T * a.ld;
    const int X = a.X, M = a.M, T = a.T, ld = a.ld, nf = X / R;
    const int tid = threadIdx.x, nth = blockDim.x;
    // tiles in 8 runs, one per XCD (workgroups go to the XCDs in turn)
    const long per = (a.tiles + 7) / 8, tile = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((long)(blockIdx.x >> 3) >= per || tile >= a.tiles) return;
    const long L0 = tile * T;
    const long nlines = a.lines - L0;          // valid lines of this tile (>= 1)

    // a thread's coefficients: mode k of the pair of lines 2 p and 2 p + 1
    constexpr int PT = xfft_per_thread(R), IT = (PT + 5) / 6;   // 3 M <= X: at most X / 3 coefficients per line
    d2v cu[IT][2], cv[IT][2], cw[IT][2];
    const int hT = T >> 1;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = tid + it * nth, p = e & (hT - 1), k = e >> (a.logT - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool ok = k < M && 2 * p + h < nlines;
            const size_t idx = ok ? (size_t)k * a.lines + L0 + 2 * p + h : 0;
            cu[it][h] = a.in[0][idx];
            cv[it][h] = a.in[1][idx];
            cw[it][h] = a.in[2][idx];
            if (!ok) cu[it][h] = cv[it][h] = cw[it][h] = d2v{0.0, 0.0};
        }
    }
    auto clear = [&](int nl) {                 // the modes that the 3/2 rule leaves empty
        const int nz = X - 2 * M + 1;
        for (int e = tid; e < nl * nz; e += nth) {
            const int l = div_by(e, a.inv_nz);
            Z[l * ld + pad8(M + e - l * nz)] = d2v{0.0, 0.0};
        }
    };

    for (int e = tid; e < X; e += nth) tw[pad8(e)] = a.tw[e];
    // ---- u and v of two lines at a time: line 2 p + i line (2 p + 1)
    auto pack = [&](d2v* z, const d2v (&c)[2], int k) {
        const d2v x = c[0], y = c[1];
        if (k == 0) {
            z[0] = d2v{x[0], y[0]};   // FFTW's c2r ignores Im of mode 0
        } else {
            z[pad8(k)] = d2v{x[0] - y[1], x[1] + y[0]};
            z[pad8(X - k)] = d2v{x[0] + y[1], y[0] - x[1]};
        }
    };
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = tid + it * nth, p = e & (hT - 1), k = e >> (a.logT - 1);
        if (k < M) {
            pack(Z + 2 * p * ld, cu[it], k);
            pack(Z + (2 * p + 1) * ld, cv[it], k);
        }
    }
    clear(T);
    lds_barrier();
    for (int i = 0; i < a.ninv; ++i) run_pass<PT, true>(Z, a.inv[i], tw, T, ld, tid, nth);

    // ---- the last inverse pass: butterfly j of the pair of lines 2 pr and 2 pr + 1
    const bool own = tid < (T >> 1) * nf;
    const int pr = own ? div_by(tid, a.inv_nf) : 0, j = own ? tid - pr * nf : 0;
    d2v uu[R], vv[R], ww[R];                   // u, v, w of the pair: (line 2 pr, line 2 pr + 1)
    auto last = [&](const d2v* src, d2v (&v)[R]) {
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = src[pad8(j + i * nf)];
#pragma unroll
        for (int i = 1; i < R; ++i) v[i] = twid<true>(v[i], tw[pad8(j * i)]);
        dft<R, true>(v);
    };
    if (own) {
        last(Z + (2 * pr) * ld, uu);
        last(Z + (2 * pr + 1) * ld, vv);
    }
    lds_barrier();

    // ---- w
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = tid + it * nth, p = e & (hT - 1), k = e >> (a.logT - 1);
        if (k < M) pack(Z + p * ld, cw[it], k);
    }
    clear(T >> 1);
    lds_barrier();
    for (int i = 0; i < a.ninv; ++i) run_pass<PT, true>(Z, a.inv[i], tw, T >> 1, ld, tid, nth);
    if (own) last(Z + pr * ld, ww);

    // ---- the products of the pair, one per complex transform: uu and vv, ww and uv, uw and vw
    for (int q = 0; q < 3; ++q) {
        // (opaque per round: the addresses of a round are cheap to form and would otherwise all be
        // kept in registers across the rounds)
        int tq = tid, jq = j, pq = pr;
        asm volatile("" : "+v"(tq), "+v"(jq), "+v"(pq));
        lds_barrier();
        if (own) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                d2v z[R];
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const d2v f = q == 0 ? (h ? vv[i] : uu[i]) : q == 1 ? (h ? uu[i] : ww[i]) : (h ? vv[i] : uu[i]);
                    z[i] = f * (q == 0 ? f : q == 1 ? (h ? vv[i] : ww[i]) : ww[i]);
                }
                dft<R, false>(z);
                d2v* out = Z + (2 * pq + h) * ld;
#pragma unroll
                for (int i = 0; i < R; ++i) out[pad8(jq * R + i)] = z[i];
            }
        }
        lds_barrier();
        for (int i = 0; i < a.nfwd; ++i) run_pass<PT, false>(Z, a.fwd[i], tw, T, ld, tq, nth);
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int e = tq + it * nth, p = e & (hT - 1), k = e >> (a.logT - 1);
            if (k >= M) continue;
            const size_t idx = (size_t)k * a.lines + L0 + 2 * p;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const d2v* z = Z + (2 * p + h) * ld;
                const d2v f = z[pad8(k)], g = z[pad8(k ? X - k : 0)];
                if (2 * p < nlines) a.out[2 * q + h][idx] = a.scale * d2v{f[0] + g[0], f[1] - g[1]};
                if (2 * p + 1 < nlines) a.out[2 * q + h][idx + 1] = a.scale * d2v{f[1] + g[1], g[0] - f[0]};
            }
        }
    }
}

// Radix sequence of an X-point transform around the fused radix R; false if X has another factor.
static bool xfft_plan(int X, int R, std::vector<int>& mids)
{
    mids.clear();
    int rest = X / R, twos = 0;
    if (X % R) return false;
    while (rest % 2 == 0) { rest /= 2; ++twos; }
    while (rest % 3 == 0) { rest /= 3; mids.push_back(3); }
    while (rest % 5 == 0) { rest /= 5; mids.push_back(5); }
    if (rest != 1) return false;
    // 2^twos as few passes as possible: 8s, then 4s for the remainder
    while (twos > 0) {
        const int b = twos == 4 || twos == 2 ? 2 : twos >= 3 ? 3 : 1;
        mids.push_back(1 << b);
        twos -= b;
    }
    std::sort(mids.begin(), mids.end(), std::greater<int>());
    return (int)mids.size() <= kXfftMaxPasses;
}

// The fused radix: 4 before 6 before 10, for the registers that its u, v and w take (48, 72 and
// 120; 3 waves per SIMD against 2).  Every even X of factors 2, 3 and 5 from 4 up has one.
static int xfft_radix(int X)
{
    std::vector<int> mids;
    for (int R : {4, 6, 10})
        if (xfft_plan(X, R, mids)) return R;
    return 0;
}

bool xprod_fft_supported(int M, int X)
{
    return M >= 1 && 3 * M <= X && X % 2 == 0 && X >= 4 && X <= kXfftMaxX && xfft_radix(X) != 0;
}

void build_xfft_table(int X, std::vector<double>& tab)
{
    tab.resize((size_t)2 * X);
    const long double tp = 2.0L * 3.14159265358979323846264338327950288L / (long double)X;
    for (int n = 0; n < X; ++n) {
        tab[2 * n] = (double)std::cos(tp * n);
        tab[2 * n + 1] = (double)std::sin(tp * n);
    }
}

hipError_t launch_xprod_fft(const XprodArgs& x, const d2v* tw, hipStream_t st)
{
    const int X = x.X, M = x.M;
    if (!xprod_fft_supported(M, X) || x.m <= 0 || !tw) return hipErrorInvalidValue;
    const int R = xfft_radix(X), nf = X / R;
    std::vector<int> mids;
    xfft_plan(X, R, mids);
    XprodFftArgs a{};
    for (int i = 0; i < 3; ++i) a.in[i] = x.in[i];
    for (int i = 0; i < 6; ++i) a.out[i] = x.out[i];
    a.tw = tw;
    a.lines = (long)x.m * x.m;
    a.M = M;
    a.X = X;
    a.scale = 0.5 / (double)X;
    a.inv_nf = 1.0f / (float)nf;
    a.inv_nz = 1.0f / (float)(X - 2 * M + 1);
    auto fill = [&](XfftPass* p, int ns0) {
        int ns = ns0;
        for (size_t i = 0; i < mids.size(); ++i) {
            const int r = mids[i];
            p[i].r = r;
            p[i].ns = ns;
            p[i].nb = X / r;
            p[i].tw = X / (ns * r);
            p[i].inv_nb = 1.0f / (float)p[i].nb;
            p[i].inv_ns = 1.0f / (float)ns;
            ns *= r;
        }
    };
    fill(a.inv, 1);
    fill(a.fwd, R);
    a.ninv = a.nfwd = (int)mids.size();
    a.ld = (X + (X >> 3) + 1) | 1;
    auto threads = [&](int T) {
        const int pt = xfft_per_thread(R), need = std::max((T / 2) * nf, (T * X + pt - 1) / pt);
        return (need + 63) / 64 * 64;
    };
    // Lines per workgroup: 8 (128 bytes of a mode per access) while 256 threads hold them (more
    // threads wait longer at each barrier: 8 lines took 1.8 times as long as 4 at 384 x 257^2), 4
    // where 8 leave fewer than two workgroups per CU (16.8 against 14.0 us at 48 x 33^2).
    int T = 2, logT = 1;
    while (T < 8 && threads(T * 2) <= 256 && !(T == 4 && a.lines < 8 * 512)) { T *= 2; ++logT; }
    a.T = T;
    a.logT = logT;
    a.tiles = (a.lines + T - 1) / T;
    const int nth = threads(T);
    const size_t lds = ((size_t)T * a.ld + X + X / 8 + 1) * sizeof(d2v);
    const dim3 grid((unsigned)((a.tiles + 7) / 8 * 8)), block(nth);
    if (R == 6) hipLaunchKernelGGL(k_xprod_fft<6>, grid, block, lds, st, a);
    else if (R == 4) hipLaunchKernelGGL(k_xprod_fft<4>, grid, block, lds, st, a);
    else hipLaunchKernelGGL(k_xprod_fft<10>, grid, block, lds, st, a);
    return hipGetLastError();
}

}  // namespace duct
