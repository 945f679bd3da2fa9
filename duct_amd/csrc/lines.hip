// Sums of derivative products along y or z with their pointwise terms, for every plane of a field:
//   y:  out(y, z) = sum_p c_p sum_k A_p(y, k) u_p(k, z) + pointwise terms
//   z:  out(y, z) = sum_p c_p sum_k A_p(z, k) u_p(y, k) + pointwise terms
// (derivyz / transyz applied along y or z, chebyshev.f90:1-540, as dense products with the matrices
// of the m CGL nodes; derivx, fourier.F:117-188, and the elementwise parts of the Runge-Kutta
// substep, main1.f90:384-655, as the pointwise terms).  One launch of each direction forms all the
// derivative sums of a step of the algorithm: the right-hand sides, the divergence, the update.
//
// Folding: A commutes with the reflection J of the nodes up to a sign, so with u split along the
// contraction into ue(k) = (u(k) + u(m-1-k)) / 2 and uo(k) = (u(k) - u(m-1-k)) / 2 a product is two
// half-size ones, Dp ue and Dm uo, and the sums are kept as their even and odd parts E and O:
// out(r) = E + O, out(m-1-r) = E - O.  An even matrix adds Dp ue to E and Dm uo to O, an odd one the
// other way round.  The centre row of odd m is one dot product per line on the vector units: as a
// 17th row it would cost a whole MFMA row tile (he = 65 rows at m = 129: 5 tiles for 4).
//
// Work decomposition: a workgroup owns 16 consecutive lines of the flattened (mode, line) index
// (the planes of odd m would waste most of a tile each) of one job and has one wave per 16 folded
// rows: a wave computes one tile of E and of O, re and im, so four accumulators, 122 registers, and
// 16 waves on a CU that hide each other's loads.  (With the next product's lines loaded under the
// present one's MFMAs, 158 registers and 12 waves: the same times to 2%.)
//
// What bounds it: HBM at the sizes whose fields do not stay in the 256 MB last-level cache.  The y
// and z launches of a substep's right-hand sides at 129^2 x 64 modes read and write 20 fields' worth
// of 17 MB each (the y launch's sums go through memory to the z launch) in 87 and 95 us, 3.6-3.8
// TB/s where a copy reaches 4.4-5.1; at 257^2 x 128 modes 816 and 878 us, 3.2 TB/s with the MFMAs
// busy half the time.  All derivative and elementwise work of an RK3 step took 1537 us at 129^2 x 64
// as nine launches per substep and takes 888 us as six; at 257^2 x 128, 12800 and 7800 us.
#include <algorithm>
#include <type_traits>

#include "lines.h"

namespace duct {

namespace {
constexpr int kLIT = 4;                          // mirrored pairs of points per thread and product

__device__ __forceinline__ d4v mfma(double a, double b, d4v c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
}  // namespace

template <bool DIRZ>
__global__ __launch_bounds__(576, 4) void k_lines(LinesArgs a, int nslab)
{
    extern __shared__ __attribute__((aligned(16))) double slab[];   // [ue re, uo re, ue im, uo im][line][k]
    const int m = a.m, he = (m + 1) / 2, ho = m / 2, KH = (he + 15) / 16 * 16;
    const int KPE = (he + 7) / 8, KPO = (ho + 7) / 8;               // fragment pairs (8 k) of the two parts
    const int LDK = 8 * KPE + 1, SL = 16 * LDK;
    const int nth = blockDim.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    // slabs in 8 runs, one per XCD; the jobs of a slab are neighbours (they share inputs)
    const int total = nslab * a.njobs, per = (total + 7) / 8;
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || id >= total) return;
    const LineJob& job = a.job[id % a.njobs];
    {   // touch the job's arguments at once: their first reads miss the scalar cache one after the other
        // otherwise, which is most of a small launch's time
        constexpr int NW = (sizeof(LineJob) + 63) / 64;
        const int* w = (const int*)&job;
        int t[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) t[i] = w[i * 16];
#pragma unroll
        for (int i = 0; i < NW; ++i) asm volatile("" : : "s"(t[i]));
    }
    const int L0 = id / a.njobs * 16;                               // first line
    const int nlines = min(16, a.nmodes * m - L0);
    double* red = slab + 4 * SL;                                    // [wave][line][re, im]

    // element offsets of a line's first point and between its points; y: line (mode, z), z: (mode, y)
    const size_t mm = (size_t)m * m;
    const int mode_first = L0 / m;
    const size_t base0 = (size_t)mode_first * mm;
    const int lrel0 = L0 - mode_first * m;
    const float invm = 1.0f / (float)m;
    auto line_off = [&](int l) -> unsigned {                        // relative to base0
        const int r = lrel0 + l;
        if constexpr (!DIRZ) return (unsigned)r * m;                // lines of consecutive planes follow each other
        const int dm = (int)(((float)r + 0.5f) * invm);             // r < m + 16
        return (unsigned)dm * (unsigned)mm + (r - dm * m);
    };
    const unsigned sk = DIRZ ? m : 1;

    // staging: the thread's mirrored pairs (line, k), k < ho (formed anew for each product: kept, their
    // offsets would cost the registers of the fourth wave per SIMD)
    const float invh = 1.0f / (float)ho;
    auto pair_at = [&](int t, int it, int& l, int& k) -> bool {
        const int e = t + it * nth, q = (int)(((float)e + 0.5f) * invh);   // e < 16 * 144
        l = DIRZ ? e & 15 : q;
        k = DIRZ ? e >> 4 : e - q * ho;
        return e < 16 * ho;
    };
    const bool odd_m = he != ho;
    const bool cok = tid < nlines;                                  // the thread stages a centre point
    const unsigned oc = line_off(cok ? tid : 0) + ho * sk;

    for (int e = tid; e < 4 * SL; e += nth) slab[e] = 0.0;          // the padding past he and ho stays zero

    d2v va[kLIT], vb[kLIT], vc = {0.0, 0.0};
    auto load = [&](const d2v* src) {      // lines past the end read line 0 and count as zero
        const d2v* U = src + base0;
        int t = tid;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int it = 0; it < kLIT; ++it) {
            int l, k;
            if (!pair_at(t, it, l, k) || l >= nlines) l = k = 0;
            const unsigned o = line_off(l);
            va[it] = U[o + k * sk];
            vb[it] = U[o + (m - 1 - k) * sk];
        }
        if (odd_m) vc = U[oc];
    };
    auto store = [&]() {
        int t = tid;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int it = 0; it < kLIT; ++it) {
            int l, k;
            if (!pair_at(t, it, l, k)) continue;
            const double f = l < nlines ? 0.5 : 0.0;
            const d2v e = f * (va[it] + vb[it]), o = f * (va[it] - vb[it]);
            double* s = slab + l * LDK + k;
            s[0] = e[0];
            s[SL] = o[0];
            s[2 * SL] = e[1];
            s[3 * SL] = o[1];
        }
        if (odd_m && tid < 16) {
            const double f = cok ? 1.0 : 0.0;
            slab[tid * LDK + ho] = f * vc[0];
            slab[2 * SL + tid * LDK + ho] = f * vc[1];
        }
    };

    d4v ere = {0.0, 0.0, 0.0, 0.0}, eim = ere, ore = ere, oim = ere;   // E and O of the wave's row tile
    d2v ctr = {0.0, 0.0};                                              // this thread's share of the centre row
    int q = 0;
    // The accumulators hold the sums over `unit`, the last product's coef: coef on the matrix rounds every element
    // once more (p's median error over 24 steps of 97^2 x 40 modes 2.64e-13 with it, 2.54e-13 without; 129^2 x 64
    // 4.07e-13 and 4.00e-13; the time is the same to 0.7%).
    auto rescale = [&](double f) {
        ere *= f;
        eim *= f;
        ore *= f;
        oim *= f;
        ctr *= f;
    };
    for (int s = 0; s < job.nstage; ++s) {
        const LineStage& st = job.stage[s];
        double unit = 1.0;
        bool empty = s == 0 || job.stage[s - 1].keep == 0.0;
        if (empty) {   // (0 times the previous output is not zero where that is infinite)
            ere = eim = ore = oim = d4v{0.0, 0.0, 0.0, 0.0};
            ctr = d2v{0.0, 0.0};
        }
        for (int pi = 0; pi < st.nprod; ++pi, ++q) {
            const LineProd& p = job.prod[q];
            const bool odd = p.odd != 0;
            const d2v* Fp = (const d2v*)p.mat + (size_t)wave * (KH / 8) * 64 + lane;
            const d2v* Fm = Fp + (size_t)KH * KH / 2;
            d2v fp = Fp[0], fm = Fm[0];
            load(p.src);
            lds_barrier();                                        // the slab's last readers are done
            store();
            lds_barrier();
            if (p.coef == 0.0) continue;                          // (1 / aspect at its limit) nothing to add
            if (!empty) rescale(unit / p.coef);
            unit = p.coef;
            empty = false;
            if (odd) {
                d4v t = ere; ere = ore; ore = t;
                t = eim; eim = oim; oim = t;
            }
            // one pair of k-steps of 4: ue against Dp and uo against Dm, the next pair's fragments in flight
            const double* S0 = slab + l16 * LDK + l4;
            auto pair = [&](int kp, const d2v& cp, const d2v& cm, d2v& np, d2v& nm) {
                const int kn = kp + 1 < KPE ? kp + 1 : kp;
                np = Fp[(size_t)kn * 64];
                nm = Fm[(size_t)kn * 64];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const double* S = S0 + (2 * kp + h) * 4;
                    const double er = S[0], orr = S[SL], ei = S[2 * SL], oi = S[3 * SL];
                    const double dp = cp[h], dm = cm[h];
                    if constexpr (!DIRZ) {
                        ere = mfma(er, dp, ere);
                        eim = mfma(ei, dp, eim);
                        ore = mfma(orr, dm, ore);
                        oim = mfma(oi, dm, oim);
                    } else {
                        ere = mfma(dp, er, ere);
                        eim = mfma(dp, ei, eim);
                        ore = mfma(dm, orr, ore);
                        oim = mfma(dm, oi, oim);
                    }
                }
            };
            d2v gp, gm;
            int kp = 0;
            for (; kp + 1 < KPO; kp += 2) {
                pair(kp, fp, fm, gp, gm);
                pair(kp + 1, gp, gm, fp, fm);
            }
            if (kp < KPO) {
                pair(kp, fp, fm, gp, gm);
                fp = gp;
            }
            if (KPE > KPO) {                                        // the even part's last pair (he = ho + 1)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const double* S = S0 + (2 * KPO + h) * 4;
                    const double er = S[0], ei = S[2 * SL];
                    const double dp = fp[h];
                    if constexpr (!DIRZ) {
                        ere = mfma(er, dp, ere);
                        eim = mfma(ei, dp, eim);
                    } else {
                        ere = mfma(dp, er, ere);
                        eim = mfma(dp, ei, eim);
                    }
                }
            }
            if (odd) {
                d4v t = ere; ere = ore; ore = t;
                t = eim; eim = oim; oim = t;
            }
            if (odd_m) {   // centre row: D2's from ue, D's from uo; k = seg, seg + nth / 16, ...
                const double* C = p.mat + (size_t)2 * KH * KH;
                const double* S = slab + (odd ? SL : 0) + l16 * LDK;
                for (int k = tid >> 4; k < he; k += nth >> 4) {
                    const double c = C[k];
                    ctr[0] += c * S[k];
                    ctr[1] += c * S[2 * SL + k];
                }
            }
        }
        if (st.nprod > 0) rescale(unit);

        // ---- the stage's output: products and terms.  Lane holds rows r (and m-1-r) of 4 lines (y) or
        // 4 rows of one line (z): D[i][j] in lane j + 16 (i % 4), element i / 4.
        if (odd_m) {
            // the previous stage's shares are read before any wave writes this one's: by the barriers of the
            // products between, or by one of its own where the stage has no product (the update's U[0] after U[2])
            if (st.nprod == 0) lds_barrier();
            const d2v c = {ctr[0] + __shfl_xor(ctr[0], 16, 64), ctr[1] + __shfl_xor(ctr[1], 16, 64)};
            const d2v w = {c[0] + __shfl_xor(c[0], 32, 64), c[1] + __shfl_xor(c[1], 32, 64)};
            if (l4 == 0) {
                red[(wave * 16 + l16) * 2] = w[0];
                red[(wave * 16 + l16) * 2 + 1] = w[1];
            }
            lds_barrier();
        }
        const bool has_c = odd_m && cok, self = st.self.cr != 0.0 || st.self.crx != 0.0 || st.self.ci != 0.0;
        d2v cv = {0.0, 0.0};
        if (has_c) {
            for (int w = 0; w < nth >> 6; ++w) cv += d2v{red[(w * 16 + tid) * 2], red[(w * 16 + tid) * 2 + 1]};
        }
        auto mode_of = [&](int l) { return a.mode0 + mode_first + (int)(((float)(lrel0 + l) + 0.5f) * invm); };
        const int mc = mode_of(l16);
        const double xc = a.alp * (double)mc;
        if (has_c) {
            for (int j = 0; j < st.nterm; ++j) {
                const LineTerm& t = st.term[j];
                const d2v y = t.t[base0 + oc];
                cv += (t.cr + t.crx * xc * xc) * y + t.ci * xc * d2v{-y[1], y[0]};
            }
            if (self) {
                const d2v y = {slab[tid * LDK + ho], slab[2 * SL + tid * LDK + ho]};
                cv += (st.self.cr + st.self.crx * xc * xc) * y + st.self.ci * xc * d2v{-y[1], y[0]};
            }
            if (mc == 0) cv[0] += st.c0;
            st.out[base0 + oc] = cv;
        }
        // (opaque: the addresses of the outputs are cheap to form and are not kept across the products)
        int q16 = l16, q4 = l4;
        asm volatile("" : "+v"(q16), "+v"(q4));
        // two of the lane's four rows at a time (the registers of all four do not fit 4 waves per SIMD)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            unsigned pa[2], pb[2];
            bool v[2];
            int md[2];
            d2v x1[2], x2[2];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int e = 2 * h + g, i = 4 * e + q4;
                const int r = 16 * wave + (DIRZ ? i : q16), l = DIRZ ? q16 : i;
                v[g] = r < ho && l < nlines;
                const unsigned o = line_off(v[g] ? l : 0), rr = v[g] ? r : 0;
                pa[g] = o + rr * sk;
                pb[g] = o + (m - 1 - rr) * sk;
                md[g] = mode_of(l);
                x1[g] = d2v{ere[e] + ore[e], eim[e] + oim[e]};
                x2[g] = d2v{ere[e] - ore[e], eim[e] - oim[e]};
            }
            for (int j = 0; j < st.nterm; ++j) {
                const LineTerm& t = st.term[j];
                const d2v* T = t.t + base0;
                d2v y1[2], y2[2];
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    y1[g] = T[pa[g]];
                    y2[g] = T[pb[g]];
                }
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const double xa = a.alp * (double)md[g], cr = t.cr + t.crx * xa * xa, ci = t.ci * xa;
                    x1[g] += cr * y1[g] + ci * d2v{-y1[g][1], y1[g][0]};
                    x2[g] += cr * y2[g] + ci * d2v{-y2[g][1], y2[g][0]};
                }
            }
            if (self) {   // the slab still holds the last product's operand
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const int i = 4 * (2 * h + g) + q4, r = 16 * wave + (DIRZ ? i : q16), l = DIRZ ? q16 : i;
                    const double* S = slab + l * LDK + (r < ho ? r : 0);
                    const d2v e = {S[0], S[2 * SL]}, o = {S[SL], S[3 * SL]};
                    const double xa = a.alp * (double)md[g], cr = st.self.cr + st.self.crx * xa * xa, ci = st.self.ci * xa;
                    const d2v y1 = e + o, y2 = e - o;
                    x1[g] += cr * y1 + ci * d2v{-y1[1], y1[0]};
                    x2[g] += cr * y2 + ci * d2v{-y2[1], y2[0]};
                }
            }
            d2v* O = st.out + base0;
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const double c0 = md[g] == 0 ? st.c0 : 0.0;
                x1[g][0] += c0;
                x2[g][0] += c0;
                if (v[g]) {
                    O[pa[g]] = x1[g];
                    O[pb[g]] = x2[g];
                }
                const int e = 2 * h + g;   // the next stage starts from keep times this output
                const d2v ev = (0.5 * st.keep) * (x1[g] + x2[g]), ov = (0.5 * st.keep) * (x1[g] - x2[g]);
                ere[e] = ev[0];
                eim[e] = ev[1];
                ore[e] = ov[0];
                oim[e] = ov[1];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        ctr = has_c ? st.keep * cv : d2v{0.0, 0.0};
    }
}

hipError_t launch_lines(const LinesArgs& a, hipStream_t st)
{
    if (a.njobs < 0 || a.njobs > kLineJobs || a.m < kMinM || a.m > kLineMaxM) return hipErrorInvalidValue;
    for (int j = 0; j < a.njobs; ++j) {
        const LineJob& J = a.job[j];
        int np = 0;
        if (J.nstage < 1 || J.nstage > kLineStages) return hipErrorInvalidValue;
        for (int s = 0; s < J.nstage; ++s) {
            const LineStage& S = J.stage[s];
            if (!S.out || S.nprod < 0 || S.nterm < 0 || S.nterm > kLineTerms) return hipErrorInvalidValue;
            for (int t = 0; t < S.nterm; ++t)
                if (!S.term[t].t) return hipErrorInvalidValue;
            np += S.nprod;
        }
        if (np < 1 || np > kLineProds) return hipErrorInvalidValue;
        for (int p = 0; p < np; ++p)
            if (!J.prod[p].src || !J.prod[p].mat) return hipErrorInvalidValue;
    }
    if (a.njobs == 0 || a.nmodes <= 0) return hipSuccess;
    const int he = (a.m + 1) / 2, ho = a.m / 2;
    const int nslab = (int)(((long)a.nmodes * a.m + 15) / 16), waves = (ho + 15) / 16;
    const size_t lds = ((size_t)4 * 16 * (8 * ((he + 7) / 8) + 1) + (size_t)waves * 32) * sizeof(double);
    const long total = (long)nslab * a.njobs;
    const dim3 grid((unsigned)((total + 7) / 8 * 8)), block(64 * waves);
    if (a.dirz) hipLaunchKernelGGL(k_lines<true>, grid, block, lds, st, a, nslab);
    else hipLaunchKernelGGL(k_lines<false>, grid, block, lds, st, a, nslab);
    return hipGetLastError();
}

// ---- one product, unfolded: D and D^T, the Chebyshev transforms (transyz), the Shen transforms -------
// out = coef A u + beta out (derivyz / transyz applied along y or z, chebyshev.f90:1-540, as a dense product with
// a matrix of the m CGL nodes: pseudomat.f90:90-107, cheb_collocation.F:19-75).  Folding halves the products but rounds each half of the rows at the scale of
// both: through D and D^T, whose large entries stand at the walls, the gradients of the projection step came
// out 1.6 times as far off (5.8e-15 against 3.6e-15 at 129^2 x 64), and one product per read is bound by
// memory or nearly so.  A workgroup owns 16 lines; a wave the row tiles w and w + W, re and im: four
// accumulators.  A last row past a multiple of 16 (m = 33, 65, 129, 257) is a dot product per line on the vector
// units: as a tile of its own 27 us per call at 129^2 x 64 instead of 23 (folded 19).
constexpr int kOneIT = 9;        // points per thread at most: 16 m over 64 ceil(tiles / 2) threads

template <bool DIRZ>
__global__ __launch_bounds__(576, 4) void k_line(LineOneArgs a, int nslab)
{
    extern __shared__ __attribute__((aligned(16))) double slab[];   // [re, im][line][k]
    const int m = a.m, mt = (m + 15) / 16, KP = (m + 7) / 8;        // the matrix's row tiles, pairs of 4 k
    const bool dot = m % 16 == 1;
    const int nt = dot ? mt - 1 : mt, W = (nt + 1) / 2;             // row tiles computed as such
    const int LDK = 8 * KP + 1, SL = 16 * LDK;
    double* red = slab + 2 * SL;                                    // [wave][line][re, im] of the last row
    const int nth = blockDim.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const int per = (nslab + 7) / 8, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);   // runs of slabs per XCD
    if ((int)(blockIdx.x >> 3) >= per || id >= nslab) return;
    const int L0 = id * 16, nlines = min(16, a.nmodes * m - L0);

    // element offsets of a line's first point and between its points, as in k_lines
    const size_t mm = (size_t)m * m;
    const int mode_first = L0 / m, lrel0 = L0 - mode_first * m;
    const size_t base0 = (size_t)mode_first * mm;
    const float invm = 1.0f / (float)m;
    auto line_off = [&](int l) -> unsigned {
        const int r = lrel0 + l;
        if constexpr (!DIRZ) return (unsigned)r * m;
        const int dm = (int)(((float)r + 0.5f) * invm);
        return (unsigned)dm * (unsigned)mm + (r - dm * m);
    };
    const unsigned sk = DIRZ ? m : 1;

    const int t0 = wave, t1 = min(wave + W, nt - 1);   // the second tile of the last wave of odd nt is not stored
    const d2v* F0 = (const d2v*)a.mat + (size_t)t0 * (2 * mt) * 64 + lane;
    const d2v* F1 = (const d2v*)a.mat + (size_t)t1 * (2 * mt) * 64 + lane;
    d2v f0 = F0[0], f1 = F1[0];
    const d2v* U = a.src + base0;
    d2v v[kOneIT];
#pragma unroll
    for (int it = 0; it < kOneIT; ++it) {              // points past the end read line 0's first and are not staged
        const int e = tid + it * nth, q = (int)(((float)e + 0.5f) * invm);   // e < 16 * 288 + 576
        int l = DIRZ ? e & 15 : q, k = DIRZ ? e >> 4 : e - q * m;
        if (e >= 16 * m || l >= nlines) l = k = 0;
        v[it] = U[line_off(l) + k * sk];
    }
#pragma unroll
    for (int it = 0; it < kOneIT; ++it) {
        const int e = tid + it * nth, q = (int)(((float)e + 0.5f) * invm);
        const int l = DIRZ ? e & 15 : q, k = DIRZ ? e >> 4 : e - q * m;
        if (e >= 16 * m) continue;
        slab[l * LDK + k] = l < nlines ? v[it][0] : 0.0;
        slab[SL + l * LDK + k] = l < nlines ? v[it][1] : 0.0;
    }
    for (int e = tid; e < 32 * (8 * KP - m); e += nth) {   // k past m, against zeros of the matrix
        const int row = e & 31, k = m + (e >> 5);
        slab[(row >> 4) * SL + (row & 15) * LDK + k] = 0.0;
    }
    lds_barrier();

    d4v re0 = {0.0, 0.0, 0.0, 0.0}, im0 = re0, re1 = re0, im1 = re0;
    const double* S0 = slab + l16 * LDK + l4;
    auto pair = [&](int kp, const d2v& c0, const d2v& c1, d2v& n0, d2v& n1) {
        const int kn = kp + 1 < KP ? kp + 1 : kp;
        n0 = F0[(size_t)kn * 64];
        n1 = F1[(size_t)kn * 64];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double re = S0[(2 * kp + h) * 4], im = S0[SL + (2 * kp + h) * 4];
            if constexpr (!DIRZ) {
                re0 = mfma(re, c0[h], re0);
                im0 = mfma(im, c0[h], im0);
                re1 = mfma(re, c1[h], re1);
                im1 = mfma(im, c1[h], im1);
            } else {
                re0 = mfma(c0[h], re, re0);
                im0 = mfma(c0[h], im, im0);
                re1 = mfma(c1[h], re, re1);
                im1 = mfma(c1[h], im, im1);
            }
        }
    };
    d2v g0, g1;
    int kp = 0;
    for (; kp + 1 < KP; kp += 2) {
        pair(kp, f0, f1, g0, g1);
        pair(kp + 1, g0, g1, f0, f1);
    }
    if (kp < KP) pair(kp, f0, f1, g0, g1);

    d2v* O = a.out + base0;
    if (dot) {
        const double* R = a.mat + (size_t)(mt - 1) * (2 * mt) * 128;   // A(m - 1, k): row 0 of the last tile
        d2v c = {0.0, 0.0};
        for (int k = tid >> 4; k < m; k += nth >> 4) {
            const double w = R[((k >> 3) * 64 + (k & 3) * 16) * 2 + ((k >> 2) & 1)];
            c += w * d2v{slab[l16 * LDK + k], slab[SL + l16 * LDK + k]};
        }
        c += d2v{__shfl_xor(c[0], 16, 64), __shfl_xor(c[1], 16, 64)};
        c += d2v{__shfl_xor(c[0], 32, 64), __shfl_xor(c[1], 32, 64)};
        if (l4 == 0) {
            red[(wave * 16 + l16) * 2] = c[0];
            red[(wave * 16 + l16) * 2 + 1] = c[1];
        }
        lds_barrier();
        if (tid < nlines) {
            c = d2v{0.0, 0.0};
            for (int w = 0; w < W; ++w) c += d2v{red[(w * 16 + tid) * 2], red[(w * 16 + tid) * 2 + 1]};
            const unsigned o = line_off(tid) + (m - 1) * sk;
            c *= a.coef;
            if (a.beta != 0.0) c += a.beta * O[o];
            O[o] = c;
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int tile = h ? wave + W : wave;
        unsigned o[4];
        bool ok[4];
        d2v y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 4 * e + l4, r = 16 * tile + (DIRZ ? i : l16), l = DIRZ ? l16 : i;
            ok[e] = r < m && tile < nt && l < nlines;
            o[e] = ok[e] ? line_off(l) + r * sk : 0;
            y[e] = d2v{0.0, 0.0};
        }
        if (a.beta != 0.0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = a.beta * O[o[e]];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (ok[e]) O[o[e]] = a.coef * (h ? d2v{re1[e], im1[e]} : d2v{re0[e], im0[e]}) + y[e];
    }
}

hipError_t launch_line(const LineOneArgs& a, hipStream_t st)
{
    if (!a.src || !a.out || !a.mat || a.m < kMinM || a.m > kLineMaxM) return hipErrorInvalidValue;
    if (a.nmodes <= 0) return hipSuccess;
    const int nslab = (int)(((long)a.nmodes * a.m + 15) / 16);
    const int tiles = a.m % 16 == 1 ? a.m / 16 : (a.m + 15) / 16, waves = (tiles + 1) / 2;
    const size_t lds = ((size_t)2 * 16 * (8 * ((a.m + 7) / 8) + 1) + (size_t)waves * 32) * sizeof(double);
    const dim3 grid((unsigned)((nslab + 7) / 8 * 8)), block(64 * waves);
    if (a.dirz) hipLaunchKernelGGL(k_line<true>, grid, block, lds, st, a, nslab);
    else hipLaunchKernelGGL(k_line<false>, grid, block, lds, st, a, nslab);
    return hipGetLastError();
}

// ---- small planes: both directions in one launch ----------------------------------------------
// A small grid's step is a chain of launches that are latency: arguments, loads, a few products, stores.  Here
// a workgroup owns one 16 x 16 tile of a job's outputs on one mode, its first wave the products along y, its
// second those along z, with the operands straight from memory into registers (the loads of all products are
// issued before the first product; the planes are a few KB and come from the caches), no staging and one
// barrier, where the second wave's sums join the first's.  Nothing is folded: at these sizes the products are
// a third of a workgroup's time.  A 33^2 x 16 step of 27 launches took 251 us, of these 18 y and z launches;
// with 9 of k_sums it takes 139 us.
template <int KP, int NPR>
__global__ __launch_bounds__(128) void k_sums(SumArgs a)
{
    __shared__ d2v ex[kSumStages][4][64];
    const int m = a.m, nt = (m + 15) / 16;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    // modes in 8 runs, one per XCD; the tiles and jobs of a mode are neighbours (they share inputs)
    const int total = a.njobs * a.nmodes * nt * nt, per = (total + 7) / 8;
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || id >= total) return;
    const int ty = id % nt, tz = id / nt % nt, jm = id / (nt * nt), mode = jm / a.njobs;
    const SumJob& job = a.job[jm % a.njobs];
    {   // touch the job's arguments at once (their first reads miss the scalar cache one after the other otherwise)
        constexpr int NW = (sizeof(SumJob) + 63) / 64;
        const int* w = (const int*)&job;
        int t[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) t[i] = w[min(i * 16, (int)sizeof(SumJob) / 4 - 1)];
#pragma unroll
        for (int i = 0; i < NW; ++i) asm volatile("" : : "s"(t[i]));
    }
    const size_t base = (size_t)mode * m * m;
    const int z16 = 16 * tz, y16 = 16 * ty;
    d4v re[kSumStages], im[kSumStages];
#pragma unroll
    for (int s = 0; s < kSumStages; ++s) re[s] = im[s] = d4v{0.0, 0.0, 0.0, 0.0};

    // k past m reads the last point against a zero of the matrix; rows and lines past m are not stored
    auto load = [&](auto dir, int p, d2v (&u)[2 * KP], d2v (&f)[KP]) {
        constexpr bool Z = decltype(dir)::value;
        const SumProd& q = job.prod[Z][p];
        const d2v* S = q.src + base;
        const d2v* F = (const d2v*)q.mat + (size_t)(Z ? tz : ty) * (2 * nt) * 64 + lane;
        const int line = min((Z ? y16 : z16) + l16, m - 1);
#pragma unroll
        for (int kp = 0; kp < KP; ++kp) {
            f[kp] = F[kp * 64];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = min(8 * kp + 4 * h + l4, m - 1);
                u[2 * kp + h] = S[Z ? k * m + line : line * m + k];
            }
        }
    };
    auto mul = [&](auto dir, double coef, const d2v (&u)[2 * KP], const d2v (&f)[KP], d4v& re, d4v& im) {
        constexpr bool Z = decltype(dir)::value;
        d4v r = {0.0, 0.0, 0.0, 0.0}, i = r;   // (scaled after the sum: coef on f would round every element once more)
#pragma unroll
        for (int kp = 0; kp < KP; ++kp)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double d = f[kp][h];
                const d2v x = u[2 * kp + h];
                r = Z ? mfma(d, x[0], r) : mfma(x[0], d, r);
                i = Z ? mfma(d, x[1], i) : mfma(x[1], d, i);
            }
        re += coef * r;
        im += coef * i;
    };
    auto products = [&](auto dir) {
        constexpr bool Z = decltype(dir)::value;
        d2v u[NPR][2 * KP], f[NPR][KP];
        const int n0 = job.stage[0].nprod[Z], n = n0 + (job.nstage > 1 ? job.stage[1].nprod[Z] : 0);
#pragma unroll
        for (int p = 0; p < NPR; ++p) load(dir, p < n ? p : 0, u[p], f[p]);
#pragma unroll
        for (int p = 0; p < NPR; ++p) {
            if (p >= n) continue;
            const double coef = job.prod[Z][p].coef;
            if (p < n0) mul(dir, coef, u[p], f[p], re[0], im[0]);
            else mul(dir, coef, u[p], f[p], re[1], im[1]);
        }
    };
    if (wave == 1) {
        products(std::true_type{});
#pragma unroll
        for (int s = 0; s < kSumStages; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) ex[s][e][lane] = d2v{re[s][e], im[s][e]};
        lds_barrier();
        return;
    }
    // the first wave: the pointwise terms of both stages (unused ones are loaded in vain), then its products
    const int y = y16 + l16;
    unsigned o[4];
    bool ok[4];
    d2v t[kSumStages][kSumTerms][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int z = z16 + 4 * e + l4;
        ok[e] = y < m && z < m;
        o[e] = ok[e] ? z * m + y : 0;
    }
#pragma unroll
    for (int s = 0; s < kSumStages; ++s)
#pragma unroll
        for (int j = 0; j < kSumTerms; ++j) {
            const d2v* T = (s < job.nstage && j < job.stage[s].nterm ? job.stage[s].term[j].t : job.stage[0].term[0].t) + base;
#pragma unroll
            for (int e = 0; e < 4; ++e) t[s][j][e] = T[o[e]];
        }
    products(std::false_type{});
    lds_barrier();
    const double xa = a.alp * (double)mode;
    d2v x[4];
#pragma unroll
    for (int s = 0; s < kSumStages; ++s) {
        if (s >= job.nstage) continue;
        const SumStage& st = job.stage[s];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const d2v p = d2v{re[s][e], im[s][e]} + ex[s][e][lane];
            x[e] = s > 0 && st.keep != 0.0 ? st.keep * x[e] + p : p;
        }
#pragma unroll
        for (int j = 0; j < kSumTerms; ++j) {
            if (j >= st.nterm) continue;
            const double cr = st.term[j].cr + st.term[j].crx * xa * xa, ci = st.term[j].ci * xa;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += cr * t[s][j][e] + ci * d2v{-t[s][j][e][1], t[s][j][e][0]};
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (mode == 0) x[e][0] += st.c0;
            if (ok[e]) (st.out + base)[o[e]] = x[e];
        }
    }
}

// Up to the size where the unfolded products cost more than the launches saved: a step of 64^2 x 48 modes
// (modes x tiles x fragment pairs 6144) takes 442 us against 461 of the y and z launches, 64^2 x 64 (8192)
// 471 against 449, 33^2 x 128 (5760) 341 against 389, 17^2 x 256 (3072) 259 against 319.
bool sums_supported(int m, int nmodes)
{
    const long nt = (m + 15) / 16;
    return m <= kSumMaxM && nmodes * nt * nt * ((m + 7) / 8) <= 7168;
}

template <int KP>
static void launch_sums_kp(const SumArgs& a, int np, dim3 grid, hipStream_t st)
{
    if (np <= 1) hipLaunchKernelGGL((k_sums<KP, 1>), grid, dim3(128), 0, st, a);
    else hipLaunchKernelGGL((k_sums<KP, kSumProds>), grid, dim3(128), 0, st, a);
}

hipError_t launch_sums(const SumArgs& a, hipStream_t st)
{
    if (a.njobs < 0 || a.njobs > kSumJobs || a.m < kMinM || a.m > kSumMaxM) return hipErrorInvalidValue;
    int most = 0;
    for (int j = 0; j < a.njobs; ++j) {
        const SumJob& J = a.job[j];
        int np[2] = {0, 0};
        if (J.nstage < 1 || J.nstage > kSumStages) return hipErrorInvalidValue;
        for (int s = 0; s < J.nstage; ++s) {
            const SumStage& S = J.stage[s];
            if (!S.out || S.nterm < 0 || S.nterm > kSumTerms || S.nprod[0] < 0 || S.nprod[1] < 0) return hipErrorInvalidValue;
            for (int t = 0; t < S.nterm; ++t)
                if (!S.term[t].t) return hipErrorInvalidValue;
            for (int d = 0; d < 2; ++d) np[d] += S.nprod[d];
        }
        if (J.stage[0].nterm < 1) return hipErrorInvalidValue;   // (the address that unused terms read)
        for (int d = 0; d < 2; ++d) {
            if (np[d] > kSumProds || !J.prod[d][0].src || !J.prod[d][0].mat) return hipErrorInvalidValue;
            for (int p = 0; p < np[d]; ++p)
                if (!J.prod[d][p].src || !J.prod[d][p].mat) return hipErrorInvalidValue;
            most = std::max(most, np[d]);
        }
    }
    if (a.njobs == 0 || a.nmodes <= 0) return hipSuccess;
    const int nt = (a.m + 15) / 16;
    const long total = (long)a.njobs * a.nmodes * nt * nt;
    if (total >= 1L << 30) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((total + 7) / 8 * 8));
    switch ((a.m + 7) / 8) {
        case 1: launch_sums_kp<1>(a, most, grid, st); break;
        case 2: launch_sums_kp<2>(a, most, grid, st); break;
        case 3: launch_sums_kp<3>(a, most, grid, st); break;
        case 4: launch_sums_kp<4>(a, most, grid, st); break;
        case 5: launch_sums_kp<5>(a, most, grid, st); break;
        case 6: launch_sums_kp<6>(a, most, grid, st); break;
        case 7: launch_sums_kp<7>(a, most, grid, st); break;
        default: launch_sums_kp<8>(a, most, grid, st); break;
    }
    return hipGetLastError();
}

}  // namespace duct
