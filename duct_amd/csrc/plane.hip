// The whole solve of one real plane in one workgroup: U = P ((P^-1 F P^-T) ./ den) P^T with the
// plane in LDS from the right-hand side to the solution (solvediag.f90:51-322, its transpose, and
// solvediag_temp.f90:2-352), boundary included.  Serves interiors up to 128 points per direction,
// whose padded plane (128 x 129 doubles, 132 KB) fits the 160 KB of a gfx950 CU.
//
// Against four k_proj launches over all planes (proj_f64.hip) it moves the field once instead of
// four times through planar intermediates, pads n to a multiple of 16 instead of a power of two,
// and needs one launch where the gauge, the edges and both boundary types took up to twelve.
//
// Work decomposition (RT = ceil(n / 16) row and column tiles of 16): a wave owns RR x CC tiles, one row
// of tiles for RT <= 5 and 7, 3 x 3 for 6 (four waves, two workgroups per CU: 86 against 114 us at 97^2
// x 40 modes x 4, where six waves left the second workgroup without a place), 2 x 4 for 8.  The basis
// rows stream from L2 in fragment order, one pair of k-steps ahead; B fragments come from LDS one k-step
// ahead (column stride N + 1: the 16 lanes of a row hit distinct banks).  A pass writes its product back
// transposed, Y = (A X)^T, so four passes close the chain:
//   X [z][y] -> P^-1 along y -> [y-eig][z] -> P^-1 along z -> G [z-eig][y-eig] -> divide
//     -> P along y -> [y][z-eig] -> P along z -> U [z][y]            ([column][row])
// Re and Im of a plane are neighbouring workgroups of one XCD: each reads and writes its half of
// the same cache lines.  Workgroups are as many as the CUs hold and walk their planes.
//
// What bounds it: the FP64 matrix cores.  At RT = 8 a plane takes ~155e3 cycles of which its MFMAs are
// 131e3; the rest is what one workgroup per CU cannot overlap: the writes between the passes (~4e3
// each), the divide (~9e3), the stores and walls.  u, v, w and p at 129^2 x 64 modes take 173 us
// (8 launches and 216 us as passes over planar intermediates), at 129^2 x 256 652 us (736), one field of
// 33^2 x 16 9 us (31), 97^2 x 40 51 us for the Neumann field, the mixed walls at 97 x 129 x 64 81 us (140)
// and at 129 x 129 x 400 362 us (483).
#include <algorithm>

#include "plane.h"
#include "temp.h"

namespace duct {

namespace {

constexpr long kLdsPerCu = 160 * 1024;

__device__ __forceinline__ double plane_wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over groups of n (a power of two) neighbouring lanes, in all of them
template <int n>
__device__ __forceinline__ double line_sum(double v)
{
#pragma unroll
    for (int off = 1; off < n; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// waves per SIMD that the LDS admits
constexpr int plane_waves(int RT, int NW, int kind)
{
    const int lds = (16 * RT * (16 * RT + 1) + (kind == PLANE_FWD ? 4 : 6) * 16 * RT + 4 * NW) * 8, wgs = (int)kLdsPerCu / lds;
    const int waves = ((wgs < 1 ? 1 : wgs) * NW + 3) / 4;
    return waves < 2 ? 2 : waves > 4 ? 4 : waves;
}

// Effective wall values of a line (mod_term_FT*: the interior correction is -D2(i, 1) g1 - D2(i, m) g2)
// and, with the interior's shares sa, sb of the derivative rows, its edge values (edge_value_*); t1, t2:
// 0 = Dirichlet, 1 = Neumann (solvediag_temp.f90:136-247)
struct WallRows {
    double d00, d0m, dm0, dmm;
};
__device__ __forceinline__ void wall_line(int t1, int t2, const WallRows& w, double v1, double v2, double sa, double sb,
                                          double& e0, double& e1)
{
    if (!t1 && !t2) {
        e0 = v1;
        e1 = v2;
    } else if (!t1) {
        e0 = v1;
        e1 = (v2 - w.dm0 * v1 - sb) / w.dmm;
    } else if (!t2) {
        e1 = v2;
        e0 = (v1 - w.d0m * v2 - sa) / w.d00;
    } else {
        const double det = w.d00 * w.dmm - w.d0m * w.dm0, ra = v1 - sa, rb = v2 - sb;
        e0 = (w.dmm * ra - w.d0m * rb) / det;
        e1 = (w.d00 * rb - w.dm0 * ra) / det;
    }
}

}  // namespace

template <int RT, int RR, int CC, int KIND>
__global__ __launch_bounds__(64 * (RT / RR) * (RT / CC), plane_waves(RT, (RT / RR) * (RT / CC), KIND)) void k_plane(PlaneArgs a)
{
    constexpr int N = 16 * RT, LD = N + 1, WC = RT / CC, NW = (RT / RR) * WC, NTH = 64 * NW;
    // One workgroup fills the LDS (RT 7 and 8): its next plane is loaded under the last pass.  All CUs
    // would otherwise load at the same time, at the rate of HBM.  Smaller planes share the CU.
    constexpr bool AHEAD = RT >= 7 && KIND != PLANE_WALL;   // (WALL's registers do not hold a plane more)
    constexpr int NV = N * N / NTH;                                  // values per thread, NTH apart
    constexpr int LPL = NTH >= 8 * N ? 8 : NTH >= 4 * N ? 4 : 2;     // lanes per line of the edge sums
    static_assert(N * N % NTH == 0 && NTH >= LPL * N, "shape");
    extern __shared__ __attribute__((aligned(16))) double sm[];
    double* X = sm;              // [column][row], stride LD
    double* lam = X + N * LD;    // eigenvalues of the two bases (WALL: along y and along z)
    double* red = lam + 2 * N;   // 4 NW: the waves' partial sums
    double* vec = red + 4 * NW;  // ADJ, WALL: 4 N, the vectors of the wall terms; FWD, WALL: rows 1 and m of D

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    const int r0 = wave / WC * RR, c0t = wave % WC * CC;   // the wave's first row and column tile
    const int my = a.my, mz = a.mz, ny = my - 2, nz = mz - 2;
    auto row_of = [](int t, int it) { return NTH % N == 0 ? t % N : (t + it * NTH) % N; };   // of a thread's values
    auto col_of = [](int t, int it) { return NTH % N == 0 ? t / N + it * (NTH / N) : (t + it * NTH) / N; };
    auto perimeter = [&](int e) -> size_t {     // e < 2 (my + mz)
        if (e < my) return e;                                              // z = 1
        if (e < 2 * my) return (size_t)(e - my) + (size_t)(mz - 1) * my;   // z = mz
        if (e < 2 * my + mz) return (size_t)(e - 2 * my) * my;             // y = 1
        return (size_t)(my - 1) + (size_t)(e - 2 * my - mz) * my;          // y = my
    };

    // Real planes in 8 runs, one per XCD, walked by the XCD's workgroups in turn; Re and Im of a plane
    // are neighbours.
    const int total = a.nf * a.nmodes * 2, per = (total + 7) / 8;
    const int step = gridDim.x >> 3, last = min(total, ((int)(blockIdx.x & 7) + 1) * per);
    auto field_of = [&](int id) { return (id >> 1) / a.nmodes; };
    auto bnd_of = [&](int id) { return KIND == PLANE_WALL ? 0 : a.bnd[field_of(id)]; };
    auto offset_of = [&](int id) { return (size_t)((id >> 1) % a.nmodes) * my * mz * 2 + (id & 1); };   // in doubles
    auto in_of = [&](int id) { return (double*)const_cast<d2v*>(a.in[field_of(id)]) + offset_of(id); };  // stride 2
    auto out_of = [&](int id) { return (double*)a.out[field_of(id)] + offset_of(id); };
    auto zero_rhs_walls = [&](int id) { return KIND == PLANE_FWD && a.bmode == BND_DIR_ZERO && bnd_of(id) == 0; };
    // the next plane to solve at or after id; Im of mode 0 is not solved but zero (int2d3d.f90:43)
    auto next_plane = [&](int id) {
        for (; id < last && (id & 1) && a.mode0 + (id >> 1) % a.nmodes == 0; id += step) {
            double* in = in_of(id);
            double* out = out_of(id);
            if (zero_rhs_walls(id))
                for (int e = tid; e < 2 * (my + mz); e += NTH) in[2 * perimeter(e)] = 0.0;
            for (int e = tid; e < my * mz; e += NTH) out[2 * (size_t)e] = 0.0;
        }
        return id;
    };
    int id = next_plane((int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3));
    if (id >= last) return;

    for (int t = tid; t < 2 * N; t += NTH) {
        const double* src = KIND == PLANE_WALL ? (t < N ? a.b[0].lamy : a.b[0].lamz) : a.b[t / N].lamy;
        lam[t] = src ? src[t % N] : 0.0;
    }
    if (KIND == PLANE_FWD && a.b[1].DC)
        for (int t = tid; t < 2 * N; t += NTH)
            vec[t] = t % N < ny ? a.b[1].DC[(t < N ? 0 : my - 1) + (size_t)(t % N + 1) * my] : 0.0;

    double v[NV];
    auto load = [&](const double* in, int it) {
        int t = tid;
        asm volatile("" : "+v"(t));   // (opaque: the offsets are not kept in registers across the loop)
        const int r = row_of(t, it), c = col_of(t, it);
        v[it] = in[r < ny && c < nz ? 2u * ((unsigned)(r + 1) + (unsigned)(c + 1) * my) : 0u];
    };
    auto load_all = [&](const double* in) {
#pragma unroll
        for (int it = 0; it < NV; ++it) load(in, it);
    };
    // basis fragments of this wave's rows
    auto frag = [&](int bnd, int p) {
        const PlaneBasis& B = a.b[bnd];
        return (const d2v*)B.A[p] + (size_t)r0 * (B.NP / 8) * 64 + lane;
    };
    auto load_a = [&](int bnd, const d2v* F, int kp, d2v (&r)[RR]) {
#pragma unroll
        for (int rr = 0; rr < RR; ++rr) r[rr] = F[((size_t)rr * (a.b[bnd].NP / 8) + kp) * 64];
    };
    d2v a0[RR], a1[RR];
    load_a(bnd_of(id), frag(bnd_of(id), 0), 0, a0);
    if (AHEAD) load_all(in_of(id));

    for (int next = 0; id < last; id = next) {
    const int mode = (id >> 1) % a.nmodes, f = field_of(id), bnd = bnd_of(id);
    const PlaneBasis& B = a.b[bnd];
    const double* ly = lam + (KIND == PLANE_WALL ? 0 : bnd * N);
    const double* lz = KIND == PLANE_WALL ? lam + N : ly;
    double* in = in_of(id);
    double* out = out_of(id);
    const double xlam = xlambda_of(a.alambda[f], a.alp, a.mode0 + mode);
    const bool dir_zero = zero_rhs_walls(id);
    next = next_plane(id + step);
    const int ahead = next < last ? next : id;   // the plane whose values and first fragments are fetched ahead

    // ---- the terms that the walls add to the interior, rank four:
    //   F(i, j) += wy0_i cy0_j + wym_i cym_j + wz0_j rz0_i + wzm_j rzm_i
    // (ADJ Neumann: E^T of the edges and corners, solvediag.f90:251-322 transposed; WALL: mod_term_FT*)
    const bool walls = KIND == PLANE_WALL || (KIND == PLANE_ADJ && bnd == 1);
    double* cy0 = vec;
    double* cym = vec + N;
    double* rz0 = vec + 2 * N;
    double* rzm = vec + 3 * N;
    const double* wy0 = nullptr;   // from index 0 of the interior, entries ws apart
    const double* wym = nullptr;
    const double* wz0 = nullptr;
    const double* wzm = nullptr;
    const int ws = KIND == PLANE_WALL ? 1 : my;
    if constexpr (KIND == PLANE_ADJ) {
        if (bnd == 1) {
            const double* DC = B.DC;
            const int m = my;
            const double DC00 = DC[0], DCmm = DC[(m - 1) + (size_t)(m - 1) * m];
            const double DC0m = DC[(size_t)(m - 1) * m], DCm0 = DC[m - 1];
            const double det = DC00 * DCmm - DC0m * DCm0;
            const size_t cidx[4] = {0, (size_t)(m - 1), (size_t)(m - 1) + (size_t)(m - 1) * m, (size_t)(m - 1) * m};
            double ffb[4];   // AM1^T of the corners
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                double v = 0.0;
#pragma unroll
                for (int r = 0; r < 4; ++r) v += B.AM1[r + 4 * c] * in[2 * cidx[r]];
                ffb[c] = v;
            }
            for (int t = tid; t < ny; t += NTH) {
                const int i = t + 1;
                const double d0 = DC[(size_t)i * m], dm = DC[(m - 1) + (size_t)i * m];
                const double eb = in[2 * (size_t)i] - d0 * ffb[0] + dm * ffb[1];
                const double et = in[2 * ((size_t)i + (size_t)(m - 1) * m)] - dm * ffb[2] - d0 * ffb[3];
                const double el = in[2 * ((size_t)i * m)] - d0 * ffb[0] + dm * ffb[3];
                const double er = in[2 * ((m - 1) + (size_t)i * m)] - d0 * ffb[1] - dm * ffb[2];
                rz0[t] = (-DCmm * eb + DCm0 * et) / det;
                rzm[t] = (DC0m * eb - DC00 * et) / det;
                cy0[t] = (-DCmm * el + DCm0 * er) / det;
                cym[t] = (DC0m * el - DC00 * er) / det;
            }
            wy0 = wz0 = DC + m;
            wym = wzm = DC + 2 * m - 1;
        }
    }
    const double* Dy0 = a.vec + 2 * my;   // WALL: the wall vectors of TempArgs
    const double* Dz0 = a.vec + 4 * my + 2 * mz;
    if constexpr (KIND == PLANE_WALL) {
        const WallRows ry = {Dy0[0], Dy0[my - 1], Dy0[my], Dy0[2 * my - 1]};
        const WallRows rz = {Dz0[0], Dz0[mz - 1], Dz0[mz], Dz0[2 * mz - 1]};
        const double* by = a.bcy + (size_t)mode * 2 * mz;
        const double* bz = a.bcz + (size_t)mode * 2 * my;
        for (int t = tid; t < nz; t += NTH) {
            double g1, g2;
            wall_line(a.by1, a.by2, ry, by[t + 1], by[mz + t + 1], 0.0, 0.0, g1, g2);
            cy0[t] = -g1;
            cym[t] = -g2;
        }
        for (int t = tid; t < ny; t += NTH) {
            double g1, g2;
            wall_line(a.bz1, a.bz2, rz, bz[t + 1], bz[my + t + 1], 0.0, 0.0, g1, g2);
            rz0[t] = -g1;
            rzm[t] = -g2;
        }
        wy0 = a.vec + 1;
        wym = a.vec + my + 1;
        wz0 = a.vec + 4 * my + 1;
        wzm = a.vec + 4 * my + mz + 1;
    }
    if (walls) lds_barrier();

    // ---- the right-hand side into LDS
    if (!AHEAD) load_all(in);
    const bool singular = KIND != PLANE_WALL && B.gauge >= 0 && fabs(xlam) <= 1.0e-10;
    double gsum = 0.0;
    {
        int t = tid;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int it = 0; it < NV; ++it) {
            const int row = row_of(t, it), col = col_of(t, it);
            if (!(row < ny && col < nz)) v[it] = 0.0;
            else {
                if (walls)
                    v[it] += (wy0[row * ws] * cy0[col] + wym[row * ws] * cym[col]) +
                             (wz0[col * ws] * rz0[row] + wzm[col * ws] * rzm[row]);
                if (KIND == PLANE_ADJ && singular) gsum += B.pcol[row] * v[it] * B.pcol[col];
            }
            X[col * LD + row] = v[it];
        }
    }
    if (KIND == PLANE_ADJ && singular) {
        gsum = plane_wave_sum(gsum);
        if (lane == 0) red[wave] = gsum;
    }
    lds_barrier();

    d4v acc[RR][CC];
    auto read_b = [&](int ks, double (&b)[CC]) {
#pragma unroll
        for (int nt = 0; nt < CC; ++nt) b[nt] = X[((c0t + nt) * 16 + l16) * LD + ks * 4 + l4];
        __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of the MFMAs that cover them
    };
    auto mma = [&](int h, const d2v (&av)[RR], const double (&b)[CC]) {
#pragma unroll
        for (int rr = 0; rr < RR; ++rr)
#pragma unroll
            for (int nt = 0; nt < CC; ++nt)
                acc[rr][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[rr][h], b[nt], acc[rr][nt], 0, 0, 0);
    };
    // acc = A X for the wave's tiles; k < kn.  a0 holds the pass's first fragments on entry and the
    // next pass's on exit.
    auto pass = [&](int p, int kn) {
        const d2v* F = frag(bnd, p);
        const int KP = (kn + 7) / 8;
        double b0[CC], b1[CC];
#pragma unroll
        for (int rr = 0; rr < RR; ++rr)
#pragma unroll
            for (int nt = 0; nt < CC; ++nt) acc[rr][nt] = d4v{0.0, 0.0, 0.0, 0.0};
        read_b(0, b0);
        auto pair = [&](int kp, const d2v (&cur)[RR], d2v (&nxt)[RR]) {
            const int kn1 = kp + 1 < KP ? kp + 1 : kp;
            load_a(bnd, F, kn1, nxt);
            read_b(2 * kp + 1, b1);
            mma(0, cur, b0);
            read_b(2 * kn1, b0);
            mma(1, cur, b1);
        };
        int kp = 0;
        for (; kp + 1 < KP; kp += 2) {
            pair(kp, a0, a1);
            pair(kp + 1, a1, a0);
        }
        if (kp < KP) pair(kp, a0, a1);
        if (p < 3) load_a(bnd, frag(bnd, p + 1), 0, a0);
        else load_a(bnd_of(ahead), frag(bnd_of(ahead), 0), 0, a0);
    };
    // Pass 3 with the next plane's values loaded a few per pair of k-steps: loads return in order, so all
    // of them at once would hold back the fragments behind them.
    auto pass_ahead = [&](int kn) {
        const d2v* F = frag(bnd, 3);
        const double* src = in_of(ahead);
        const int KP = (kn + 7) / 8;
        constexpr int LP = NV / (2 * RT);
        static_assert(!AHEAD || LP * 2 * RT == NV, "loads per pair");
        double b0[CC], b1[CC];
#pragma unroll
        for (int rr = 0; rr < RR; ++rr)
#pragma unroll
            for (int nt = 0; nt < CC; ++nt) acc[rr][nt] = d4v{0.0, 0.0, 0.0, 0.0};
        read_b(0, b0);
        auto pair = [&](int kp, const d2v (&cur)[RR], d2v (&nxt)[RR]) {
            const int kn1 = kp + 1 < KP ? kp + 1 : KP - 1;
            load_a(bnd, F, kn1, nxt);
#pragma unroll
            for (int l = 0; l < LP && next < last; ++l) load(src, kp * LP + l);
            if (kp < KP) {
                read_b(2 * kp + 1, b1);
                mma(0, cur, b0);
                read_b(2 * kn1, b0);
                mma(1, cur, b1);
            }
        };
#pragma unroll
        for (int kp = 0; kp < 2 * RT; kp += 2) {
            pair(kp, a0, a1);
            pair(kp + 1, a1, a0);
        }
        load_a(bnd_of(ahead), frag(bnd_of(ahead), 0), 0, a0);
    };
    // X <- acc^T: D[i][j] of a tile in lane j + 16 (i % 4), element i / 4
    auto put = [&]() {
        lds_barrier();
#pragma unroll
        for (int rr = 0; rr < RR; ++rr)
#pragma unroll
            for (int nt = 0; nt < CC; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    X[(16 * (r0 + rr) + 4 * r + l4) * LD + (c0t + nt) * 16 + l16] = acc[rr][nt][r];
        lds_barrier();
    };

    pass(0, ny);
    put();
    pass(1, nz);
    // ---- divide (solvediag.f90:61-66, :151-159): row i is the z-eigenvector, column j the y one (the
    // padding is zero and stays zero)
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
        double li[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) li[r] = lz[16 * (r0 + rr) + 4 * r + l4];
#pragma unroll
        for (int nt = 0; nt < CC; ++nt) {
            const int j = (c0t + nt) * 16 + l16;
            const double lj = ly[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool ok = 16 * (r0 + rr) + 4 * r + l4 < nz && j < ny;
                acc[rr][nt][r] = acc[rr][nt][r] / (ok ? lj + li[r] - xlam : 1.0);
            }
        }
    }
    if (KIND != PLANE_WALL && singular) {   // the null mode's entry (a, a): solvediag.f90:161-206, U(a, a) = wanted
        double c = 0.0, s = 0.0;
        if (KIND == PLANE_ADJ) {
            for (int w = 0; w < NW; ++w) c += red[w];
            c /= B.pdiag * B.pdiag;
        }
        // the entries (i, j) of the wave's tiles, one after the other
        auto each = [&](auto&& fn) {
#pragma unroll
            for (int rr = 0; rr < RR; ++rr)
#pragma unroll
                for (int nt = 0; nt < CC; ++nt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = 16 * (r0 + rr) + 4 * r + l4, j = (c0t + nt) * 16 + l16;
                        if (i < nz && j < ny) acc[rr][nt][r] = fn(i, j, acc[rr][nt][r]);
                    }
        };
        each([&](int i, int j, double g) {
            if (i == B.gauge && j == B.gauge) return 0.0;
            if (KIND == PLANE_ADJ) return g - c * B.prow[j] * B.prow[i] / (ly[j] + lz[i] - xlam);
            s += B.prow[j] * g * B.prow[i];
            return g;
        });
        if (KIND == PLANE_FWD) {
            s = plane_wave_sum(s);
            if (lane == 0) red[wave] = s;
            lds_barrier();
            s = 0.0;
            for (int w = 0; w < NW; ++w) s += red[w];
            const double v = (B.wanted - s) / (B.pdiag * B.pdiag);
            each([&](int i, int j, double g) { return i == B.gauge && j == B.gauge ? v : g; });
        }
    }
    put();
    pass(2, ny);
    put();
    if constexpr (AHEAD) pass_ahead(nz);
    else pass(3, nz);

    // ---- the solution: row i is z, column j is y (contiguous over the lanes)
    int q16 = l16, q4 = l4;
    asm volatile("" : "+v"(q16), "+v"(q4));
#pragma unroll
    for (int rr = 0; rr < RR; ++rr)
#pragma unroll
        for (int nt = 0; nt < CC; ++nt) {
            const int j = (c0t + nt) * 16 + q16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * (r0 + rr) + 4 * r + q4;
                if (i < nz && j < ny) out[2u * ((unsigned)(j + 1) + (unsigned)(i + 1) * my)] = acc[rr][nt][r];
            }
        }
    if (KIND == PLANE_ADJ || (KIND == PLANE_FWD && bnd == 0)) {
        // by the waves that finish the pass first (the older ones of their SIMDs)
        constexpr int NE = NTH >= 512 ? NTH / 2 : NTH;
        for (int e = tid; e < 2 * (my + mz) && tid < NE; e += NE) {
            const size_t idx = 2 * perimeter(e);
            const double v = KIND == PLANE_FWD && a.bmode == BND_DIR_KEEP ? in[idx] : 0.0;
            if (dir_zero) in[idx] = 0.0;
            out[idx] = v;
        }
        lds_barrier();   // the last pass's reads of X are done
        continue;
    }

    // ---- edges of the Neumann field (solvediag.f90:251-322) and of the walls (solvediag_temp.f90): the
    // sums along y and z with the derivative rows, several threads per line
    if (KIND == PLANE_WALL)
        for (int t = tid; t < 4 * N; t += NTH) {   // (the wall vectors of the right-hand side are used up)
            const int i = t % N, d = t / N;
            vec[t] = i < (d < 2 ? ny : nz) ? (d < 2 ? Dy0 + d * my : Dz0 + (d - 2) * mz)[i + 1] : 0.0;
        }
    put();
    // LPL lanes per line: line z = c over y, line y = c over z (threads past the last line repeat it)
    const int c = min(tid / LPL, N - 1), q = tid % LPL;
    const bool line = tid / LPL < N;
    double s0y = 0.0, smy = 0.0, s0z = 0.0, smz = 0.0;
    // each sum ends with its largest terms, at its own wall: the other way round the small ones would be
    // rounded to the large ones' last place, and phi's walls are what grad(phi) multiplies by m^2 / 3
    const double* vz = KIND == PLANE_WALL ? vec + 2 * N : vec;
#pragma unroll 4
    for (int i = 0; i < N / LPL; ++i) {
        const int t = q + i * LPL, r = N - LPL + q - i * LPL;
        s0y += vec[r] * X[c * LD + r];
        smy += vec[N + t] * X[c * LD + t];
        s0z += vz[r] * X[r * LD + c];
        smz += vz[N + t] * X[t * LD + c];
    }
    s0y = line_sum<LPL>(s0y);
    smy = line_sum<LPL>(smy);
    s0z = line_sum<LPL>(s0z);
    smz = line_sum<LPL>(smz);
    if constexpr (KIND == PLANE_WALL) {
        const WallRows ry = {Dy0[0], Dy0[my - 1], Dy0[my], Dy0[2 * my - 1]};
        const WallRows rz = {Dz0[0], Dz0[mz - 1], Dz0[mz], Dz0[2 * mz - 1]};
        const double* by = a.bcy + (size_t)mode * 2 * mz;
        const double* bz = a.bcz + (size_t)mode * 2 * my;
        if (line && q == 0 && c < nz) {
            double e0, e1;
            wall_line(a.by1, a.by2, ry, by[c + 1], by[mz + c + 1], s0y, smy, e0, e1);
            out[2 * ((size_t)(c + 1) * my)] = e0;
            out[2 * ((size_t)(c + 1) * my + my - 1)] = e1;
        }
        if (line && q == 1 && c < ny) {
            double e0, e1;
            wall_line(a.bz1, a.bz2, rz, bz[c + 1], bz[my + c + 1], s0z, smz, e0, e1);
            out[2 * (size_t)(c + 1)] = e0;
            out[2 * ((size_t)(c + 1) + (size_t)(mz - 1) * my)] = e1;
        }
        if (tid < 4) {   // corners keep the right-hand side's values
            const size_t c = (tid & 1 ? my - 1 : 0) + (tid & 2 ? (size_t)(mz - 1) * my : 0);
            out[2 * c] = in[2 * c];
        }
        lds_barrier();
        continue;
    }
    const int m = my;
    const double* DC = B.DC;
    const double DC00 = DC[0], DCmm = DC[(m - 1) + (size_t)(m - 1) * m];
    const double DC0m = DC[(size_t)(m - 1) * m], DCm0 = DC[m - 1];
    const double det = DC00 * DCmm - DC0m * DCm0;
    double f1 = 0.0, f2 = 0.0, f3 = 0.0, f4 = 0.0;
    if (line && q == 0 && c < ny) {
        const double d0 = DC[(size_t)(c + 1) * m], dm = DC[(m - 1) + (size_t)(c + 1) * m];
        const double el = (-DCmm * s0y + DC0m * smy) / det, er = (DCm0 * s0y - DC00 * smy) / det;
        const double vb = (-DCmm * s0z + DC0m * smz) / det, vt = (DCm0 * s0z - DC00 * smz) / det;
        out[2 * ((size_t)(c + 1) * m)] = el;
        out[2 * ((m - 1) + (size_t)(c + 1) * m)] = er;
        out[2 * (size_t)(c + 1)] = vb;
        out[2 * ((size_t)(c + 1) + (size_t)(m - 1) * m)] = vt;
        f1 = -d0 * vb - d0 * el;
        f2 = dm * vb - d0 * er;
        f3 = -dm * vt - dm * er;
        f4 = -d0 * vt + dm * el;
    }
    f1 = plane_wave_sum(f1);
    f2 = plane_wave_sum(f2);
    f3 = plane_wave_sum(f3);
    f4 = plane_wave_sum(f4);
    if (lane == 0) {
        red[wave * 4] = f1;
        red[wave * 4 + 1] = f2;
        red[wave * 4 + 2] = f3;
        red[wave * 4 + 3] = f4;
    }
    lds_barrier();
    if (tid < 4) {   // corners: AM1 of the four sums
        double ff[4] = {0.0, 0.0, 0.0, 0.0};
        for (int w = 0; w < NW; ++w)
#pragma unroll
            for (int c = 0; c < 4; ++c) ff[c] += red[w * 4 + c];
        const double* A = B.AM1;
        const double v = A[tid] * ff[0] + A[tid + 4] * ff[1] + A[tid + 8] * ff[2] + A[tid + 12] * ff[3];
        size_t idx;
        if (tid == 0) idx = 0;
        else if (tid == 1) idx = (size_t)(m - 1);
        else if (tid == 2) idx = (size_t)(m - 1) + (size_t)(m - 1) * m;
        else idx = (size_t)(m - 1) * m;
        out[2 * idx] = v;
    }
    lds_barrier();
    }
}

bool plane_supported(int my, int mz)
{
    return my >= kMinM && mz >= kMinM && my - 2 <= kPlaneMaxN && mz - 2 <= kPlaneMaxN;
}

template <int RT, int RR, int CC>
static hipError_t launch_plane_rt(int kind, const PlaneArgs& a, hipStream_t st)
{
    constexpr int N = 16 * RT, NW = (RT / RR) * (RT / CC);
    const size_t lds = ((size_t)N * (N + 1) + (kind == PLANE_FWD ? 4 : 6) * N + 4 * NW) * sizeof(double);
    // as many workgroups as fit the CUs' LDS at once (and 16 waves of each), a multiple of the XCDs
    int dev = 0, ncu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    const long total = (long)a.nf * a.nmodes * 2;
    const long per_cu = std::max<long>(1, std::min<long>(kLdsPerCu / (long)lds, 16 / NW));
    const long wgs = std::min(total, per_cu * std::max(ncu, 8));
    const dim3 grid((unsigned)((wgs + 7) / 8 * 8)), block(64 * NW);
    if (kind == PLANE_FWD) hipLaunchKernelGGL((k_plane<RT, RR, CC, PLANE_FWD>), grid, block, lds, st, a);
    else if (kind == PLANE_ADJ) hipLaunchKernelGGL((k_plane<RT, RR, CC, PLANE_ADJ>), grid, block, lds, st, a);
    else if (kind == PLANE_WALL) hipLaunchKernelGGL((k_plane<RT, RR, CC, PLANE_WALL>), grid, block, lds, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_plane(int kind, const PlaneArgs& a, hipStream_t st)
{
    if (!plane_supported(a.my, a.mz) || a.nf < 0 || a.nf > kMaxFields) return hipErrorInvalidValue;
    if (a.nf == 0 || a.nmodes <= 0) return hipSuccess;
    const int n = (a.my > a.mz ? a.my : a.mz) - 2;
    switch ((n + 15) / 16) {
        case 1: return launch_plane_rt<1, 1, 1>(kind, a, st);
        case 2: return launch_plane_rt<2, 1, 2>(kind, a, st);
        case 3: return launch_plane_rt<3, 1, 3>(kind, a, st);
        case 4: return launch_plane_rt<4, 1, 4>(kind, a, st);
        case 5: return launch_plane_rt<5, 1, 5>(kind, a, st);
        case 6: return launch_plane_rt<6, 3, 3>(kind, a, st);
        case 7: return launch_plane_rt<7, 1, 7>(kind, a, st);
        case 8: return launch_plane_rt<8, 2, 4>(kind, a, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace duct
