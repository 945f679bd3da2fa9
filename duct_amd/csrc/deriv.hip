// Collocation derivative products on whole complex(8) planes:
//   y:  out(y, z) = beta out + scal sum_k D(y, k) u(k, z)      (D u, along the contiguous y)
//   z:  out(y, z) = beta out + scal sum_k D(z, k) u(y, k)      (u D^T, along z)
// for every plane of one or more fields (derivyz / transyz applied along y or z,
// chebyshev.f90:1-540, as a dense product with the matrices of the m CGL nodes).
//
// Work decomposition: a workgroup owns one 16-line slab of one plane of one op, the lines being
// the direction that is not contracted (16 z for y, 16 y for z), and stages that slab of u, all
// K = 16 ceil(m/16) contraction points, re and im, in LDS once. Its three waves then cover the
// NT = ceil(m/16) output tiles along the contracted direction, TPW tiles each, streaming the
// matrix fragments from L2. At m = 129 the padding costs (144/129)^3 = 1.4x the useful MFMA work,
// against 2.5x for 64 x 64 output blocks, and a slab is 37 KB of LDS, so four workgroups share a
// CU (static LDS sized for NP <= 48 TPW).
//
// One launch runs a list of independent ops (its own field, matrix, direction, scale and beta
// each): a single field's planes give about two waves per SIMD at m = 129, too few to hide the
// L2 latency of the fragments or to balance the CUs, so callers group the products that do not
// depend on each other.
#include "common.h"
#include "proj_lp.h"

namespace duct {

namespace {
constexpr int kWaves = 3;
constexpr int kThreads = 64 * kWaves;
}  // namespace

template <bool DIRZ, int TPW>
__device__ __forceinline__ void cline_slab(const d2v* __restrict__ U, d2v* O, const double* Dfrag, int m, int NP,
                                           int lb, double scal, double beta, double* slab)
{
    const int NT = NP / 16, K = NP, LDK = K + 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: scalar branches only
    const int l16 = lane & 15, l4 = lane >> 4;
    const int L0 = lb * 16;

    // stage the slab: y: u(k, z = L0 + l) is contiguous in k;  z: u(y = L0 + l, k) has y contiguous.
    // All loads of a thread are issued before its LDS stores, so their latencies overlap; they are
    // unconditional (points outside the plane read u(0, 0) and are stored as zeros).
    double* Sre = slab;
    double* Sim = slab + 16 * LDK;
    constexpr int IT = (16 * 16 * kWaves * TPW + kThreads - 1) / kThreads;
    const float invK = 1.0f / (float)K;       // e / K below is exact: e < 2^13, K <= 288
    d2v v[IT];
    bool ok[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = tid + it * kThreads;
        int l, k;
        if constexpr (DIRZ) {
            l = e & 15;
            k = e >> 4;
        } else {
            l = (int)(((float)e + 0.5f) * invK);
            k = e - l * K;
        }
        ok[it] = e < 16 * K && L0 + l < m && k < m;
        const size_t idx = DIRZ ? (size_t)(L0 + l) + (size_t)k * m : (size_t)k + (size_t)(L0 + l) * m;
        v[it] = U[ok[it] ? idx : 0];
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int e = tid + it * kThreads;
        if (e < 16 * K) {
            int l, k;
            if constexpr (DIRZ) {
                l = e & 15;
                k = e >> 4;
            } else {
                l = (int)(((float)e + 0.5f) * invK);
                k = e - l * K;
            }
            Sre[l * LDK + k] = ok[it] ? v[it][0] : 0.0;
            Sim[l * LDK + k] = ok[it] ? v[it][1] : 0.0;
        }
    }
    __syncthreads();

    // tiles of this wave: t = wave + kWaves s
    const d2v* Df = (const d2v*)Dfrag;
    d4v acc[TPW][2];
#pragma unroll
    for (int s = 0; s < TPW; ++s) acc[s][0] = acc[s][1] = d4v{0.0, 0.0, 0.0, 0.0};
    const int KP = K / 8;                         // fragment pairs of k-steps
    // Tiles past NT (when 3 TPW > NT) recompute the last tile and are not stored: the loop has
    // no branches, so the prefetch of the next pair's fragments overlaps this pair's products.
    const d2v* Dt[TPW];
#pragma unroll
    for (int s = 0; s < TPW; ++s) {
        const int t = wave + kWaves * s;
        Dt[s] = Df + (size_t)(t < NT ? t : NT - 1) * KP * 64 + lane;
    }
    d2v df[TPW], dn[TPW];                         // this pair's fragments, the next pair's (prefetched)
    auto fetch = [&](int kp, d2v (&dst)[TPW]) {
#pragma unroll
        for (int s = 0; s < TPW; ++s) dst[s] = Dt[s][(size_t)kp * 64];
    };
    // One fragment pair: prefetch the next pair's fragments into `nxt`, then the products with `cur`.
    // The loop below calls it twice per iteration with the buffers swapped (KP = NP / 8 is even), so
    // the prefetched fragments are never copied: a copy at the bottom of the loop would wait for the
    // very loads it rotates in (and the compiler does not unroll loops holding MFMAs when that would
    // need a remainder).
    auto step = [&](int kp, d2v (&cur)[TPW], d2v (&nxt)[TPW]) {
        fetch(kp + 1 < KP ? kp + 1 : kp, nxt);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = (kp * 2 + h) * 4 + l4;
            const double ure = Sre[l16 * LDK + k], uim = Sim[l16 * LDK + k];
#pragma unroll
            for (int s = 0; s < TPW; ++s) {
                if constexpr (!DIRZ) {
                    // acc[i = z][j = y] = sum_k u(k, z) D(y, k): A = slab [z][k], B = D fragment [k][y]
                    acc[s][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ure, cur[s][h], acc[s][0], 0, 0, 0);
                    acc[s][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(uim, cur[s][h], acc[s][1], 0, 0, 0);
                } else {
                    // acc[i = z][j = y] = sum_k D(z, k) u(y, k): A = D fragment [z][k], B = slab [k][y]
                    acc[s][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s][h], ure, acc[s][0], 0, 0, 0);
                    acc[s][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s][h], uim, acc[s][1], 0, 0, 0);
                }
            }
        }
    };
    fetch(0, df);
    for (int kp = 0; kp < KP; kp += 2) {
        step(kp, df, dn);
        step(kp + 1, dn, df);
    }

    // epilogue: D[i][j] in lane j + 16 (i % 4), element i / 4; y runs along lanes (coalesced).
    // The accumulated outputs are all loaded before the first store: out and u may be the same
    // allocation for the compiler, which would otherwise serialise every load behind a store.
    d2v ov[TPW][4];
    if (beta != 0.0) {
#pragma unroll
        for (int s = 0; s < TPW; ++s) {
            const int t = wave + kWaves * s;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 4 * e + l4;
                const int z = DIRZ ? 16 * t + i : L0 + i;
                const int y = DIRZ ? L0 + l16 : 16 * t + l16;
                ov[s][e] = (t < NT && z < m && y < m) ? O[(size_t)y + (size_t)z * m] : d2v{0.0, 0.0};
            }
        }
    }
#pragma unroll
    for (int s = 0; s < TPW; ++s) {
        const int t = wave + kWaves * s;
        if (t >= NT) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 4 * e + l4;
            const int z = DIRZ ? 16 * t + i : L0 + i;
            const int y = DIRZ ? L0 + l16 : 16 * t + l16;
            if (z < m && y < m) {
                d2v r = {scal * acc[s][0][e], scal * acc[s][1][e]};
                if (beta != 0.0) r += beta * ov[s][e];
                O[(size_t)y + (size_t)z * m] = r;
            }
        }
    }
}

template <int TPW>
__global__ __launch_bounds__(kThreads, 2) void k_cline(ClineArgs a)
{
    __shared__ double slab[2 * 16 * (16 * kWaves * TPW + 1)];   // [part][line 0..15][k 0..K-1], stride LDK
    const int NT = a.NP / 16, m = a.m;
    const long per_op = (long)a.nmodes * NT;
    const int o = (int)(blockIdx.x / per_op);
    const long r = blockIdx.x % per_op;
    const int mode = (int)(r / NT), lb = (int)(r % NT);
    const ClineOp& op = a.op[o];
    const d2v* U = op.in + (size_t)mode * m * m;
    d2v* O = op.out + (size_t)mode * m * m;
    if (op.dirz)
        cline_slab<true, TPW>(U, O, op.Dfrag, m, a.NP, lb, op.scal, op.beta, slab);
    else
        cline_slab<false, TPW>(U, O, op.Dfrag, m, a.NP, lb, op.scal, op.beta, slab);
}

hipError_t launch_cline_ops(const ClineArgs& a, hipStream_t st)
{
    // the matrix fragments cover NP = 16 ceil(m/16) >= m; at most 6 tiles per wave (m <= 288)
    if (a.NP % 16 || a.NP < a.m || a.NP > 16 * kWaves * 6 || a.nops < 0 || a.nops > kMaxClineOps)
        return hipErrorInvalidValue;
    for (int i = 0; i < a.nops; ++i) {
        if (!a.op[i].in || !a.op[i].out || !a.op[i].Dfrag) return hipErrorInvalidValue;
        for (int j = 0; j < a.nops; ++j)   // every output is written by one op and read by no other
            if ((j != i && a.op[j].out == a.op[i].out) || a.op[j].in == a.op[i].out) return hipErrorInvalidValue;
    }
    if (a.nops == 0 || a.nmodes <= 0) return hipSuccess;
    const int NT = a.NP / 16;
    const long blocks = (long)a.nops * a.nmodes * NT;
    switch ((NT + kWaves - 1) / kWaves) {
        case 1: hipLaunchKernelGGL(k_cline<1>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 2: hipLaunchKernelGGL(k_cline<2>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 3: hipLaunchKernelGGL(k_cline<3>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 4: hipLaunchKernelGGL(k_cline<4>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 5: hipLaunchKernelGGL(k_cline<5>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        case 6: hipLaunchKernelGGL(k_cline<6>, dim3((unsigned)blocks), dim3(kThreads), 0, st, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_cline(int dirz, const CollocArgs& a, hipStream_t st)
{
    if (a.g.nf < 1 || a.g.nf > kMaxClineOps) return hipErrorInvalidValue;
    ClineArgs c{};
    c.nops = a.g.nf;
    c.nmodes = a.g.nmodes;
    c.m = a.g.m;
    c.NP = a.NP;
    for (int f = 0; f < a.g.nf; ++f) c.op[f] = ClineOp{a.g.in[f], a.g.out[f], a.Dfrag, a.scal, a.beta, dirz};
    return launch_cline_ops(c, st);
}

}  // namespace duct
