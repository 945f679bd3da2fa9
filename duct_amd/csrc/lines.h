// Derivative sums along y or z on whole complex planes (lines.hip).
#pragma once
#include "common.h"

namespace duct {

constexpr int kLineProds = 3;    // matrix products of a job
constexpr int kLineStages = 3;   // outputs of a job
constexpr int kLineTerms = 2;    // pointwise terms of an output
constexpr int kLineJobs = 6;     // jobs of a launch
constexpr int kLineMaxM = 288;   // 9 row tiles of 16 folded rows

// coef * A u along the launch's direction; mat: A folded (build_colloc); odd: J A J = -A (the
// first derivative), else J A J = A (the second).
struct LineProd {
    const d2v* src;
    const double* mat;
    double coef;
    int odd;
};
// (cr + crx xa^2) t + ci xa (i t), xa = alp (mode0 + mode) of the point's Fourier mode
struct LineTerm {
    const d2v* t;
    double cr, crx, ci;
};
// out = carried + the stage's products + terms + self + c0 (on the real part of Fourier mode 0);
// carried = keep * out of the job's previous stage.  self: a term on the operand of the stage's last
// product (of an earlier stage's if it has none), which is at hand (self.t is not read).
struct LineStage {
    d2v* out;
    double keep;                 // factor on out for the next stage
    double c0;
    int nprod, nterm;            // products of this stage (the job's next ones), terms
    LineTerm term[kLineTerms];
    LineTerm self;
};
// A job's stages run in order for each of its lines; the shares of the centre row (odd m) that a stage passes
// between the waves are guarded by the barriers of its products, or by one of its own if it has none.  An output
// may be one of its own stage's terms (read before it is written, at the same point), and no product's source or
// other job's term.
struct LineJob {
    LineProd prod[kLineProds];
    LineStage stage[kLineStages];
    int nstage;
};
struct LinesArgs {
    LineJob job[kLineJobs];
    int njobs, m, nmodes, mode0, dirz;
    double alp;
};
hipError_t launch_lines(const LinesArgs& a, hipStream_t st);

// out = coef * A src + beta * out along y or z; mat: A in fragments of 16 rows (build_frag); m <= kLineMaxM
struct LineOneArgs {
    const d2v* src;
    d2v* out;
    const double* mat;
    double coef, beta;
    int m, nmodes, dirz;
};
hipError_t launch_line(const LineOneArgs& a, hipStream_t st);

// The same sums along both directions in one launch, for small planes (k_sums).
constexpr int kSumProds = 3;     // products of a job per direction
constexpr int kSumTerms = 3;     // pointwise terms of an output
constexpr int kSumStages = 2;    // outputs of a job
constexpr int kSumJobs = 3;      // jobs of a launch
constexpr int kSumMaxM = 64;

// coef * A u along the list's direction; mat: A in fragments of 16 rows (build_frag of build_colloc)
struct SumProd {
    const d2v* src;
    const double* mat;
    double coef;
};
// out = keep * the previous stage's out + the stage's products + terms + c0 (on the real part of Fourier
// mode 0).  The terms of a job are read before its outputs are written, at the same point; no output is a
// product's source or another job's term.
struct SumStage {
    d2v* out;
    double keep, c0;
    int nprod[2], nterm;         // products along y, z (the job's next ones), terms
    LineTerm term[kSumTerms];
};
struct SumJob {
    SumProd prod[2][kSumProds];  // along y, along z
    SumStage stage[kSumStages];
    int nstage;
};
struct SumArgs {
    SumJob job[kSumJobs];
    int njobs, m, nmodes;
    double alp;
};
// planes small and few enough for k_sums
bool sums_supported(int m, int nmodes);
hipError_t launch_sums(const SumArgs& a, hipStream_t st);

}  // namespace duct
