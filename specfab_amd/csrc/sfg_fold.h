// Small-batch stepper: one workgroup per parcel, the operator folded over its
// parameters into one value per coupled pair, held in registers.
#pragma once
#include <vector>

#include "sfg_kernels.h"

namespace sfg {

// How the operator of one truncation is laid out over the threads of a
// workgroup (host side, built once per L by fold_layout).  A "pair" is the
// complex coefficient (Re, Im) of n_l^m, m >= 0; thread t evaluates up to
// `slots` sources of one target pair (a chunk), the chunks of a target are
// consecutive threads.  The weighted sum of the first 15 rows that <D> needs
// is one more target.
struct FoldLayout {
    int L = 0, n = 0, npairs = 0, threads = 0, slots = 0, npat = 0;
    int g0 = 0, gn = 0;                 // chunks (threads) of the <D> sum
    int chunks = 0;                     // most chunks of a target
    std::vector<int> src;               // [slot][thread] source pair
    std::vector<int> cnt, base;         // [wave][slot] entries of the slot (largest of the wave's), first row
    std::vector<double> c;              // [row][lane] coupling value (0 past a thread's own entries)
    std::vector<unsigned char> pat;     // [row][lane] weight pattern
    std::vector<signed char> pcode;     // [pattern][4] weight of cell (row part, source part): +-(index + 1), 0 none;
                                        // index: theta 0..22, omega 23..37
    std::vector<int> pos;               // [row] 2 * pair + part
    std::vector<int> chunk0, chunkn;    // [row] chunks of the row's target
    std::vector<int> blk;               // [row] l / 2
};
const FoldLayout& fold_layout(int L);
constexpr int FOLD_PAIRS = 121;         // pairs at L = 20
constexpr int FOLD_THREADS = 512;
constexpr int FOLD_PATTERNS = 64;
constexpr int FOLD_G = 5;               // most chunks of the <D> sum
// (slots, most chunks of a target) of every truncation
#define SFG_FOLD_SHAPES(X) X(2, 5) X(5, 4) X(9, 3) X(8, 5) X(6, 7) X(8, 6) X(5, 9) X(7, 7) X(9, 5)

// the same tables on the device
struct FoldTab {
    int threads = 0, slots = 0, chunks = 0, npat = 0, npairs = 0, g0 = 0, gn = 0;
    const int* src = nullptr;
    const int *cnt = nullptr, *base = nullptr;
    const double* c = nullptr;
    const unsigned char* pat = nullptr;
    const signed char* pcode = nullptr;
    const int *pos = nullptr, *chunk0 = nullptr, *chunkn = nullptr, *blk = nullptr;
};

struct FoldArgs {
    FoldTab t;
    ParamArgs pa;        // kinematics; pa.theta null: the workgroup forms the parameters itself,
                         // else they are read from pa.theta, pa.omega, pa.sl
    int64_t p0, np;      // the launch's parcels p0 .. p0 + np - 1 of pa.P
    int n, scheme, nsteps, use_ddrx;
    int* steps;          // as EvolveArgs
    int steps_dec;
    double dt;
    double* X;
    int* status;
    float* traj;         // or null: (nsteps + 1, P, n complex) float pairs, see evolve_trajectory
    const int *cre, *cim, *csgn, *cneg;   // complex rows of the trajectory (as state_to_nlm)
};

// Batches up to this many parcels take the small-batch stepper: its time grows
// with the parcels from about 250 on (one per CU), while a generated stepper's
// stays until all CUs hold a group of 64.  The line is where both measured the
// same, which is a ratio of two functions linear in the stages of the launch: the
// generated steppers' second launch, for the parameters, and the folding of the
// operator are paid once.
int64_t fold_limit(int L, int prec, int64_t stages);

const void* fold_kernel_fn(const FoldTab& t, int prec, bool own);
inline unsigned fold_grid(int64_t np) { return (unsigned)((np + 7) / 8 * 8); }
// parcels of one launch at most: the runtime takes fewer than 2^32 work-items
inline int64_t fold_most(int threads) { return (((int64_t(1) << 32) - 1) / threads) / 8 * 8; }
hipError_t launch_fold(const FoldArgs& a, int prec, hipStream_t s);

}  // namespace sfg
