// CPU emulation of the small-batch stepper (tests only): the kernel of
// sfg_fold.hip compiled as plain C++ (-DSFG_HOST_EMUL), one workgroup at a
// time with its threads concurrent, over the host layout of sfg_fold_host.cpp.
#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <thread>
#include <vector>

#include "sfg_internal.h"
#include "sfg_fold.hip"

thread_local sfg_dim3 threadIdx, blockIdx, blockDim;

namespace {
struct Barrier {
    std::mutex m;
    std::condition_variable cv;
    int expected = 0, arrived = 0;
    long gen = 0;
    void release() {
        arrived = 0;
        gen++;
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> lk(m);
        const long g = gen;
        if (++arrived == expected) release();
        else cv.wait(lk, [&] { return gen != g; });
    }
    void drop() {
        std::lock_guard<std::mutex> lk(m);
        expected--;
        if (arrived > 0 && arrived == expected) release();
    }
};
thread_local Barrier* cur_barrier = nullptr;

template <class T, bool OWN>
void run(const sfg::FoldArgs& a) {
#define SFG_FOLD(K, C) \
    if (a.t.slots == K && a.t.chunks == C) return sfg::fold_kernel<T, K, C, OWN>(a);
    SFG_FOLD_SHAPES(SFG_FOLD)
#undef SFG_FOLD
}
}  // namespace

void sfg_emul_syncthreads() { cur_barrier->wait(); }

// x: real SoA state (n, P), advanced in place; steps: per-parcel counts or
// null; given: read the parameters from arrays (as a plan does) instead of
// forming them in the kernel; traj: (nsteps + 1, P, n, 2) or null; split: the
// parcels of a first launch, the rest in a second (0: one launch).
extern "C" int emul_fold(int L, int64_t P, int prec, int procs, int scheme, int nsteps, double dt, const double* ugrad,
                         const double* tau, const double* gam0, const double* lam, double* x, int* steps, int steps_dec,
                         int* status, int given, float* traj, int64_t split) {
    const sfg::RealOperator& op = sfg::real_operator(L);
    const sfg::FoldLayout& f = sfg::fold_layout(L);
    const int nblk = L / 2 + 1;
    std::vector<double> A2(6 * 15), A4(36 * 15);
    for (int i = 0; i < 6; i++) for (int q = 0; q < 15; q++) A2[i * 15 + q] = op.A2[i][q];
    for (int i = 0; i < 36; i++) for (int q = 0; q < 15; q++) A4[i * 15 + q] = op.A4[i][q];
    sfg::FoldArgs a{};
    a.t.threads = f.threads; a.t.slots = f.slots; a.t.chunks = f.chunks; a.t.npat = f.npat; a.t.npairs = f.npairs; a.t.g0 = f.g0; a.t.gn = f.gn;
    a.t.src = f.src.data(); a.t.cnt = f.cnt.data(); a.t.base = f.base.data(); a.t.c = f.c.data(); a.t.pat = f.pat.data();
    a.t.pcode = f.pcode.data(); a.t.pos = f.pos.data(); a.t.chunk0 = f.chunk0.data(); a.t.chunkn = f.chunkn.data();
    a.t.blk = f.blk.data();
    sfg::ParamArgs& pa = a.pa;
    pa.P = P; pa.nblk = nblk; pa.nq = 15; pa.procs = procs; pa.iota = 1.0; pa.zeta = 0.0; pa.reg_nu = op.reg_nu;
    pa.ugrad = ugrad; pa.tau = tau; pa.gam0 = gam0; pa.lam = lam; pa.A2 = A2.data(); pa.A4 = A4.data();
    for (int b = 0; b < nblk; b++) pa.reg_shape[b] = op.reg_shape[b];
    std::vector<double> theta, omega, sl;
    if (given) {
        theta.resize(23 * P); omega.resize(15 * P); sl.resize(nblk * P);
        for (int64_t p = 0; p < P; p++) {
            sfg::ParcelParams q;
            double th[23];
            sfg::parcel_kinematics(pa, p, q);
            sfg::parcel_theta(pa, q, th);
            for (int i = 0; i < 23; i++) theta[i * P + p] = th[i];
            for (int i = 0; i < 15; i++) omega[i * P + p] = (procs & 2) ? sfg::parcel_omega(pa, q, i) : 0.0;
            for (int b = 0; b < nblk; b++) sl[b * P + p] = sfg::parcel_sl(pa, q, b);
        }
        pa.theta = theta.data(); pa.omega = omega.data(); pa.sl = sl.data();
    }
    a.n = op.n; a.scheme = scheme; a.nsteps = nsteps; a.use_ddrx = (procs & 2) ? 1 : 0;
    a.steps = steps; a.steps_dec = steps_dec; a.dt = dt; a.X = x; a.status = status; a.traj = traj;
    a.cre = op.cre.data(); a.cim = op.cim.data(); a.csgn = op.csgn.data(); a.cneg = op.cneg.data();
    for (int64_t p0 : {int64_t(0), split}) {
        a.p0 = p0;
        a.np = p0 || !split ? P - p0 : split;
        for (unsigned b = 0; b < sfg::fold_grid(a.np); b++) {
            Barrier bar;
            bar.expected = f.threads;
            std::vector<std::thread> th;
            for (int t = 0; t < f.threads; t++)
                th.emplace_back([&, t] {
                    blockIdx.x = b;
                    blockDim.x = (unsigned)f.threads;
                    threadIdx.x = (unsigned)t;
                    cur_barrier = &bar;
                    if (given) prec ? run<float, false>(a) : run<double, false>(a);
                    else prec ? run<float, true>(a) : run<double, true>(a);
                    bar.drop();
                });
            for (auto& t : th) t.join();
        }
        if (!split) break;
    }
    return 0;
}
