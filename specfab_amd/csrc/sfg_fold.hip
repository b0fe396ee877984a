// Small-batch stepper: one workgroup per parcel.
//
// The steppers of sfg_fast_* step 64 parcels per workgroup, so a batch of a
// few thousand parcels leaves most of the chip idle and every stage costs the
// whole operator's instruction stream.  Here a parcel's operator is summed
// over its 23 parameters once per launch into one real 2 x 2 block per coupled
// pair of complex coefficients (1,187 blocks instead of 8,581 terms at L =
// 12), which stay in registers: thread t holds up to K sources of one target
// (sfg_fold.h), so a stage is K LDS reads of a complex coefficient and 4 K
// FMAs per thread, a reduction of the target's chunks through LDS and the
// Runge-Kutta update by the thread of each row.  <D> is one more target.
#include <algorithm>

#include "sfg_fold.h"
#include "sfg_params.h"

namespace sfg {

namespace {

template <class T> struct Vec2;
template <> struct Vec2<double> { typedef double type __attribute__((vector_size(16))); };
template <> struct Vec2<float> { typedef float type __attribute__((vector_size(8))); };

}  // namespace

// waves per SIMD that the registers are limited to: four in FP64 (4 K operator
// values of two registers; forming the operator parameters takes 122), in FP32
// as many as 4 K + 50 registers allow, where what the parameters need beyond
// that spills once per launch (8,000 parcels, L = 12, ten steps: 305 -> 207 us;
// the same in FP64 costs more than it gives: 341 -> 355 us)
constexpr int fold_waves(int bytes, int K) { return bytes == 8 ? 4 : (K > 6 ? 5 : 512 / (4 * K + 50)); }

// K sources per thread, at most C chunks per target, OWN: the workgroup forms
// its operator parameters (else they are read from the params kernel's arrays)
template <class T, int K, int C, bool OWN>
__global__ void __launch_bounds__(FOLD_THREADS, fold_waves(sizeof(T), K)) fold_kernel(FoldArgs a) {
    typedef typename Vec2<T>::type V2;
    __shared__ V2 xs[FOLD_PAIRS + 1];
    __shared__ V2 part[FOLD_THREADS];
    __shared__ T w4[FOLD_PATTERNS][4];
    __shared__ double th[NPAR_K + 15 + 11];
    const int tid = threadIdx.x, NT = a.t.threads;
    const int64_t P = a.pa.P;
    // workgroups go round the eight XCDs: neighbouring parcels share 64-byte
    // lines of the state rows, so each XCD takes one contiguous range
    const int64_t chunk = (a.np + 7) / 8, i0 = (int64_t)(blockIdx.x % 8) * chunk + blockIdx.x / 8, p = a.p0 + i0;
    if (i0 >= a.np || (int64_t)(blockIdx.x / 8) >= chunk) return;
    const int rem = a.steps ? a.steps[p] : a.nsteps;
    const int ns = (a.steps && a.steps_dec) ? (rem < a.nsteps ? rem : a.nsteps) : rem;
    const bool row = tid < a.n;
    double s = row ? a.X[(int64_t)tid * P + p] : 0.0;
    if (ns > 0) {   // uniform over the workgroup
        T* xf = (T*)xs;
        for (int i = tid; i < 2 * (FOLD_PAIRS + 1); i += NT) xf[i] = (T)0;
        const int nblk = a.pa.nblk;
        if constexpr (!OWN) {
            for (int i = tid; i < NPAR_K + 15 + nblk; i += NT)
                th[i] = i < NPAR_K ? a.pa.theta[(int64_t)i * P + p]
                                   : (i < NPAR_K + 15 ? a.pa.omega[(int64_t)(i - NPAR_K) * P + p]
                                                      : a.pa.sl[(int64_t)(i - NPAR_K - 15) * P + p]);
        } else if (tid < 64) {
            ParcelParams q;
            parcel_kinematics(a.pa, p, q);
            double t[NPAR_K];
            parcel_theta(a.pa, q, t);
            if (tid == 0)
                for (int i = 0; i < NPAR_K; i++) th[i] = t[i];
            if (tid < 15) th[NPAR_K + tid] = (a.pa.procs & 2) && tid < a.pa.nq ? parcel_omega(a.pa, q, tid) : 0.0;
            if (tid < nblk) th[NPAR_K + 15 + tid] = parcel_sl(a.pa, q, tid);
        }
        __syncthreads();
        for (int i = tid; i < 4 * a.t.npat; i += NT) {
            const int code = a.t.pcode[i];
            w4[i / 4][i % 4] = code > 0 ? (T)th[code - 1] : (code < 0 ? (T)-th[-code - 1] : (T)0);
        }
        int pos = 0, c0 = 0, cn = 0;
        T sl = 0;
        if (row) {
            pos = a.t.pos[tid];
            c0 = a.t.chunk0[tid];
            cn = a.t.chunkn[tid];
            sl = (T)th[NPAR_K + 15 + a.t.blk[tid]];
            xf[pos] = (T)s;
        }
        __syncthreads();
        // the operator, summed over its weights
        T M[K][4];
        int src[K];
        const int wv = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid & 63;
#pragma unroll
        for (int j = 0; j < K; j++) {
            src[j] = a.t.src[j * NT + tid];
#pragma unroll
            for (int q = 0; q < 4; q++) M[j][q] = (T)0;
            const int cnt = a.t.cnt[wv * K + j], base = a.t.base[wv * K + j];
            for (int e = 0; e < cnt; e++) {
                const T c = (T)a.t.c[(int64_t)(base + e) * 64 + lane];
                const T* w = w4[a.t.pat[(int64_t)(base + e) * 64 + lane]];
#pragma unroll
                for (int q = 0; q < 4; q++) M[j][q] = fma(c, w[q], M[j][q]);
            }
        }
        const int nstage = a.scheme ? 4 : 1;
        const double h = a.dt;
        const T* pf = (const T*)part;
        const int g0 = a.t.g0, gn = a.use_ddrx ? a.t.gn : 0;
        T y = 0;
        for (int step = 0; step < ns; step++) {
            for (int k = 0; k < nstage; k++) {
                T re = 0, im = 0;
                // read before the barrier: the rows' threads overwrite xs after it
                const T xr = xf[pos], ix0 = (T)1 / xf[0];
#pragma unroll
                for (int j = 0; j < K; j++) {
                    const V2 x = xs[src[j]];
                    re = fma(M[j][0], x[0], re);
                    re = fma(M[j][1], x[1], re);
                    im = fma(M[j][2], x[0], im);
                    im = fma(M[j][3], x[1], im);
                }
                part[tid] = V2{re, im};
                __syncthreads();
                if (row) {
                    T acc = 0, g = 0;
#pragma unroll
                    for (int i = 0; i < C; i++) acc += i < cn ? pf[2 * (c0 + i) + (pos & 1)] : (T)0;
#pragma unroll
                    for (int i = 0; i < FOLD_G; i++) g += i < gn ? pf[2 * (g0 + i)] : (T)0;
                    if (gn) g *= ix0;
                    const T f = fma(sl - g, xr, acc);
                    const bool last = k == nstage - 1;
                    const T cy = (T)(nstage == 1 ? h : (k == 0 || k == 3 ? h / 6 : h / 3)), cx = (T)(k == 2 ? h : h / 2);
                    y = fma(cy, f, y);
                    if (last) {
                        s += (double)y;
                        y = 0;
                        if (a.traj) s = (double)(float)s;
                    }
                    xf[pos] = last ? (T)s : fma(cx, f, (T)s);
                }
                __syncthreads();
            }
            if (a.traj && row) {   // complex row tid; xs is next written after the next barrier
                float* o = a.traj + (((int64_t)(step + 1) * P + p) * a.n + tid) * 2;
                const int ci = a.cim[tid];
                const float sg = (float)a.csgn[tid];
                o[0] = sg * (float)xf[a.t.pos[a.cre[tid]]];
                o[1] = ci < 0 ? 0.0f : (a.cneg[tid] ? -sg : sg) * (float)xf[a.t.pos[ci]];
            }
        }
        if (row) a.X[(int64_t)tid * P + p] = s;
    }
    if (row && a.status && !isfinite(s)) atomicOr(a.status + p, 1);
    if (tid == 0 && a.steps && a.steps_dec) a.steps[p] = rem - ns;
}

#ifndef SFG_HOST_EMUL
const void* fold_kernel_fn(const FoldTab& t, int prec, bool own) {
    if (t.threads > FOLD_THREADS || t.npairs > FOLD_PAIRS || t.npat > FOLD_PATTERNS || t.gn > FOLD_G) return nullptr;
#define SFG_FOLD(K, C)                                                                                              \
    if (t.slots == K && t.chunks == C) {                                                                            \
        if (prec) return own ? (const void*)&fold_kernel<float, K, C, true> : (const void*)&fold_kernel<float, K, C, false>; \
        return own ? (const void*)&fold_kernel<double, K, C, true> : (const void*)&fold_kernel<double, K, C, false>; \
    }
    SFG_FOLD_SHAPES(SFG_FOLD)
#undef SFG_FOLD
    return nullptr;
}

hipError_t launch_fold(const FoldArgs& a, int prec, hipStream_t s) {
    const void* fn = fold_kernel_fn(a.t, prec, a.pa.theta == nullptr);
    if (!fn || a.n > a.t.threads) return hipErrorInvalidValue;
    FoldArgs b = a;
    void* args[] = {&b};
    const int64_t most = fold_most(a.t.threads);
    for (b.p0 = a.p0; b.p0 < a.p0 + a.np; b.p0 += most) {
        b.np = std::min(most, a.p0 + a.np - b.p0);
        const hipError_t e = hipLaunchKernel(fn, dim3(fold_grid(b.np)), dim3(a.t.threads), args, 0, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
#endif

}  // namespace sfg
