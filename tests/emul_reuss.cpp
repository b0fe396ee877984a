// CPU build of the two Reuss acoustic tensors of sfg_wave.hip (tests only).
#include "sfg_wave.hip"

thread_local sfg_dim3 threadIdx, blockIdx, blockDim, gridDim;
void sfg_emul_syncthreads() {}

// N compliances: a2 (N, 6) Mandel, a4 entries (N, 15), coefficients k (N, 5);
// Q (N, 9) by the symmetric elimination (ok 0 where it passes the matrix on)
// and by the pivoted solve
extern "C" void emul_reuss(int64_t N, const double* a2v, const double* u, const double* k, double* Qs, int* ok, double* Ql) {
    for (int64_t i = 0; i < N; i++) {
        double Q[9];
        ok[i] = sfg::qnorm_reuss_spd(a2v + 6 * i, u + 15 * i, k + 5 * i, Q);
        for (int j = 0; j < 9; j++) Qs[9 * i + j] = Q[j];
        sfg::qnorm_reuss(a2v + 6 * i, u + 15 * i, k + 5 * i, Q);
        for (int j = 0; j < 9; j++) Ql[9 * i + j] = Q[j];
    }
}
