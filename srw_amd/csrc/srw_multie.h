// srw_multie.h - partially coherent (multi-electron) accumulation kernels.
#pragma once
#include <hip/hip_runtime.h>

// Propagated mesh of one electron.
struct srwm_emesh {
    double xStart, xStep, zStart, zStep;
    int nx, nz;
};

// Result mesh.
struct srwm_rmesh {
    double xStart, xStep, zStart, zStep;
    int nx, nz;
};

extern "C" {
// Srep (optional): electrons j of the batch in groups of perRep also add
// their weighted intensity into Srep[(j / perRep) * nr + point] (per-replicate
// sums of the randomized quasi-Monte Carlo sampler).
int srwm_launch_accum(const float* I, long long iStride, const srwm_emesh* em, const float* w, int nb,
                      srwm_rmesh rm, double* S1, double* S2, double* norm2, double* Srep, int perRep,
                      hipStream_t st);
// Sums of the error estimate after n electrons: out[0] = sum S1^2, out[1] = sum
// S2, out[2] = the squared deviations of the R replicate means from the mean
// over points and replicates (0 when Srep is nullptr), in work[0..2]; work
// holds SRWM_ERR_WORK doubles.
#define SRWM_ERR_WORK (3 + 3 * 512)
int srwm_launch_err_sums(const double* S1, const double* S2, const double* Srep, int R, double n, long long nr,
                         double* work, hipStream_t st);
int srwm_launch_stokes_out(const double* S1, double scale, long long n, float* out, hipStream_t st);
}
