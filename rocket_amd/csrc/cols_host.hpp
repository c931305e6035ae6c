// Launchers of the extraction chain's column passes (cols.hip).
#pragma once

#include "fft_device.hpp"
#include "prnu_internal.hpp"

namespace prnu {

int launch_cols_power(const FftDesc &d, const float2 *A, int lda, int wh, float2 *B, float *P, int64_t plane, int nb,
                      hipStream_t st);
int launch_cols_inverse(const FftDesc &d, const float2 *B, const float *S, int wh, float2 *A, int lda,
                        int64_t plane, int nb, hipStream_t st);
int launch_cols_spectrum(const FftDesc &d, const float2 *A, int lda, int wh, int64_t plane, float2 *out,
                         int64_t out_stride, int nb, hipStream_t st);

}  // namespace prnu
