// The extraction chain's column passes (cols_device.hpp): forward with the
// power spectrum, scaled inverse, and the spectrum's in-place forward pass.
// Each frame's half spectrum is a row-major plane A of h rows of wh = w/2 + 1
// values, lda apart; B, P and S are transposed (column j at j * h).
#include "prnu_internal.hpp"
#include "cols_device.hpp"
#include "cols_host.hpp"

namespace prnu {
namespace {

// Forward FFT of every column of A into B and |F|^2 into P.  grid (8 per, frames)
template <class P>
__global__ __launch_bounds__(P::kThreads) void cols_power_kernel(P pl, const float2 *__restrict__ A, int lda, int wh,
                                                                  float2 *__restrict__ B, float *__restrict__ Pw,
                                                                  int64_t plane, int per) {
    extern __shared__ __attribute__((aligned(16))) float2 cols_smem[];
    const int strip = cols_strip<P>(per);
    if (strip >= (wh + P::COLS - 1) / P::COLS) return;
    const int j0 = strip * P::COLS;
    stage_cols(pl, A + (int64_t)blockIdx.y * plane, lda, j0, wh, cols_smem);
    const int c = (int)threadIdx.x / P::T, col = j0 + c, n = pl.n();
    float2 *buf = cols_smem + c * pl.stride();
    const bool store = col < wh;
    float2 *row = B + (int64_t)blockIdx.y * plane + (int64_t)col * n;
    float *prow = Pw + (int64_t)blockIdx.y * plane + (int64_t)col * n;
    pl.template run<-1, true>(
        buf, [&](int i) { return buf[pl.pad(i)]; },
        [&](int j, float2 f) {
            if (store) {
                row[j] = f;
                prow[j] = f.x * f.x + f.y * f.y;
            }
        });
}

// Column r of B times its row of the scale S (column 0: the mean of S(0, c) and
// S(0, -c), which the other rows hold already), inverse FFT, into A's columns.
// grid (8 per, frames)
template <class P>
__global__ __launch_bounds__(P::kThreads) void cols_inverse_kernel(P pl, const float2 *__restrict__ B,
                                                                   const float *__restrict__ S, int wh,
                                                                   float2 *__restrict__ A, int lda, int64_t plane,
                                                                   int per) {
    extern __shared__ __attribute__((aligned(16))) float2 cols_smem[];
    const int strip = cols_strip<P>(per);
    if (strip >= (wh + P::COLS - 1) / P::COLS) return;
    const int j0 = strip * P::COLS, n = pl.n();
    const int c = (int)threadIdx.x / P::T;
    const int col = min(j0 + c, wh - 1);  // a column past wh transforms the last one again and stores nothing
    float2 *buf = cols_smem + c * pl.stride();
    const float2 *row = B + (int64_t)blockIdx.y * plane + (int64_t)col * n;
    const float *srow = S + (int64_t)blockIdx.y * plane + (int64_t)col * n;
    // column 0 is its own mirror; the others add their own value again (no branch
    // around the loads, which then stay batched)
    const int flip = col == 0 ? -1 : 1, at = col == 0 ? n : 0;
    pl.template run<1, false>(
        buf,
        [&](int j) { return cscale(row[j], 0.5f * (srow[j] + srow[j == 0 ? 0 : at + flip * j])); },
        [&](int j, float2 f) { buf[pl.pad(j)] = f; });  // the last pass has read buf before it writes
    __syncthreads();
    unstage_cols(pl, cols_smem, A + (int64_t)blockIdx.y * plane, lda, j0, wh);
}

// Forward FFT of every column of A into the same columns of out (rows wh
// apart, frames out_stride apart).  grid (8 per, frames)
template <class P>
__global__ __launch_bounds__(P::kThreads) void cols_spectrum_kernel(P pl, const float2 *__restrict__ A, int lda,
                                                                     int wh, int64_t plane, float2 *__restrict__ out,
                                                                     int64_t out_stride, int per) {
    extern __shared__ __attribute__((aligned(16))) float2 cols_smem[];
    const int strip = cols_strip<P>(per);
    if (strip >= (wh + P::COLS - 1) / P::COLS) return;
    const int j0 = strip * P::COLS;
    stage_cols(pl, A + (int64_t)blockIdx.y * plane, lda, j0, wh, cols_smem);
    float2 *buf = cols_smem + (int)threadIdx.x / P::T * pl.stride();
    // the last pass has read buf before it writes (a barrier between)
    pl.template run<-1, true>(
        buf, [&](int i) { return buf[pl.pad(i)]; }, [&](int j, float2 f) { buf[pl.pad(j)] = f; });
    __syncthreads();
    unstage_cols(pl, cols_smem, out + (int64_t)blockIdx.y * out_stride, wh, j0, wh);
}

}  // namespace

int launch_cols_power(const FftDesc &d, const float2 *A, int lda, int wh, float2 *B, float *P, int64_t plane, int nb,
                      hipStream_t st) {
    return with_cols_plan(d, [&](auto pl) -> int {
        typedef decltype(pl) Plan;
        const int per = cols_per<Plan>(wh);
        hipLaunchKernelGGL(cols_power_kernel<Plan>, dim3(8 * per, nb), dim3(Plan::kThreads), cols_lds(pl), st, pl, A,
                           lda, wh, B, P, plane, per);
        PRNU_CHECK_LAUNCH();
        return PRNU_OK;
    });
}

int launch_cols_inverse(const FftDesc &d, const float2 *B, const float *S, int wh, float2 *A, int lda,
                        int64_t plane, int nb, hipStream_t st) {
    return with_cols_plan(d, [&](auto pl) -> int {
        typedef decltype(pl) Plan;
        const int per = cols_per<Plan>(wh);
        hipLaunchKernelGGL(cols_inverse_kernel<Plan>, dim3(8 * per, nb), dim3(Plan::kThreads), cols_lds(pl), st, pl, B,
                           S, wh, A, lda, plane, per);
        PRNU_CHECK_LAUNCH();
        return PRNU_OK;
    });
}

int launch_cols_spectrum(const FftDesc &d, const float2 *A, int lda, int wh, int64_t plane, float2 *out,
                         int64_t out_stride, int nb, hipStream_t st) {
    return with_cols_plan(d, [&](auto pl) -> int {
        typedef decltype(pl) Plan;
        const int per = cols_per<Plan>(wh);
        hipLaunchKernelGGL(cols_spectrum_kernel<Plan>, dim3(8 * per, nb), dim3(Plan::kThreads), cols_lds(pl), st, pl, A,
                           lda, wh, plane, out, out_stride, per);
        PRNU_CHECK_LAUNCH();
        return PRNU_OK;
    });
}

}  // namespace prnu
