// Column transforms of a row-major complex plane, strip by strip through LDS.
//
// A workgroup takes a strip of COLS adjacent columns: it stages
// them row by row (pieces of COLS values of each row, two adjacent columns per
// thread) into one padded LDS buffer per column, T threads transform each
// column there, and the results leave as the caller likes.  Workgroup g takes
// strip (g mod 8) * per + g / 8: workgroup ids go to the 8 XCDs round-robin,
// so the strips that share 128-byte lines of a row run on one XCD and its L2
// serves each line once.
//
// Why strips: a column pass over a transposed plane needs two transposes
// around it (16 bytes per value read and written twice more; four frames of
// 4000x3000: 160 us), and a column read straight from the plane takes 64 lines
// per load.  A strip is 8 columns of up to 1023 values or 2 of up to 8192 (136
// KiB of LDS), at 16 values per thread (ColsRt); the hot lengths 1024 and 1536
// have compile-time plans on one wave per column, 8 columns a strip (ColsC).
#pragma once

#include "fft_device.hpp"

namespace prnu {

// Columns of N values, N known at compile time, one wave each.
template <int N>
struct ColsC {
    static constexpr int T = 64, COLS = 8, kThreads = T * COLS;
    static constexpr bool kConst = true;
    const float2 *tw;
    __host__ __device__ static constexpr int n() { return N; }
    // +4 spreads the staging writes of the 8 buffers over the banks
    __host__ __device__ static constexpr int stride() { return fft_wave_lds<N>() + 4; }
    __device__ static int pad(int i) { return fft_wave_pad<FftWavePlan<N>::kPadShift>(i); }
    template <int DIR, bool SYNC_FIRST, class Get, class Put>
    __device__ void run(float2 *buf, Get get, Put put) const {
        fft_wave<DIR, N, SYNC_FIRST, true>(buf, tw, get, put);
    }
};

// Columns of d.n <= 16 T values on T threads each.
template <int T_, int COLS_>
struct ColsRt {
    static constexpr int T = T_, COLS = COLS_, kThreads = T * COLS;
    static constexpr bool kConst = false;
    FftDesc d;
    __host__ __device__ int n() const { return d.n; }
    __host__ __device__ int stride() const { return fft_pad_lds(d.n) + 4; }
    __device__ static int pad(int i) { return fft_pad(i); }
    template <int DIR, bool SYNC_FIRST, class Get, class Put>
    __device__ void run(float2 *buf, Get get, Put put) const {
        fft_rt<DIR, T, 16 * T, T == 64, SYNC_FIRST>(buf, d, (int)threadIdx.x & (T - 1), get, put);
    }
};

template <class P>
size_t cols_lds(const P &pl) {
    return sizeof(float2) * (size_t)P::COLS * pl.stride();
}

// Calls f(plan) with the plan of columns of d.n values.
// Strips of 2 columns where a column takes two waves or more: up to four
// workgroups a CU, which stage and transform in turn, and enough of them for a
// narrow frame (wide strips of 8 columns up to 2048 values and 4 up to 4096
// against these, the chain: one frame of 100x2000 102 -> 86 us, 4 of 4000x3000
// 895 -> 842, 32 of 2000x1500 1623 -> 1528; 8 of 4096x4096 2316 -> 2355).  One
// wave a column: 8 columns (8 frames of 1000x2000 267 us, 289 by 2).  (At 1536
// rows the run-time plan on two waves per column, strips of 8, measured 333 and
// 356 us for the chain's two passes over 32 frames of 2048x1536, the
// compile-time plan 263 and 291, by 4 columns 277 and 328.)
template <class F>
auto with_cols_plan(const FftDesc &d, F f) {
    if (d.n == 1024) return f(ColsC<1024>{d.tw});
    if (d.n == 1536) return f(ColsC<1536>{d.tw});
    if (d.n < 1024) return f(ColsRt<64, 8>{d});
    if (d.n <= 2048) return f(ColsRt<128, 2>{d});
    if (d.n <= 4096) return f(ColsRt<256, 2>{d});
    return f(ColsRt<512, 2>{d});
}

// Strips of `cols` columns and the workgroups that take them.
template <class P>
int cols_per(int cols) {
    return ((cols + P::COLS - 1) / P::COLS + 7) / 8;
}
template <class P>
__device__ __forceinline__ int cols_strip(int per) {
    return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
}

// f(i) for i = first, first + STEP, ... below n (first < STEP); a constant
// number of times where n is known.
template <class P, int STEP, class F>
__device__ __forceinline__ void rows_of(const P &pl, int first, F f) {
    if constexpr (P::kConst) {
        static_assert(P::n() % STEP == 0, "rows_of: whole steps");
#pragma unroll 4
        for (int k = 0; k < P::n() / STEP; ++k) f(first + STEP * k);
    } else {
#pragma unroll 4
        for (int i = first; i < pl.n(); i += STEP) f(i);
    }
}

// Stages columns [j0, j0 + COLS) of A (rows lda values apart, `cols` columns),
// those below `cols`, and waits.  The second column of the last pair may lie
// past `cols`: it is read where the row's pitch or the next row holds a value
// (j0 + c2 + 1 <= cols <= lda, and a plane holds more than rows * cols values),
// and never used.
template <class P>
__device__ __forceinline__ void stage_cols(const P &pl, const float2 *__restrict__ A, int lda, int j0, int cols,
                                           float2 *lds) {
    constexpr int kPer = P::COLS / 2, kRows = P::kThreads / kPer;  // threads per row, rows per step
    const int t = (int)threadIdx.x, c2 = (t % kPer) * 2, sb = pl.stride();
    const bool wide = (lda & 1) == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;  // 16-byte aligned pairs (j0 is even)
    if (j0 + c2 < cols) {
        const float2 *src = A + j0 + c2;
        float2 *l0 = lds + c2 * sb, *l1 = l0 + sb;
        const bool both = j0 + c2 + 1 < cols;
        // (the choice outside the loops: inside, the loads are not batched)
        if (wide)
            rows_of<P, kRows>(pl, t / kPer, [&](int i) {
                const float4 v = *reinterpret_cast<const float4 *>(src + (int64_t)i * lda);
                l0[pl.pad(i)] = make_float2(v.x, v.y);
                l1[pl.pad(i)] = make_float2(v.z, v.w);
            });
        else
            rows_of<P, kRows>(pl, t / kPer, [&](int i) {
                const float2 *q = src + (int64_t)i * lda;
                const float2 a = q[0], b = both ? q[1] : a;
                l0[pl.pad(i)] = a;
                l1[pl.pad(i)] = b;
            });
    }
    __syncthreads();
}

// The staged strip back to rows: out[i * ldo + j0 + c] for c < COLS, j0 + c < cols.
template <class P>
__device__ __forceinline__ void unstage_cols(const P &pl, const float2 *lds, float2 *__restrict__ out, int64_t ldo,
                                             int j0, int cols) {
    const int t = (int)threadIdx.x, c = t % P::COLS, sb = pl.stride();
    if (j0 + c < cols)
        rows_of<P, P::kThreads / P::COLS>(pl, t / P::COLS, [&](int i) {
            out[(int64_t)i * ldo + j0 + c] = lds[c * sb + pl.pad(i)];
        });
}

}  // namespace prnu
