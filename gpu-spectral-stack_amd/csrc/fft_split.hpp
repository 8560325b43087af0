#pragma once

// Column and row passes whose tile does not fit LDS as complex values: the tile lives in registers,
// 32 values per lane, and the stage exchanges cross through LDS a part at a time (run_stages_split),
// so a tile of 16 transforms of 1024 points needs 70 KB (two workgroups per compute unit) and one
// of 2048 points 139 KB, where complex exchanges hold 8 and 4. Every global access is then a run of
// 16 values, a whole 128-byte line: tiles of 8 columns read half a line per row, whose other half
// belongs to another workgroup. A column pass of 1024-point columns over 2^24 points went from
// 69.9 to 58.8 us (4.6 TB/s, what a copy in that pattern reaches; in place, behind a row pass, 44.5).
// Rows of 1024 points keep 8 to a workgroup (46.6 us; 16 split rows 47.5 us, and 9.2 against 11.8 us
// for one 2^20 transform).

#include "stockham.hpp"

namespace spx::dev {

template <int N_>
struct SplitPlan : Plan<N_, 16, 32> {
    using Base = Plan<N_, 16, 32>;
    static constexpr int kTile = 16;                     // transforms per workgroup
    static constexpr int kLanes = kTile * Base::L;
    static constexpr int kWavesPerSimd = kLanes <= 512 ? 4 : kLanes / 256;
    static_assert(Base::L >= 32 && kLanes <= 1024, "1024 or 2048 points");
};

// Columns: the lanes of a wave walk 16 neighbouring columns, so its LDS exchanges cross waves.
template <int N>
struct SplitColumnPlan : SplitPlan<N> {
    static constexpr bool kWaveLocal = false;
    static constexpr int kLds = (pad(N - 1) + 1) * SplitPlan<N>::kTile;  // floats
};

// Unpruned strided columns (StridedIo), in place or not: tile b holds columns 16 b .. 16 b + 15 of
// the slabs' columns laid end to end. An exchange row holds one float of each column, with a spare
// row after every 16 (PaddedRows): the four rows that a wave's 64 lanes touch lie on four distinct
// quarters of the 64 banks. Consecutive tiles, which share lines when a row of the arrays is no
// multiple of 16 values, run on one XCD, and the loads leave those lines in its L2 (nontemporal
// loads: 1024 x 33 out of place, 528 tiles, 76.6 against 64 us; whole lines 1 % slower too). Fewer than
// 256 tiles of 1024-point columns in place keep the hint (fft2 of 32 arrays of 1024 x 64, 128 tiles,
// 22.5 against 23.2 us, of 96 of 1024 x 32, 192 tiles, 24.8 against 26.0; 256 tiles 34.3 against 33.3,
// 512 49.7 against 44.7).
template <class P, bool Inv, bool Table>
__global__ void __launch_bounds__(P::kLanes, P::kWavesPerSimd)
    columns_split_kernel(StridedIo io, long long batch, const cf32* table)
{
    using Lay = PaddedRows<P::kTile>;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    __shared__ float s[P::kLds];
    const int tid = threadIdx.x;
    const int c = tid % P::kTile;
    const int lane = tid / P::kTile;
    const long long t = xcd_order<32>(blockIdx.x, gridDim.x) * P::kTile + c;
    const bool live = t < batch;
    const long long slab = (live ? t : batch - 1) / io.cols;
    const long long at = slab * P::N * io.cols + ((live ? t : batch - 1) - slab * io.cols)
                         + static_cast<long long>(lane) * io.cols;
    const bool once = P::N == 1024 && io.stream_out && io.x == io.y && gridDim.x < 256;
    cf32 v[P::E];
    const cf32* const src = io.x + at;
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        constexpr long long off = (e / R0) * P::L + (e % R0) * (P::N / R0);
        v[e] = once ? ld_stream(src + off * io.cols) : src[off * io.cols];
    });
    run_stages_split<P, 0, Inv, Table, Lay>(v, s + c, lane, table);
    if (live) {
        cf32* const dst = io.y + at;
        static_for<0, P::E>([&](auto ei) {
            constexpr int e = decltype(ei)::value;
            constexpr long long off = (e / RL) * P::L + (e % RL) * (P::N / RL);
            const cf32 z = cscale(v[e], io.scale);
            if (io.stream_out) {
                st_stream(dst + off * io.cols, z);
            } else {
                dst[off * io.cols] = z;
            }
        });
    }
}

// The second of two passes of a large transform (TwiddleRowsTransposedIo): 16 twiddled rows per
// workgroup, stored transposed in runs of 16 values. The twiddle of element lane + L m of row k1 is
// w^(k1 lane) w^(k1 L m); the second factors, one per row and m, go to LDS once per workgroup. Rows
// exchange 32 mod 64 floats apart, and the transposition writes element k2 of row u at 17 k2 + u.
template <class P, bool Inv, bool Table, class Io>
__global__ void __launch_bounds__(P::kLanes, P::kWavesPerSimd)
    rows_split_kernel(Io io, const cf32* table)
{
    constexpr int T = P::kTile;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    constexpr int kStride = (pad(P::N - 1) + 1 + 31) / 64 * 64 + 32;
    constexpr int kTurned = T + 1;
    static_assert(kStride >= pad(P::N - 1) + 1 && T * kStride >= P::N * kTurned, "LDS");
    __shared__ float s[T * kStride];
    __shared__ cf32 factor[T * P::E];
    const int tid = threadIdx.x;
    const int u = tid / P::L;
    const int lane = tid % P::L;
    const long long first = static_cast<long long>(blockIdx.x) * T;  // T divides n1
    const long long slab = first / io.rows.n1;
    const int k1 = static_cast<int>(first - slab * io.rows.n1);
    const cf32* const row = io.rows.x + (first + u) * P::N + lane;
    cf32 v[P::E];
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        v[e] = row[(e / R0) * P::L + (e % R0) * (P::N / R0)];
    });
    if (tid < T * P::E) {
        const int step = (k1 + tid / P::E) * P::L * (tid % P::E);  // below n, exact in float
        cf32 w = expi_pi(static_cast<float>(step) * io.rows.two_over_n);
        w.im *= io.rows.sign;
        factor[tid] = w;
    }
    cf32 base = expi_pi(static_cast<float>((k1 + u) * lane) * io.rows.two_over_n);
    base.im *= io.rows.sign;
    __syncthreads();
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        constexpr int m = e / R0 + (e % R0) * (P::E / R0);
        v[e] = cmul(v[e], cmul(base, factor[u * P::E + m]));
    });
    run_stages_split<P, 0, Inv, Table>(v, s + u * kStride, lane, table);

    // Element k2 of row u to column u of the matrix of k2 rows, k1 fastest: two parts again.
    constexpr int kStep = P::kLanes / T;  // k2 rows per store
    const int tu = tid % T;
    const int tk = tid / T;
    cf32* const dst = io.rows.y + slab * io.n + k1 + tu;
    float re[P::E];
    static_for<0, 2>([&](auto part) {
        constexpr bool kIm = decltype(part)::value != 0;
        __syncthreads();
        static_for<0, P::E>([&](auto ei) {
            constexpr int e = decltype(ei)::value;
            constexpr int off = (e / RL) * P::L + (e % RL) * (P::N / RL);
            s[(lane + off) * kTurned + u] = kIm ? v[e].im : v[e].re;
        });
        __syncthreads();
        static_for<0, P::E>([&](auto ei) {
            constexpr int e = decltype(ei)::value;
            const int k2 = tk + e * kStep;
            const float x = s[k2 * kTurned + tu];
            if constexpr (kIm) {
                st_stream(dst + static_cast<long long>(io.rows.n1) * k2,
                          cscale(cf32{re[e], x}, io.rows.scale));
            } else {
                re[e] = x;
            }
        });
    });
}

}  // namespace spx::dev
