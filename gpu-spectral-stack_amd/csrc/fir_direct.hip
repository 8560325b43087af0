// Short real FIR filters (rf.fir, reference python/spectral/rf.py:120-153) as products with a
// Toeplitz matrix on the fp32 matrix cores, in place of overlap-save blocks: for few taps the
// convolution sum itself is less arithmetic than two FFTs per block, needs no filter spectrum and
// rounds less.
//
// Sixteen segments of sixteen outputs are one 16 x 16 product Y = X T: Y[m][i] = y[s + 16 m + i],
// X[m][u] = x[s - Kp + 16 m + u] and T[u][i] = h[i + Kp - u] for u below U, the multiple of 16 that
// holds K + 15 (Kp = U - 16): U / 4 v_mfma_f32_16x16x4_f32 for the real parts and as many for the
// imaginary parts, of which K / (K + 15) and up is the sum's own work. X is read from LDS in place,
// each sample U / 16 times; samples lie 18 per 16 there, so that a half-wave's 32 values fall on
// distinct banks. Results come out 16 consecutive outputs to a run, whole lines.
//
// A workgroup walks consecutive steps of 1024 outputs, 256 per wave, and has the next step's samples
// in flight while it multiplies. 2^22 samples, 63 taps: 8.5 us of matrix work and 10.7 us of HBM
// traffic at the copy rate; the call went from 22.1 us (256-point blocks and the launch for their
// filter spectrum) to 18.2 us, of which about 4 us are the first step's loads and the last one's
// stores. 2^14 to 2^20 samples: 12.8 -> 7 us (129 taps 8). Against 64 bits 1.4e-7, where blocks are
// 3e-7 off. Twice as many or half as many workgroups were 1 to 2 us slower. Every row takes whole
// steps, short of its end too (65536 rows of 16 samples: 1.7 ns a step with 15 taps, 3.2 with 63), so
// the caller keeps short rows to few.

#include "stockham.hpp"

#include "fft_api.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace spx {
namespace dev {
namespace {

constexpr int kFirThreads = 256;
constexpr int kFirStep = 1024;                       // outputs per workgroup and step
constexpr int kFirMaxU = 16 * ((kFirDirectTaps + 15 + 15) / 16);
constexpr int kFirMaxWindow = kFirStep - 16 + kFirMaxU;  // samples per step
constexpr int kFirLoads = (kFirMaxWindow + kFirThreads - 1) / kFirThreads;
constexpr int kFirRow = 18;                          // LDS values per 16 samples
constexpr int kFirBuffer = kFirMaxWindow / 16 * kFirRow;

using f4v = float __attribute__((ext_vector_type(4)));

// Steps [first, last) of all rows' steps, `steps` per row of n samples, by this workgroup.
__global__ void __launch_bounds__(kFirThreads)
    fir_direct_kernel(const cf32* __restrict__ x, const float* __restrict__ h,
                      cf32* __restrict__ y, long long n, int taps, int u_groups, long long steps,
                      long long all_steps, long long per_block)
{
    __shared__ cf32 buffer[2][kFirBuffer];
    __shared__ float reversed[kFirMaxU + 16];  // h[d] at d + 15, zeros around
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid / 64;
    const int kp = 16 * u_groups - 16;
    const int window = kFirStep + kp;
    for (int e = tid; e < kFirMaxU + 16; e += kFirThreads) {
        const int d = e - 15;
        reversed[e] = d >= 0 && d < taps ? h[d] : 0.0f;
    }

    // Samples tid + 256 k of a step's window (the last one of them only for tid < kp), LDS slots
    // 288 apart. An inner step has its whole window inside the row: a uniform base and constant
    // offsets, no branch around a load or a store. The others replace samples outside the row by zeros.
    static_assert(kFirThreads % 16 == 0 && kFirMaxWindow <= kFirStep + kFirThreads, "window");
    constexpr int kSlots = kFirThreads / 16 * kFirRow;
    const int slot = tid / 16 * kFirRow + tid % 16;
    const unsigned tail = static_cast<unsigned>(cmin(tid + kFirStep, window - 1));
    cf32 next[kFirLoads];
    const auto fetch = [&](long long row, long long step) {
        const cf32* const src = x + (row * n + step * kFirStep - kp);
#pragma unroll
        for (int k = 0; k < kFirLoads; ++k) {
            next[k] = ld_stream(
                src + (k + 1 < kFirLoads ? static_cast<unsigned>(tid + k * kFirThreads) : tail));
        }
    };
    const auto fetch_edge = [&](long long row, long long step) {
        const long long at = step * kFirStep - kp + tid;
#pragma unroll
        for (int k = 0; k < kFirLoads; ++k) {
            const long long i = at + k * kFirThreads;
            next[k] = czero();
            if (tid + k * kFirThreads < window && i >= 0 && i < n) {
                next[k] = ld_stream(x + row * n + i);
            }
        }
    };
    const auto park = [&](cf32* samples) {
#pragma unroll
        for (int k = 0; k < kFirLoads; ++k) {
            if (k + 1 < kFirLoads || tid < kp) {
                samples[slot + k * kSlots] = next[k];
            }
        }
        __syncthreads();
    };
    // Lane: segment (and offset) lane % 16, samples 4 q + lane / 16; then output lane % 16 of
    // segments 4 (lane / 16) + r.
    const auto multiply = [&](const cf32* samples, f4v& re, f4v& im) {
        const cf32* a = samples + (16 * wave + lane % 16) * kFirRow + lane / 16;
        const float* b = reversed + 15 + lane % 16 + kp - lane / 16;
        re = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        im = re;
        for (int g = 0; g < u_groups; ++g) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const cf32 v = a[4 * q];
                const float t = b[-4 * q];
                re = __builtin_amdgcn_mfma_f32_16x16x4f32(v.re, t, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f32_16x16x4f32(v.im, t, im, 0, 0, 0);
            }
            a += kFirRow;
            b -= 16;
        }
    };
    const int out = 256 * wave + 64 * (lane / 16) + lane % 16;

    const long long first = static_cast<long long>(blockIdx.x) * per_block;
    long long left = (first + per_block < all_steps ? first + per_block : all_steps) - first;
    long long row = first / steps;
    long long step = first - row * steps;
    // The buffer written for a step was last read two steps before it, ahead of a barrier.
    int half = 0;
    f4v re;
    f4v im;
    while (left > 0) {
        cf32* const dst = y + row * n;
        const auto store = [&](long long at) {
            cf32* const to = dst + at * kFirStep;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                st_stream(to + static_cast<unsigned>(out + 16 * r), cf32{re[r], im[r]});
            }
        };
        const long long in_row = n / kFirStep - step;  // whole steps left in this row
        const long long whole = in_row < left ? in_row : left;
        if (whole > 0 && (step > 0 || kp == 0)) {
            // A step's results are stored once the next step's samples have landed, ahead of the
            // loads after them: the wait for loads is then never a wait for fresh stores (stored
            // at once, 2^22 samples took the sum of the matrix and the memory time).
            fetch(row, step);
            park(buffer[half]);
            for (long long w = 1; w < whole; ++w, ++step) {
                if (w > 1) {
                    store(step - 1);
                }
                fetch(row, step + 1);
                multiply(buffer[half], re, im);
                half ^= 1;
                park(buffer[half]);
            }
            if (whole > 1) {
                store(step - 1);
            }
            multiply(buffer[half], re, im);
            store(step);
            left -= whole;
        } else {  // the row's first step, or its last and partial one
            fetch_edge(row, step);
            park(buffer[half]);
            multiply(buffer[half], re, im);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const long long i = step * kFirStep + out + 16 * r;
                if (i < n) {
                    st_stream(dst + i, cf32{re[r], im[r]});
                }
            }
            --left;
        }
        half ^= 1;
        if (++step == steps) {
            step = 0;
            ++row;
        }
    }
}

}  // namespace
}  // namespace dev

void fir_direct(const cf32* x, const float* taps, cf32* y, long long n, int count,
                long long rows, hipStream_t stream)
{
    if (n < 1 || rows < 1 || count < 1 || count > kFirDirectTaps) {
        throw InvalidArgument("fir_direct: need n and rows >= 1 and 1 to " + str(kFirDirectTaps)
                              + " taps, got n = " + str(n) + ", rows = " + str(rows) + ", taps = "
                              + str(count));
    }
    const auto* a = reinterpret_cast<const char*>(x);
    const auto* b = reinterpret_cast<const char*>(y);
    const std::size_t bytes = static_cast<std::size_t>(n) * static_cast<std::size_t>(rows)
                              * sizeof(cf32);
    if (a < b + bytes && b < a + bytes) {
        throw InvalidArgument("fir_direct: x and y must not overlap");
    }
    const int u_groups = (count + 15 + 15) / 16;
    const long long steps = (n + dev::kFirStep - 1) / dev::kFirStep;
    const long long all = steps * rows;
    // Four workgroups per compute unit once there is more than one step for each.
    const long long resident = 4LL * device_cus();
    const long long per_block = std::max(1LL, (all + resident - 1) / resident);
    const long long blocks = (all + per_block - 1) / per_block;
    hipLaunchKernelGGL(dev::fir_direct_kernel, dim3(static_cast<unsigned>(blocks)),
                       dim3(dev::kFirThreads), 0, stream, x, taps, y, n, count, u_groups, steps,
                       all, per_block);
    SPX_LAUNCH_CHECK();
}

}  // namespace spx
