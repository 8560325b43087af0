// Navier-Stokes steps on grids whose field does not fit one workgroup's LDS, or whose state keeps
// the full half spectrum: three kernels per IMEX stage, in place of the reference's two batched
// transforms and about fifteen elementwise kernels (python/spectral/flow/gpu.py:115-129).
//
// State: omega_hat per field, `rows` x W complex values: the pruned (FNO) layout, rows ky = 0 ..
// m-1 then -m .. -1 and W = m columns with m = n/3 + 1, or the rfft2 layout, n rows and
// W = n/2 + 1 columns.
//
// The nonlinear term is N = u wx + v wy. Two real fields share one complex transform: with
// z1 = u + i v and z2 = wx + i wy, N = Re z1 Re z2 + Im z1 Im z2. Both fields of a pair have the
// same scale, so neither's rounding spoils the other's. For a pair A + i B of real fields, the
// row spectrum is P[k] = (A~ + i B~)[k] at k >= 0 and Q[k] = conj((A~ - i B~)[k]) at -k, and as
// the column transforms are linear, P and Q are column transforms of the state times one complex
// multiplier per mode each. Per stage:
//   ns_columns_kernel  the inverse column transforms of P1, Q1, P2, Q2, one tile of columns of one
//                      of them per workgroup: state -> work (field, grid row, 4, pitch)
//   ns_rows_kernel     two grid rows per lane group: each row's z1 and z2 (n-point complex inverses
//                      read straight from P and Q), their product, then ONE complex forward of both
//                      rows' products, split into the two rows' first W bins: work -> work, over
//                      the rows it read
//   ns_update_kernel   the forward columns of those bins and the IMEX update of the kept rows
//                        stage 0: out_f = F, out_w = (e w + dt F) i
//                        stage 1: out_w = (e w0 + dt/2 (f0 + F)) i
//                      with F = f_hat - mask N_hat, e = 1 + dt/2 L, i = 1 / (1 - dt/2 L),
//                      L = -nu |k|^2 - alpha.
// Every pass moves its arrays once; the derived spectra (4 n pitch values per field) are the one
// large intermediate. Normalization: inverse 1 / n^2, forward none, as numpy. The imaginary parts
// of a row's zero and n/2 frequencies are dropped, as numpy's irfft drops them.
//
// Measured on MI355X (256^2 pruned, 48 fields): columns 12.8 us (38 MB written), rows 13.0 us
// (38 MB read, 8 MB written), update 10.3 us; a stage was about 105 us composed. About 4 us of
// each launch is its ramp and drain; neither fewer stages (radix 16) nor the update's loads issued
// ahead of its transform moved the rest.

#include "stockham.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace spx {
namespace dev {
namespace {

// A plan whose transforms span waves: the column passes hold kT neighbouring columns per tile,
// the columns fastest over the lanes, so that every global access of a wave is whole runs of kT
// values (128 bytes).
template <int N, int R, int E>
struct ColumnPlan : Plan<N, R, E> {
    static constexpr bool kWaveLocal = false;
};

template <int N_, bool Pruned_>
struct NsGrid {
    static constexpr int N = N_;
    static constexpr bool kPruned = Pruned_;
    static constexpr int m = N / 3 + 1;
    static constexpr int kRows = Pruned_ ? 2 * m : N;      // state rows per field
    static constexpr int kW = Pruned_ ? m : N / 2 + 1;     // state columns
    static constexpr int kPitch = (kW + 15) / 16 * 16;     // of P and Q rows: whole 128-byte lines
    static constexpr int kT = N <= 512 ? 16 : 8;           // columns per tile
    static constexpr int kTiles = (kW + kT - 1) / kT;
    // Radix and values per lane of the columns: 8 while a tile then takes at most 512 lanes. At 256
    // the update waits on its loads, not on its stages: 12.4 us with 16 values, 10.3 us with 8.
    static constexpr int kR = N <= 256 ? 8 : 16;
    using PC = ColumnPlan<N, kR, kR>;
    static constexpr int kColumnThreads = kT * PC::L;
    static constexpr int kColumnLds = pad(N - 1) * kT + kT;
    static constexpr int kRE = N <= 512 ? 8 : 16;          // rows: one wave or less per transform
    using PR = Plan<N, kRE, kRE>;
    static constexpr int kRowLds = PR::T * PR::kStride;

    static_assert(PR::L <= 64 && kColumnThreads <= 1024, "workgroup shapes");
    static_assert(slots_match<PR>(), "inverse outputs must be forward inputs");
    static_assert(kColumnLds * sizeof(cf32) <= 80 * 1024, "two column tiles per compute unit");
};

// State row of full-spectrum row i (0 .. N-1), or -1 when the layout drops it.
template <class G>
__device__ __forceinline__ int state_row(int i)
{
    if constexpr (!G::kPruned) {
        return i;
    } else {
        return i < G::m ? i : (i >= G::N - G::m ? i - G::N + 2 * G::m : -1);
    }
}

template <class G>
__device__ __forceinline__ float ky_of(int i)
{
    return static_cast<float>(i < G::N / 2 ? i : i - G::N);
}

// 1 / x to the last bit or the one before it: the hardware's approximation and one Newton step
// (a correctly rounded division is four times the instructions).
__device__ __forceinline__ float reciprocal(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}

// Multiplier of omega_hat for set 0 .. 3 (P1, Q1 before its conjugation, P2, Q2 likewise):
//   u + i v: (i ky + kx) / k^2, u - i v: (i ky - kx) / k^2   (u = i ky psi, v = -i kx psi)
//   wx + i wy: i kx - ky, wx - i wy: i kx + ky
// times 1 / n^2.
template <class G>
__device__ __forceinline__ cf32 multiplier(int set, float kx, float ky)
{
    constexpr float kScale = 1.0f / (static_cast<float>(G::N) * static_cast<float>(G::N));
    if (set < 2) {
        const float k2 = kx * kx + ky * ky;
        const float f = k2 > 0.0f ? kScale * reciprocal(k2) : 0.0f;
        return {(set == 0 ? kx : -kx) * f, ky * f};
    }
    return {(set == 2 ? -ky : ky) * kScale, kx * kScale};
}

// One tile of kT columns of one set. Blocks run set fastest within an XCD's share (consecutive
// blocks go to consecutive XCDs), so the four sets of a tile read the state from one L2.
template <class G>
__global__ void __launch_bounds__(G::kColumnThreads)
    ns_columns_kernel(const cf32* __restrict__ state, cf32* __restrict__ work, int items)
{
    using P = typename G::PC;
    using Lay = PaddedRows<G::kT>;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    __shared__ cf32 s[G::kColumnLds];
    const int slot = static_cast<int>(blockIdx.x) / 8;
    const int item = (slot / 4) * 8 + static_cast<int>(blockIdx.x) % 8;  // (field, tile)
    const int set = slot % 4;
    if (item >= items) {
        return;  // the whole workgroup
    }
    const int field = item / G::kTiles;
    const int tid = threadIdx.x;
    const int c = tid % G::kT;
    const int lane = tid / G::kT;
    const int col = (item % G::kTiles) * G::kT + c;
    const bool live = col < G::kW;
    const cf32* const w = state + static_cast<long long>(field) * G::kRows * G::kW;
    const float kx = static_cast<float>(col);
    cf32 v[P::E];
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int i = input_index<P, 0>(lane, e / R0, e % R0);
        const int r = state_row<G>(i);
        v[e] = live && r >= 0 ? w[r * G::kW + col] : czero();
    }
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int i = input_index<P, 0>(lane, e / R0, e % R0);
        v[e] = cmul(v[e], multiplier<G>(set, kx, ky_of<G>(i)));
    }
    run_stages<P, 0, true, false, Lay>(v, s + c, lane, nullptr);
    cf32* const out = work + (static_cast<long long>(field) * G::N * 4 + set) * G::kPitch + col;
    const float sign = (set & 1) != 0 ? -1.0f : 1.0f;
    if (col < G::kPitch) {
        static_for<0, P::E>([&](auto ei) {
            constexpr int e = decltype(ei)::value;
            const int y = lane + (e / RL) * P::L + (e % RL) * (P::N / RL);
            out[y * (4 * G::kPitch)] = cf32{v[e].re, sign * v[e].im};
        });
    }
}

// Stage-0 inputs of a grid row's inverse from its P and Q.
template <class G>
__device__ __forceinline__ void load_pair(const cf32* __restrict__ p, cf32 (&v)[G::PR::E], int lane)
{
    using P = typename G::PR;
    constexpr int R0 = P::template radix<0>();
    const cf32* const q = p + G::kPitch;
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        constexpr int off = (e / R0) * P::L + (e % R0) * (P::N / R0);
        const int k = lane + off;
        cf32 z = czero();
        if constexpr (off < G::kW) {
            if (k < G::kW) {
                z = p[k];
            }
        }
        if constexpr (off + P::L > G::N - G::kW) {
            if (k > G::N - G::kW && k > G::N / 2) {
                z = q[G::N - k];
            }
        }
        // P + i 0 and Q meet at the frequencies whose imaginary parts are dropped.
        if constexpr (off == 0 || off == G::N / 2) {
            if (lane == 0 && k < G::kW) {
                z = cscale(cadd(z, q[k]), 0.5f);
            }
        }
        v[e] = z;
    });
}

template <class G>
__global__ void __launch_bounds__(G::PR::kThreads) ns_rows_kernel(cf32* work, long long pairs)
{
    using P = typename G::PR;
    constexpr int RL = P::template radix<P::kStages - 1>();
    __shared__ cf32 lds[G::kRowLds];
    const int lane = static_cast<int>(threadIdx.x) % P::L;
    const int t = static_cast<int>(threadIdx.x) / P::L;
    const long long pair = static_cast<long long>(blockIdx.x) * P::T + t;
    cf32* const s = lds + t * P::kStride;
    const bool live = pair < pairs;
    // Lane groups past the end repeat the last pair and store nothing.
    cf32* const row0 = work + (live ? pair : pairs - 1) * (2LL * 4 * G::kPitch);
    cf32* const row1 = row0 + 4 * G::kPitch;
    cf32 g[P::E];  // both rows' products, in the forward's input slots
#pragma unroll
    for (int y = 0; y < 2; ++y) {
        const cf32* const row = y == 0 ? row0 : row1;
        cf32 a[P::E];
        cf32 b[P::E];
        load_pair<G>(row, a, lane);
        load_pair<G>(row + 2 * G::kPitch, b, lane);
        run_stages<P, 0, true, false>(a, s, lane, nullptr);
        run_stages<P, 0, true, false>(b, s, lane, nullptr);
        static_for<0, P::E>([&](auto ei) {
            constexpr int e = decltype(ei)::value;
            const float product = a[e].re * b[e].re + a[e].im * b[e].im;
            if (y == 0) {
                g[forward_slot_of<P>(e)].re = product;
            } else {
                g[forward_slot_of<P>(e)].im = product;
            }
        });
    }
    run_stages<P, 0, false, false>(g, s, lane, nullptr);
    lds_sync<true>();  // the last exchange's reads are done
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        constexpr int k = (e / RL) * P::L + (e % RL) * (P::N / RL);
        s[pad(lane) + pad(k)] = g[e];
    });
    lds_sync<true>();
    if (live) {
        // G = G0 + i G1 of two real rows: G0[k] = (G[k] + conj G[-k]) / 2 and
        // G1[k] = (G[k] - conj G[-k]) / 2i.
        for (int k = lane; k < G::kW; k += P::L) {
            const cf32 f = s[pad(k)];
            const cf32 h = s[pad((G::N - k) & (G::N - 1))];
            row0[k] = cf32{0.5f * (f.re + h.re), 0.5f * (f.im - h.im)};
            row1[k] = cf32{0.5f * (f.im + h.im), 0.5f * (h.re - f.re)};
        }
    }
}

// One tile of kT columns: the forward column transforms and the update of the kept rows. out_f and
// out_w may be w0 or f0 (each lane reads the elements it is about to write), so none is restrict.
template <class G>
__global__ void __launch_bounds__(G::kColumnThreads)
    ns_update_kernel(const cf32* __restrict__ work, const cf32* w0, const cf32* f0, cf32* out_f,
                     cf32* out_w, const cf32* __restrict__ forcing_hat,
                     const float* __restrict__ nu, int nu_stride, float drag, float dt, int stage)
{
    using P = typename G::PC;
    using Lay = PaddedRows<G::kT>;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    __shared__ cf32 s[G::kColumnLds];
    const int field = static_cast<int>(blockIdx.x) / G::kTiles;
    const int tid = threadIdx.x;
    const int c = tid % G::kT;
    const int lane = tid / G::kT;
    const int col = (static_cast<int>(blockIdx.x) % G::kTiles) * G::kT + c;
    const cf32* const in = work + static_cast<long long>(field) * G::N * 4 * G::kPitch + col;
    const float nu_f = nu[static_cast<long long>(field) * nu_stride];
    cf32 v[P::E];
    const bool live = col < G::kW;
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int y = input_index<P, 0>(lane, e / R0, e % R0);
        v[e] = live ? in[y * (4 * G::kPitch)] : czero();
    }
    run_stages<P, 0, false, false, Lay>(v, s + c, lane, nullptr);
    if (!live) {
        return;  // past the last barrier
    }
    const long long base = static_cast<long long>(field) * G::kRows * G::kW;
    const float kmax = static_cast<float>(G::N) / 3.0f;
    const float kx = static_cast<float>(col);
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        const int i = lane + (e / RL) * P::L + (e % RL) * (P::N / RL);
        const int r = state_row<G>(i);
        if (r >= 0) {
            const int at = r * G::kW + col;
            const float ky = ky_of<G>(i);
            const bool kept = kx <= kmax && fabsf(ky) <= kmax;
            const cf32 F = csub(forcing_hat[at], kept ? v[e] : czero());
            const float linear = -nu_f * (kx * kx + ky * ky) - drag;
            const float ex = 1.0f + 0.5f * dt * linear;
            const float im = reciprocal(1.0f - 0.5f * dt * linear);
            const cf32 w = w0[base + at];
            if (stage == 0) {
                out_f[base + at] = F;
                out_w[base + at] = cscale(cadd(cscale(w, ex), cscale(F, dt)), im);
            } else {
                const cf32 sum = cadd(f0[base + at], F);
                out_w[base + at] = cscale(cadd(cscale(w, ex), cscale(sum, 0.5f * dt)), im);
            }
        }
    });
}

struct NsArrays {
    const cf32* w_in;
    cf32* w_out;
    cf32* work;
    const cf32* forcing_hat;
    const float* nu;
    int nu_stride;
    float drag;
    float dt;
};

template <class G>
void stage(const NsArrays& a, const cf32* state, const cf32* w0, const cf32* f0, cf32* out_f,
           cf32* out_w, cf32* spectra, const float* nu, int fields, int which, hipStream_t stream)
{
    const int items = fields * G::kTiles;
    const unsigned column_blocks = static_cast<unsigned>((items + 7) / 8) * 32u;
    hipLaunchKernelGGL(ns_columns_kernel<G>, dim3(column_blocks), dim3(G::kColumnThreads), 0,
                       stream, state, spectra, items);
    SPX_LAUNCH_CHECK();
    const long long pairs = static_cast<long long>(fields) * (G::N / 2);
    const auto row_blocks = static_cast<unsigned>((pairs + G::PR::T - 1) / G::PR::T);
    hipLaunchKernelGGL(ns_rows_kernel<G>, dim3(row_blocks), dim3(G::PR::kThreads), 0, stream,
                       spectra, pairs);
    SPX_LAUNCH_CHECK();
    hipLaunchKernelGGL(ns_update_kernel<G>, dim3(static_cast<unsigned>(items)),
                       dim3(G::kColumnThreads), 0, stream, spectra, w0, f0, out_f, out_w,
                       a.forcing_hat, nu, a.nu_stride, a.drag, a.dt, which);
    SPX_LAUNCH_CHECK();
}

// Fields advanced together: as many as keep the derived spectra (the array that every kernel
// streams) within half of the 256 MB Infinity Cache.
template <class G>
constexpr int fields_per_group()
{
    constexpr long long bytes = 8LL * 4 * G::N * G::kPitch;
    return static_cast<int>(std::max(1LL, (128LL << 20) / bytes));
}

template <class G>
std::size_t workspace(int batch)
{
    const int group = std::min(batch, fields_per_group<G>());
    return static_cast<std::size_t>(group) * (4 * G::N * G::kPitch + 2 * G::kRows * G::kW);
}

template <class G>
void advance(const NsArrays& a, int batch, int steps, hipStream_t stream)
{
    constexpr long long kField = static_cast<long long>(G::kRows) * G::kW;
    const int most = std::min(batch, fields_per_group<G>());
    const int groups = (batch + most - 1) / most;
    cf32* const spectra = a.work;
    cf32* const tendency = spectra + static_cast<long long>(most) * 4 * G::N * G::kPitch;
    cf32* const predicted = tendency + most * kField;
    for (int g = 0; g < groups; ++g) {
        // Even shares, so that no group is left with a few fields.
        const int first = static_cast<int>(static_cast<long long>(batch) * g / groups);
        const int fields = static_cast<int>(static_cast<long long>(batch) * (g + 1) / groups) - first;
        cf32* const out = a.w_out + first * kField;
        const float* const nu = a.nu + static_cast<long long>(first) * a.nu_stride;
        const cf32* w = a.w_in + first * kField;
        for (int s = 0; s < steps; ++s) {
            stage<G>(a, w, w, nullptr, tendency, predicted, spectra, nu, fields, 0, stream);
            stage<G>(a, predicted, w, tendency, nullptr, out, spectra, nu, fields, 1, stream);
            w = out;
        }
    }
}

// f.template operator()<G>() for the kernels' grid of this size and layout.
template <class F>
auto dispatch(int n, bool pruned, F&& f)
{
    const auto layout = [&](auto size) {
        constexpr int N = decltype(size)::value;
        return pruned ? f(NsGrid<N, true>{}) : f(NsGrid<N, false>{});
    };
    switch (n) {
    case 32: return layout(std::integral_constant<int, 32>{});
    case 64: return layout(std::integral_constant<int, 64>{});
    case 128: return layout(std::integral_constant<int, 128>{});
    case 256: return layout(std::integral_constant<int, 256>{});
    case 512: return layout(std::integral_constant<int, 512>{});
    case 1024: return layout(std::integral_constant<int, 1024>{});
    default:
        throw InvalidArgument("ns_grid_steps: supports n = 32 to 1024, a power of two, got "
                              + str(n));
    }
}

}  // namespace
}  // namespace dev

bool ns_grid_supports(int n) { return is_pow2(n) && n >= 32 && n <= 1024; }

std::size_t ns_grid_workspace(int n, bool pruned, int batch)
{
    if (batch < 1) {
        throw InvalidArgument("ns_grid_workspace: need batch >= 1");
    }
    return dev::dispatch(
        n, pruned, [&](auto g) { return dev::workspace<decltype(g)>(batch); });
}

void ns_grid_steps(const cf32* w_in, cf32* w_out, cf32* work, const cf32* forcing_hat,
                   const float* nu, int nu_stride, float drag, float dt, int n, bool pruned,
                   int batch, int steps, hipStream_t stream)
{
    if (batch < 1 || steps < 1 || (nu_stride != 0 && nu_stride != 1)) {
        throw InvalidArgument("ns_grid_steps: need batch >= 1, steps >= 1, nu_stride 0 or 1");
    }
    if (w_in == nullptr || w_out == nullptr || work == nullptr || forcing_hat == nullptr
        || nu == nullptr) {
        throw InvalidArgument(
            "ns_grid_steps: w_in, w_out, work, forcing_hat and nu must not be null");
    }
    const dev::NsArrays arrays{w_in, w_out, work, forcing_hat, nu, nu_stride, drag, dt};
    dev::dispatch(n, pruned,
                  [&](auto g) { dev::advance<decltype(g)>(arrays, batch, steps, stream); });
}

}  // namespace spx
