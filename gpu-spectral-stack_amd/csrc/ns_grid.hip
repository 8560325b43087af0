// Navier-Stokes steps on grids whose field does not fit one workgroup's LDS, or whose state keeps
// the full half spectrum: two kernels per IMEX stage, in place of the reference's two batched
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
//   ns_rows_kernel     two grid rows per lane group: each row's z1 and z2 (n-point complex inverses
//                      read straight from P and Q), their product, then ONE complex forward of both
//                      rows' products, split into the two rows' first W bins: work -> bins
//   ns_update_columns_kernel  the forward columns of those bins and the IMEX update of the kept
//                      rows, then, from the same registers, the inverse column transforms of the
//                      next stage's P1, Q1, P2, Q2: bins -> state, work (field, grid row, 4, pitch)
//                        stage 0: out_f = F, state (e w + dt F) i, which only the columns see
//                        stage 1: out_w = (e w0 + dt/2 (f0 + F)) i
//                      with F = f_hat - mask N_hat, e = 1 + dt/2 L, i = 1 / (1 - dt/2 L),
//                      L = -nu |k|^2 - alpha.
// A call's first stage takes its columns from ns_columns_kernel and its last one ends in
// ns_update_kernel: 4 steps + 1 launches per group of fields. The derived spectra (4 n pitch values
// per field) are the one large intermediate. Normalization: inverse 1 / n^2, forward none, as numpy.
// The imaginary parts of a row's zero and n/2 frequencies are dropped, as numpy's irfft drops them.
//
// Measured on MI355X (256^2 pruned, 48 fields, six steps and a frame): 434 us with the update and
// the columns apart (10.3 and 12.8 us; rows 13.0 us), 349 us as here (rows 13.0, update and
// columns 17 us a launch). Both kernels issue vector instructions for 6 us of a launch and wait on
// loads and exchanges for the rest, two to three waves per SIMD; 4 us of each launch is its ramp
// and drain. Rows with the second row's loads ahead of the first row's transforms were 1.7 us slower
// (registers), with one row per lane group 4 us slower (the pair's forward then runs on both).

#include "stockham.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace spx {
namespace dev {
namespace {

// A plan whose transforms span waves: the column passes hold kT neighbouring columns per tile,
// the columns fastest over the lanes, so that every global access of a wave is whole runs of kT
// values.
template <int N, int R, int E>
struct ColumnPlan : Plan<N, R, E> {
    static constexpr bool kWaveLocal = false;
};

// Few: few fields of 256^2, which take 4 values per lane, twice the waves, each half as long.
template <int N_, bool Pruned_, bool Few = false>
struct NsGrid {
    static constexpr int N = N_;
    static constexpr bool kPruned = Pruned_;
    static constexpr int m = N / 3 + 1;
    static constexpr int kRows = Pruned_ ? 2 * m : N;      // state rows per field
    static constexpr int kW = Pruned_ ? m : N / 2 + 1;     // state columns
    static constexpr int kPitch = (kW + 15) / 16 * 16;     // of P and Q rows: whole 128-byte lines
    // Columns per tile. From 256 on 8, half a line per access, twice as many workgroups to balance:
    // with both halves read on one XCD, 48 fields of 256^2 362 -> 334 us for six steps, 30 of 512^2
    // 825 -> 722 us.
    static constexpr int kT = N <= 128 ? 16 : 8;
    static constexpr int kTiles = (kW + kT - 1) / kT;
    // Radix and values per lane of the columns: 8 while a tile then takes at most 512 lanes. At 256
    // the update waits on its loads, not on its stages: 12.4 us with 16 values, 10.3 us with 8.
    static constexpr int kR = Few ? 4 : N <= 256 ? 8 : 16;
    using PC = ColumnPlan<N, kR, kR>;
    static constexpr int kColumnThreads = kT * PC::L;
    static constexpr int kColumnLds = pad(N - 1) * kT + kT;
    static constexpr int kRE = Few ? 4 : N <= 512 ? 8 : 16;          // rows: one wave or less per transform
    using PR = Plan<N, kRE, kRE>;
    static constexpr int kRowParts = cmax(1, N / 2 / PR::T);  // row workgroups per field
    static constexpr int kRowLds = PR::T * PR::kStride;

    static_assert(!Few || N == 256, "the shape measured");
    static_assert(PR::L <= 64 && kColumnThreads <= 1024, "workgroup shapes");
    static_assert(slots_match<PR>() && slots_match<PC>(),
                  "one direction's outputs must be the other's inputs");
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

// 1 / x to the last bit or the one before it: the hardware's approximation and one Newton step. With
// correctly rounded divisions the state and the frame are as far off 64 bits after six steps, to four
// digits (256^2 pruned 3.0e-7 and 3.9e-7, 512^2 2.9e-7 and 3.7e-7), and a call takes 2-3 % longer.
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

// A workgroup's field and its part (0 .. Parts-1) of that field.
struct NsBlock {
    int field;
    int part;
};

// Consecutive blocks go to consecutive XCDs. by_xcd: a field's blocks on one XCD; otherwise Share
// consecutive parts on one XCD.
template <int Parts, int Share>
__device__ __forceinline__ NsBlock block_of(bool by_xcd)
{
    const int xcd = static_cast<int>(blockIdx.x) % 8;
    const int slot = static_cast<int>(blockIdx.x) / 8;
    if (by_xcd) {
        return {slot / Parts * 8 + xcd, slot % Parts};
    }
    const int item = slot / Share * 8 + xcd;
    return {item / (Parts / Share), item % (Parts / Share) * Share + slot % Share};
}

template <int Parts, int Share>
unsigned blocks_of(int fields, bool by_xcd)
{
    return by_xcd ? static_cast<unsigned>((fields + 7) / 8) * (8u * Parts)
                  : static_cast<unsigned>((fields * (Parts / Share) + 7) / 8) * (8u * Share);
}

// One set's inverse columns of a tile. v: the state in the transform's input slots.
template <class G>
__device__ __forceinline__ void derived_columns(cf32 (&v)[G::PC::E], cf32* s,
                                                cf32* __restrict__ work, int field, int col,
                                                int lane, int set)
{
    using P = typename G::PC;
    using Lay = PaddedRows<G::kT>;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    const float kx = static_cast<float>(col);
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int i = input_index<P, 0>(lane, e / R0, e % R0);
        v[e] = cmul(v[e], multiplier<G>(set, kx, ky_of<G>(i)));
    }
    run_stages<P, 0, true, false, Lay>(v, s, lane, nullptr);
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

// The first stage of a call: one tile of kT columns of one set. Blocks run set fastest within an
// XCD's share (consecutive blocks go to consecutive XCDs), so the four sets of a tile read the state
// from one L2.
template <class G>
__global__ void __launch_bounds__(G::kColumnThreads)
    ns_columns_kernel(const cf32* __restrict__ state, cf32* __restrict__ work, int fields,
                      bool by_xcd)
{
    using P = typename G::PC;
    constexpr int R0 = P::template radix<0>();
    __shared__ cf32 s[G::kColumnLds];
    const auto [field, part] = block_of<4 * G::kTiles, 4>(by_xcd);
    if (field >= fields) {
        return;  // the whole workgroup
    }
    const int c = static_cast<int>(threadIdx.x) % G::kT;
    const int lane = static_cast<int>(threadIdx.x) / G::kT;
    const int col = part / 4 * G::kT + c;
    const bool live = col < G::kW;
    const cf32* const w = state + static_cast<long long>(field) * G::kRows * G::kW;
    cf32 v[P::E];
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int i = input_index<P, 0>(lane, e / R0, e % R0);
        const int r = state_row<G>(i);
        v[e] = live && r >= 0 ? w[r * G::kW + col] : czero();
    }
    derived_columns<G>(v, s + c, work, field, col, lane, part % 4);
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
__global__ void __launch_bounds__(G::PR::kThreads)
    ns_rows_kernel(const cf32* __restrict__ work, cf32* __restrict__ bins, int fields, bool by_xcd)
{
    using P = typename G::PR;
    constexpr int RL = P::template radix<P::kStages - 1>();
    __shared__ cf32 lds[G::kRowLds];
    const int lane = static_cast<int>(threadIdx.x) % P::L;
    const int t = static_cast<int>(threadIdx.x) / P::L;
    const auto [field, part] = block_of<G::kRowParts, 1>(by_xcd);
    const long long pairs = static_cast<long long>(fields) * (G::N / 2);
    const long long pair = G::kRowParts > 1
                               ? static_cast<long long>(field) * (G::N / 2) + part * P::T + t
                               : static_cast<long long>(blockIdx.x) * P::T + t;
    if (pair - t >= pairs) {
        return;  // the whole workgroup
    }
    cf32* const s = lds + t * P::kStride;
    const bool live = pair < pairs;
    // Lane groups past the end repeat the last pair and store nothing.
    const cf32* const row0 = work + (live ? pair : pairs - 1) * (2LL * 4 * G::kPitch);
    const cf32* const row1 = row0 + 4 * G::kPitch;
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
        cf32* const out = bins + pair * (2LL * G::kPitch);
        for (int k = lane; k < G::kW; k += P::L) {
            const cf32 f = s[pad(k)];
            const cf32 h = s[pad((G::N - k) & (G::N - 1))];
            out[k] = cf32{0.5f * (f.re + h.re), 0.5f * (f.im - h.im)};
            out[G::kPitch + k] = cf32{0.5f * (f.im + h.im), 0.5f * (h.re - f.re)};
        }
    }
}

// What a stage's update reads and writes. The stores of stage 0 go to out_f, those of stage 1 to
// out_w.
struct NsUpdate {
    const cf32* bins;
    const cf32* w0;
    const cf32* f0;
    cf32* out_f;
    cf32* out_w;
    const cf32* forcing_hat;
    const float* nu;
    int nu_stride;
    float drag;
    float dt;
};

// One tile of kT columns: the forward column transforms of the rows' bins and the update. v: the
// state that the stage arrives at, element lane + (e / RL) L + (e % RL) N / RL in slot e, zeros where
// the layout keeps no row. Every load comes before the first store, which may alias w0.
template <class G, int Stage>
__device__ __forceinline__ void update_columns(cf32 (&v)[G::PC::E], cf32* s, const NsUpdate& a,
                                               int field, int col, int lane, bool store)
{
    using P = typename G::PC;
    using Lay = PaddedRows<G::kT>;
    constexpr int R0 = P::template radix<0>();
    constexpr int RL = P::template radix<P::kStages - 1>();
    const cf32* const in = a.bins + static_cast<long long>(field) * G::N * G::kPitch + col;
    const float nu_f = a.nu[static_cast<long long>(field) * a.nu_stride];
    const bool live = col < G::kW;
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int y = input_index<P, 0>(lane, e / R0, e % R0);
        v[e] = live ? in[y * G::kPitch] : czero();
    }
    const long long base = static_cast<long long>(field) * G::kRows * G::kW;
    const auto row_of = [lane](int e) {
        return lane + (e / RL) * P::L + (e % RL) * (P::N / RL);
    };
    run_stages<P, 0, false, false, Lay>(v, s, lane, nullptr);
    cf32 w[P::E];
    cf32 f[P::E];
    cf32 forcing[P::E];
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int r = state_row<G>(row_of(e));
        const bool has = live && r >= 0;
        const int at = has ? r * G::kW + col : 0;
        w[e] = has ? a.w0[base + at] : czero();
        forcing[e] = has ? a.forcing_hat[at] : czero();
        if constexpr (Stage == 1) {
            f[e] = has ? a.f0[base + at] : czero();
        }
    }
    const float kmax = static_cast<float>(G::N) / 3.0f;
    const float kx = static_cast<float>(col);
#pragma unroll
    for (int e = 0; e < P::E; ++e) {
        const int i = row_of(e);
        const int r = state_row<G>(i);
        const float ky = ky_of<G>(i);
        // A product, so that a field that has overflowed spreads to every mode, as N_hat * mask does.
        const float mask = kx <= kmax && fabsf(ky) <= kmax ? 1.0f : 0.0f;
        const cf32 F = csub(forcing[e], cscale(v[e], mask));
        const float linear = -nu_f * (kx * kx + ky * ky) - a.drag;
        const float ex = 1.0f + 0.5f * a.dt * linear;
        const float im = reciprocal(1.0f - 0.5f * a.dt * linear);
        const cf32 add = Stage == 0 ? cscale(F, a.dt) : cscale(cadd(f[e], F), 0.5f * a.dt);
        const cf32 next = cscale(cadd(cscale(w[e], ex), add), im);
        const bool has = live && r >= 0;
        if (has && store) {
            (Stage == 0 ? a.out_f : a.out_w)[base + r * G::kW + col] = Stage == 0 ? F : next;
        }
        v[e] = has ? next : czero();
    }
}

// The last stage of a call.
template <class G>
__global__ void __launch_bounds__(G::kColumnThreads)
    ns_update_kernel(NsUpdate a, int fields, bool by_xcd)
{
    __shared__ cf32 s[G::kColumnLds];
    const auto [field, part] = block_of<G::kTiles, 1>(by_xcd);
    if (field >= fields) {
        return;  // the whole workgroup
    }
    const int c = static_cast<int>(threadIdx.x) % G::kT;
    const int col = part * G::kT + c;
    cf32 v[G::PC::E];
    update_columns<G, 1>(v, s + c, a, field, col, static_cast<int>(threadIdx.x) / G::kT, true);
}

// The update of a stage and the derived columns of the next one, Sets of a tile's four per workgroup.
// The workgroups of a tile each form its new state, which one of them stores.
template <class G, int Stage, int Sets>
__global__ void __launch_bounds__(G::kColumnThreads)
    ns_update_columns_kernel(NsUpdate a, cf32* __restrict__ work, int fields, bool by_xcd)
{
    using P = typename G::PC;
    __shared__ cf32 s[G::kColumnLds];
    constexpr int kShare = 4 / Sets;
    const auto [field, part] = block_of<kShare * G::kTiles, kShare>(by_xcd);
    const int first = part % kShare * Sets;
    if (field >= fields) {
        return;  // the whole workgroup
    }
    const int c = static_cast<int>(threadIdx.x) % G::kT;
    const int lane = static_cast<int>(threadIdx.x) / G::kT;
    const int col = part / kShare * G::kT + c;
    cf32 state[P::E];
    update_columns<G, Stage>(state, s + c, a, field, col, lane, first == 0);
    cf32 next[P::E];  // in the inverse's input slots
    static_for<0, P::E>([&](auto ei) {
        constexpr int e = decltype(ei)::value;
        next[forward_slot_of<P>(e)] = state[e];
    });
#pragma unroll
    for (int set = 0; set < Sets; ++set) {
        cf32 v[P::E];
#pragma unroll
        for (int e = 0; e < P::E; ++e) {
            v[e] = next[e];
        }
        derived_columns<G>(v, s + c, work, field, col, lane, first + set);
    }
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

// Whether a field's blocks all run on one XCD, so that what one kernel writes is in the L2 the next
// one reads it from. Always up to 256^2 (six steps, best of either order: one field of 128^2 in the
// full layout 186 -> 146 us, nine 209 -> 170, one field of 256^2 164 -> 155, 48 357 -> 334). Larger
// fields do not fit an L2, and an idle XCD costs more: only if at most an eighth of the XCDs are
// idle (512^2: one field 222 against 299 us, 12 fields 404 against 414, 8 fields 331 -> 322, 30 797
// -> 722; 1024^2: four fields 542 against 880 us, 8 fields 981 -> 899).
template <class G>
bool by_xcd(int fields)
{
    const int rounds = (fields + 7) / 8;
    return G::N <= 256 || fields >= 7 * rounds;
}

template <class G>
void launch_rows(const cf32* spectra, cf32* bins, int fields, hipStream_t stream)
{
    const int pairs = fields * (G::N / 2);
    const unsigned blocks = G::kRowParts > 1 ? blocks_of<G::kRowParts, 1>(fields, by_xcd<G>(fields))
                                             : static_cast<unsigned>((pairs + G::PR::T - 1) / G::PR::T);
    hipLaunchKernelGGL(ns_rows_kernel<G>, dim3(blocks), dim3(G::PR::kThreads), 0, stream, spectra,
                       bins, fields, by_xcd<G>(fields));
    SPX_LAUNCH_CHECK();
}

template <class G, int Stage, int Sets>
void launch_update_columns(const NsUpdate& a, cf32* spectra, int fields, hipStream_t stream)
{
    const unsigned blocks = blocks_of<4 / Sets * G::kTiles, 4 / Sets>(fields, by_xcd<G>(fields));
    hipLaunchKernelGGL((ns_update_columns_kernel<G, Stage, Sets>), dim3(blocks),
                       dim3(G::kColumnThreads), 0, stream, a, spectra, fields, by_xcd<G>(fields));
    SPX_LAUNCH_CHECK();
}

// One, two or all four sets per workgroup: the fewest workgroups that repeat a tile's update while
// there are at most two waves per SIMD of the chip. 256^2 pruned, six steps with 1 / 2 / 4 sets:
// 8 fields 169 / 167 / 185 us, 16 fields 199 / 195 / 200, 48 fields 377 / 339 / 334, 100 fields
// 641 / 559 / 547; 1024^2: one field 368 / 394 / 451, two 447 / 401 / 457, four 618 / 632 / 542.
template <class G, int Stage>
void update_and_columns(const NsUpdate& a, cf32* spectra, int fields, hipStream_t stream)
{
    const long long waves = static_cast<long long>(fields) * G::kTiles * (G::kColumnThreads / 64);
    const long long filled = 8LL * device_cus();
    if (4 * waves <= filled) {
        launch_update_columns<G, Stage, 1>(a, spectra, fields, stream);
    } else if (2 * waves <= filled) {
        launch_update_columns<G, Stage, 2>(a, spectra, fields, stream);
    } else {
        launch_update_columns<G, Stage, 4>(a, spectra, fields, stream);
    }
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
    return static_cast<std::size_t>(group) * (5 * G::N * G::kPitch + 2 * G::kRows * G::kW);
}

template <class G>
void advance(const NsArrays& a, int batch, int steps, hipStream_t stream)
{
    constexpr long long kField = static_cast<long long>(G::kRows) * G::kW;
    const int most = std::min(batch, fields_per_group<G>());
    const int groups = (batch + most - 1) / most;
    constexpr long long kGrid = static_cast<long long>(G::N) * G::kPitch;
    cf32* const spectra = a.work;
    cf32* const bins = spectra + most * 4 * kGrid;
    cf32* const tendency = bins + most * kGrid;
    cf32* const spare = tendency + most * kField;
    for (int g = 0; g < groups; ++g) {
        // Even shares, so that no group is left with a few fields.
        const int first = static_cast<int>(static_cast<long long>(batch) * g / groups);
        const int fields = static_cast<int>(static_cast<long long>(batch) * (g + 1) / groups) - first;
        cf32* const out = a.w_out + first * kField;
        NsUpdate u{bins, a.w_in + first * kField, tendency, tendency, nullptr, a.forcing_hat,
                   a.nu + static_cast<long long>(first) * a.nu_stride, a.nu_stride, a.drag, a.dt};
        hipLaunchKernelGGL(ns_columns_kernel<G>, dim3(blocks_of<4 * G::kTiles, 4>(fields, by_xcd<G>(fields))),
                           dim3(G::kColumnThreads), 0, stream, u.w0, spectra, fields, by_xcd<G>(fields));
        SPX_LAUNCH_CHECK();
        for (int s = 0; s < steps; ++s) {
            launch_rows<G>(spectra, bins, fields, stream);
            update_and_columns<G, 0>(u, spectra, fields, stream);
            launch_rows<G>(spectra, bins, fields, stream);
            if (s + 1 < steps) {
                // Not into w0, which other workgroups of the tile still read.
                u.out_w = u.w0 == spare ? out : spare;
                update_and_columns<G, 1>(u, spectra, fields, stream);
                u.w0 = u.out_w;
            }
        }
        u.out_w = out;
        hipLaunchKernelGGL(ns_update_kernel<G>, dim3(blocks_of<G::kTiles, 1>(fields, by_xcd<G>(fields))),
                           dim3(G::kColumnThreads), 0, stream, u, fields, by_xcd<G>(fields));
        SPX_LAUNCH_CHECK();
    }
}

// f(G{}) for the kernels' grid of this size, layout and number of fields. Up to 16 fields of 256^2
// (two per XCD) leave SIMDs without a wave, and shorter waves are then faster: six steps, 8 / 4
// values per lane, one field 160 -> 146 us, 8 fields 168 -> 152 (204 -> 190 in the full layout), 16
// fields 194 -> 191, 33 fields 284 -> 311.
template <class F>
auto dispatch(int n, bool pruned, int batch, F&& f)
{
    const auto layout = [&](auto size) {
        constexpr int N = decltype(size)::value;
        return pruned ? f(NsGrid<N, true>{}) : f(NsGrid<N, false>{});
    };
    switch (n) {
    case 32: return layout(std::integral_constant<int, 32>{});
    case 64: return layout(std::integral_constant<int, 64>{});
    case 128: return layout(std::integral_constant<int, 128>{});
    case 256:
        if (batch <= 16) {
            return pruned ? f(NsGrid<256, true, true>{}) : f(NsGrid<256, false, true>{});
        }
        return layout(std::integral_constant<int, 256>{});
    case 512: return layout(std::integral_constant<int, 512>{});
    case 1024: return layout(std::integral_constant<int, 1024>{});
    default:
        throw InvalidArgument("ns_grid_steps: supports n = 32 to 1024, a power of two, got "
                              + str(n));
    }
}

}  // namespace
}  // namespace dev

namespace {

// An array in memory.
struct Span {
    const void* first;
    std::uintptr_t bytes;

    bool overlaps(const Span& other) const
    {
        const auto a = reinterpret_cast<std::uintptr_t>(first);
        const auto b = reinterpret_cast<std::uintptr_t>(other.first);
        return a < b + other.bytes && b < a + bytes;
    }
};

}  // namespace

bool ns_grid_supports(int n) { return is_pow2(n) && n >= 32 && n <= 1024; }

std::size_t ns_grid_workspace(int n, bool pruned, int batch)
{
    if (batch < 1) {
        throw InvalidArgument("ns_grid_workspace: need batch >= 1");
    }
    return dev::dispatch(
        n, pruned, batch, [&](auto g) { return dev::workspace<decltype(g)>(batch); });
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
    dev::dispatch(n, pruned, batch, [&](auto g) {
        using G = decltype(g);
        constexpr std::uintptr_t kField = sizeof(cf32) * G::kRows * G::kW;
        const Span in{w_in, batch * kField};
        const Span out{w_out, batch * kField};
        const Span wk{work, dev::workspace<G>(batch) * sizeof(cf32)};
        const Span forcing{forcing_hat, kField};
        const Span nus{nu, (nu_stride == 0 ? 1 : batch) * sizeof(float)};
        if (wk.overlaps(in) || wk.overlaps(out) || wk.overlaps(forcing) || wk.overlaps(nus)) {
            throw InvalidArgument("ns_grid_steps: work must not overlap another array");
        }
        if (w_in != w_out && in.overlaps(out)) {
            throw InvalidArgument(
                "ns_grid_steps: w_in and w_out must be the same array or not overlap");
        }
        dev::advance<G>(arrays, batch, steps, stream);
    });
}

}  // namespace spx
