// Device pieces shared by the one-workgroup-per-system kernels
// (getrf_wg.hip, getrs_wg.hip): MFMA operand layouts, the pivot search of a
// wave, and the blocked triangular sweep on a system's right-hand sides.
#pragma once

#include "lu_device.h"
#include "magma_internal.h"

#include <climits>
#include <type_traits>
#include <utility>

namespace mgi {

constexpr int kWgNB = 32;           // block width of the LU and of the sweeps

// v_mfma_*_16x16x4 layouts (lane l, lr = l % 16, lq = l / 16): first operand
// P[lr][k = lq], second operand Q[k = lq][lr], result rows row(r, lq), column
// lr, r = 0..3. With the product's depth index taken in the order row(r, lq)
// the result registers of one product are the operand registers of the next.
template <typename T> struct WgMfma;
template <> struct WgMfma<double> {
    typedef double acc_t __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ int row(int r, int lq) { return 4 * r + lq; }
    __device__ static __forceinline__ acc_t mma(double p, double q, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, c, 0, 0, 0);
    }
};
template <> struct WgMfma<float> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ int row(int r, int lq) { return 4 * lq + r; }
    __device__ static __forceinline__ acc_t mma(float p, float q, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(p, q, c, 0, 0, 0);
    }
};
// depth index of step kk (0..7) of a 32-deep product
template <typename T>
__device__ __forceinline__ int wg_k(int kk, int lq) { return 16 * (kk >> 2) + WgMfma<T>::row(kk & 3, lq); }

// Zero that the compiler cannot see through: lane indices that a phase
// offsets by it keep the phase's address arithmetic inside the phase (hoisted
// out of the block loop, the addresses of all phases live in registers at
// once and the LU kernels spill far more than the FP64 forms do now).
__device__ __forceinline__ int wg_opaque_zero()
{
    int z = 0;
    asm volatile("" : "+r"(z));
    return z;
}

// This thread's wave, as a wave-uniform (scalar) value.
__device__ __forceinline__ int wg_wave() { return __builtin_amdgcn_readlane((int)threadIdx.x / kWave, 0); }

template <int... Js, typename F>
__device__ __forceinline__ void wg_for(std::integer_sequence<int, Js...>, F&& f)
{
    (f(std::integral_constant<int, Js>{}), ...);
}

template <typename T> struct WgLim;
template <> struct WgLim<double> { static constexpr double sfmin = kSfminD; };
template <> struct WgLim<float>  { static constexpr float sfmin = kSfminF; };

// Maximum of an int over each group of G lanes (G = 64: the whole wave), as
// a wave-uniform value; for G < 64 every group must hold the same values.
// (Every stage is one DPP-sourced v_max_i32: the quad and mirror patterns
// read a valid lane everywhere, and the row broadcasts leave the masked rows
// at the identity.)
template <int G>
__device__ __forceinline__ int wg_group_max(int v)
{
    if constexpr (G >= 2) v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppQuadXor1, 0xF, 0xF, true));
    if constexpr (G >= 4) v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppQuadXor2, 0xF, 0xF, true));
    if constexpr (G >= 8) v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppHalfMirror, 0xF, 0xF, true));
    if constexpr (G >= 16) v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppMirror, 0xF, 0xF, true));
    if constexpr (G >= 32) {
        v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppBcast15, 0xA, 0xF, false));
        v = max(v, __builtin_amdgcn_update_dpp(INT_MIN, v, kDppBcast31, 0xC, 0xF, false));
    }
    return __builtin_amdgcn_readlane(v, 63);
}

// Lane (of the first group) that holds the largest v, ties to the lowest
// pos; lanes without a candidate pass v = -1. A non-negative floating value
// orders like its bits, so the search runs on the upper 32 bits alone (one
// DPP-sourced v_max per stage) and looks at the rest only when they tie.
// (The 64-bit search costs two moves and a v_max_f64 per stage: about twice
// the latency of the pivot chain.)
template <int G>
__device__ __forceinline__ int wg_pick(double v, int pos)
{
    constexpr unsigned long long kMask = G == 64 ? ~0ull : ((1ull << G) - 1);
    const int hi = __double2hiint(v);
    const int mh = wg_group_max<G>(hi);
    unsigned long long b = __ballot(hi == mh) & kMask;
    if ((b & (b - 1)) != 0ull) {
        const int lo = hi == mh ? (__double2loint(v) ^ INT_MIN) : INT_MIN;
        const int ml = wg_group_max<G>(lo);
        const bool c = hi == mh && lo == ml;
        b = __ballot(c) & kMask;
        if ((b & (b - 1)) != 0ull) {
            const int mp = -wg_group_max<G>(c ? -pos : -INT_MAX);
            b = __ballot(c && pos == mp) & kMask;
        }
    }
    return __ffsll((long long)b) - 1;
}
template <int G>
__device__ __forceinline__ int wg_pick(float v, int pos)
{
    constexpr unsigned long long kMask = G == 64 ? ~0ull : ((1ull << G) - 1);
    const int hi = __float_as_int(v);
    const int mh = wg_group_max<G>(hi);
    unsigned long long b = __ballot(hi == mh) & kMask;
    if ((b & (b - 1)) != 0ull) {
        const bool c = hi == mh;
        const int mp = -wg_group_max<G>(c ? -pos : -INT_MAX);
        b = __ballot(c && pos == mp) & kMask;
    }
    return __ffsll((long long)b) - 1;
}

// Broadcast lane Q of every quad to the whole quad.
template <int Q>
__device__ __forceinline__ double wg_quad(double v) { return quad_bcast_d<Q>(v); }
template <int Q>
__device__ __forceinline__ float wg_quad(float v)
{
    constexpr int ctrl = Q | (Q << 2) | (Q << 4) | (Q << 6);
    return dpp_f<ctrl>(v);
}

// One 32 x 32 triangular system per four lanes: lane 4c + q holds rows q,
// q+4, .. (y[0..7]) of column c; the solved entry of each step reaches the
// other lanes of the quad by DPP. d (LDS, row stride 33) is lower triangular,
// or upper triangular and solved from the last row up with BACK; with DIAG its
// diagonal holds reciprocal pivots, without it is one. A row that a step does
// not reach keeps its value whatever the step's factors are (a select, not a
// zero factor: an infinite entry stays in its row). Rows from nb on are an
// identity with a zero right-hand side; the groups of four steps that hold
// only such rows are skipped. The branch between the groups also bounds the
// compiler's scheduling: without it the FP64 solves spilled up to 52 registers
// (8,192 x 8^2 with five right-hand sides 106 us instead of 62).
template <typename T, bool BACK, bool DIAG = false>
__device__ __forceinline__ void wg_solve_block(const T* d, T (&y)[8], int q, int nb = kWgNB)
{
    constexpr int LD = kWgNB + 1;
    wg_for(std::make_integer_sequence<int, kWgNB / 4>{}, [&](auto gc) {
        constexpr int g = BACK ? kWgNB / 4 - 1 - decltype(gc)::value : decltype(gc)::value;
        if (4 * g >= nb) return;
        // four steps' coefficients in flight at a time
        __builtin_amdgcn_sched_barrier(0);
        wg_for(std::make_integer_sequence<int, 4>{}, [&](auto kc) {
            constexpr int qk = BACK ? 3 - decltype(kc)::value : decltype(kc)::value;
            constexpr int sk = g, k = 4 * g + qk;
            if constexpr (DIAG) {
                const T v = y[sk] * d[k * LD + k];
                y[sk] = q == qk ? v : y[sk];
            }
            const T xk = wg_quad<qk>(y[sk]);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                if (BACK ? 4 * s >= k : 4 * s + 3 <= k) continue;          // every row of the slot is done
                const int i = q + 4 * s;
                const T v = fma(-d[i * LD + k], xk, y[s]);
                const bool whole = BACK ? 4 * s + 3 < k : 4 * s > k;       // every row of the slot is reached
                y[s] = (whole || (BACK ? i < k : i > k)) ? v : y[s];
            }
        });
    });
}

// ---------------------------------------------------------------------------
// Triangular sweep: B := E^{-1} B for one n x n triangle of the factors in A
// (E = its transpose with TRANS), B column-major with nr <= MAXR columns
// in global memory or in LDS (PB), all waves of the workgroup. BACK runs from
// the last row up. Per block of 32 rows: the diagonal block goes to LDS; one
// wave per 16 right-hand sides solves it (wg_solve_block); then every wave takes
// 16-row tiles of the remaining rows and removes the block's contribution by
// MFMA, its operand read straight from the factors. The next diagonal block
// and each wave's first tile are loaded while the block is solved. Each entry
// of the triangle is read once, so the sweep is bound by HBM once enough
// workgroups hide the chain of blocks.
// ---------------------------------------------------------------------------
template <typename T, int MAXR>
struct WgSweepSmem {
    static constexpr int LD = kWgNB + 1;
    T d[kWgNB * LD];               // d[i*LD + j] = E(kb + i, kb + j)
    T x[MAXR * LD];                // the block's right-hand sides, x[c*LD + i]
};

template <typename T, int NTH, bool BACK, bool TRANS, bool UNIT, typename PB, int MAXR>
__device__ __forceinline__ void wg_sweep(const MGI_GLOBAL_AS T* A, int ld, int n, PB B, int ldb, int nr,
                                         WgSweepSmem<T, MAXR>& sm)
{
    constexpr int LD = WgSweepSmem<T, MAXR>::LD;
    constexpr int W = NTH / kWave;
    constexpr int ND = kWgNB * kWgNB / NTH;        // diagonal-block entries per thread
    using M = WgMfma<T>;
    const int nblk = (n + kWgNB - 1) / kWgNB;
    const int nstr = (nr + 15) / 16;
    auto block = [&](int ib) { return kWgNB * (BACK ? nblk - 1 - ib : ib); };
    T dreg[ND];
    // memory runs down i (or j when transposed); outside the block: identity
    auto load_d = [&](int kb) {
        const int nb = min(kWgNB, n - kb);
#pragma unroll
        for (int u = 0; u < ND; ++u) {
            const int e = (int)threadIdx.x + NTH * u;
            const int p = min(e % kWgNB, nb - 1), q = min(e / kWgNB, nb - 1);
            dreg[u] = A[(kb + p) + (size_t)(kb + q) * ld];
        }
    };
    load_d(block(0));
    for (int ib = 0; ib < nblk; ++ib) {
        const int t = threadIdx.x + wg_opaque_zero(), w = wg_wave(), l = t % kWave;
        const int lr = l % 16, lq = l / 16;
        const int kb = block(ib);
        const int nb = min(kWgNB, n - kb);
        T dg = T(1);
#pragma unroll
        for (int u = 0; u < ND; ++u) {
            const int p = (t + NTH * u) % kWgNB, q = (t + NTH * u) / kWgNB;
            const int i = TRANS ? q : p, j = TRANS ? p : q;
            T v = i == j ? T(1) : T(0);
            if (p < nb && q < nb && !(UNIT && i == j) && (BACK ? j >= i : j <= i)) v = dreg[u];
            dg = i == j ? v : dg;
            sm.d[i * LD + j] = v;
        }
        if constexpr (!UNIT) {
            // the diagonal as reciprocals: each thread holds at most one of
            // its entries, so one division serves the block
            const int p = t % kWgNB;
            if (p % (NTH / kWgNB) == t / kWgNB) sm.d[p * LD + p] = T(1) / dg;
        }
        for (int e = t; e < kWgNB * 16 * nstr; e += NTH) {
            const int i = e % kWgNB, c = e / kWgNB;
            sm.x[c * LD + i] = (i < nb && c < nr) ? B[(kb + i) + (size_t)c * ldb] : T(0);
        }
        if (ib + 1 < nblk) load_d(block(ib + 1));
        // the rows not yet solved: below the block (a block with rows below
        // is full), or above it
        const int r0 = BACK ? 0 : kb + kWgNB, r1 = BACK ? kb : n;
        const int tiles = r1 > r0 ? (r1 - r0 + 15) / 16 : 0;
        auto load_e = [&](int ti, T (&ef)[8]) {
            const int row = min(r0 + 16 * ti + lr, r1 - 1);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                const int kc = kb + min(wg_k<T>(kk, lq), nb - 1);
                ef[kk] = TRANS ? A[kc + (size_t)row * ld] : A[row + (size_t)kc * ld];
            }
        };
        T ef[8];
        if (w < tiles) load_e(w, ef);
        __syncthreads();
        for (int sw = w; sw < nstr; sw += W) {
            const int c = 16 * sw + (l >> 2), q = l & 3;
            T y[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) y[s] = sm.x[c * LD + q + 4 * s];
            wg_solve_block<T, BACK, !UNIT>(sm.d, y, q, nb);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int i = q + 4 * s;
                sm.x[c * LD + i] = y[s];
                if (i < nb && c < nr) B[(kb + i) + (size_t)c * ldb] = y[s];
            }
        }
        __syncthreads();
        // the first tile was loaded during the solve; with it waited for here
        // the loop's own waits leave the next tile's loads in flight (in the
        // loop, the wait for either would be for both)
        __builtin_amdgcn_s_waitcnt(0x0F70);                    // vmcnt(0)
        for (int ti = w; ti < tiles; ti += W) {
            const int row = r0 + 16 * ti + lr;
            const bool rin = row < r1;
            T en[8];
            if (ti + W < tiles) load_e(ti + W, en);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) ef[kk] = wg_k<T>(kk, lq) < nb ? ef[kk] : T(0);
            for (int s = 0; s < nstr; ++s) {
                T bv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    bv[r] = B[min(row, r1 - 1) + (size_t)min(16 * s + M::row(r, lq), nr - 1) * ldb];
                typename M::acc_t acc = {0, 0, 0, 0};
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) acc = M::mma(sm.x[(16 * s + lr) * LD + wg_k<T>(kk, lq)], ef[kk], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int c = 16 * s + M::row(r, lq);
                    if (rin && c < nr) B[row + (size_t)c * ldb] = bv[r] - acc[r];
                }
            }
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) ef[kk] = en[kk];
        }
        __syncthreads();
    }
}

}  // namespace mgi
