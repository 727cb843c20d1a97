// Batched LU (and LU + solve) with one workgroup per system: the whole
// right-looking factorisation of a matrix of up to 512 rows runs inside one
// kernel, one thread per row, so the panel's chain of pivot steps of one
// system overlaps the updates of the others on the same CU and no launch
// boundary separates the steps. Per block of 32 columns:
//   panel    thread t holds row k + t of the block in registers; per column
//            every wave publishes its best candidate with its whole row in
//            LDS, one barrier, and every thread applies the rank-1 update.
//            Rows are not moved: each carries its LAPACK position and is
//            written to it after the last column;
//   swaps    the block's row permutation on the columns to the right,
//   + U12    together with U12 = L11^{-1} A12, 16 columns per wave pass: the
//            32 pivot rows are gathered (four lanes per column) and forward
//            substituted, the displaced top rows move down;
//   update   A22 -= L21 U12, each wave a strip of 32 rows: its L21 operands
//            stay in registers for the whole step, U12 and A22 stream through
//            L1 / L2.
// The factored columns' later interchanges are composed and applied once at
// the end. With right-hand sides (gesv) B is carried along as more columns
// on the right and the back substitution follows in the same kernel.
//
// What bounds it: traffic past the L2 at the copy rate (each block reads and
// writes the trailing matrix twice). At most 128 VGPRs (four waves per SIMD)
// keeps 16 waves per CU in flight; the panel's dependent chain (about one
// microsecond per column when alone) is hidden by the other systems of the CU.
// The FP64 forms spill 23 registers at that bound (96 bytes of scratch a lane):
// values kept across a block, and a diagonal block's entries in the back
// substitution, none in the column steps or the update's MFMA loops. The FP32
// forms do not spill.
//
// Reference behaviour: magmablas/zgetf2_devicefunc.cuh:218-294 (panel step),
// magmablas/magma_templates.h:44-60 (ties), src/zgetrf_panel_batched.cpp:102-196
// (panel / laswp / trsm / gemm order), src/xshgetrf_gpu.cpp:214-350 (FP32
// panel, low-precision trailing update).
#include "magma_internal.h"
#include "getrf_kernels.h"
#include "wg_lu.h"

namespace mgi {

namespace {

typedef __bf16 wbf8_t __attribute__((ext_vector_type(8)));
typedef _Float16 wh8_t __attribute__((ext_vector_type(8)));

constexpr int kWgGesvRhs = 16;      // right-hand sides carried along with the matrix

template <typename T, int NTH>
struct WgSmem {
    static constexpr int W = NTH / kWave;
    static constexpr int NB = kWgNB;
    static constexpr int LD = NB + 1;
    union {
        struct {
            alignas(16) T cand[2][W][16];  // each wave's candidate row, by step parity
            T rinv[2][W];
            T val[2][W];
            int pos[2][W];
            T l11[NB * LD];                // the block's top 32 rows, l11[i*LD + j]
            int dst[NB];                   // where top row i went (below the block), or -1
        } f;
        WgSweepSmem<T, kWgGesvRhs> sweep;
    };
    unsigned short map[NTH / NB][NTH];     // per block: position -> row before the block's interchanges
};

// Operands of the trailing update: KK values per lane and MFMA step.
template <typename T, int MODE>
struct UpdOperand {
    static constexpr bool kWide = MODE == kUpdBF16 || MODE == kUpdFP16 || MODE == kUpdBF16x3;
    // depth index of value v (0..7) of a lane
    __device__ static __forceinline__ int k(int v, int lq) { return kWide ? 8 * lq + v : wg_k<T>(v, lq); }
    T x[8];
    __device__ __forceinline__ void finish() {}
};
template <>
struct UpdOperand<float, kUpdFP16> {
    __device__ static __forceinline__ int k(int v, int lq) { return 8 * lq + v; }
    float x[8];
    wh8_t h;
    __device__ __forceinline__ void finish()
    {
#pragma unroll
        for (int v = 0; v < 8; ++v) h[v] = (_Float16)x[v];
    }
};
template <>
struct UpdOperand<float, kUpdBF16> {
    __device__ static __forceinline__ int k(int v, int lq) { return 8 * lq + v; }
    float x[8];
    wbf8_t h;
    __device__ __forceinline__ void finish()
    {
#pragma unroll
        for (int v = 0; v < 8; ++v) h[v] = (__bf16)x[v];
    }
};
template <>
struct UpdOperand<float, kUpdBF16x3> {
    __device__ static __forceinline__ int k(int v, int lq) { return 8 * lq + v; }
    float x[8];
    wbf8_t h, lo;
    __device__ __forceinline__ void finish()
    {
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            h[v] = (__bf16)x[v];
            lo[v] = (__bf16)(x[v] - (float)h[v]);
        }
    }
};

// acc += U^T L^T over a depth of 32 (first operand U, second L: lane lr is a
// row of the tile, the registers its columns)
template <typename T, int MODE>
__device__ __forceinline__ typename WgMfma<T>::acc_t upd_mma(const UpdOperand<T, MODE>& u, const UpdOperand<T, MODE>& l,
                                                             typename WgMfma<T>::acc_t acc)
{
    if constexpr (MODE == kUpdFP16) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(u.h, l.h, acc, 0, 0, 0);
    } else if constexpr (MODE == kUpdBF16) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u.h, l.h, acc, 0, 0, 0);
    } else if constexpr (MODE == kUpdBF16x3) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u.h, l.lo, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u.lo, l.h, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u.h, l.h, acc, 0, 0, 0);
    } else {
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) acc = WgMfma<T>::mma(u.x[kk], l.x[kk], acc);
    }
    return acc;
}

// one 16-column strip of what lies right of the block: A's columns, then B's
template <typename T>
struct Strip {
    MGI_GLOBAL_AS T* p;     // row k (the block's first row) of the strip's first column
    int ld, nc;             // leading dimension, columns in the strip (<= 16)
};

}  // namespace

template <typename T, int MODE, int NTH>
__global__ void __launch_bounds__(NTH, 4)
getrf_wg_kernel(SizeArgs sz, T** __restrict__ dA_array, int** __restrict__ ipiv_array, int* __restrict__ info_array,
                WgRhs<T> rhs)
{
    constexpr int W = NTH / kWave, NB = kWgNB;
    constexpr int kVec = 16 / sizeof(T);              // values per 16-byte LDS access
    typedef T vec_t __attribute__((ext_vector_type(kVec)));
    using M = WgMfma<T>;
    using acc_t = typename M::acc_t;
    using Smem = WgSmem<T, NTH>;
    constexpr int LD = Smem::LD;
    __shared__ Smem sm;
    const int b = sz.mat(blockIdx.x);
    int m, n, ld;
    sz.get(b, m, n, ld);
    const int t = threadIdx.x, w = wg_wave();
    const int minmn = min(m, n);
    if (minmn <= 0) {
        if (t == 0) info_array[b] = 0;
        return;
    }
    auto A = gptr(dA_array[b]);
    // a null pivot array asks for the factorisation without pivoting
    // (src/zgetrf_nopiv_batched.cpp): the diagonal entry is the pivot
    const bool nopiv = ipiv_array == nullptr;
    auto ipiv = gptr(nopiv ? nullptr : ipiv_array[b]);
    const bool solve = rhs.dB_array != nullptr;
    auto B = gptr(solve ? rhs.dB_array[b] : nullptr);
    const int nr = solve ? (rhs.nrhs_arr ? rhs.nrhs_arr[b] : rhs.nrhs) : 0;
    const int ldb = solve ? (rhs.lddb_arr ? rhs.lddb_arr[b] : rhs.lddb) : 0;
    int info = 0;

    for (int k = 0, st = 0; k < minmn; k += NB, ++st) {
        const int jb = min(NB, minmn - k);
        const int mloc = m - k;
        auto P = A + k + (size_t)k * ld;
        // ---- panel ---------------------------------------------------------
        {
            T a[NB];
            const int l = t % kWave;
            // rows and columns outside the panel read a valid element and
            // become zero (a select costs less than a branch per load)
            auto Pt = P + min(t, mloc - 1);
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const T v = Pt[(size_t)min(c, jb - 1) * ld];
                a[c] = (t < mloc && c < jb) ? v : T(0);
            }
            int pos = t, piv = 0;
            bool active = t < mloc;
            // Two halves of 16 columns through the same code (the phases share
            // the instruction cache): each half keeps its update to itself, the
            // first then updates the second, whose registers take its place
#pragma unroll 1
            for (int h = 0; h < 2; ++h) {
                const int j0 = 16 * h;
                wg_for(std::make_integer_sequence<int, 16>{}, [&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    constexpr int par = j & 1;
                    constexpr int ja = j / kVec * kVec;    // first column of the vectors that hold column j
                    if (j0 + j < jb) {
                        // candidate of this row (LAPACK idamax: a NaN wins only at
                        // the first position, where it counts as infinite)
                        const bool first = pos == j0 + j;
                        const T alt = first ? T(INFINITY) : T(-1);
                        T v = fabs(a[j]);
                        v = ((v == v) & !nopiv) ? v : alt;
                        v = active ? v : T(-1);
                        if (__ballot(active) != 0ull) {
                            // every lane's reciprocal, formed while the search runs
                            const T ri = T(1) / a[j];
                            const int pl = wg_pick<64>(v, pos);
                            const T rw = readlane_t(ri, pl);
                            if (l == pl) {
                                sm.f.val[par][w] = v;
                                sm.f.pos[par][w] = v >= T(0) ? pos : INT_MAX;
                                sm.f.rinv[par][w] = rw;
#pragma unroll
                                for (int c = ja; c < 16; c += kVec) {
                                    vec_t x;
#pragma unroll
                                    for (int e = 0; e < kVec; ++e) x[e] = a[c + e];
                                    *reinterpret_cast<vec_t*>(&sm.f.cand[par][w][c]) = x;
                                }
                            }
                        } else if (l == 0) {
                            sm.f.val[par][w] = T(-1);
                            sm.f.pos[par][w] = INT_MAX;
                        }
                        __syncthreads();
                        const int posv = sm.f.pos[par][l % W];
                        const T rv = sm.f.rinv[par][l % W];
                        const int pw = wg_pick<W>(sm.f.val[par][l % W], posv);
                        // the whole pivot row at once (one LDS round trip)
                        T u[16];
#pragma unroll
                        for (int c = ja; c < 16; c += kVec) {
                            const vec_t x = *reinterpret_cast<const vec_t*>(&sm.f.cand[par][pw][c]);
#pragma unroll
                            for (int e = 0; e < kVec; ++e) u[c + e] = x[e];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        const int p = __builtin_amdgcn_readlane(posv, pw);
                        const T rinv = readlane_t(rv, pw);
                        const T pv = u[j];
                        const bool zero = __ballot(pv == T(0)) != 0ull;
                        piv = l == j0 + j ? p : piv;
                        if (zero && info == 0) info = k + j0 + j + 1;
                        // interchange of positions j0 + j and p
                        const bool win = active & (pos == p);
                        pos = (active & first) ? p : pos;
                        pos = win ? j0 + j : pos;
                        active = active & !win;
                        // a zero pivot leaves its column unscaled; the step
                        // is applied all the same (LAPACK dgetf2)
                        T f = a[j] * rinv;
                        if (__ballot(fabs(pv) < WgLim<T>::sfmin) != 0ull) {
                            asm volatile("" ::: "memory");     // no division outside this branch
                            f = zero ? a[j] : a[j] / pv;
                        }
                        if (active) {
                            a[j] = f;
#pragma unroll
                            for (int c = j + 1; c < 16; ++c) a[c] = fma(-f, u[c], a[c]);
                        }
                    }
                });
                if (h == 0 && jb > 16) {
                    // U12 of the second half: the first half's pivot rows
                    // forward-substituted by one wave (lane 4c + q: column c,
                    // rows q, q+4, ..), then removed from the rows below
                    if (t < mloc && pos < 16) {
#pragma unroll
                        for (int c = 0; c < NB; ++c) sm.f.l11[pos * LD + c] = a[c];
                    }
                    __syncthreads();
                    if (w == 0) {
                        const int c = 16 + (l >> 2), q = l & 3;
                        T x[4];
#pragma unroll
                        for (int s = 0; s < 4; ++s) x[s] = sm.f.l11[(q + 4 * s) * LD + c];
                        wg_for(std::make_integer_sequence<int, 15>{}, [&](auto kc) {
                            constexpr int kk = decltype(kc)::value;
                            const T xk = wg_quad<kk & 3>(x[kk >> 2]);
#pragma unroll
                            for (int s = 0; s < 4; ++s) {
                                if (4 * s + 3 <= kk) continue;
                                const int i = q + 4 * s;
                                const T y = fma(-sm.f.l11[i * LD + kk], xk, x[s]);
                                x[s] = (4 * s > kk || i > kk) ? y : x[s];
                            }
                        });
#pragma unroll
                        for (int s = 0; s < 4; ++s) sm.f.l11[(q + 4 * s) * LD + c] = x[s];
                    }
                    __syncthreads();
                    if (t < mloc && pos < 16) {
#pragma unroll
                        for (int c = 16; c < NB; ++c) a[c] = sm.f.l11[pos * LD + c];
                    }
                    if (active) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            if (r % 2 == 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int c = 16; c < NB; ++c) a[c] = fma(-a[r], sm.f.l11[r * LD + c], a[c]);
                        }
                    }
                }
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const T x = a[c];
                    a[c] = a[16 + c];
                    a[16 + c] = x;
                }
            }
            // rows to their positions: memory, the block's top rows in LDS, the map
            if (t < mloc) {
                sm.map[st][pos] = (unsigned short)t;
#pragma unroll
                for (int c = 0; c < NB; ++c)
                    if (c < jb) P[pos + (size_t)c * ld] = a[c];
                if (pos < NB) {
#pragma unroll
                    for (int c = 0; c < NB; ++c) sm.f.l11[pos * LD + c] = a[c];
                }
            } else if (t < NB) {
#pragma unroll
                for (int c = 0; c < NB; ++c) sm.f.l11[t * LD + c] = T(0);
            }
            if (t < NB) sm.f.dst[t] = (t < mloc && pos >= NB) ? pos : -1;
            if (t < jb && !nopiv) ipiv[k + t] = k + piv + 1;
        }
        __syncthreads();
        const int ncolA = n - k - jb;
        const int nsA = ncolA > 0 ? (ncolA + 15) / 16 : 0;
        const int ns = nsA + (nr + 15) / 16;
        if (ns == 0) continue;
        auto strip = [&](int s) {
            Strip<T> x;
            if (s < nsA) {
                x.ld = ld;
                x.nc = min(16, ncolA - 16 * s);
                x.p = A + k + (size_t)(k + jb + 16 * s) * ld;
            } else {
                x.ld = ldb;
                x.nc = min(16, nr - 16 * (s - nsA));
                x.p = B + k + (size_t)(16 * (s - nsA)) * ldb;
            }
            return x;
        };
        // ---- interchanges and U12 on the strips ----------------------------
        if (w < ns) {
            // lane 4c + q: column c, rows q, q+4, .. of the block
            const int l = (t + wg_opaque_zero()) % kWave, cl = l >> 2, q = l & 3;
            int src[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) src[i] = sm.map[st][min(q + 4 * i, mloc - 1)];
            const int dsp = sm.f.dst[l & 31];
            for (int s = w; s < ns; s += W) {
                const Strip<T> x = strip(s);
                T y[8], dv[8];
                // lanes outside the strip read its last column; rows outside
                // the block have zero multipliers and are not stored
                auto Cc = x.p + (size_t)min(cl, x.nc - 1) * x.ld;
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = Cc[src[i]];
                // displaced top rows: lane l moves row l % 32 of two columns per step
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    dv[u] = x.p[min(l & 31, mloc - 1) + (size_t)min(2 * u + (l >> 5), x.nc - 1) * x.ld];
                wg_solve_block<T, false>(sm.f.l11, y, q);
                // every load of the wave has returned before its first store
                __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0)
                __builtin_amdgcn_wave_barrier();
                if (cl < x.nc) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (q + 4 * i < jb) Cc[q + 4 * i] = y[i];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int c = 2 * u + (l >> 5);
                    if (dsp >= 0 && c < x.nc) x.p[dsp + (size_t)c * x.ld] = dv[u];
                }
            }
        }
        __syncthreads();
        // ---- trailing update (a block with rows below it is full, or
        //      nothing lies right of it) ------------------------------------
        const int Mr = mloc - NB;
        if (Mr > 0 && jb == NB) {
            using Op = UpdOperand<T, MODE>;
            const int l = (t + wg_opaque_zero()) % kWave, lr = l % 16, lq = l / 16;
            const int nch = (Mr + 31) / 32;                    // 32-row strips
            const int ncg = max(1, W / nch);                   // waves sharing one strip's columns
            const int nfull = ncolA / 16;                      // full column strips of A
            for (int task = w; task < nch * ncg; task += W) {
                const int rc = task % nch;
                const int row0 = NB + 32 * rc;                 // first row of the strip
                Op lf[2];
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
                    for (int v = 0; v < 8; ++v)
                        lf[rt].x[v] = P[min(row0 + 16 * rt + lr, mloc - 1) + (size_t)Op::k(v, lq) * ld];
                    lf[rt].finish();
                }
                // Strips from the right: those that the interchanges touched
                // last come first, and the next panel's columns are written
                // last, while the L2 still holds them
                const int s0 = task / nch;
                const bool whole = row0 + 32 <= mloc;
                const int last = s0 < ns ? s0 + (ns - 1 - s0) / ncg * ncg : -1;    // this wave's last strip
                for (int s = last; s >= (whole ? max(nfull, s0) : s0); s -= ncg) {
                    const Strip<T> x = strip(s);
                    Op u;
                    T c[2][4];
                    auto Uc = x.p + (size_t)min(lr, x.nc - 1) * x.ld;
#pragma unroll
                    for (int v = 0; v < 8; ++v) u.x[v] = Uc[Op::k(v, lq)];
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            c[rt][r] = x.p[min(row0 + 16 * rt + lr, mloc - 1) +
                                           (size_t)min(M::row(r, lq), x.nc - 1) * x.ld];
                    u.finish();
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) {
                        acc_t acc = {0, 0, 0, 0};
                        acc = upd_mma<T, MODE>(u, lf[rt], acc);
                        if (row0 + 16 * rt + lr < mloc) {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (M::row(r, lq) < x.nc)
                                    x.p[row0 + 16 * rt + lr + (size_t)M::row(r, lq) * x.ld] = c[rt][r] - acc[r];
                        }
                    }
                }
                if (whole && s0 < nfull) {
                    // whole tiles: no guards, so that the loads of the next
                    // strip stay in flight over the stores of this one (a
                    // guarded store makes the wait counts unknown)
                    const size_t offu = (size_t)lr * ld + Op::k(0, lq);
                    const size_t offc = (size_t)M::row(0, lq) * ld + row0 + lr;
                    const size_t stepc = (size_t)(M::row(1, 0) - M::row(0, 0)) * ld;
                    auto load_u = [&](int q, Op& u) {
                        auto Uc = A + k + (size_t)(k + NB + 16 * q) * ld + offu;
#pragma unroll
                        for (int v = 0; v < 8; ++v) u.x[v] = Uc[Op::k(v, 0)];
                    };
                    auto tile = [&](int q, Op& u, Op& un) {
                        auto Cc = A + k + (size_t)(k + NB + 16 * q) * ld + offc;
                        T c[2][4];
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int rt = 0; rt < 2; ++rt) c[rt][r] = Cc[r * stepc + 16 * rt];
                        load_u(max(q - ncg, 0), un);
                        u.finish();
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) {
                            acc_t acc = {0, 0, 0, 0};
                            acc = upd_mma<T, MODE>(u, lf[rt], acc);
#pragma unroll
                            for (int r = 0; r < 4; ++r) Cc[r * stepc + 16 * rt] = c[rt][r] - acc[r];
                        }
                    };
                    Op u0, u1;
                    int s = s0 + (nfull - 1 - s0) / ncg * ncg;
                    load_u(s, u0);
                    for (; s >= 0; s -= 2 * ncg) {
                        tile(s, u0, u1);
                        if (s - ncg >= 0) tile(s - ncg, u1, u0);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (t == 0) info_array[b] = info;

    // ---- later interchanges of the factored columns, composed and applied
    //      once: row t of block s's columns comes from the row that the maps
    //      of the blocks after s trace it back to -----------------------------
    if (!nopiv) {
        const int nst = (minmn + NB - 1) / NB;
        int cur = t;
        for (int s = nst - 1; s >= 1; --s) {
            const int ks = NB * s;
            const bool in = t >= ks && t < m;
            if (in) cur = ks + sm.map[s][cur - ks];
            const bool mv = in && cur != t;
            auto Lc = A + (size_t)(ks - NB) * ld;
            T v[NB];
            if (mv) {
#pragma unroll
                for (int c = 0; c < NB; ++c) v[c] = Lc[cur + (size_t)c * ld];
            }
            __builtin_amdgcn_s_waitcnt(0x0F70);                // vmcnt(0)
            __syncthreads();
            if (mv) {
#pragma unroll
                for (int c = 0; c < NB; ++c) Lc[t + (size_t)c * ld] = v[c];
            }
        }
    }
    if (solve) {
        __syncthreads();
        wg_sweep<T, NTH, true, false, false>(A, ld, n, B, ldb, nr, sm.sweep);
    }
}

bool getrf_wg_supported(int max_m) { return max_m >= 1 && max_m <= 512; }

// One workgroup per system pays where its panel chain is the larger part or
// the batch fills the device: measured against the launch-per-step blocked LU
// (FP64, us) 2,000 x 256^2 5750 -> 2776, 1 x 512^2 2215 -> 1573, 32 x 512^2
// 2444 -> 1702. A few wide systems want their columns spread over many
// workgroups instead (1 x 512 x 1024: 2266 against 3020; 64 x 512 x 4096:
// 8904 against 16535). Up to 12 pivots the LDS kernel's shorter start wins
// (20,000 x 8 x 10: 171 against 226; 1,000 x 24 x 40: 86 against 77).
bool getrf_wg_preferred(int max_m, int max_n, int batch)
{
    return getrf_wg_supported(max_m) && (max_m < max_n ? max_m : max_n) > 12 && (max_n <= max_m || batch >= 512);
}

// The register-tile kernel has the shorter chain per system, but a CU holds
// only two to four of them; from about six systems per CU on (1,536) the eight
// that fit here win above 64 rows. Measured (gesv, FP64, us, tile against
// this): 1,024 x 100^2 255 / 267, 2,048 x 100^2 478 / 371, 8,192 x 100^2 1781
// / 1384, 20,000 x 128^2 5463 / 4560; at 64 rows 8,192 systems 508 / 588.
// Without right-hand sides the tile fits three systems of up to 80 rows per CU,
// all of the time of 80, while here the time grows with the rows: from 69 to 80
// the tile wins (getrf, 1,536 x 80^2 151 / 176, 2,304 x 72^2 209 / 251, 10,000 x
// 80^2 743 / 879; 10,000 x 72^2 764 / 805 but 4,000 x 72^2 345 / 323; 4,000 x
// 65^2 344 / 295, 4,000 x 81^2 496 / 408), but for the batches of up to 76 rows
// that run at once here and in three rounds there (2,048 x 72^2 197 / 179).
bool getrf_wg_over_tile(int max_n, int batch, bool solve)
{
    const bool one_round = max_n <= 76 && batch > 1536 && batch <= 2048;
    return max_n > 64 && batch >= 1536 && (solve || max_n <= 68 || max_n > 80 || one_round);
}

template <typename T, int MODE>
static magma_int_t wg_launch(const SizeArgs& sz, int max_m, T** dA_array, int** ipiv_array, int* info_array,
                             const WgRhs<T>& rhs, int batch, hipStream_t stream)
{
    if (!getrf_wg_supported(max_m) || rhs.max_nrhs > kWgGesvRhs) return MAGMA_ERR_NOT_SUPPORTED;
    if (max_m <= 128)
        getrf_wg_kernel<T, MODE, 128><<<batch, 128, 0, stream>>>(sz, dA_array, ipiv_array, info_array, rhs);
    else if (max_m <= 256)
        getrf_wg_kernel<T, MODE, 256><<<batch, 256, 0, stream>>>(sz, dA_array, ipiv_array, info_array, rhs);
    else
        getrf_wg_kernel<T, MODE, 512><<<batch, 512, 0, stream>>>(sz, dA_array, ipiv_array, info_array, rhs);
    MGI_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

magma_int_t getrf_wg_launch(const SizeArgs& sz, int max_m, double** dA_array, int** ipiv_array, int* info_array,
                            const WgRhs<double>& rhs, int batch, hipStream_t stream)
{
    return wg_launch<double, kUpdF64>(sz, max_m, dA_array, ipiv_array, info_array, rhs, batch, stream);
}

magma_int_t sgetrf_wg_launch(int mode, const SizeArgs& sz, int max_m, float** dA_array, int** ipiv_array,
                             int* info_array, const WgRhs<float>& rhs, int batch, hipStream_t stream)
{
    switch (mode) {
        case kUpdF32:    return wg_launch<float, kUpdF32>(sz, max_m, dA_array, ipiv_array, info_array, rhs, batch, stream);
        case kUpdBF16:   return wg_launch<float, kUpdBF16>(sz, max_m, dA_array, ipiv_array, info_array, rhs, batch, stream);
        case kUpdFP16:   return wg_launch<float, kUpdFP16>(sz, max_m, dA_array, ipiv_array, info_array, rhs, batch, stream);
        case kUpdBF16x3: return wg_launch<float, kUpdBF16x3>(sz, max_m, dA_array, ipiv_array, info_array, rhs, batch, stream);
        default: return MAGMA_ERR_NOT_SUPPORTED;
    }
}

}  // namespace mgi
