// Batched LU, and LU + solve, of square systems of up to 64 rows (FP32; 48
// in FP64): one wave per system, lane l holds row l in registers, so there is
// no LDS, no barrier and no pass over memory but the first read and the last
// write.
//
// Columns are taken 16 at a time through the same code (the registers rotate
// by 16 after each group, so that the code stays within the instruction
// cache): per column the wave picks the pivot (32-bit DPP search, every lane's
// reciprocal beside it), reads the pivot row's entries out of its lane into
// scalar registers and updates the group's columns; after the group the same
// steps run over each later group of 16 columns. Rows are not moved: each
// carries its LAPACK position and is stored at it. Right-hand sides are solved
// four at a time from the registers.
//
// What bounds it: vector issue (about two lane reads per FP64 entry of each
// pivot row), with three (FP64) or four waves per SIMD to hide the pivot
// chain. At that bound two of the FP64 forms with right-hand sides spill (up to
// 16 rows 57 registers, 164 bytes of scratch a lane; up to 48 rows 18, 76
// bytes); the others do not. FP32 8,192 x 64^2: 787 us on the LDS kernel that served it, 364 on
// one workgroup per system, 228 here (1.2 TB/s).
//
// Reference behaviour: magmablas/zgetf2_devicefunc.cuh:218-294 (panel step),
// magmablas/magma_templates.h:44-60 (ties),
// magmablas/zgetrf_batched_smallsq_noshfl.cu (register LU with row tracking).
#include "magma_internal.h"
#include "getrf_kernels.h"
#include "wg_lu.h"

namespace mgi {

constexpr int kLwWaves = 4;         // systems per workgroup
constexpr int kLwRhs = 4;           // right-hand sides solved at a time

// The 16-column groups of a row move up by one (the first becomes the last),
// or down with BACK.
template <typename T, int NC, bool BACK>
__device__ __forceinline__ void lw_rotate(T (&a)[NC])
{
    T keep[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) keep[c] = a[BACK ? NC - 16 + c : c];
    if constexpr (BACK) {
#pragma unroll
        for (int c = NC - 1; c >= 16; --c) a[c] = a[c - 16];
    } else {
#pragma unroll
        for (int c = 0; c < NC - 16; ++c) a[c] = a[c + 16];
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) a[BACK ? c : NC - 16 + c] = keep[c];
}

template <typename T, int NCH, bool WITH_B>
__global__ void __launch_bounds__(kLwWaves * kWave, (sizeof(T) == 8 && NCH > 2) ? 3 : 4)
lu_wave_kernel(TileArgs ta, T** __restrict__ dA_array, int** __restrict__ ipiv_array, int* __restrict__ info_array,
               T** __restrict__ dB_array, int batch)
{
    constexpr int NC = 16 * NCH;
    const int sys = blockIdx.x * kLwWaves + wg_wave();
    if (sys >= batch) return;
    const int mat = ta.map ? ta.map[sys] : sys;
    const int n = ta.n_arr ? ta.n_arr[mat] : ta.n;
    const int ld = ta.ldda_arr ? ta.ldda_arr[mat] : ta.ldda;
    if (n <= 0) return;                            // empty system: nothing to factor
    const int l = threadIdx.x % kWave;
    auto A = gptr(dA_array[mat]);
    auto ipiv = gptr(ipiv_array[mat]);

    T a[NC];
    auto Al = A + min(l, n - 1);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const T v = Al[(size_t)min(c, n - 1) * ld];
        a[c] = (l < n && c < n) ? v : T(0);
    }
    int pos = l;                                   // LAPACK position of this lane's row
    bool active = l < n;
    int info = 0;
    int piv = 0, lane_of = 0;                      // lane k: step k's pivot position and lane
    T rdiag = T(1);                                // reciprocal of this row's pivot
#pragma unroll 1
    for (int h = 0; h < NCH; ++h) {
        int step = active ? 16 : -1;               // step of this group that takes this row
        wg_for(std::make_integer_sequence<int, 16>{}, [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const int k = 16 * h + j;
            if (k < n) {
                // LAPACK idamax: a NaN wins only at the first position, where
                // it counts as infinite
                const bool first = pos == k;
                const T alt = first ? T(INFINITY) : T(-1);
                T v = fabs(a[j]);
                v = v == v ? v : alt;
                v = active ? v : T(-1);
                const T ri = T(1) / a[j];
                const int pl = wg_pick<64>(v, pos);
                const T pv = readlane_t(a[j], pl);
                const T rinv = readlane_t(ri, pl);
                const int pp = __builtin_amdgcn_readlane(pos, pl);
                T u[16];
#pragma unroll
                for (int c = j + 1; c < 16; ++c) u[c] = readlane_t(a[c], pl);
                piv = l == k ? pp : piv;
                lane_of = l == k ? pl : lane_of;
                const bool win = l == pl;
                pos = (active & first) ? pp : pos;
                pos = win ? k : pos;
                active = active & !win;
                step = win ? j : step;
                rdiag = win ? rinv : rdiag;
                const bool zero = __ballot(pv == T(0)) != 0ull;
                if (zero && info == 0) info = k + 1;
                // a zero pivot leaves its column unscaled; the step is applied
                // all the same (LAPACK dgetf2)
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
        // the same steps on the later groups
        const int steps = min(16, n - 16 * h);
        wg_for(std::make_integer_sequence<int, NCH - 1>{}, [&](auto gc) {
            constexpr int g = decltype(gc)::value + 1;
            if (g < NCH - h) {
                wg_for(std::make_integer_sequence<int, 16>{}, [&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    if (r < steps) {
                        const int pl = __builtin_amdgcn_readlane(lane_of, 16 * h + r);
                        T u[16];
#pragma unroll
                        for (int c = 0; c < 16; ++c) u[c] = readlane_t(a[16 * g + c], pl);
                        if (step > r) {
#pragma unroll
                            for (int c = 0; c < 16; ++c) a[16 * g + c] = fma(-a[r], u[c], a[16 * g + c]);
                        }
                    }
                });
            }
        });
        lw_rotate<T, NC, false>(a);                // the next group takes the place of this one
    }
    if (l < n) {
        ipiv[l] = piv + 1;
        auto Ap = A + pos;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (c < n) Ap[(size_t)c * ld] = a[c];
    }
    if (l == 0) info_array[mat] = info;

    if constexpr (WITH_B) {
        const int nrhs = ta.nrhs_arr ? ta.nrhs_arr[mat] : ta.nrhs;
        const int ldb = ta.lddb_arr ? ta.lddb_arr[mat] : ta.lddb;
        auto B = gptr(dB_array[mat]);
#pragma unroll 1
        for (int c0 = 0; c0 < nrhs; c0 += kLwRhs) {
            T b[kLwRhs];
#pragma unroll
            for (int c = 0; c < kLwRhs; ++c) {
                const T v = B[min(l, n - 1) + (size_t)min(c0 + c, nrhs - 1) * ldb];
                b[c] = l < n ? v : T(0);
            }
            // unit lower, forward: step k's entry comes from its pivot's lane;
            // 16 steps at a time, as above
#pragma unroll 1
            for (int h = 0; h < NCH; ++h) {
                wg_for(std::make_integer_sequence<int, 16>{}, [&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    const int k = 16 * h + j;
                    const int pl = __builtin_amdgcn_readlane(lane_of, min(k, n - 1));
#pragma unroll
                    for (int c = 0; c < kLwRhs; ++c) {
                        const T y = fma(-a[j], readlane_t(b[c], pl), b[c]);
                        b[c] = (pos > k && k < n) ? y : b[c];
                    }
                });
                lw_rotate<T, NC, false>(a);
            }
            // upper, backward
#pragma unroll 1
            for (int h = NCH - 1; h >= 0; --h) {
                lw_rotate<T, NC, true>(a);
                wg_for(std::make_integer_sequence<int, 16>{}, [&](auto jc) {
                    constexpr int j = 15 - decltype(jc)::value;
                    const int k = 16 * h + j;
                    const int pl = __builtin_amdgcn_readlane(lane_of, min(k, n - 1));
#pragma unroll
                    for (int c = 0; c < kLwRhs; ++c) {
                        const T xk = readlane_t(b[c] * rdiag, pl);
                        const T y = fma(-a[j], xk, b[c]);
                        const T z = pos < k ? y : (pos == k ? xk : b[c]);
                        b[c] = k < n ? z : b[c];
                    }
                });
            }
            if (l < n) {
#pragma unroll
                for (int c = 0; c < kLwRhs; ++c)
                    if (c0 + c < nrhs) B[pos + (size_t)(c0 + c) * ldb] = b[c];
            }
        }
    }
}

template <typename T, bool WITH_B>
static magma_int_t wave_launch(int nch, const TileArgs& a, T** dA_array, int** ipiv_array, int* info_array,
                               T** dB_array, int batch, hipStream_t stream)
{
    const dim3 grid(ceildiv(batch, kLwWaves)), block(kLwWaves * kWave);
    switch (nch) {
        case 1: lu_wave_kernel<T, 1, WITH_B><<<grid, block, 0, stream>>>(a, dA_array, ipiv_array, info_array, dB_array, batch); break;
        case 2: lu_wave_kernel<T, 2, WITH_B><<<grid, block, 0, stream>>>(a, dA_array, ipiv_array, info_array, dB_array, batch); break;
        case 3: lu_wave_kernel<T, 3, WITH_B><<<grid, block, 0, stream>>>(a, dA_array, ipiv_array, info_array, dB_array, batch); break;
        default:
            if constexpr (sizeof(T) == 4) {
                if (nch != 4) return MAGMA_ERR_NOT_SUPPORTED;
                lu_wave_kernel<T, 4, WITH_B><<<grid, block, 0, stream>>>(a, dA_array, ipiv_array, info_array, dB_array, batch);
            } else {
                return MAGMA_ERR_NOT_SUPPORTED;
            }
    }
    MGI_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

magma_int_t lu_wave_launch(int nch, const TileArgs& a, double** dA_array, int** ipiv_array, int* info_array,
                           double** dB_array, int batch, hipStream_t stream)
{
    return dB_array ? wave_launch<double, true>(nch, a, dA_array, ipiv_array, info_array, dB_array, batch, stream)
                    : wave_launch<double, false>(nch, a, dA_array, ipiv_array, info_array, dB_array, batch, stream);
}

magma_int_t slu_wave_launch(int nch, const TileArgs& a, float** dA_array, int** ipiv_array, int* info_array, int batch,
                            hipStream_t stream)
{
    return wave_launch<float, false>(nch, a, dA_array, ipiv_array, info_array, nullptr, batch, stream);
}

}  // namespace mgi
