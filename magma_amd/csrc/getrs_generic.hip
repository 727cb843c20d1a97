// Batched triangular solve with LU factors: the choice of kernel, and the
// kernel for up to four right-hand sides (FP64 or FP32, fixed or per-matrix
// sizes). Everything else goes to getrs_wg.hip.
#include "magma_internal.h"
#include "lu_device.h"
#include "getrf_kernels.h"

namespace mgi {

constexpr int kRsThreads = 256;

// ---------------------------------------------------------------------------
// NoTrans for n <= 64 R (n <= 256), one wave per (system, group of up to
// kWaveCols right-hand sides): lane l keeps rows l + 64 s (s < R) of x in registers,
// so the sweeps need neither LDS nor a workgroup barrier. Row k's solved
// value reaches the other lanes through a cross-lane read, and the factor is
// streamed down its columns (64 contiguous elements per slot, loads issued
// ahead of the dependent updates). The interchanges are applied by tracing
// every row back through them; each row's updates run in the order of the
// columns, forward and then backward.
// ---------------------------------------------------------------------------
constexpr int kWaveCols = 4;
constexpr int kFewSystems = 1024;     // FP64 batches that do not fill the chip with one wave per system

template <typename T, int R>
__global__ void __launch_bounds__(kRsThreads)
getrs_wave_kernel(RsSizes sz, int groups, int nsys, T** __restrict__ dA_array, int** __restrict__ ipiv_array,
                  T** __restrict__ dB_array)
{
    const int gw = blockIdx.x * (kRsThreads / kWave) + threadIdx.x / kWave;
    const int sys = gw / groups;
    if (sys >= nsys) return;
    const int b = sz.map ? sz.map[sys] : sys;
    int n, nrhs, ldda, lddb;
    sz.get(b, n, nrhs, ldda, lddb);
    const int c0 = (gw % groups) * kWaveCols;
    if (n <= 0 || c0 >= nrhs) return;
    const int nr = min(kWaveCols, nrhs - c0);
    const int l = threadIdx.x % kWave;
    auto A = gptr(dA_array[b]);
    auto ipiv = gptr(ipiv_array ? ipiv_array[b] : nullptr);   // null: factors without pivoting
    auto B = gptr(dB_array[b]) + (size_t)c0 * lddb;

    // (P^T B)(i,:) = B(src(i),:)
    int src[R];
#pragma unroll
    for (int s = 0; s < R; ++s) src[s] = l + 64 * s;
    for (int k = ipiv ? n - 1 : -1; k >= 0; --k) {
        int p = ipiv[k] - 1;
        p = (p > k && p < n) ? p : k;
#pragma unroll
        for (int s = 0; s < R; ++s) src[s] = (src[s] == k) ? p : (src[s] == p ? k : src[s]);
    }
    T x[R][kWaveCols];
#pragma unroll
    for (int s = 0; s < R; ++s)
#pragma unroll
        for (int c = 0; c < kWaveCols; ++c)
            x[s][c] = (l + 64 * s < n && c < nr) ? B[src[s] + (size_t)c * lddb] : T(0);

    // Columns are processed in chunks of CH; the factor entries of the next
    // chunk are loaded while the current one is applied.
    constexpr int CH = R <= 2 ? 8 : (R <= 4 ? 4 : 2);
    // unit lower, forward: step k = 64 s + kk
#pragma unroll
    for (int s = 0; s < R; ++s) {
        const int kend = min(64, n - 1 - 64 * s);
        if (kend <= 0) continue;
        T cur[CH][R], nxt[CH][R];
        auto load_l = [&](T (&buf)[CH][R], int kk0) {
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const int k = 64 * s + kk0 + j;
                const bool kin = kk0 + j < kend;
                auto Lk = A + (size_t)(kin ? k : 0) * ldda;
#pragma unroll
                for (int s2 = s; s2 < R; ++s2) {
                    const int i = l + 64 * s2;
                    buf[j][s2] = (kin && i > k && i < n) ? Lk[i] : T(0);
                }
            }
        };
        load_l(cur, 0);
        for (int kk0 = 0; kk0 < kend; kk0 += CH) {
            if (kk0 + CH < kend) load_l(nxt, kk0 + CH);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const int kk = kk0 + j;
                if (kk < kend) {
                    const int k = 64 * s + kk;
#pragma unroll
                    for (int c = 0; c < kWaveCols; ++c) {
                        if (c < nr) {
                            const T xk = readlane_t(x[s][c], kk);
#pragma unroll
                            for (int s2 = s; s2 < R; ++s2)
                                if (l + 64 * s2 > k) x[s2][c] = fma(-cur[j][s2], xk, x[s2][c]);
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int s2 = s; s2 < R; ++s2) cur[j][s2] = nxt[j][s2];
        }
    }
    // non-unit upper, backward: step k = 64 s + kk, kk descending
#pragma unroll
    for (int s = R - 1; s >= 0; --s) {
        if (64 * s >= n) continue;
        const int ktop = min(63, n - 1 - 64 * s);        // first kk processed
        T cur[CH][R], nxt[CH][R], dcur[CH], dnxt[CH];
        auto load_u = [&](T (&buf)[CH][R], T (&dg)[CH], int kk0) {
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const int kk = kk0 - j;
                const bool kin = kk >= 0;
                const int k = 64 * s + (kin ? kk : 0);
                auto Uk = A + (size_t)k * ldda;
                dg[j] = Uk[k];
#pragma unroll
                for (int s2 = 0; s2 <= s; ++s2) {
                    const int i = l + 64 * s2;
                    buf[j][s2] = (kin && i < k) ? Uk[i] : T(0);
                }
            }
        };
        load_u(cur, dcur, ktop);
        for (int kk0 = ktop; kk0 >= 0; kk0 -= CH) {
            if (kk0 - CH >= 0) load_u(nxt, dnxt, kk0 - CH);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                const int kk = kk0 - j;
                if (kk >= 0) {
                    const int k = 64 * s + kk;
                    // one reciprocal per step, independent of the chain
                    const T rk = T(1) / dcur[j];
#pragma unroll
                    for (int c = 0; c < kWaveCols; ++c) {
                        if (c < nr) {
                            const T xk = readlane_t(x[s][c], kk) * rk;
                            if (l == kk) x[s][c] = xk;
#pragma unroll
                            for (int s2 = 0; s2 <= s; ++s2)
                                if (l + 64 * s2 < k) x[s2][c] = fma(-cur[j][s2], xk, x[s2][c]);
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                dcur[j] = dnxt[j];
#pragma unroll
                for (int s2 = 0; s2 <= s; ++s2) cur[j][s2] = nxt[j][s2];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < R; ++s)
#pragma unroll
        for (int c = 0; c < kWaveCols; ++c)
            if (l + 64 * s < n && c < nr) B[l + 64 * s + (size_t)c * lddb] = x[s][c];
}

template <typename T, int R>
static magma_int_t getrs_wave_launch(const RsSizes& sz, int max_nrhs, T** dA_array, int** ipiv_array, T** dB_array,
                                     int batch, hipStream_t stream)
{
    const int groups = ceildiv(max_nrhs, kWaveCols);
    const long waves = (long)batch * groups;
    const int wpb = kRsThreads / kWave;
    getrs_wave_kernel<T, R><<<(int)ceildiv(waves, (long)wpb), kRsThreads, 0, stream>>>(sz, groups, batch, dA_array,
                                                                                     ipiv_array, dB_array);
    MGI_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

// The largest order the solve accepts keeps a system's pivots and eight
// right-hand sides within a workgroup's LDS.
size_t getrs_generic_bytes(int n, int elem) { return (size_t)n * 8 * elem + 2 * (size_t)n * sizeof(int); }
size_t getrs_generic_bytes(int n) { return getrs_generic_bytes(n, sizeof(double)); }

template <typename T>
magma_int_t getrs_generic_launch_t(int trans, const RsSizes& sz, int max_nrhs, T** dA_array, int** ipiv_array,
                                   T** dB_array, int batch, hipStream_t stream)
{
    if (batch <= 0 || max_nrhs <= 0) return MAGMA_SUCCESS;
    if (getrs_generic_bytes(sz.max_n, sizeof(T)) > max_dynamic_lds()) return MAGMA_ERR_NOT_SUPPORTED;
    // up to four right-hand sides of many systems of up to 256 rows read the
    // factors once in one wave, without barriers (FP64 us, wave against
    // workgroup: 2,000 x 256^2 r1 276 / 379, r4 320 / 382; 20,000 x 16^2 r2 85 /
    // 222; 8,192 x 64^2 r1 134 / 212; 5,000 x 100^2 r4 219 / 284); with more, or
    // above 256 rows, the workgroup's MFMA sweeps win (2,000 x 256^2 r16 935 /
    // 486, 5,000 x 100^2 r5 361 / 286). Up to four systems per CU the wave's
    // chain of columns is what counts, and the workgroup's chain of blocks is
    // shorter (64 x 256^2 r1 174 / 106, r4 221 / 106; 1,024 x 256^2 r1 231 / 199;
    // 1,024 x 64^2 r4 56 / 38; even at 16 rows). FP32 batches, whose waves
    // stream half the bytes, stay with the wave at every size (8,192 x 64^2 r1
    // 80 / 89), and so do mapped buckets, beside which other buckets run.
    const bool few = sizeof(T) == 8 && sz.map == nullptr && batch <= kFewSystems;
    if (trans == 0 && sz.max_n <= 256 && max_nrhs <= kWaveCols && !few) {
        if (sz.max_n <= 64) return getrs_wave_launch<T, 1>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        if (sz.max_n <= 128) return getrs_wave_launch<T, 2>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        return getrs_wave_launch<T, 4>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
    }
    return getrs_wg_launch<T>(trans, sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
}

template magma_int_t getrs_generic_launch_t<double>(int, const RsSizes&, int, double**, int**, double**, int,
                                                    hipStream_t);
template magma_int_t getrs_generic_launch_t<float>(int, const RsSizes&, int, float**, int**, float**, int,
                                                   hipStream_t);

magma_int_t getrs_generic_launch(int trans, int n, int nrhs, double** dA_array, int ldda, int** ipiv_array,
                                 double** dB_array, int lddb, int batch, hipStream_t stream)
{
    RsSizes sz{n, nrhs, ldda, lddb, n, nullptr, nullptr, nullptr, nullptr, nullptr};
    return getrs_generic_launch_t<double>(trans, sz, nrhs, dA_array, ipiv_array, dB_array, batch, stream);
}

}  // namespace mgi
