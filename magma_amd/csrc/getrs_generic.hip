// Batched triangular solve with LU factors: the choice of kernel, and the
// kernels for up to four right-hand sides at a time (FP64 or FP32, fixed or
// per-matrix sizes). Everything else goes to getrs_wg.hip.
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

// ---------------------------------------------------------------------------
// Trans with up to four right-hand sides: one workgroup per system, the
// right-hand sides in LDS, blocks of 64 rows. Wave w solves the block's
// triangle for right-hand side w (lane l holds row l of the triangle in
// registers, the solved entry of each step reaches the others by a lane read);
// then every thread applies the block to the rows left, one row each, with 32
// of its contiguous factor entries in flight. Bound: the chain of blocks in
// few systems, HBM in many. Three workgroups per CU (147 registers in FP64):
// without the bound two, and 768 systems of 256 rows take 1.4 times as long.
// (The reason to keep it beside the workgroup's sweeps stands at the choice.)
// ---------------------------------------------------------------------------
constexpr int kFewRhs = 4;

template <typename T, bool BACK, bool UNIT>
__device__ __forceinline__ void few_sweep(const MGI_GLOBAL_AS T* __restrict__ A, int ld, int n, T* sB, int nr)
{
    const int tid = threadIdx.x, l = tid % kWave, w = tid / kWave;
    for (int done = 0; done < n; done += kWave) {
        const int kb = BACK ? max(0, n - done - kWave) : done;
        const int nb = min(kWave, n - done);
        if (w < nr) {
            const int r = kb + l;
            const bool in = l < nb;
            T f[kWave];
            auto Fr = A + kb + (size_t)r * ld;
#pragma unroll
            for (int j = 0; j < kWave; ++j) f[j] = (in && (BACK ? j > l && j < nb : j < l)) ? Fr[j] : T(0);
            const T rd = (!UNIT && in) ? T(1) / A[r + (size_t)r * ld] : T(1);
            T x = in ? sB[r + w * n] : T(0);
#pragma unroll
            for (int jj = 0; jj < kWave; ++jj) {
                const int j = BACK ? kWave - 1 - jj : jj;
                if (j < nb) {
                    T xj = readlane_t(x, j);
                    if constexpr (!UNIT) {
                        xj *= readlane_t(rd, j);
                        if (l == j) x = xj;
                    }
                    if (BACK ? l < j : l > j) x = fma(-f[j], xj, x);
                }
            }
            if (in) sB[r + w * n] = x;
        }
        __syncthreads();
        // the rows left exist only beside a full block
        const int i0 = BACK ? 0 : kb + kWave, i1 = BACK ? kb : n;
        for (int i = i0 + tid; i < i1; i += kRsThreads) {
            T acc[kFewRhs];
#pragma unroll
            for (int c = 0; c < kFewRhs; ++c) acc[c] = sB[i + c * n];
            auto Fi = A + kb + (size_t)i * ld;
            constexpr int CH = 32;
            for (int j0 = 0; j0 < kWave; j0 += CH) {
                T f[CH];
#pragma unroll
                for (int u = 0; u < CH; ++u) f[u] = Fi[BACK ? kWave - 1 - (j0 + u) : j0 + u];
#pragma unroll
                for (int u = 0; u < CH; ++u) {
                    const int j = BACK ? kWave - 1 - (j0 + u) : j0 + u;
#pragma unroll
                    for (int c = 0; c < kFewRhs; ++c) acc[c] = fma(-f[u], sB[kb + j + c * n], acc[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < kFewRhs; ++c)
                if (c < nr) sB[i + c * n] = acc[c];
        }
        __syncthreads();
    }
}

template <typename T>
__global__ void __launch_bounds__(kRsThreads, sizeof(T) == 8 ? 3 : 4)
getrs_few_kernel(RsSizes sz, T** __restrict__ dA_array, int** __restrict__ ipiv_array, T** __restrict__ dB_array)
{
    extern __shared__ __align__(16) unsigned char rf_raw[];
    const int b = sz.map ? sz.map[blockIdx.x] : blockIdx.x;
    int n, nrhs, ldda, lddb;
    sz.get(b, n, nrhs, ldda, lddb);
    if (n <= 0 || nrhs <= 0) return;
    const int nr = min(nrhs, kFewRhs);
    const int tid = threadIdx.x;
    T* sB = reinterpret_cast<T*>(rf_raw);                     // n x kFewRhs, the unused columns zero
    int* perm = reinterpret_cast<int*>(rf_raw + (size_t)sz.max_n * kFewRhs * sizeof(T));
    int* spiv = perm + sz.max_n;
    auto A = gptr(dA_array[b]);
    auto B = gptr(dB_array[b]);
    auto ipiv = gptr(ipiv_array ? ipiv_array[b] : nullptr);   // null: factors without pivoting
    // (P^T B)(i,:) = B(perm[i],:): each row is traced back through the
    // interchanges, last to first; one outside [k, n) is none
    for (int i = tid; i < n; i += kRsThreads) {
        const int p = ipiv ? ipiv[i] - 1 : i;
        spiv[i] = (p > i && p < n) ? p : i;
#pragma unroll
        for (int c = 0; c < kFewRhs; ++c) sB[i + c * n] = c < nr ? B[i + (size_t)c * lddb] : T(0);
    }
    __syncthreads();
    for (int r = tid; r < n; r += kRsThreads) {
        int src = r;
        for (int k = n - 1; k >= 0; --k) {
            const int p = spiv[k];
            src = (src == k) ? p : (src == p ? k : src);
        }
        perm[r] = src;
    }
    few_sweep<T, false, false>(A, ldda, n, sB, nr);           // U^T
    few_sweep<T, true, true>(A, ldda, n, sB, nr);             // L^T
    for (int i = tid; i < n; i += kRsThreads)
#pragma unroll
        for (int c = 0; c < kFewRhs; ++c)
            if (c < nr) B[perm[i] + (size_t)c * lddb] = sB[i + c * n];
}

template <typename T>
static magma_int_t getrs_few_launch(const RsSizes& sz, T** dA_array, int** ipiv_array, T** dB_array, int batch,
                                    hipStream_t stream)
{
    const size_t lds = (size_t)sz.max_n * (kFewRhs * sizeof(T) + 2 * sizeof(int));
    MGI_HIP_CHECK(hipFuncSetAttribute((const void*)getrs_few_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)lds));
    getrs_few_kernel<T><<<batch, kRsThreads, lds, stream>>>(sz, dA_array, ipiv_array, dB_array);
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
    const bool f64 = sizeof(T) == 8;
    const int n = sz.max_n;
    if (trans != 0) {
        // The workgroup's sweeps work on 16 right-hand sides whatever their
        // number; the row-per-thread kernel is ahead (us, workgroup / few) in
        // FP64 with one or two of them in systems of a few blocks that the chip
        // holds all at once (1 x 64^2 r1 43 / 36, 512 x 128^2 r1 72 / 59; 1,024 x
        // 64^2 r1 49 / 58; from 160 rows on the two are level), and with up to
        // four that do not stay in the workgroup's LDS (64 x 2,000^2 r4 2975 /
        // 2262); in FP32, where its contiguous loads count, with one or two from
        // 193 rows on (3,000 x 512^2 r2 1355 / 1020; 1,100 x 200^2 r1 133 / 136;
        // 8,192 x 128^2 r1 242 / 292), with up to four from 481 (64 x 1,000^2 r4
        // 635 / 513; 3,000 x 200^2 r4 263 / 404).
        const bool few = f64 ? (max_nrhs <= 2 && n > 32 && n <= 128 && batch <= 768) ||
                                   (size_t)n * max_nrhs * sizeof(T) > kGetrsRhsLds
                             : max_nrhs <= 2 ? n > 192 : n > 480;
        if (max_nrhs <= kFewRhs && few) return getrs_few_launch<T>(sz, dA_array, ipiv_array, dB_array, batch, stream);
        return getrs_wg_launch<T>(trans, sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
    }
    // Up to four right-hand sides of many systems of up to 256 rows read the
    // factors once in one wave, without barriers (us, wave / workgroup: 20,000 x
    // 16^2 r2 92 / 124, 8,192 x 33^2 r1 79 / 114, 8,192 x 64^2 r1 135 / 135; above
    // that the workgroup has overtaken it, 8,192 x 128^2 r4 426 / 312, so the
    // line could come down). Up to four FP64 systems per CU the wave's chain of
    // columns is what counts, and the workgroup's chain of blocks is shorter
    // (64 x 256^2 r4 231 / 95; 1,024 x 256^2 r1 234 / 152); mapped buckets, beside
    // which other buckets run, stay with the wave. With more right-hand sides
    // the workgroup wins (8,192 x 128^2 r5 705 / 313, FP32 3,000 x 256^2 r5 501 /
    // 270), except in systems so small that a wave's work on them is a few
    // columns (20,000 x 4^2 r5 75 / 108, 20,000 x 8^2 r8 110 / 116, r9 144 / 123;
    // with more right-hand sides while the waves nearly all run at once: 64 x
    // 4^2 r64 29 / 33, 64 x 8^2 r32 31 / 33, 2,000 x 8^2 r17 49 / 42).
    const long waves = (long)batch * ceildiv(max_nrhs, kWaveCols);
    const bool tiny = n <= 8 && (n * max_nrhs <= 64 || n * waves <= 40960);
    const bool few = f64 && sz.map == nullptr && batch <= kFewSystems;
    if (n <= 256 && (tiny || (max_nrhs <= kWaveCols && !few))) {
        if (n <= 64) return getrs_wave_launch<T, 1>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        if (n <= 128) return getrs_wave_launch<T, 2>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        return getrs_wave_launch<T, 4>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
    }
    return getrs_wg_launch<T>(0, sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
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
