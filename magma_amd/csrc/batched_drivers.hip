// Public batched LU drivers: argument checking, quick returns and kernel
// selection. Argument codes and return conventions follow
// src/zgetrf_batched.cpp:82-105, src/zgetrs_batched.cpp:86-117 and
// src/zgesv_batched.cpp:93-154.
#include "magma_internal.h"
#include "getrf_kernels.h"

#include <algorithm>

namespace mgi {

// Asynchronous factorisation; the public entry point adds the host sync.
magma_int_t getrf_batched_async(int m, int n, double** dA_array, int ldda, int** ipiv_array,
                                int* info_array, int batch, hipStream_t stream)
{
    if (m == n && getrf_tile_supported(n) && !getrf_wg_over_tile(n, batch, false))
        return getrf_tile_launch(n, dA_array, ldda, ipiv_array, info_array, batch, stream);
    // Wide systems of few rows leave most of the workgroup kernel's lanes and
    // strips empty: the LDS kernel wins (us, LDS / workgroup: 20,000 x 13 x 20 238 / 274,
    // 20,000 x 20 x 24 348 / 372, 20 x 40 381 / 379; 24 x 40 452 / 408)
    const bool short_wide = n > m && m <= 20 && n <= 48;
    if (!short_wide && getrf_wg_preferred(m, n, batch)) {
        SizeArgs sz{m, n, ldda, nullptr, nullptr, nullptr, nullptr};
        return getrf_wg_launch(sz, m, dA_array, ipiv_array, info_array, WgRhs<double>{}, batch, stream);
    }
    if (getrf_lds_bytes(m, n) <= max_dynamic_lds())
        return getrf_lds_launch(m, n, dA_array, ldda, ipiv_array, info_array, batch, stream);
    if (getrf_blocked_supported(m))
        return getrf_blocked_launch(m, n, ldda, nullptr, nullptr, nullptr, m, n, dA_array, ipiv_array,
                                    info_array, batch, stream);
    return MAGMA_ERR_NOT_SUPPORTED;
}

magma_int_t getrs_batched_async(int trans, int n, int nrhs, double** dA_array, int ldda, int** ipiv_array,
                                double** dB_array, int lddb, int batch, hipStream_t stream)
{
    if (getrs_generic_bytes(n) <= max_dynamic_lds())
        return getrs_generic_launch(trans, n, nrhs, dA_array, ldda, ipiv_array, dB_array, lddb, batch, stream);
    return MAGMA_ERR_NOT_SUPPORTED;
}

}  // namespace mgi

extern "C" {

magma_int_t magma_dgetrf_batched(magma_int_t m, magma_int_t n, double** dA_array, magma_int_t ldda,
                                 magma_int_t** ipiv_array, magma_int_t* info_array,
                                 magma_int_t batchCount, magma_queue_t queue)
{
    magma_int_t arginfo = 0;
    if (m < 0)
        arginfo = -1;
    else if (n < 0)
        arginfo = -2;
    else if (ldda < std::max(1, m))
        arginfo = -4;
    else if (batchCount < 0)
        arginfo = -7;
    if (arginfo != 0) {
        magma_xerbla(__func__, -arginfo);
        return arginfo;
    }
    if (m == 0 || n == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    magma_int_t rc = mgi::getrf_batched_async(m, n, dA_array, ldda, ipiv_array, info_array,
                                              batchCount, queue->stream);
    if (rc != MAGMA_SUCCESS) return rc;
    MGI_HIP_CHECK(hipStreamSynchronize(queue->stream));
    return 0;
}

magma_int_t magma_dgetrs_batched(magma_trans_t trans, magma_int_t n, magma_int_t nrhs,
                                 double** dA_array, magma_int_t ldda, magma_int_t** dipiv_array,
                                 double** dB_array, magma_int_t lddb,
                                 magma_int_t batchCount, magma_queue_t queue)
{
    const bool notran = (trans == MagmaNoTrans);
    magma_int_t info = 0;
    if (!notran && trans != MagmaTrans && trans != MagmaConjTrans)
        info = -1;
    else if (n < 0)
        info = -2;
    else if (nrhs < 0)
        info = -3;
    else if (ldda < std::max(1, n))
        info = -5;
    else if (lddb < std::max(1, n))
        info = -8;
    else if (batchCount < 0)
        info = -9;
    if (info != 0) {
        magma_xerbla(__func__, -info);
        return info;
    }
    if (n == 0 || nrhs == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    return mgi::getrs_batched_async(notran ? 0 : 1, n, nrhs, dA_array, ldda, dipiv_array,
                                    dB_array, lddb, batchCount, queue->stream);
}

magma_int_t magma_dgesv_batched(magma_int_t n, magma_int_t nrhs, double** dA_array, magma_int_t ldda,
                                magma_int_t** dipiv_array, double** dB_array, magma_int_t lddb,
                                magma_int_t* dinfo_array, magma_int_t batchCount, magma_queue_t queue)
{
    magma_int_t info = 0;
    if (n < 0)
        info = -1;
    else if (nrhs < 0)
        info = -2;
    else if (ldda < std::max(1, n))
        info = -4;
    else if (lddb < std::max(1, n))
        info = -6;
    else if (batchCount < 0)
        info = -9;
    if (info != 0) {
        magma_xerbla(__func__, -info);
        return info;
    }
    if (n == 0 || nrhs == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    if (mgi::gesv_tile_supported(n, nrhs) && !mgi::getrf_wg_over_tile(n, batchCount, true))
        return mgi::gesv_tile_launch(n, nrhs, dA_array, ldda, dipiv_array, dinfo_array, dB_array, lddb,
                                     batchCount, queue->stream);
    if (mgi::getrf_wg_preferred(n, n, batchCount) && nrhs <= 16) {
        mgi::SizeArgs sz{n, n, ldda, nullptr, nullptr, nullptr, nullptr};
        mgi::WgRhs<double> rhs;
        rhs.dB_array = dB_array;
        rhs.nrhs = rhs.max_nrhs = nrhs;
        rhs.lddb = lddb;
        return mgi::getrf_wg_launch(sz, n, dA_array, dipiv_array, dinfo_array, rhs, batchCount, queue->stream);
    }
    info = mgi::getrf_batched_async(n, n, dA_array, ldda, dipiv_array, dinfo_array, batchCount, queue->stream);
    if (info != MAGMA_SUCCESS) return info;
    return mgi::getrs_batched_async(0, n, nrhs, dA_array, ldda, dipiv_array, dB_array, lddb,
                                    batchCount, queue->stream);
}

void magma_get_dgetrf_batched_nbparam(magma_int_t n, magma_int_t* nb, magma_int_t* recnb)
{
    // The blocking a caller that sizes its own workspace may plan with: 16 for
    // the register-tile orders, the whole matrix where it fits a workgroup's
    // LDS, and above that the blocked LU's nb-wide blocks of 32-wide panels.
    // The one-workgroup kernel takes some of these orders with 32-wide panels
    // in place; it needs no workspace, so the answer does not depend on it.
    int b = 16, r = 16;
    if (!mgi::getrf_tile_supported(n)) {
        if (mgi::getrf_lds_bytes(n, n) <= mgi::max_dynamic_lds()) {
            b = std::max(1, n);
            r = 1;
        } else {
            b = std::max(mgi::getrf_blocked_nb(n), 1);
            r = std::min(b, 32);
        }
    }
    if (nb) *nb = b;
    if (recnb) *recnb = r;
}

void magma_get_dgetrf_vbatched_nbparam(magma_int_t max_m, magma_int_t max_n, magma_int_t* nb, magma_int_t* recnb)
{
    // 16 (the register tile's panels) up to 128 rows, the blocked LU's block
    // for the largest row count above that; see the square form above for the
    // one-workgroup kernel.
    int b = 16, r = 16;
    if (max_m > 128 || max_n > 128) {
        b = std::max(mgi::getrf_blocked_nb(max_m), 1);
        r = std::min(b, 32);
    }
    if (nb) *nb = b;
    if (recnb) *recnb = r;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Single precision (the "s" forms of the same drivers).
// ---------------------------------------------------------------------------
namespace mgi {

magma_int_t sgetrf_batched_async(int m, int n, float** dA_array, int ldda, int** ipiv_array, int* info_array,
                                 int batch, hipStream_t stream)
{
    // FP32 has no register-tile kernel: the wave kernel takes every batch (one
    // system of 64 rows 160 -> 90 us, 20,000 x 8^2 156 -> 71, 8,192 x 64^2 787 -> 228)
    if (m == n && n <= 64) {
        TileArgs a{n, 0, ldda, 0, nullptr, nullptr, nullptr, nullptr, nullptr};
        return slu_wave_launch((n + 15) / 16, a, dA_array, ipiv_array, info_array, batch, stream);
    }
    if (getrf_wg_preferred(m, n, batch)) {
        SizeArgs sz{m, n, ldda, nullptr, nullptr, nullptr, nullptr};
        return sgetrf_wg_launch(kUpdF32, sz, m, dA_array, ipiv_array, info_array, WgRhs<float>{}, batch, stream);
    }
    if (getrf_lds_bytes(m, n, sizeof(float)) <= max_dynamic_lds())
        return sgetrf_lds_launch(m, n, dA_array, ldda, ipiv_array, info_array, batch, stream);
    if (getrf_blocked_supported(m))
        return sgetrf_blocked_launch(kUpdF32, m, n, ldda, nullptr, nullptr, nullptr, m, n, dA_array, ipiv_array,
                                     info_array, batch, stream);
    return MAGMA_ERR_NOT_SUPPORTED;
}

magma_int_t sgetrs_batched_async(int trans, int n, int nrhs, float** dA_array, int ldda, int** ipiv_array,
                                 float** dB_array, int lddb, int batch, hipStream_t stream)
{
    RsSizes rs{n, nrhs, ldda, lddb, n, nullptr, nullptr, nullptr, nullptr, nullptr};
    return getrs_generic_launch_t<float>(trans, rs, nrhs, dA_array, ipiv_array, dB_array, batch, stream);
}

}  // namespace mgi

extern "C" {

magma_int_t magma_sgetrf_batched(magma_int_t m, magma_int_t n, float** dA_array, magma_int_t ldda,
                                 magma_int_t** ipiv_array, magma_int_t* info_array,
                                 magma_int_t batchCount, magma_queue_t queue)
{
    magma_int_t arginfo = 0;
    if (m < 0)
        arginfo = -1;
    else if (n < 0)
        arginfo = -2;
    else if (ldda < std::max(1, m))
        arginfo = -4;
    else if (batchCount < 0)
        arginfo = -7;
    if (arginfo != 0) {
        magma_xerbla(__func__, -arginfo);
        return arginfo;
    }
    if (m == 0 || n == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    magma_int_t rc = mgi::sgetrf_batched_async(m, n, dA_array, ldda, ipiv_array, info_array, batchCount,
                                               queue->stream);
    if (rc != MAGMA_SUCCESS) return rc;
    MGI_HIP_CHECK(hipStreamSynchronize(queue->stream));
    return 0;
}

magma_int_t magma_sgetrs_batched(magma_trans_t trans, magma_int_t n, magma_int_t nrhs,
                                 float** dA_array, magma_int_t ldda, magma_int_t** dipiv_array,
                                 float** dB_array, magma_int_t lddb,
                                 magma_int_t batchCount, magma_queue_t queue)
{
    const bool notran = (trans == MagmaNoTrans);
    magma_int_t info = 0;
    if (!notran && trans != MagmaTrans && trans != MagmaConjTrans)
        info = -1;
    else if (n < 0)
        info = -2;
    else if (nrhs < 0)
        info = -3;
    else if (ldda < std::max(1, n))
        info = -5;
    else if (lddb < std::max(1, n))
        info = -8;
    else if (batchCount < 0)
        info = -9;
    if (info != 0) {
        magma_xerbla(__func__, -info);
        return info;
    }
    if (n == 0 || nrhs == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    return mgi::sgetrs_batched_async(notran ? 0 : 1, n, nrhs, dA_array, ldda, dipiv_array, dB_array, lddb,
                                     batchCount, queue->stream);
}

magma_int_t magma_sgesv_batched(magma_int_t n, magma_int_t nrhs, float** dA_array, magma_int_t ldda,
                                magma_int_t** dipiv_array, float** dB_array, magma_int_t lddb,
                                magma_int_t* dinfo_array, magma_int_t batchCount, magma_queue_t queue)
{
    magma_int_t info = 0;
    if (n < 0)
        info = -1;
    else if (nrhs < 0)
        info = -2;
    else if (ldda < std::max(1, n))
        info = -4;
    else if (lddb < std::max(1, n))
        info = -6;
    else if (batchCount < 0)
        info = -9;
    if (info != 0) {
        magma_xerbla(__func__, -info);
        return info;
    }
    if (n == 0 || nrhs == 0 || batchCount == 0) return 0;
    if (queue == nullptr) return MAGMA_ERR_NOT_INITIALIZED;
    hipSetDevice(queue->device);
    info = mgi::sgetrf_batched_async(n, n, dA_array, ldda, dipiv_array, dinfo_array, batchCount, queue->stream);
    if (info != MAGMA_SUCCESS) return info;
    return mgi::sgetrs_batched_async(0, n, nrhs, dA_array, ldda, dipiv_array, dB_array, lddb, batchCount,
                                     queue->stream);
}

}  // extern "C"
