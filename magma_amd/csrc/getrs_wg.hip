// Batched triangular solve with LU factors (LAPACK dgetrs semantics), one
// workgroup per system and up to 32 right-hand sides: the interchanges on the
// right-hand sides, then two blocked sweeps (wg_sweep, wg_lu.h) that read
// each factor once, 32 columns at a time, and apply it by MFMA.
//
// NoTrans: B := U \ (L \ (P^T B))          (src/zgetrs_batched.cpp:119-145)
// Trans:   B := P (L^T \ (U^T \ B))        (src/zgetrs_gpu.cpp:203-227; the
//          batched reference's transposed branch uses the wrong triangles and
//          pivot order, so the non-batched LAPACK order is followed here).
//
// Bound: HBM on the factors once a CU holds several workgroups; a single
// system is bound by the chain of its 32-row blocks. Against the sweeps with
// per-row FMA that it replaced (kernel, us): FP64 1,000 x 384^2 transposed, 16
// right-hand sides 1219 -> 524 (2.3 TB/s on the factors); FP64 8,192 x 64^2
// transposed, 8 right-hand sides 562 -> 130; FP32 the same 372 -> 71; FP32
// 1,000 x 300^2, 8 right-hand sides 6849 -> 138.
//
// At small orders the chain of one wave counts. What shortened it, in whole
// calls of FP64 8,192 x 64^2 r8 and 20,000 x 16^2 r16: one division per diagonal
// block instead of one per entry that a thread holds, and eight columns of B in
// flight (265 -> 230, 377 -> 255 us); steps past a block's rows skipped, which
// also ended the spills, and the first tile waited for before the loop over
// tiles (216 -> 139, 257 -> 138; 1,100 x 512^2 r1 811 -> 594). The forms of more
// than one wave fit four waves per SIMD without scratch (one of them spills one
// register); the FP64 one-wave forms take 160..167 + 8 registers, two or three
// waves per SIMD.
#include "magma_internal.h"
#include "getrf_kernels.h"
#include "wg_lu.h"

namespace mgi {

constexpr int kMaxRhs = 32;      // right-hand sides per workgroup (16 if the batch has no more)
constexpr long kOneStrip = 1024; // one-wave workgroups on one wave per SIMD
constexpr int kPermCols = 4;     // right-hand sides permuted at a time in global memory

template <typename T, int NTH, bool TRANS, bool INLDS, int MAXR>
__global__ void __launch_bounds__(NTH, 4)
getrs_wg_kernel(RsSizes sz, T** __restrict__ dA_array, int** __restrict__ ipiv_array, T** __restrict__ dB_array)
{
    extern __shared__ __align__(16) unsigned char rw_raw[];
    __shared__ WgSweepSmem<T, MAXR> sm;
    const int b = sz.map ? sz.map[blockIdx.x] : blockIdx.x;
    int n, nrhs, ldda, lddb;
    sz.get(b, n, nrhs, ldda, lddb);
    const int c0 = blockIdx.y * MAXR;
    if (n <= 0 || c0 >= nrhs) return;
    const int nr = min(MAXR, nrhs - c0);
    auto A = gptr(dA_array[b]);
    auto B = gptr(dB_array[b]) + (size_t)c0 * lddb;
    // (P^T B)(i,:) = B(perm[i],:), P the product of the interchanges
    // k <-> ipiv[k]-1 in order: each row is traced back through them (last to
    // first); one outside [k, n) cannot come from a valid LU and is none
    int* perm = reinterpret_cast<int*>(rw_raw);
    int* spiv = perm + sz.max_n;
    T* buf = reinterpret_cast<T*>(rw_raw + (size_t)sz.max_n * 2 * sizeof(int));
    const int tid = threadIdx.x;
    const bool swaps = ipiv_array != nullptr;                           // null: factors without pivoting
    if (swaps) {
        auto ipiv = gptr(ipiv_array[b]);
        for (int i = tid; i < n; i += NTH) {
            const int p = ipiv[i] - 1;
            spiv[i] = (p > i && p < n) ? p : i;
        }
        __syncthreads();
    }
    for (int r = tid; r < n; r += NTH) {
        int src = r;
        if (swaps) {
#pragma unroll 8
            for (int k = n - 1; k >= 0; --k) {
                const int p = spiv[k];
                src = (src == k) ? p : (src == p ? k : src);
            }
        }
        perm[r] = src;
    }
    __syncthreads();
    if constexpr (INLDS) {
        const int ldx = n | 1;                 // odd: the columns start in different banks
        // eight columns' loads in flight at a time (those past the last one
        // read it again and are dropped)
        for (int i = tid; i < n; i += NTH) {
            auto Bi = B + (TRANS ? i : perm[i]);
            for (int c = 0; c < nr; c += 8) {
                T v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = Bi[(size_t)min(c + e, nr - 1) * lddb];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (c + e < nr) buf[i + (c + e) * ldx] = v[e];
            }
        }
        __syncthreads();
        if constexpr (TRANS) {
            wg_sweep<T, NTH, false, true, false>(A, ldda, n, buf, ldx, nr, sm);     // U^T
            wg_sweep<T, NTH, true, true, true>(A, ldda, n, buf, ldx, nr, sm);       // L^T
        } else {
            wg_sweep<T, NTH, false, false, true>(A, ldda, n, buf, ldx, nr, sm);     // L
            wg_sweep<T, NTH, true, false, false>(A, ldda, n, buf, ldx, nr, sm);     // U
        }
        for (int c = 0; c < nr; ++c)
            for (int i = tid; i < n; i += NTH) B[(TRANS ? perm[i] : i) + (size_t)c * lddb] = buf[i + c * ldx];
    } else {
        auto permute = [&]() {
            if (!swaps) return;
            for (int c = 0; c < nr; c += kPermCols) {
                const int nc = min(kPermCols, nr - c);
                for (int q = 0; q < nc; ++q)
                    for (int i = tid; i < n; i += NTH)
                        buf[q * n + (TRANS ? perm[i] : i)] = B[i + (size_t)(c + q) * lddb];
                __syncthreads();
                for (int q = 0; q < nc; ++q)
                    for (int i = tid; i < n; i += NTH)
                        B[i + (size_t)(c + q) * lddb] = buf[q * n + (TRANS ? i : perm[i])];
                __syncthreads();
            }
        };
        if constexpr (TRANS) {
            wg_sweep<T, NTH, false, true, false>(A, ldda, n, B, lddb, nr, sm);
            wg_sweep<T, NTH, true, true, true>(A, ldda, n, B, lddb, nr, sm);
            permute();
        } else {
            permute();
            wg_sweep<T, NTH, false, false, true>(A, ldda, n, B, lddb, nr, sm);
            wg_sweep<T, NTH, true, false, false>(A, ldda, n, B, lddb, nr, sm);
        }
    }
}

template <typename T, int NTH, bool TRANS, bool INLDS, int MAXR>
static magma_int_t launch_one(const RsSizes& sz, int max_nrhs, size_t lds, T** dA_array, int** ipiv_array, T** dB_array,
                              int batch, hipStream_t stream)
{
    MGI_HIP_CHECK(hipFuncSetAttribute((const void*)getrs_wg_kernel<T, NTH, TRANS, INLDS, MAXR>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const dim3 grid(batch, ceildiv(max_nrhs, MAXR));
    getrs_wg_kernel<T, NTH, TRANS, INLDS, MAXR><<<grid, NTH, lds, stream>>>(sz, dA_array, ipiv_array, dB_array);
    MGI_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

template <typename T, int NTH, bool TRANS>
static magma_int_t launch_nth(const RsSizes& sz, int max_nrhs, T** dA_array, int** ipiv_array, T** dB_array, int batch,
                              hipStream_t stream)
{
    const size_t perm = (size_t)sz.max_n * 2 * sizeof(int);
    // one wave solves its strips of 16 right-hand sides one after the other: a
    // workgroup takes one strip while the strips all run at once (us, two strips
    // / one: 64 x 64^2 r32 60 / 47, 512 x 64^2 r32 64 / 52; 1,024 x 64^2 r32 69 / 80)
    const bool one = max_nrhs <= 16 || (NTH == kWave && (long)batch * ceildiv(max_nrhs, 16) <= kOneStrip);
    const int cols = one ? 16 : kMaxRhs;
    const size_t rhs = (size_t)(sz.max_n | 1) * (max_nrhs < cols ? max_nrhs : cols) * sizeof(T);
    const size_t gl = perm + (size_t)sz.max_n * kPermCols * sizeof(T);
    if (one)
        return rhs <= kGetrsRhsLds
                   ? launch_one<T, NTH, TRANS, true, 16>(sz, max_nrhs, perm + rhs, dA_array, ipiv_array, dB_array, batch, stream)
                   : launch_one<T, NTH, TRANS, false, 16>(sz, max_nrhs, gl, dA_array, ipiv_array, dB_array, batch, stream);
    return rhs <= kGetrsRhsLds
               ? launch_one<T, NTH, TRANS, true, kMaxRhs>(sz, max_nrhs, perm + rhs, dA_array, ipiv_array, dB_array, batch, stream)
               : launch_one<T, NTH, TRANS, false, kMaxRhs>(sz, max_nrhs, gl, dA_array, ipiv_array, dB_array, batch, stream);
}

template <typename T>
magma_int_t getrs_wg_launch(int trans, const RsSizes& sz, int max_nrhs, T** dA_array, int** ipiv_array, T** dB_array,
                            int batch, hipStream_t stream)
{
    // threads by order: one wave up to 64 rows; eight where a block's update
    // covers more than 512 rows
    auto go = [&](auto tr) {
        constexpr bool TR = decltype(tr)::value;
        if (sz.max_n <= 64) return launch_nth<T, 64, TR>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        if (sz.max_n <= 128) return launch_nth<T, 128, TR>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        if (sz.max_n <= 512) return launch_nth<T, 256, TR>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
        return launch_nth<T, 512, TR>(sz, max_nrhs, dA_array, ipiv_array, dB_array, batch, stream);
    };
    return trans ? go(std::true_type{}) : go(std::false_type{});
}

template magma_int_t getrs_wg_launch<double>(int, const RsSizes&, int, double**, int**, double**, int, hipStream_t);
template magma_int_t getrs_wg_launch<float>(int, const RsSizes&, int, float**, int**, float**, int, hipStream_t);

}  // namespace mgi
