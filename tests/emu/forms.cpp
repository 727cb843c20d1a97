// C entries to the launchers that the dispatch reaches only with large
// batches, so that the emulation can run their kernels on a few systems.
#include "getrf_kernels.h"

using namespace mgi;

// One wave per system; B may be null (LU only), and so may the map and the
// per-matrix arrays.
extern "C" int emu_lu_wave_d(int nch, int n, int ld, const int* map, const int* n_arr, const int* ld_arr, double** A,
                             int** ipiv, int* info, double** B, int nrhs, int ldb, int batch)
{
    const TileArgs a{n, nrhs, ld, ldb, map, n_arr, nullptr, ld_arr, nullptr};
    return lu_wave_launch(nch, a, A, ipiv, info, B, batch, nullptr);
}

extern "C" int emu_lu_wave_s(int nch, int n, int ld, float** A, int** ipiv, int* info, int batch)
{
    const TileArgs a{n, 0, ld, 0, nullptr, nullptr, nullptr, nullptr, nullptr};
    return slu_wave_launch(nch, a, A, ipiv, info, batch, nullptr);
}

// One workgroup per system; ipiv may be null (no pivoting), and so may B.
extern "C" int emu_lu_wg_d(int m, int n, int ld, double** A, int** ipiv, int* info, double** B, int nrhs, int ldb,
                           int batch)
{
    const SizeArgs sz{m, n, ld, nullptr, nullptr, nullptr, nullptr};
    WgRhs<double> rhs;
    if (B) {
        rhs.dB_array = B;
        rhs.nrhs = rhs.max_nrhs = nrhs;
        rhs.lddb = ldb;
    }
    return getrf_wg_launch(sz, m, A, ipiv, info, rhs, batch, nullptr);
}
