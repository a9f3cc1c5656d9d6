// Chirp-z form of the two tau <-> iw sums and the definiteness test of the
// causality checks (ft_czt.hip).  All pointers are device pointers.
#pragma once
#include <hip/hip_runtime.h>

#include "dev_common.hpp"

namespace dg {

constexpr int kCztM = 4096;         // FFT length: one tile in the LDS of a workgroup
constexpr int kCztTile = kCztM / 2; // inputs and outputs of a tile

// E [2 n_tau] e^{i pi m / n_tau}, then tw [kCztM] e^{-2 pi i k / kCztM}, then filt [kCztM]
inline size_t czt_table_count(int n_tau) { return 2 * (size_t)n_tau + 2 * kCztM; }
hipError_t launch_czt_tables(int n_tau, cd* tab, hipStream_t s);

// in_tiles are shared out over in_groups workgroups, each adding its tiles, as many groups as there
// are tiles while their partial sums, m2 n_out each, fit kCztPartBytes
struct CztPlan {
    int n_tau, n_in, n_out, in_tiles, in_groups, out_tiles, ld_in, ld_out;
};
constexpr size_t kCztPartBytes = (size_t)512 << 20;
CztPlan czt_plan(int n_tau, int n_in, int n_out, int m2);

// parts [in_group][e][n_out] of sum_i exp(-+ i pi (2f+1) t / n_tau) in[e][i]:
// to_w false: i = frequency f, output t = tau index; true: i = t, output f (phase +)
hipError_t launch_czt(const CztPlan& p, bool to_w, int m2, const cd* tab, const cd* in, cd* parts, hipStream_t s);

// bad[0] += number of matrices X_b (d x d, count of them) for which -X_b (X_b Hermitian), or with
// anti -(X_b - X_b^H)/2i, is not positive definite by a margin; with anti, those that have a
// negative eigenvalue by a margin are counted in bad[1] instead; bad preset by the caller
hipError_t launch_not_posdef(const cd* X, int d, int count, bool anti, int* bad, hipStream_t s);

}  // namespace dg
