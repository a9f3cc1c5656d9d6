// Upfolding of up to 32 Kohn-Sham orbitals, one pass per k, and the k -> R sums of R lists
// dense in (R, element) (upfold_small.hip).  Device pointers unless noted.
#pragma once
#include <hip/hip_runtime.h>

#include "dev_common.hpp"

namespace dg {

constexpr int kUpfoldSmall = 32;

struct UpfoldArgs {
    int n, n_orb, nk;
    double beta, mu;
    const cd *X, *C, *T, *Ko, *S;  // [nk][...]; S null: identity overlap
    const double* eps;             // [nk][n_orb]
    const int* v2k;                // [nk][n]
    cd *D, *DDir, *DD;             // [nk][n_orb][n_orb]; DDir, DD with S only
    int* singular;                 // preset by the caller
};
hipError_t launch_upfold_small(const UpfoldArgs& a, hipStream_t s);

// R sums of nx matrices per k: part [seg][x][R][e] = sum over the segment's k of
// ph(k, R) Y_x(k)(e), ph [nk][n_r padded to kRsTile] from launch_r_phases (phase +)
// (14: the 27 R of the first shell of neighbours are two tiles with one column of padding; 14
// sums take 66 vector registers, seven wavefronts per SIMD, and a tile's phases 84 scalar ones.
// NumOrbit = 28, 12^3 k, the whole call, a workgroup per run of entries -> tiles, ms: 125 R
// (126 padded) 6.8 -> 0.75, 343 R (350) 20.4 -> 1.72)
constexpr int kRsTile = 14;
inline int rs_pad(int n_r) { return (n_r + kRsTile - 1) / kRsTile * kRsTile; }
hipError_t launch_r_phases(const int4* R, int n_r, const double* kphase, int nk, cd* ph, hipStream_t s);
hipError_t launch_r_sums(const cd* const Y[3], int nx, int oo, int nk, int n_r, const cd* ph, int nseg, cd* part,
                         hipStream_t s);
// dmr[x][entry] += scale * sum_seg part[seg][x or 0][of[entry].x][of[entry].y], x = 0..2
hipError_t launch_r_scatter(const cd* part, int nseg, int nx, int n_r, int oo, const int2* of, int n_entries,
                            double scale, cd* dmr, hipStream_t s);

}  // namespace dg
