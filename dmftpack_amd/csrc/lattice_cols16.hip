// Column-per-lane Schur kernels, bucket N = 16 (n_c up to 16); see lattice_schur_cols.hpp.
#include "lattice_schur_cols.hpp"

namespace dg {

hipError_t launch_cols_16(const LatArgs& a, int mode, const cd* sig_all, hipStream_t s)
{
    return launch_cols_bucket<16>(a, mode, sig_all, s);
}

hipError_t launch_cols_multi_16(const LatArgs& proto, int mode, hipStream_t s, const SchurMulti& m)
{
    return launch_cols_bucket<16>(proto, mode, nullptr, s, &m);
}

}  // namespace dg
