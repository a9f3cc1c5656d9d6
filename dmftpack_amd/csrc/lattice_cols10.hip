// Column-per-lane Schur kernels, bucket N = 10 (n_c up to 10); see lattice_schur_cols.hpp.
#include "lattice_schur_cols.hpp"

namespace dg {

hipError_t launch_cols_10(const LatArgs& a, int mode, const cd* sig_all, hipStream_t s)
{
    return launch_cols_bucket<10>(a, mode, sig_all, s);
}

hipError_t launch_cols_multi_10(const LatArgs& proto, int mode, hipStream_t s, const SchurMulti& m)
{
    return launch_cols_bucket<10>(proto, mode, nullptr, s, &m);
}

}  // namespace dg
