// Distinct R vectors of a hopping or R list.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <map>
#include <set>
#include <vector>

namespace dgi {

// Index of each row's R = (row[0], row[1], row[2]) among the distinct ones, in order of first
// appearance; rows of five ints (hopping and R lists), host only
struct RIndex {
    std::vector<int4> R;
    std::vector<int> of;  // per row
};

// Empty (R and of) where there are more than max_r distinct ones.  64 rows spread over the list
// show that at once for most lists that are sparse, whose sums make no use of the index
// (indexing them all took 10 of 108 us of an H(k) with n = 32, 4096 k and 30 % of 19 R).
inline RIndex index_r(int n_rows, const int* rows, size_t max_r)
{
    RIndex x;
    {
        std::set<std::array<int, 3>> some;
        const int n = std::min(n_rows, 64);
        for (int s = 0; s < n && some.size() <= max_r; ++s) {
            const int* v = rows + 5 * (size_t)((long long)n_rows * s / n);
            some.insert({v[0], v[1], v[2]});
        }
        if (some.size() > max_r) return x;
    }
    x.of.resize(n_rows);
    long long lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    for (int q = 0; q < n_rows; ++q)
        for (int c = 0; c < 3; ++c) {
            lo[c] = std::min<long long>(lo[c], rows[5 * (size_t)q + c]);
            hi[c] = std::max<long long>(hi[c], rows[5 * (size_t)q + c]);
        }
    const long long e0 = hi[0] - lo[0] + 1, e1 = hi[1] - lo[1] + 1, e2 = hi[2] - lo[2] + 1;
    const bool grid = e0 < 65536 && e1 < 65536 && e2 < 65536 && e0 * e1 < 65536 && e0 * e1 * e2 < 65536;
    std::vector<int> at(grid ? e0 * e1 * e2 : 0, -1);
    std::map<std::array<int, 3>, int> far;  // scattered R vectors
    int last = -1;
    for (int q = 0; q < n_rows; ++q) {
        const int* v = rows + 5 * (size_t)q;
        if (last < 0 || x.R[last].x != v[0] || x.R[last].y != v[1] || x.R[last].z != v[2]) {
            int* slot = grid ? &at[((v[0] - lo[0]) * e1 + (v[1] - lo[1])) * e2 + (v[2] - lo[2])]
                             : &far.emplace(std::array<int, 3>{v[0], v[1], v[2]}, -1).first->second;
            if (*slot < 0) {
                if (x.R.size() == max_r) return RIndex();
                *slot = (int)x.R.size();
                x.R.push_back(int4{v[0], v[1], v[2], 0});
            }
            last = *slot;
        }
        x.of[q] = last;
    }
    return x;
}

}  // namespace dgi
