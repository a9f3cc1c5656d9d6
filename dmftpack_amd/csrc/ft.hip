// Matsubara tail moments and the iw <-> tau transforms.
//
//   dmftgpu_moments   getAsymto_moments   (FourierTransform.cpp:184-465)
//   dmftgpu_ft_w2tau  FourierTransform_ + FourierTransform_tau (:126-178, :16-118)
//   dmftgpu_ft_tau2w  FT_t_to_w           (:521-561)
//
// GPU work: the sliding-window least-squares fits (one thread per window start
// and matrix element, summing in the reference's ascending order), the window
// averages, the batched positivity tests, and both transforms: on the uniform tau grid as
// chirp-z transforms (ft_czt.hip), at arbitrary tau values as a dense complex product.  The
// tail of FourierTransform_tau does not depend on tau, so it is subtracted once per
// frequency, not once per (tau, frequency) as in the reference loop (:55-61).
// Host work: the small d x d set-up (square roots, inverses, eigenbases) and
// the sequential selection / patch logic, restated from the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/dmftgpu.h"
#include "api_internal.hpp"
#include "ft_czt.hpp"
#include "host_linalg.hpp"
#include "lattice_kernels.hpp"

using dg::cd;
using dgi::fail;

namespace {

using namespace dg;

// ---------------------------------------------------------------------------
// getAsymto_moments kernels
// ---------------------------------------------------------------------------
// Partial-pivot LU inverse of the real n x n (n <= 4) normal matrix, the
// steps of Eigen's PartialPivLU::inverse: pivot = the first largest |entry|
// of the column, multipliers by the reciprocal pivot, fused updates, forward
// then backward substitution per unit column.  Every multiply-add is an
// explicit fma and nothing else is contracted, so the oracle's restatement
// (which does the same) gives the same bits.
__device__ void lu_inverse4(const double (&A)[16], int n, double (&X)[16])
{
#pragma clang fp contract(off)
    double lu[16];
    int perm[4];
    for (int e = 0; e < 16; ++e) lu[e] = A[e];
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int k = 0; k < n; ++k) {
        int p = k;
        double best = fabs(lu[k + k * 4]);
        for (int i = k + 1; i < n; ++i)
            if (fabs(lu[i + k * 4]) > best) {
                best = fabs(lu[i + k * 4]);
                p = i;
            }
        if (p != k) {
            for (int j = 0; j < n; ++j) {
                double t = lu[k + j * 4];
                lu[k + j * 4] = lu[p + j * 4];
                lu[p + j * 4] = t;
            }
            int t = perm[k];
            perm[k] = perm[p];
            perm[p] = t;
        }
        if (best != 0.0) {
            const double inv = 1.0 / lu[k + k * 4];
            for (int i = k + 1; i < n; ++i) lu[i + k * 4] *= inv;
        }
        for (int j = k + 1; j < n; ++j) {
            const double u = lu[k + j * 4];
            for (int i = k + 1; i < n; ++i) lu[i + j * 4] = fma(-lu[i + k * 4], u, lu[i + j * 4]);
        }
    }
    for (int c = 0; c < n; ++c) {
        double x[4];
        for (int i = 0; i < n; ++i) x[i] = (perm[i] == c) ? 1.0 : 0.0;
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < i; ++j) x[i] = fma(-lu[i + j * 4], x[j], x[i]);
        for (int i = n - 1; i >= 0; --i) {
            for (int j = i + 1; j < n; ++j) x[i] = fma(-lu[i + j * 4], x[j], x[i]);
            x[i] /= lu[i + i * 4];
        }
        for (int i = 0; i < n; ++i) X[i + c * 4] = x[i];
    }
}

// columns of the design matrix for row pair jj (Re row 2jj, Im row 2jj+1)
// non-G: Re: [1, 0, -1/z^2, 0]   Im: [0, -1/z, 0, 1/z^3]   (:227-230)
// G    : Re: [-1/z^2, 0]          Im: [0, 1/z^3]             (:366-367)
// basis values per frequency, tab[wn] = {-1/z, -1/z^2, 1/z^3, 1/z}, formed on
// the host with std::pow as the reference forms them (dmftgpu_moments)
// K^T K of window w, entry (a, b) with a <= b (the matrix is symmetric): one
// thread per (window, entry), summing the rows in order, Re row then Im row of
// each frequency, one fma per row (zero entries included).
__global__ void k_mom_ktk(int n_freq, int range, int green, const double4* __restrict__ tab, double* __restrict__ ktk)
{
#pragma clang fp contract(off)
    const int nm = green ? 2 : 4;
    const int npair = nm * (nm + 1) / 2;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= range * npair) return;
    const int w = t / npair;
    int q = t % npair, b = 0;
    while (q > b) {  // pair index q -> (a, b), a <= b, column by column
        q -= b + 1;
        ++b;
    }
    const int a = q;
    double K = 0.0;
    for (int wn = w; wn < n_freq; ++wn) {
        const double4 c = tab[wn];
        double re[4] = {0, 0, 0, 0}, im[4] = {0, 0, 0, 0};
        if (!green) {
            re[0] = 1.0;
            im[1] = c.x;
            re[2] = c.y;
            im[3] = c.z;
        } else {
            re[0] = c.y;
            im[1] = c.z;
        }
        K = fma(re[a], re[b], K);
        K = fma(im[a], im[b], K);
    }
    ktk[(size_t)w * 16 + a + b * 4] = K;
    ktk[(size_t)w * 16 + b + a * 4] = K;
}

// inverse of each window's normal matrix, in place (one thread per window)
__global__ void k_mom_kinv(int range, int green, double* __restrict__ kinv)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= range) return;
    const int nm = green ? 2 : 4;
    double K[16], X[16];
    for (int e = 0; e < 16; ++e) K[e] = kinv[(size_t)w * 16 + e];
    lu_inverse4(K, nm, X);
    for (int e = 0; e < 16; ++e) kinv[(size_t)w * 16 + e] = X[e];
}

// mt[a][w][e] = sum_rows KM_solve[w][a][row] g_e[row], with the rows of
// KM_solve = (K^T K)^{-1} K^T formed first, as the reference associates the
// product (FourierTransform.cpp:239-243): per frequency the Re row of the
// design matrix contributes sum_b Kinv[a][b] Re_b and the Im row
// sum_b Kinv[a][b] Im_b (the rows' zero entries left out), each taken times
// its half of g and added, Re row first, in ascending frequency order.
// One thread per (moment, window, element pair al <= be): the transposed element's row
// values are the conjugates, term by term, so its sum is the conjugate and is written with
// it.  The sum is a serial chain, so the time is that of the longest window.  A wavefront's
// frequencies are uniform (its windows are neighbours; each waits for its own start), so
// the basis values come as scalar operands and a frequency costs two vector loads, those of
// kFitAhead frequencies issued ahead of their use.  With the basis loaded by each lane and
// an element a thread, d = 5 and N_freq = 1000 took 220 us, bound by the L1 loads; this
// form 75 us.  From kFitAll (window, pair) fits on, a thread takes all NA moments: the data
// are read once instead of once a moment, which counts where they leave the caches.  us of the
// call, one moment / all a thread: d = 5, 1000 frequencies (15000 fits) 193 / 238, 2500 (37500)
// 489 / 506, d = 10, 1000 (55000) 499 / 464, d = 28, 1500 (609000) 7475 / 3177 (an element a
// thread: 7057), d = 32, 2500 (1.32e6) 38950 / 12920 (25420).
constexpr int kFitAhead = 8;
constexpr size_t kFitAll = 40960;

template <bool GREEN, int NA>
__global__ __launch_bounds__(64) void k_mom_fit(const cd* __restrict__ fw, int d, int n_freq, int range,
                                                const double* __restrict__ tab_, const double* __restrict__ kinv,
                                                cd* __restrict__ mt)
{
#pragma clang fp contract(off)
    const int m2 = d * d, np = d * (d + 1) / 2, a0 = blockIdx.y * NA;
    const kconst_double* tab = (const kconst_double*)tab_;
    const unsigned first = blockIdx.x * 64, last = min(first + 63, (unsigned)(range * np - 1));
    const unsigned t = min(first + threadIdx.x, last);  // spare lanes repeat the last entry
    const int w = (int)(t / np), q = (int)(t % np);
    int be = 0, al = q;
    while (al > be) al -= ++be;  // pair q -> (al, be), al <= be
    double x[NA][4];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        const double* X = kinv + (size_t)w * 16 + a0 + a;  // Kinv(a, b) at X[4 b]
#pragma unroll
        for (int b = 0; b < 4; ++b) x[a][b] = GREEN && b > 1 ? 0.0 : X[4 * b];
    }
    // element addresses: the frequency's uniform base and the lane's offset
    const unsigned oa = (al + be * d) * sizeof(cd), ob = (be + al * d) * sizeof(cd);
    auto at = [&](int wn, unsigned o) -> cd { return *(const cd*)((const char*)(fw + (size_t)wn * m2) + o); };
    cd s[NA];  // twice the sums: the halves of Re and Im are taken at the end (exactly)
#pragma unroll
    for (int a = 0; a < NA; ++a) s[a] = cd{0, 0};
    // basis values {-1/z, -1/z^2, 1/z^3, 1/z} of a frequency at c
    auto add = [&](double c0, double c1, double c2, double c3, cd fab, cd fba) {
        // 2 Re = F_ab + conj(F_ba) ; 2 Im = (F_ab - conj(F_ba))/i
        const cd re = cd{fab.x + fba.x, fab.y - fba.y};
        cd im = cd{fab.y + fba.y, fba.x - fab.x};
        if (GREEN && al == be) im.x += 2.0 * c3;  // (:373)
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            double kr, ki;
            if (!GREEN) {
                // Re row [1, 0, -1/z^2, 0], Im row [0, -1/z, 0, 1/z^3]   (:227-230)
                kr = fma(x[a][2], c1, x[a][0]);
                ki = fma(x[a][3], c2, x[a][1] * c0);
            } else {
                // Re row [-1/z^2, 0], Im row [0, 1/z^3]   (:366-367)
                kr = x[a][0] * c1;
                ki = x[a][1] * c2;
            }
            s[a] = cadd(s[a], cd{fma(ki, im.x, kr * re.x), fma(ki, im.y, kr * re.y)});
        }
    };
    auto add1 = [&](int wn) {
        const kconst_double* c = tab + 4 * wn;
        add(c[0], c[1], c[2], c[3], at(wn, oa), at(wn, ob));
    };
    int wn = (int)(first / np);       // the first window of the wavefront
    const int w1 = (int)(last / np);  // and its last
    for (; wn < w1; ++wn)
        if (wn >= w) add1(wn);
    if (wn + kFitAhead <= n_freq) {
        // the next kFitAhead frequencies' loads are under way while these are added, and
        // the scalar loads of a group are waited for together
        cd p[2][kFitAhead], r[2][kFitAhead];
        auto load = [&](int h, int w0) {
#pragma unroll
            for (int u = 0; u < kFitAhead; ++u) {
                const int f = min(w0 + u, n_freq - 1);
                p[h][u] = at(f, oa);
                r[h][u] = at(f, ob);
            }
        };
        auto sum = [&](int h, int w0) {
            double c[kFitAhead][4];
#pragma unroll
            for (int u = 0; u < kFitAhead; ++u)
#pragma unroll
                for (int x = GREEN ? 1 : 0; x < (GREEN ? 4 : 3); ++x) c[u][x] = tab[4 * (w0 + u) + x];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < kFitAhead; ++u) add(c[u][0], c[u][1], c[u][2], c[u][3], p[h][u], r[h][u]);
            __builtin_amdgcn_sched_barrier(0);
        };
        load(0, wn);
        for (; wn + 2 * kFitAhead <= n_freq; wn += 2 * kFitAhead) {
            load(1, wn + kFitAhead);
            sum(0, wn);
            load(0, wn + 2 * kFitAhead);
            sum(1, wn + kFitAhead);
        }
        if (wn + kFitAhead <= n_freq) {
            sum(0, wn);
            wn += kFitAhead;
        }
    }
    for (; wn < n_freq; ++wn) add1(wn);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        const cd v = cd{0.5 * s[a].x, 0.5 * s[a].y};
        cd* out = mt + ((size_t)(a0 + a) * range + w) * m2;
        out[be + al * d] = cconj(v);
        out[al + be * d] = v;
    }
}

// trace[a][w] = sum_alpha Re mt[a][w][alpha alpha]     (:244-247)
__global__ void k_mom_trace(const cd* __restrict__ mt, int d, int range, int nm, double* __restrict__ trace)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= range * nm) return;
    const int a = t / range, w = t % range;
    double s = 0.0;
    for (int al = 0; al < d; ++al) s += mt[((size_t)a * range + w) * d * d + al + al * d].x;
    trace[t] = s;
}

// avg[a][c][e] = mean_{iw=c..c+2Nv} mt[a][iw][e]     (:259-283)
__global__ void k_mom_avg(const cd* __restrict__ mt, int m2, int range, int nm, int Nv, cd* __restrict__ avg)
{
    const int ncent = range - 2 * Nv;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nm * ncent * m2) return;
    const int e = (int)(t % m2);
    const int c = (int)((t / m2) % ncent);
    const int a = (int)(t / ((size_t)m2 * ncent));
    cd s = cd{0, 0};
    const cd* m = mt + ((size_t)a * range + c) * m2 + e;
#pragma unroll 8
    for (int iw = 0; iw <= 2 * Nv; ++iw) s = cadd(s, m[(size_t)iw * m2]);
    const double cnt = 2 * Nv + 1;
    avg[t] = cd{s.x / cnt, s.y / cnt};
}

// positivity matrix per window centre:
//   non-G: T = Vi m3 Vi - (Vi m2 Vi)^2, Vi = (m1)^{-1/2}   (:298-308)
//   G    : T = m1 - m0^2                                   (:423-424)
// (w1, U1) = eig(m1avg) for the non-G branch.  One wavefront per centre, the products
// one after the other in LDS (Vi, tmp, P2), an entry's sum in the order of its inner index.  A
// centre whose m1 is not positive gets T = -1 (the window is rejected anyway).
__global__ __launch_bounds__(64) void k_mom_posmat(const cd* __restrict__ avg, int d, int ncent, int green,
                                                   const double* __restrict__ w1, const cd* __restrict__ U1,
                                                   cd* __restrict__ T)
{
    extern __shared__ cd pm[];
    const int m2 = d * d, c = blockIdx.x, t = threadIdx.x;
    auto A = [&](int a) { return avg + ((size_t)a * ncent + c) * m2; };
    cd* out = T + (size_t)c * m2;
    if (green) {
        const cd* m0 = A(0);
        for (int e = t; e < m2; e += 64) {
            cd s = A(1)[e];
            for (int l = 0; l < d; ++l) s = cfms(m0[e % d + l * d], m0[l + (e / d) * d], s);
            out[e] = s;
        }
        return;
    }
    const double* w = w1 + (size_t)c * d;
    if (!(w[0] > 0.0)) {
        for (int e = t; e < m2; e += 64) out[e] = cd{-1.0, 0.0};
        return;
    }
    cd *Vi = pm, *tmp = pm + m2, *P2 = pm + 2 * m2, *mq = pm + 3 * m2;
    const cd* U = U1 + (size_t)c * m2;
    for (int e = t; e < m2; e += 64) mq[e] = U[e];
    wave_sync();
    for (int e = t; e < m2; e += 64) {
        const int i = e % d, j = e / d;
        cd s = cd{0, 0};
        for (int l = 0; l < d; ++l) s = cadd(s, cscale(cmulc(mq[i + l * d], mq[j + l * d]), 1.0 / sqrt(w[l])));
        Vi[e] = s;
    }
    auto product = [&](const cd* X, const cd* Y, cd* Z) {
        wave_sync();
        for (int e = t; e < m2; e += 64) {
            const int i = e % d, j = e / d;
            cd s = cd{0, 0};
            for (int l = 0; l < d; ++l) s = cfma(X[i + l * d], Y[l + j * d], s);
            Z[e] = s;
        }
        wave_sync();
    };
    wave_sync();
    for (int e = t; e < m2; e += 64) mq[e] = A(2)[e];
    product(Vi, mq, tmp);
    product(tmp, Vi, P2);
    for (int e = t; e < m2; e += 64) mq[e] = A(3)[e];
    product(Vi, mq, tmp);
    for (int e = t; e < m2; e += 64) {
        const int i = e % d, j = e / d;
        cd s = cd{0, 0};
        for (int l = 0; l < d; ++l) s = cfma(tmp[i + l * d], Vi[l + j * d], s);
        for (int l = 0; l < d; ++l) s = cfms(P2[i + l * d], P2[l + j * d], s);
        out[e] = s;
    }
}

// threads of the window-selection workgroup (one workgroup per moment, the
// window centres spread over its threads)
constexpr int kSelThreads = 1024;

// Window choice of getAsymto_moments (:289-315) for moment a = blockIdx.x:
// the spread of the moment's trace over the 2 Nv + 1 windows around each
// centre (mean, then the squared deviations, in the reference's order), and
// the scan "minPos = ncent-1; for i: if ok[i] && var[i] < var[minPos] then
// minPos = i", i.e. the first admissible centre of least spread if that
// spread is below the last centre's, else the last centre.  ok[i] is the
// positivity test on the window-averaged moments (:301-312, :432).
// cen[target] = minPos + Nv, target = a (a + 2 for the G branch).
__global__ __launch_bounds__(kSelThreads) void k_mom_select(const double* __restrict__ trace, const double* __restrict__ w1,
                                                    const double* __restrict__ wT, int d, int range, int ncent, int Nv,
                                                    int green, int* __restrict__ cen)
{
    __shared__ double bv[kSelThreads];
    __shared__ int bi[kSelThreads];
    const int a = blockIdx.x, t = threadIdx.x;
    auto spread = [&](int i) {
#pragma clang fp contract(off)
        const double* v = trace + (size_t)a * range + i;  // centre i + Nv, window [i, i + 2 Nv]
        double mean = 0.0;
#pragma unroll 8
        for (int j = 0; j < 2 * Nv + 1; ++j) mean += v[j];
        mean /= (2 * Nv + 1);
        double ss = 0.0;
#pragma unroll 8
        for (int j = 0; j < 2 * Nv + 1; ++j) {
            const double dv = v[j] - mean;
            ss += dv * dv;
        }
        return sqrt(ss / (2 * Nv + 1));
    };
    double best = 0.0;
    int besti = -1;
    for (int i = t; i < ncent; i += kSelThreads) {
        const bool ok = green ? wT[(size_t)i * d] > 1 : (w1[(size_t)i * d] > 0 && wT[(size_t)i * d] > 0);
        if (!ok) continue;
        const double v = spread(i);
        if (besti < 0 || v < best) {  // ascending i within a thread: the first of equals stays
            best = v;
            besti = i;
        }
    }
    bv[t] = best;
    bi[t] = besti;
    __syncthreads();
    for (int w = kSelThreads / 2; w > 0; w >>= 1) {
        if (t < w) {
            const int oi = bi[t + w];
            const double ov = bv[t + w];
            if (oi >= 0 && (bi[t] < 0 || ov < bv[t] || (ov == bv[t] && oi < bi[t]))) {
                bv[t] = ov;
                bi[t] = oi;
            }
        }
        __syncthreads();
    }
    if (t == 0) {
        const int last = ncent - 1;
        const int minPos = (bi[0] >= 0 && bv[0] < spread(last)) ? bi[0] : last;
        cen[green ? a + 2 : a] = minPos + Nv;
    }
}

// moments[4][d][d] = 0 and windows = -1, then m1 = I on the G branch (:451-452)
__global__ void k_mom_init(cd* __restrict__ mom, int d, int green, int* __restrict__ cen)
{
    const int m2 = d * d;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 4) cen[t] = -1;
    if (t >= 4 * m2) return;
    const int q = t / m2, e = t % m2;
    mom[t] = cd{(green && q == 1 && e % d == e / d) ? 1.0 : 0.0, 0.0};
}

// final moment of the chosen window: mean over the window of (mt_ab + conj(mt_ba))/2,
// then Hermitised (:319-330, :458-461); blockIdx.y = moment index
__global__ void k_mom_final(const cd* __restrict__ mt, int d, int range, int green, const int* __restrict__ cen_all,
                            int Nv, cd* __restrict__ mom)
{
    const int m2 = d * d;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= m2) return;
    const int mom_idx = blockIdx.y;
    const int target = green ? mom_idx + 2 : mom_idx;
    const int cen = cen_all[target];
    cd* out = mom + (size_t)target * m2;
    const int al = e % d, be = e / d;
    cd s = cd{0, 0}, st = cd{0, 0};
#pragma unroll 4
    for (int w = cen - Nv; w <= cen + Nv; ++w) {
        const cd* m = mt + ((size_t)mom_idx * range + w) * m2;
        s = cadd(s, cscale(cadd(m[al + be * d], cconj(m[be + al * d])), 0.5));
        st = cadd(st, cscale(cadd(m[be + al * d], cconj(m[al + be * d])), 0.5));
    }
    const double cnt = 2 * Nv + 1;
    s = cd{s.x / cnt, s.y / cnt};
    st = cd{st.x / cnt, st.y / cnt};
    out[e] = cscale(cadd(s, cconj(st)), 0.5);
}

// ---------------------------------------------------------------------------
// iw -> tau
// ---------------------------------------------------------------------------
// Tiles of 16 rows (frequency or tau) x 16 elements, 256 threads: reads and writes of
// either order move 256-byte runs, the transpose going through LDS.
constexpr int kTile = 16;

// D_i = F_i - tail_i,  tail_i = 1/2 sum_h A_h diag(1/(i w_i - e_h)) A_h^H   (:55-61), written to
// D[i*si + e*se].  The d factors 1/(i w_i - e_h) of a row and the d products
// A_h(a,l) conj(A_h(b,l)) of an element are formed once per tile.
__global__ __launch_bounds__(256) void k_ft_subtract_tail(const cd* __restrict__ fw, int d, int n_freq, double beta,
                                                          const cd* __restrict__ A1, const double* __restrict__ e1,
                                                          const cd* __restrict__ A2, const double* __restrict__ e2,
                                                          cd* __restrict__ D, size_t si, size_t se,
                                                          int* __restrict__ bad)
{
    __shared__ cd sg[2][kTile][33], sp[2][kTile][33], st[kTile][kTile + 1];
    const int m2 = d * d, i0 = blockIdx.x * kTile, f0 = blockIdx.y * kTile;
    if (bad && i0 == 0 && f0 == 0 && threadIdx.x == 0) *bad = 0;  // for the definiteness test that follows
    for (int t = threadIdx.x; t < kTile * d; t += 256) {
        const int r = t / d, l = t % d;
        const double w = (kPi / beta) + (i0 + r) * ((2 * kPi) / beta);
        sg[0][r][l] = crcp(cd{-e1[l], w});
        sg[1][r][l] = crcp(cd{-e2[l], w});
        const int e = min(f0 + r, m2 - 1), a = e % d, b = e / d;
        sp[0][r][l] = cmulc(A1[a + l * d], A1[b + l * d]);
        sp[1][r][l] = cmulc(A2[a + l * d], A2[b + l * d]);
    }
    __syncthreads();
    {
        const int q = threadIdx.x % kTile, r = threadIdx.x / kTile, i = i0 + r, e = f0 + q;
        cd v = cd{0.0, 0.0};
        if (i < n_freq && e < m2) {
            cd tail = cd{0.0, 0.0};
            for (int l = 0; l < d; ++l) {
                tail = cfma(sp[0][q][l], sg[0][r][l], tail);
                tail = cfma(sp[1][q][l], sg[1][r][l], tail);
            }
            v = csub(fw[(size_t)i * m2 + e], cscale(tail, 0.5));
        }
        st[r][q] = v;
    }
    __syncthreads();
    const bool rows = si < se;  // consecutive threads along the faster index of D
    const int r = rows ? threadIdx.x % kTile : threadIdx.x / kTile, q = rows ? threadIdx.x / kTile : threadIdx.x % kTile;
    if (i0 + r < n_freq && f0 + q < m2) D[(i0 + r) * si + (f0 + q) * se] = st[r][q];
}

// ---------------------------------------------------------------------------
// The sum over frequencies at arbitrary tau values (FourierTransform_tau called with its
// own points): out[j][e] = sum_i exp(-i w_i tau_j) in[i][e], a dense complex product.  The
// uniform grids take the chirp-z form (ft_czt.hip).
// ---------------------------------------------------------------------------
struct TauPoints {
    double w0, dw;
    const double* taus;
    __device__ cd operator()(int j, int i) const  // exp(-i w_i tau_j), the reference's FP64 w*tau
    {
        double s, c;
        sincos((w0 + i * dw) * taus[j], &s, &c);
        return cd{c, -s};
    }
    __device__ cd step4(int j) const  // from i to i + 4
    {
        double s, c;
        sincos(4.0 * dw * taus[j], &s, &c);
        return cd{c, -s};
    }
};

// VALU form, any m2: a workgroup takes TJ consecutive rows j and all elements over its share
// of i, [y*ichunk, min(ni, (y+1)*ichunk)), inputs staged in LDS TI rows at a time; with more
// than one range the results are partial sums, out + y*nj*m2, which k_dft_sum_parts adds in
// range order.
template <int OPT>
__global__ __launch_bounds__(256) void k_dft(int nj, int ni, int m2, int TJ, int TI, int ichunk,
                                             const cd* __restrict__ in, cd* __restrict__ out, TauPoints coef)
{
    extern __shared__ cd sm[];
    cd* sc = sm;            // [TJ][TI]
    cd* sx = sm + TJ * TI;  // [TI][m2]
    const int j0 = blockIdx.x * TJ;
    const int ib = blockIdx.y * ichunk;
    const int ie = min(ni, ib + ichunk);
    out += (size_t)blockIdx.y * nj * m2;
    const int nout = TJ * m2;
    cd acc[OPT];
#pragma unroll
    for (int q = 0; q < OPT; ++q) acc[q] = cd{0, 0};
    for (int i0 = ib; i0 < ie; i0 += TI) {
        __syncthreads();
        for (int t = threadIdx.x; t < TJ * TI; t += 256) {
            const int jj = t / TI, ii = t % TI;
            sc[t] = (j0 + jj < nj && i0 + ii < ie) ? coef(j0 + jj, i0 + ii) : cd{0, 0};
        }
        for (int t = threadIdx.x; t < TI * m2; t += 256) sx[t] = i0 + t / m2 < ie ? in[(size_t)i0 * m2 + t] : cd{0, 0};
        __syncthreads();
#pragma unroll
        for (int q = 0; q < OPT; ++q) {
            const int o = threadIdx.x + q * 256;
            if (o >= nout) break;
            const int jj = o / m2, e = o % m2;
            cd s = acc[q];
            for (int ii = 0; ii < TI; ++ii) s = cfma(sc[jj * TI + ii], sx[ii * m2 + e], s);
            acc[q] = s;
        }
    }
#pragma unroll
    for (int q = 0; q < OPT; ++q) {
        const int o = threadIdx.x + q * 256;
        if (o >= nout) break;
        const int jj = o / m2, e = o % m2;
        if (j0 + jj < nj) out[(size_t)(j0 + jj) * m2 + e] = acc[q];
    }
}

// G(tau_j) = Herm[ (X + X^H)/beta + 1/2 sum_h A_h diag(-1/(e^{e tau} + e^{e (tau-beta)})) A_h^H ]   (:62-90),
// X_j(e) = sum_q X[q*sq + j*sj + e*se] over nq partial sums; with wrap, X_{n_tau} = -X_0 (the
// phase there is e^{-i pi (2n+1)}).  The upper triangle of the tail is the conjugate of the
// lower one, so the result is Hermitian to the last bit.  The 2d exponential factors of a tau
// are formed once per tile (they were 4d exponentials per element: 81 -> 12 us at d = 10,
// N_tau = 8192).
struct FtSums {
    const cd* X;
    int nq;
    size_t sq, sj, se;
    int wrap;  // n_tau, or -1
};

__global__ __launch_bounds__(256) void k_ft_finish(FtSums x, int d, int ntau1, double beta, double tstep,
                                                   const double* __restrict__ taus, const cd* __restrict__ A1,
                                                   const double* __restrict__ e1, const cd* __restrict__ A2,
                                                   const double* __restrict__ e2, cd* __restrict__ out)
{
    __shared__ double sg[2][kTile][33];
    __shared__ cd sp[2][kTile][33], st[kTile][kTile + 1];
    const int m2 = d * d, j0 = blockIdx.x * kTile, f0 = blockIdx.y * kTile;
    for (int t = threadIdx.x; t < kTile * d; t += 256) {
        const int r = t / d, l = t % d;
        const int j = min(j0 + r, ntau1 - 1);
        const double tau = taus ? taus[j] : j * tstep;
        sg[0][r][l] = -1.0 / (exp(e1[l] * tau) + exp(e1[l] * (tau - beta)));
        sg[1][r][l] = -1.0 / (exp(e2[l] * tau) + exp(e2[l] * (tau - beta)));
        const int e = min(f0 + r, m2 - 1), a = e % d, b = e / d, hi = max(a, b), lo = min(a, b);
        sp[0][r][l] = cmulc(A1[hi + l * d], A1[lo + l * d]);
        sp[1][r][l] = cmulc(A2[hi + l * d], A2[lo + l * d]);
    }
    __syncthreads();
    {
        const bool rows = x.sj < x.se;
        const int r = rows ? threadIdx.x % kTile : threadIdx.x / kTile;
        const int q = rows ? threadIdx.x / kTile : threadIdx.x % kTile;
        const int j = j0 + r, e = f0 + q;
        cd v = cd{0.0, 0.0};
        if (j < ntau1 && e < m2) {
            const int a = e % d, b = e / d;
            const bool wr = j == x.wrap;
            const cd* p = x.X + (wr ? 0 : j) * x.sj;
            cd xab = cd{0.0, 0.0}, xba = cd{0.0, 0.0};
            for (int y = 0; y < x.nq; ++y) {
                xab = cadd(xab, p[y * x.sq + (size_t)e * x.se]);
                xba = cadd(xba, p[y * x.sq + (size_t)(b + a * d) * x.se]);
            }
            v = cscale(cadd(xab, cconj(xba)), (wr ? -1.0 : 1.0) / beta);
            cd s = cd{0.0, 0.0};
            for (int l = 0; l < d; ++l) {
                s = cadd(s, cscale(sp[0][q][l], sg[0][r][l]));
                s = cadd(s, cscale(sp[1][q][l], sg[1][r][l]));
            }
            v = cadd(v, cscale(a >= b ? s : cconj(s), 0.5));
            if (a == b) v.y = 0.0;
        }
        st[r][q] = v;
    }
    __syncthreads();
    const int r = threadIdx.x / kTile, q = threadIdx.x % kTile;
    if (j0 + r < ntau1 && f0 + q < m2) out[(size_t)(j0 + r) * m2 + f0 + q] = st[r][q];
}

// G(tau_t), t = 1..n_tau-1, as [e][t] with a zero at t = 0 (the chirp-z input of tau -> iw), and
// G(0), G(beta) to ends: the output may be the input's own buffer; clears the counters of the
// definiteness test that follows
__global__ __launch_bounds__(256) void k_ft_gather_tau(const cd* __restrict__ gt, int m2, int n_tau,
                                                       cd* __restrict__ out, cd* __restrict__ ends,
                                                       int* __restrict__ bad)
{
    __shared__ cd st[kTile][kTile + 1];
    const int i0 = blockIdx.x * kTile, f0 = blockIdx.y * kTile;
    if (i0 == 0 && f0 == 0 && threadIdx.x < 2) bad[threadIdx.x] = 0;
    int r = threadIdx.x / kTile, q = threadIdx.x % kTile;
    if (i0 == 0 && r < 2 && f0 + q < m2) ends[r * m2 + f0 + q] = gt[(r ? (size_t)n_tau * m2 : 0) + f0 + q];
    st[r][q] = (i0 + r > 0 && i0 + r < n_tau && f0 + q < m2) ? gt[(size_t)(i0 + r) * m2 + f0 + q] : cd{0.0, 0.0};
    __syncthreads();
    r = threadIdx.x % kTile;
    q = threadIdx.x / kTile;
    if (i0 + r < n_tau && f0 + q < m2) out[(size_t)(f0 + q) * n_tau + i0 + r] = st[r][q];
}

// FT_t_to_w (:531-547) from the plain sums S = sum_{0<t<n_tau} e^{i w tau_t} G(tau_t): the
// integral of the piecewise linear interpolant is, with theta = w dt and
// alpha = int_0^1 (1-u) e^{i theta u} du,
//   dt [ (sin(theta/2)/(theta/2))^2 S + alpha G(0) - conj(alpha) G(beta) ]
// (e^{i w beta} = -1).  alpha by its Taylor series below theta = 1, where the closed form
// cancels.
struct LinearWeights {
    double sum;  // of S
    cd ends;     // of G(0); -conj of G(beta)
};

__device__ __forceinline__ LinearWeights linear_weights(int n, int n_tau, double dt)
{
    const double th = kPi * (2.0 * n + 1.0) / n_tau;
    const double h = sin(0.5 * th) / (0.5 * th);
    cd al;
    if (th < 1.0) {
        const double t2 = th * th;
        double x = 0.0, y = 0.0;
        for (int p = 9; p >= 0; --p) {  // x = sum (-1)^p th^2p/(2p+2)!,  y = sum (-1)^p th^2p/(2p+3)!
            x = 1.0 - t2 * x / ((2.0 * p + 3.0) * (2.0 * p + 4.0));
            y = 1.0 - t2 * y / ((2.0 * p + 4.0) * (2.0 * p + 5.0));
        }
        al = cd{0.5 * x, th * y / 6.0};
    } else {
        double s, c;
        sincos(th, &s, &c);
        al = cd{(1.0 - c) / (th * th), (th - s) / (th * th)};
    }
    return LinearWeights{h * h * dt, cscale(al, dt)};
}

__device__ __forceinline__ cd linear_total(cd S, const LinearWeights& w, cd g0, cd gbeta)
{
    return csub(cfma(w.ends, g0, cscale(S, w.sum)), cmulc(gbeta, w.ends));
}

__global__ __launch_bounds__(256) void k_ft_w_finish(const cd* __restrict__ parts, int nq, const cd* __restrict__ ends,
                                                     int m2, int n_freq, int n_tau, double dt, cd* __restrict__ fw)
{
    __shared__ cd st[kTile][kTile + 1];
    __shared__ LinearWeights sw[kTile];
    const int n0 = blockIdx.x * kTile, f0 = blockIdx.y * kTile;
    if (threadIdx.x < kTile) sw[threadIdx.x] = linear_weights(n0 + threadIdx.x, n_tau, dt);
    {
        const int r = threadIdx.x % kTile, q = threadIdx.x / kTile;
        cd v = cd{0.0, 0.0};
        if (n0 + r < n_freq && f0 + q < m2)
            for (int y = 0; y < nq; ++y) v = cadd(v, parts[((size_t)y * m2 + f0 + q) * n_freq + n0 + r]);
        st[r][q] = v;
    }
    __syncthreads();
    const int r = threadIdx.x / kTile, q = threadIdx.x % kTile, e = f0 + q;
    if (n0 + r < n_freq && e < m2)
        fw[(size_t)(n0 + r) * m2 + e] = linear_total(st[r][q], sw[r], ends[e], ends[m2 + e]);
}

// The whole tau -> iw transform of a small grid in one launch: four lanes share an entry
// of F(iw_n), each with every fourth tau, the phases e^{i pi (2n+1) t/n_tau} looked up in the
// chirp-z form's table.  The chirp-z form's three launches and two FFTs take 44 us of a call at any
// such size: 64 frequencies x 128 tau 30 us against 44 (d = 1), 36 against 50 (d = 10); 200 x 400 37
// against 45 (d = 1), 42 against 47 (d = 5), 65 against 61 (d = 10); 100 x 1000 59 against 45 (d = 1).
constexpr int kDirectLanes = 4;

__global__ __launch_bounds__(256) void k_ft_tau2w_direct(const cd* __restrict__ gt, int m2, int n_freq, int n_tau,
                                                         double dt, const cd* __restrict__ tab, cd* __restrict__ fw,
                                                         int* __restrict__ bad)
{
    if (blockIdx.x == 0 && threadIdx.x < 2) bad[threadIdx.x] = 0;
    const int part = threadIdx.x % kDirectLanes;
    const size_t o = (size_t)blockIdx.x * (256 / kDirectLanes) + threadIdx.x / kDirectLanes;
    const bool live = o < (size_t)n_freq * m2;
    const int n = live ? (int)(o / m2) : 0, e = live ? (int)(o % m2) : 0;
    const int n2 = 2 * n_tau;
    const long long f = 2 * n + 1;
    int at = (int)(f * (1 + part) % n2);  // of the table, at tau t
    const int step = (int)(f * kDirectLanes % n2);
    cd S = cd{0.0, 0.0};
#pragma unroll 8
    for (int t = 1 + part; t < n_tau; t += kDirectLanes) {
        S = cfma(tab[at], gt[(size_t)t * m2 + e], S);
        at += step;
        if (at >= n2) at -= n2;
    }
#pragma unroll
    for (int x = 1; x < kDirectLanes; x <<= 1) {
        S.x += __shfl_xor(S.x, x);
        S.y += __shfl_xor(S.y, x);
    }
    if (live && part == 0)
        fw[o] = linear_total(S, linear_weights(n, n_tau, dt), gt[e], gt[(size_t)n_tau * m2 + e]);
}

// the sizes that the direct form takes: products in all, and the length of a lane's chain
constexpr double kDirectMax = 5e6;

inline bool tau2w_direct(int n_freq, int n_tau, int m2)
{
    return n_tau <= 512 && (double)n_freq * n_tau * m2 <= kDirectMax;
}

// (F - F^H)/(2i), for the causality test of FT_t_to_w (:552)
__global__ void k_antiherm(const cd* __restrict__ f, int d, int count, cd* __restrict__ out)
{
    const int m2 = d * d;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)count * m2) return;
    const int e = (int)(t % m2), a = e % d, b = e / d;
    const size_t base = t - e;
    const cd x = f[t], y = f[base + b + a * d];
    const cd dlt = cd{x.x - y.x, x.y + y.y};  // x - conj(y)
    out[t] = cd{0.5 * dlt.y, -0.5 * dlt.x};  // dlt / (2i)
}

// parts[y][j][e] -> out[j][e], y ascending
__global__ void k_dft_sum_parts(const cd* __restrict__ parts, int nparts, size_t count, cd* __restrict__ out)
{
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    cd s = parts[t];
    for (int y = 1; y < nparts; ++y) s = cadd(s, parts[(size_t)y * count + t]);
    out[t] = s;
}

// The same sum on the matrix cores (FP64 MFMA), for m2 <= 16 * NE: complex products split
// into real v_mfma_f64_16x16x4 (D = A B + D, A 16 x 4, B 4 x 16).  A wavefront owns 16
// consecutive rows j and every e tile (NE tiles of 16 elements), so each phase factor it
// forms serves NE tiles.  Per step of 4 summed indices, lane l = r + 16 k holds the factor
// (j0 + r, i0 + k), the A operand's (r, k) entry, walked along i by a per-row constant and
// formed again exactly every 16th step (rounding ~1e-15), and loads in[i0 + k][16 t + r], the
// B operand's (k, r) entry of tile t; the accumulator of tile t holds out[j0 + c][16 t + r'] at
// lane r' + 16 (c % 4), register c / 4.  blockIdx.y selects the range of i, as in k_dft.
typedef double dmfma4 __attribute__((ext_vector_type(4)));

template <int NE>
__global__ __launch_bounds__(256) void k_dft_mfma(int nj, int ni, int m2, int ichunk, const cd* __restrict__ in,
                                                  cd* __restrict__ out, TauPoints coef)
{
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, k = lane >> 4;
    const int j0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;
    const int ib = blockIdx.y * ichunk;
    const int ie = min(ni, ib + ichunk);
    out += (size_t)blockIdx.y * nj * m2;
    dmfma4 accR[NE], accI[NE];
#pragma unroll
    for (int t = 0; t < NE; ++t) {
        accR[t] = dmfma4{0.0, 0.0, 0.0, 0.0};
        accI[t] = dmfma4{0.0, 0.0, 0.0, 0.0};
    }
    const int j = j0 + r;
    const bool jok = j < nj;
    const cd m4 = coef.step4(jok ? j : 0);
    cd p = cd{0, 0};
    for (int i0 = ib, step = 0; i0 < ie; i0 += 4, ++step) {
        const int i = i0 + k;
        if ((step & 15) == 0) p = coef(jok ? j : 0, i);
        else p = cmul(p, m4);
        const cd c = (i < ie && jok) ? p : cd{0, 0};
        cd b[NE];
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            const int e = 16 * t + r;
            b[t] = (i < ie && e < m2) ? in[(size_t)i * m2 + e] : cd{0, 0};
        }
        // four passes over the tiles: consecutive MFMAs update different accumulators
        const double ar = c.x, ai = c.y;
#pragma unroll
        for (int t = 0; t < NE; ++t) accR[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, b[t].x, accR[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < NE; ++t) accI[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, b[t].y, accI[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < NE; ++t) accR[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, b[t].y, accR[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < NE; ++t) accI[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, b[t].x, accI[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NE; ++t) {
        const int e = 16 * t + r;
        if (e >= m2) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int jj = j0 + k + 4 * g;
            if (jj < nj) out[(size_t)jj * m2 + e] = cd{accR[t][g], accI[t][g]};
        }
    }
}

struct DftShape {
    int TJ, TI, ks, ichunk;
    bool mfma;
};

// Tiles of the dense sum and the split of the summed index i over workgroups: about 1024
// workgroups.  m2 <= 128 on the matrix cores, rows in tiles of 64 per workgroup (16 per
// wavefront), i split in multiples of 4.
inline DftShape dft_shape(int nj, int ni, int m2)
{
    DftShape d{};
    d.mfma = m2 <= 128;
    if (d.mfma) {
        d.TJ = 64;
        d.TI = 4;
    } else {
        d.TJ = std::max(1, std::min(32, 2048 / m2));
        d.TI = std::max(1, std::min(32, 2048 / m2));
    }
    const int gx = (nj + d.TJ - 1) / d.TJ;
    const int steps = (ni + d.TI - 1) / d.TI;
    const int ks = std::max(1, std::min({(1024 + gx - 1) / gx, steps, d.mfma ? 32 : 16}));
    d.ichunk = (steps + ks - 1) / ks * d.TI;
    d.ks = (ni + d.ichunk - 1) / d.ichunk;
    return d;
}

// scratch (in cd) the split sum needs for its partial sums
inline size_t dft_part_count(int nj, int ni, int m2)
{
    const DftShape d = dft_shape(nj, ni, m2);
    return d.ks > 1 ? (size_t)d.ks * nj * m2 : 0;
}

hipError_t launch_dft(int nj, int ni, int m2, const cd* in, cd* out, TauPoints coef, cd* parts, hipStream_t s)
{
    const DftShape d = dft_shape(nj, ni, m2);
    if (d.ks > 1 && !parts) return hipErrorInvalidValue;
    cd* dst = d.ks > 1 ? parts : out;
    const dim3 grid((nj + d.TJ - 1) / d.TJ, d.ks);
    if (d.mfma) {
#define M_(NE)                                                                                                          if (m2 <= 16 * NE) {                                                                                                    hipLaunchKernelGGL((k_dft_mfma<NE>), grid, dim3(256), 0, s, nj, ni, m2, d.ichunk, in, dst, coef);               } else
        M_(1) M_(2) M_(4) M_(6) M_(7) M_(8) return hipErrorInvalidValue;
#undef M_
    } else {
        const int opt = (d.TJ * m2 + 255) / 256;
        const size_t shm = sizeof(cd) * ((size_t)d.TJ * d.TI + (size_t)d.TI * m2);
#define L_(O)                                                                                                            {                                                                                                                        hipError_t e = hipFuncSetAttribute((const void*)k_dft<O>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);         if (e != hipSuccess) return e;                                                                                       hipLaunchKernelGGL((k_dft<O>), grid, dim3(256), shm, s, nj, ni, m2, d.TJ, d.TI, d.ichunk, in, dst, coef);        }
        if (opt <= 4) L_(4) else L_(8)
#undef L_
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || d.ks == 1) return e;
    const size_t cnt = (size_t)nj * m2;
    hipLaunchKernelGGL(k_dft_sum_parts, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, s, parts, d.ks, cnt, out);
    return hipGetLastError();
}

unsigned nblk(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

#define HIPCHK(expr)                                                                                    \
    do {                                                                                                \
        hipError_t e_ = (expr);                                                                         \
        if (e_ != hipSuccess) return fail(h, DMFTGPU_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

static char* ft_ws(dmftgpu_handle h, size_t bytes, int* rc)
{
    hipError_t e;
    char* p = (char*)h->ft.get(bytes, &e);
    if (!p) *rc = fail(h, DMFTGPU_ERR_HIP, "ft workspace %zu bytes: %s", bytes, hipGetErrorString(e));
    return p;
}

struct Carve {
    char* base;
    size_t off = 0;
    template <class T>
    T* take(size_t count)
    {
        T* p = (T*)(base + off);
        off += (count * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

extern "C" int dmftgpu_moments(dmftgpu_handle h, int d, int n_freq, double beta, const double* fw, int green_asym,
                               double* moments, int* windows)
{
    (void)hipGetLastError();  // drop an error left by an earlier failed call
    if (!h) return DMFTGPU_ERR_ARG;
    if (d < 1 || d > 32) return fail(h, DMFTGPU_ERR_UNSUPPORTED, "d=%d outside 1..32", d);
    if (!fw || !moments) return fail(h, DMFTGPU_ERR_ARG, "fw and moments are required");
    if (!(beta > 0.0)) return fail(h, DMFTGPU_ERR_ARG, "beta=%g", beta);
    const int nm = green_asym ? 2 : 4;
    const int range = (green_asym ? n_freq - 2 : n_freq - 4) + 1;
    int Nv = n_freq / 20;
    if (Nv == 0) Nv = 1;
    const int ncent = range - 2 * Nv;
    // the reference asserts on the window bounds (:321, :440)
    if (range < 1 || ncent < 1) return fail(h, DMFTGPU_ERR_ARG, "n_freq=%d too small for the window search", n_freq);
    const int m2 = d * d;
    // the basis table and the inverted normal matrices depend on (n_freq, beta,
    // green_asym) only: kept in the handle and formed again when those change
    dmftgpu_handle_s::MomEntry* ent = nullptr;
    for (auto& m : h->mom_cache)
        if (m.valid && m.nf == n_freq && m.beta == beta && m.green == green_asym) ent = &m;
    const bool hit = ent != nullptr;
    if (!hit) {  // the least recently used entry (an unused one first)
        ent = &h->mom_cache[0];
        for (auto& m : h->mom_cache)
            if (!m.valid || m.used < ent->used) {
                ent = &m;
                if (!m.valid) break;
            }
    }
    ent->used = ++h->mom_clock;
    hipError_t eg;
    char* kbase = (char*)ent->buf.get((size_t)n_freq * sizeof(double4) + 256 + (size_t)range * 16 * 8, &eg);
    if (!kbase) return fail(h, DMFTGPU_ERR_HIP, "moment cache: %s", hipGetErrorString(eg));
    double4* tab = (double4*)kbase;
    double* kinv = (double*)(kbase + ((size_t)n_freq * sizeof(double4) + 255) / 256 * 256);
    size_t need = (size_t)nm * range * m2 * 16 + (size_t)nm * range * 8 +
                  (size_t)nm * ncent * m2 * 16 + (size_t)ncent * m2 * 16 * 3 + (size_t)ncent * d * 8 * 2 + 64 * 256;
    int rc = 0;
    char* base = ft_ws(h, need, &rc);
    if (!base) return rc;
    Carve cv{base};
    cd* mt = cv.take<cd>((size_t)nm * range * m2);
    double* trace = cv.take<double>((size_t)nm * range);
    cd* avg = cv.take<cd>((size_t)nm * ncent * m2);
    double* w1 = cv.take<double>((size_t)ncent * d);
    cd* U1 = cv.take<cd>((size_t)ncent * m2);
    cd* T = cv.take<cd>((size_t)ncent * m2);
    double* wT = cv.take<double>((size_t)ncent * d);
    int* cen = cv.take<int>(4);
    hipStream_t s = h->stream;
    if (!hit) {
        ent->valid = false;
        std::vector<double4> htab(n_freq);
        for (int wn = 0; wn < n_freq; ++wn) {
            const double z = (2 * wn + 1) * kPi / beta;  // (:224, :364)
            htab[wn] = double4{-1. / std::pow(z, 1), -1. / std::pow(z, 2), 1. / std::pow(z, 3), 1.0 / z};
        }
        HIPCHK(hipMemcpyAsync(tab, htab.data(), sizeof(double4) * n_freq, hipMemcpyHostToDevice, s));
        HIPCHK(hipStreamSynchronize(s));  // htab is a host temporary
        const int npair = green_asym ? 3 : 10;
        hipLaunchKernelGGL(k_mom_ktk, dim3(nblk((size_t)range * npair)), dim3(256), 0, s, n_freq, range, green_asym, tab,
                           kinv);
        HIPCHK(hipGetLastError());
        hipLaunchKernelGGL(k_mom_kinv, dim3(nblk(range)), dim3(256), 0, s, range, green_asym, kinv);
        HIPCHK(hipGetLastError());
        ent->valid = true;
        ent->nf = n_freq;
        ent->beta = beta;
        ent->green = green_asym;
    }
    const size_t fits = (size_t)range * (d * (d + 1) / 2);
    const bool all = fits >= kFitAll;
    const dim3 gfit((unsigned)((fits + 63) / 64), all ? 1 : nm);
    auto fit = green_asym ? all ? k_mom_fit<true, 2> : k_mom_fit<true, 1> : all ? k_mom_fit<false, 4> : k_mom_fit<false, 1>;
    hipLaunchKernelGGL(fit, gfit, dim3(64), 0, s, (const cd*)fw, d, n_freq, range, (const double*)tab, kinv, mt);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_mom_trace, dim3(nblk((size_t)range * nm)), dim3(256), 0, s, mt, d, range, nm, trace);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_mom_avg, dim3(nblk((size_t)nm * ncent * m2)), dim3(256), 0, s, mt, m2, range, nm, Nv, avg);
    HIPCHK(hipGetLastError());
    if (!green_asym) HIPCHK(dg::launch_herm_eig(avg + (size_t)1 * ncent * m2, d, 0, d, nullptr, 0, w1, U1, ncent, s));
    const int pshm = (int)(4 * (size_t)m2 * sizeof(cd));
    HIPCHK(hipFuncSetAttribute((const void*)k_mom_posmat, hipFuncAttributeMaxDynamicSharedMemorySize, pshm));
    hipLaunchKernelGGL(k_mom_posmat, dim3(ncent), dim3(64), pshm, s, avg, d, ncent, green_asym, w1, U1, T);
    HIPCHK(hipGetLastError());
    HIPCHK(dg::launch_herm_eig(T, d, 0, d, nullptr, 0, wT, nullptr, ncent, s));
    // window choice and final moments on the device: no host round trip
    cd* dm = (cd*)moments;
    hipLaunchKernelGGL(k_mom_init, dim3(nblk((size_t)4 * m2)), dim3(256), 0, s, dm, d, green_asym, cen);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_mom_select, dim3(nm), dim3(kSelThreads), 0, s, trace, w1, wT, d, range, ncent, Nv, green_asym, cen);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_mom_final, dim3(nblk(m2), nm), dim3(256), 0, s, mt, d, range, green_asym, cen, Nv, dm);
    HIPCHK(hipGetLastError());
    if (windows) {  // the only wait of the call
        int win[4];
        HIPCHK(hipMemcpyAsync(win, cen, sizeof(win), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        std::memcpy(windows, win, sizeof(win));
    }
    return DMFTGPU_OK;
}

// Two-pole tail set-up of FourierTransform_tau (:22-44): returns V^H U_h and eig values e_h.
static void tail_setup(int d, const std::vector<hl::cx>& m1, const std::vector<hl::cx>& m2, const std::vector<hl::cx>& m3,
                       std::vector<hl::cx>& A1, std::vector<double>& e1, std::vector<hl::cx>& A2, std::vector<double>& e2)
{
    using namespace hl;
    Mat V = zeros(d), H1 = zeros(d), H2 = zeros(d);
    std::vector<double> w;
    Mat Q;
    eigh(d, m1, w, Q);
    if (w[0] > 0) {
        V = herm_func(d, w, Q, [](double x) { return std::sqrt(x > 0 ? x : 0.0); });
        Mat Vi, ViH;
        inverse(d, V, Vi);
        inverse(d, adj(d, V), ViH);
        Mat M2 = mul(d, mul(d, ViH, lin(m2, 2.0, m2, 0.0)), Vi);
        Mat M3 = mul(d, mul(d, ViH, lin(m3, 2.0, m3, 0.0)), Vi);
        Mat X = lin(M3, 0.5, mul(d, M2, M2), -0.25);
        eigh(d, X, w, Q);
        if (w[0] > 0) {
            Mat sq = herm_func(d, w, Q, [](double x) { return std::sqrt(x > 0 ? x : 0.0); });
            H1 = lin(M2, 0.5, sq, 1.0);
        } else {
            H1 = lin(M2, 0.5, M2, 0.0);
        }
        H2 = lin(M2, 1.0, H1, -1.0);
    }
    Mat U;
    Mat VH = adj(d, V);
    eigh(d, H1, e1, U);
    A1 = mul(d, VH, U);
    eigh(d, H2, e2, U);
    A2 = mul(d, VH, U);
}

// The two-pole tail on the device, one copy from host, which the caller keeps until it has
// waited for the stream
struct TailDev {
    std::vector<double> host;
    const cd *A1, *A2;
    const double *e1, *e2;
};

static TailDev tail_upload(dmftgpu_handle h, int d, const std::vector<hl::cx>& A1, const std::vector<double>& e1,
                           const std::vector<hl::cx>& A2, const std::vector<double>& e2, Carve& cv, int* rc)
{
    const size_t m2 = (size_t)d * d;
    TailDev t;
    t.host.resize(4 * m2 + 2 * d);
    double* dev = cv.take<double>(t.host.size());
    auto put = [&](size_t at, const void* src, size_t count) {
        std::memcpy(t.host.data() + at, src, sizeof(double) * count);
        return dev + at;
    };
    t.A1 = (const cd*)put(0, A1.data(), 2 * m2);
    t.A2 = (const cd*)put(2 * m2, A2.data(), 2 * m2);
    t.e1 = put(4 * m2, e1.data(), d);
    t.e2 = put(4 * m2 + d, e2.data(), d);
    const hipError_t e =
        hipMemcpyAsync(dev, t.host.data(), sizeof(double) * t.host.size(), hipMemcpyHostToDevice, h->stream);
    if (e != hipSuccess) *rc = fail(h, DMFTGPU_ERR_HIP, "tail upload: %s", hipGetErrorString(e));
    return t;
}

// Tables of the chirp-z form for n_tau, kept in the handle for the last n_tau
static const cd* czt_tables(dmftgpu_handle h, int n_tau, int* rc)
{
    hipError_t e;
    if (h->czt_n != n_tau) {
        h->czt_n = 0;
        cd* t = (cd*)h->czt.get(dg::czt_table_count(n_tau) * sizeof(cd), &e);
        if (t) e = dg::launch_czt_tables(n_tau, t, h->stream);
        if (e != hipSuccess) {
            *rc = fail(h, DMFTGPU_ERR_HIP, "transform tables: %s", hipGetErrorString(e));
            return nullptr;
        }
        h->czt_n = n_tau;
    }
    return (const cd*)h->czt.ptr;
}

extern "C" int dmftgpu_ft_w2tau(dmftgpu_handle h, int d, int n_freq, int n_tau, double beta, const double* fw,
                                const double* moments, double* gtau, int* patched)
{
    (void)hipGetLastError();  // drop an error left by an earlier failed call
    if (!h) return DMFTGPU_ERR_ARG;
    if (d < 1 || d > 32) return fail(h, DMFTGPU_ERR_UNSUPPORTED, "d=%d outside 1..32", d);
    if (!fw || !moments || !gtau) return fail(h, DMFTGPU_ERR_ARG, "fw, moments and gtau are required");
    if (n_freq < 1 || n_tau < 1 || !(beta > 0.0)) return fail(h, DMFTGPU_ERR_ARG, "n_freq=%d n_tau=%d beta=%g", n_freq, n_tau, beta);
    const int m2 = d * d, ntau1 = n_tau + 1;
    hipStream_t s = h->stream;
    std::vector<hl::cx> hm(4 * (size_t)m2);
    HIPCHK(hipMemcpyAsync(hm.data(), moments, sizeof(cd) * 4 * m2, hipMemcpyDefault, s));
    HIPCHK(hipStreamSynchronize(s));
    std::vector<hl::cx> m1(hm.begin() + m2, hm.begin() + 2 * m2), mm2(hm.begin() + 2 * m2, hm.begin() + 3 * m2),
        m3(hm.begin() + 3 * m2, hm.begin() + 4 * m2);
    std::vector<hl::cx> A1, A2;
    std::vector<double> e1, e2;
    tail_setup(d, m1, mm2, m3, A1, e1, A2, e2);
    const dg::CztPlan cp = dg::czt_plan(n_tau, n_freq, n_tau, m2);
    const size_t npart = (size_t)cp.in_groups * m2 * n_tau;
    size_t need = (size_t)n_freq * m2 * 16 + 4 * (size_t)m2 * 16 + 4 * (size_t)d * 8 +
                  (size_t)ntau1 * d * 8 + npart * 16 + 16 * 256;
    int rc = 0;
    char* base = ft_ws(h, need, &rc);
    if (!base) return rc;
    Carve cv{base};
    cd* D = cv.take<cd>((size_t)n_freq * m2);
    cd* parts = cv.take<cd>(npart);
    const TailDev tl = tail_upload(h, d, A1, e1, A2, e2, cv, &rc);
    if (rc) return rc;
    double* wmin = cv.take<double>((size_t)ntau1 * d);
    int* bad = cv.take<int>(1);
    const dim3 gf((n_freq + kTile - 1) / kTile, (m2 + kTile - 1) / kTile);
    const cd* tab = czt_tables(h, n_tau, &rc);
    if (!tab) return rc;
    hipLaunchKernelGGL(k_ft_subtract_tail, gf, dim3(256), 0, s, (const cd*)fw, d, n_freq, beta, tl.A1, tl.e1, tl.A2, tl.e2,
                       D, (size_t)1, (size_t)n_freq, bad);
    HIPCHK(hipGetLastError());
    HIPCHK(dg::launch_czt(cp, false, m2, tab, D, parts, s));
    const FtSums xs{parts, cp.in_groups, (size_t)m2 * n_tau, 1, (size_t)n_tau, n_tau};
    cd* out = (cd*)gtau;
    hipLaunchKernelGGL(k_ft_finish, dim3((ntau1 + kTile - 1) / kTile, (m2 + kTile - 1) / kTile), dim3(256), 0, s, xs, d,
                       ntau1, beta, beta / n_tau, (const double*)nullptr, tl.A1, tl.e1, tl.A2, tl.e2, out);
    HIPCHK(hipGetLastError());
    // causality patch (:145-175): it acts where the smallest eigenvalue of G(tau_j) is not
    // negative.  G(tau_j) negative definite by a margin for every j settles that there is nothing
    // to do; otherwise the eigenvalues decide
    HIPCHK(dg::launch_not_posdef(out, d, ntau1, false, bad, s));
    int hbad = 0;
    HIPCHK(hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    std::vector<double> hw;
    bool any = false;
    if (hbad) {
        HIPCHK(dg::launch_herm_eig(out, d, 0, d, nullptr, 0, wmin, nullptr, ntau1, s));
        hw.resize((size_t)ntau1 * d);
        HIPCHK(hipMemcpyAsync(hw.data(), wmin, sizeof(double) * hw.size(), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        for (int t = 0; t <= n_tau; ++t) any |= hw[(size_t)t * d] >= 0;
    }
    int check = 0;
    if (any) {  // rare path: restate the reference loop on the host
        std::vector<hl::cx> g((size_t)ntau1 * m2);
        HIPCHK(hipMemcpyAsync(g.data(), out, sizeof(cd) * g.size(), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        double mine11 = 0.0;
        for (int t = 0; t < ntau1; ++t) {
            const double tau = t * beta / n_tau;
            const double mine = hw[(size_t)t * d];
            mine11 = mine;
            if (mine >= 0 && (t != 0 && t != n_tau)) {
                check = 1;
                for (int t1 = t + 1; t1 < ntau1; ++t1) {
                    const double tau1 = t1 * beta / n_tau, taup = (t - 1) * beta / n_tau;
                    for (int e = 0; e < m2; ++e)
                        g[(size_t)t * m2 + e] = (g[(size_t)t1 * m2 + e] - g[(size_t)(t - 1) * m2 + e]) / (tau1 - taup) *
                                                    (tau - taup) + g[(size_t)(t - 1) * m2 + e];
                    hl::Mat gm(g.begin() + (size_t)t * m2, g.begin() + (size_t)(t + 1) * m2);
                    mine11 = hl::min_eig(d, gm);
                    if (mine11 < 0) break;
                }
            }
            if (mine11 >= 0) {
                check = 1;
                for (int e = 0; e < m2; ++e) g[(size_t)t * m2 + e] = 0.0;
                for (int l = 0; l < d; ++l) g[(size_t)t * m2 + l + (size_t)l * d] = -1e-10;
            }
        }
        HIPCHK(hipMemcpyAsync(out, g.data(), sizeof(cd) * g.size(), hipMemcpyHostToDevice, s));
        HIPCHK(hipStreamSynchronize(s));
    }
    if (patched) *patched = check;
    return DMFTGPU_OK;
}

extern "C" int dmftgpu_ft_tau2w(dmftgpu_handle h, int d, int n_freq, int n_tau, double beta, const double* gtau,
                                double* fw, int* violations)
{
    (void)hipGetLastError();  // drop an error left by an earlier failed call
    if (!h) return DMFTGPU_ERR_ARG;
    if (d < 1 || d > 32) return fail(h, DMFTGPU_ERR_UNSUPPORTED, "d=%d outside 1..32", d);
    if (!gtau || !fw) return fail(h, DMFTGPU_ERR_ARG, "gtau and fw are required");
    if (n_freq < 1 || n_tau < 1 || !(beta > 0.0)) return fail(h, DMFTGPU_ERR_ARG, "n_freq=%d n_tau=%d beta=%g", n_freq, n_tau, beta);
    const int m2 = d * d;
    const double dt = beta / n_tau;
    hipStream_t s = h->stream;
    // the direct form reads gtau while it writes fw
    const cd *g0 = (const cd*)gtau, *g1 = g0 + (size_t)(n_tau + 1) * m2;
    const bool apart = (const cd*)fw >= g1 || (const cd*)fw + (size_t)n_freq * m2 <= g0;
    const bool direct = apart && tau2w_direct(n_freq, n_tau, m2);
    const dg::CztPlan cp = dg::czt_plan(n_tau, n_tau, n_freq, m2);
    const size_t npart = direct ? 0 : (size_t)cp.in_groups * m2 * n_freq, ngin = direct ? 0 : (size_t)n_tau * m2;
    size_t need = (ngin + npart + 2 * m2 + (size_t)n_freq * m2) * 16 + (size_t)n_freq * d * 8 + 9 * 256;
    int rc = 0;
    char* base = ft_ws(h, need, &rc);
    if (!base) return rc;
    Carve cv{base};
    cd* gin = cv.take<cd>(ngin);
    cd* ends = cv.take<cd>(2 * (size_t)m2);
    cd* ah = cv.take<cd>((size_t)n_freq * m2);
    double* wmax = cv.take<double>((size_t)n_freq * d);
    int* bad = cv.take<int>(2);
    cd* parts = cv.take<cd>(npart);
    const cd* tab = czt_tables(h, n_tau, &rc);
    if (!tab) return rc;
    if (direct) {
        hipLaunchKernelGGL(k_ft_tau2w_direct, dim3(nblk((size_t)n_freq * m2 * kDirectLanes)), dim3(256), 0, s, g0, m2,
                           n_freq, n_tau, dt, tab, (cd*)fw, bad);
    } else {
        hipLaunchKernelGGL(k_ft_gather_tau, dim3((n_tau + kTile - 1) / kTile, (m2 + kTile - 1) / kTile), dim3(256), 0, s,
                           g0, m2, n_tau, gin, ends, bad);
        HIPCHK(hipGetLastError());
        HIPCHK(dg::launch_czt(cp, true, m2, tab, gin, parts, s));
        hipLaunchKernelGGL(k_ft_w_finish, dim3((n_freq + kTile - 1) / kTile, (m2 + kTile - 1) / kTile), dim3(256), 0, s,
                           parts, cp.in_groups, ends, m2, n_freq, n_tau, dt, (cd*)fw);
    }
    HIPCHK(hipGetLastError());
    // causality test (:551-558): a frequency violates it where (F - F^H)/2i has a positive
    // eigenvalue.  The elimination settles that for all but the matrices with an eigenvalue
    // within rounding of zero; with one of those the eigenvalues are counted
    HIPCHK(dg::launch_not_posdef((const cd*)fw, d, n_freq, true, bad, s));
    int hbad[2] = {0, 0};
    HIPCHK(hipMemcpyAsync(hbad, bad, sizeof(hbad), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (!hbad[0]) {
        if (violations) *violations = hbad[1];
        return DMFTGPU_OK;
    }
    hipLaunchKernelGGL(k_antiherm, dim3(nblk((size_t)n_freq * m2)), dim3(256), 0, s, (const cd*)fw, d, n_freq, ah);
    HIPCHK(hipGetLastError());
    HIPCHK(dg::launch_herm_eig(ah, d, 0, d, nullptr, 0, wmax, nullptr, n_freq, s));
    std::vector<double> hw((size_t)n_freq * d);
    HIPCHK(hipMemcpyAsync(hw.data(), wmax, sizeof(double) * hw.size(), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    int viol = 0;
    for (int n = 0; n < n_freq; ++n) viol += hw[(size_t)n * d + d - 1] > 0;
    if (violations) *violations = viol;
    return DMFTGPU_OK;
}


// FourierTransform_tau (FourierTransform.cpp:16-118) at arbitrary tau values
// (no causality patch: the single-tau overloads of FourierTransform have none).
extern "C" int dmftgpu_ft_w2tau_points(dmftgpu_handle h, int d, int n_freq, double beta, const double* fw,
                                       const double* moments, int n_points, const double* taus_host, double* out)
{
    (void)hipGetLastError();  // drop an error left by an earlier failed call
    if (!h) return DMFTGPU_ERR_ARG;
    if (d < 1 || d > 32) return fail(h, DMFTGPU_ERR_UNSUPPORTED, "d=%d outside 1..32", d);
    if (!fw || !moments || !out || !taus_host || n_points < 1 || n_freq < 1 || !(beta > 0.0))
        return fail(h, DMFTGPU_ERR_ARG, "bad arguments to ft_w2tau_points");
    const int m2 = d * d;
    hipStream_t s = h->stream;
    std::vector<hl::cx> hm(4 * (size_t)m2);
    HIPCHK(hipMemcpyAsync(hm.data(), moments, sizeof(cd) * 4 * m2, hipMemcpyDefault, s));
    HIPCHK(hipStreamSynchronize(s));
    std::vector<hl::cx> m1(hm.begin() + m2, hm.begin() + 2 * m2), mm2(hm.begin() + 2 * m2, hm.begin() + 3 * m2),
        m3(hm.begin() + 3 * m2, hm.begin() + 4 * m2);
    std::vector<hl::cx> A1, A2;
    std::vector<double> e1, e2;
    tail_setup(d, m1, mm2, m3, A1, e1, A2, e2);
    const size_t npart = dft_part_count(n_points, n_freq, m2);
    size_t need = (size_t)n_freq * m2 * 16 + (size_t)n_points * m2 * 16 + 4 * (size_t)m2 * 16 + 4 * (size_t)d * 8 +
                  (size_t)n_points * 8 + npart * 16 + 16 * 256;
    int rc = 0;
    char* base = ft_ws(h, need, &rc);
    if (!base) return rc;
    Carve cv{base};
    cd* D = cv.take<cd>((size_t)n_freq * m2);
    cd* X = cv.take<cd>((size_t)n_points * m2);
    cd* parts = npart ? cv.take<cd>(npart) : nullptr;
    const TailDev tl = tail_upload(h, d, A1, e1, A2, e2, cv, &rc);
    if (rc) return rc;
    double* dtau = cv.take<double>(n_points);
    HIPCHK(hipMemcpyAsync(dtau, taus_host, sizeof(double) * n_points, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_ft_subtract_tail, dim3((n_freq + kTile - 1) / kTile, (m2 + kTile - 1) / kTile), dim3(256), 0, s,
                       (const cd*)fw, d, n_freq, beta, tl.A1, tl.e1, tl.A2, tl.e2, D, (size_t)m2, (size_t)1, (int*)nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(launch_dft(n_points, n_freq, m2, D, X, TauPoints{kPi / beta, (2 * kPi) / beta, dtau}, parts, s));
    hipLaunchKernelGGL(k_ft_finish, dim3((n_points + kTile - 1) / kTile, (m2 + kTile - 1) / kTile), dim3(256), 0, s,
                       FtSums{X, 1, 0, (size_t)m2, 1, -1}, d, n_points, beta, 0.0, (const double*)dtau, tl.A1, tl.e1, tl.A2,
                       tl.e2, (cd*)out);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s));
    return DMFTGPU_OK;
}
