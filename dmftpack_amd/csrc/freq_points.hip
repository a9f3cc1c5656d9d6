// Frequency points of the density sums (NumMatrix, N, dN/dmu, densityMatDFT).
//
// GreenFtn_w and GiwToNele sum over high_freq * N_freq Matsubara frequencies, and
// beyond N_freq Sigma is its moment expansion (GreenFtn.cpp:224-240), so there the
// summand f(w) (entries of G_cc, tr G, tr G^2) is an analytic function of w.  Its
// sum over a run of frequencies w_a..w_b with w_b <= 2 w_a is taken by the Gauss
// rule of the discrete measure itself: 16 points and positive weights that
// integrate every polynomial in u = 1/w of degree <= 31 over that set exactly.
//
// Error: f is analytic where A(w) = (iw + mu) - H - P Sigma(w) P^H is invertible.
// On the Bernstein ellipse rho = 4.5 around [1/w_b, 1/w_a] both Re w and |w| are
// >= 0.746 w_a =: r, and the Hermitian part of -iA is >= r - s there, with s a bound
// of |Sigma - Herm m0| (H and mu drop out: H is Hermitian).  k_freq_points takes
// the rule only if s <= r/2, from the moments' Frobenius norms; then
// |G| <= 2/r on the ellipse and the rule is off by <= 4.3 |f| rho^-32 < 1e-20 of
// the sum, far below the rounding of adding the terms one by one.  Otherwise (short
// grids at low temperature, moments that are not finite) every frequency is a point
// with weight 1, as it is for a run of at most kGaussMin frequencies.
//
// What it gives: the kernels solve N_freq + 16 frequencies instead of 2 N_freq.
// The plain method keeps every frequency (the reference's algorithm as it stands).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "lattice_kernels.hpp"

namespace dg {

namespace {

// Gauss rule of the measure with unit mass at each t_n = 1/(2n+1), n0 <= n < n1:
// x[i] = 1/node (a real-valued "2n+1"), w[i] its weight.  Stieltjes recurrence to the
// 16 x 16 Jacobi matrix; its eigenvalues, all at once, by bisection on Sturm counts
// (Barth, Martin and Wilkinson, Numer. Math. 9, 386 (1967)); the weights are the
// Christoffel numbers len / sum_k p_k(node)^2 (Golub and Welsch, Math. Comp. 23, 221
// (1969)).  The sums over the measure take 8 partial sums, which vectorise: about 70 us of
// host time at 2048 frequencies, 20 at 64 (freq_tail keeps the rules).
void gauss_rule(int n0, int n1, double* x, double* w)
{
    constexpr int m = kGaussPoints, V = 8;
    const int len = n1 - n0, lv = (len + V - 1) / V * V;
    const double hi = 1.0 / (2.0 * n0 + 1.0), lo = 1.0 / (2.0 * (n1 - 1) + 1.0);
    std::vector<double> s(lv, 0.0), p0(lv, 0.0), p1(lv, 0.0);
    for (int i = 0; i < len; ++i) {
        // (2 t - lo - hi)/(hi - lo) as differences of t, which do not cancel at the ends
        const double t = 1.0 / (2.0 * (n0 + i) + 1.0);
        s[i] = ((t - lo) - (hi - t)) / (hi - lo);
        p1[i] = 1.0 / std::sqrt((double)len);
    }
    double d[m], e[m], beta = 0.0;
    for (int k = 0; k < m; ++k) {
        double sa[V] = {}, sn[V] = {};
        for (int i = 0; i < lv; i += V)
            for (int v = 0; v < V; ++v) sa[v] += s[i + v] * p1[i + v] * p1[i + v];
        const double al = ((sa[0] + sa[1]) + (sa[2] + sa[3])) + ((sa[4] + sa[5]) + (sa[6] + sa[7]));
        for (int i = 0; i < lv; i += V)
            for (int v = 0; v < V; ++v) {
                const double q = (s[i + v] - al) * p1[i + v] - beta * p0[i + v];
                p0[i + v] = p1[i + v];
                p1[i + v] = q;
                sn[v] += q * q;
            }
        beta = std::sqrt(((sn[0] + sn[1]) + (sn[2] + sn[3])) + ((sn[4] + sn[5]) + (sn[6] + sn[7])));
        for (int i = 0; i < lv; ++i) p1[i] /= beta;
        d[k] = al;
        e[k] = beta;
    }
    double lower[m], upper[m];  // node j has j eigenvalues above it
    for (int j = 0; j < m; ++j) {
        lower[j] = -1.0;
        upper[j] = 1.0;
    }
    for (int it = 0; it < 54; ++it) {
        double mid[m], q[m], above[m];
        for (int j = 0; j < m; ++j) {
            mid[j] = 0.5 * (lower[j] + upper[j]);
            q[j] = d[0] - mid[j];
            above[j] = q[j] > 0.0 ? 1.0 : 0.0;
        }
        for (int k = 1; k < m; ++k)
            for (int j = 0; j < m; ++j) {  // pivots of T - mid; a zero one passes as +-infinity
                q[j] = d[k] - mid[j] - e[k - 1] * e[k - 1] / q[j];
                above[j] += q[j] > 0.0 ? 1.0 : 0.0;
            }
        for (int j = 0; j < m; ++j) {
            const bool right = above[j] > j;
            lower[j] = right ? mid[j] : lower[j];
            upper[j] = right ? upper[j] : mid[j];
        }
    }
    for (int j = 0; j < m; ++j) {
        const double node = 0.5 * (lower[j] + upper[j]);
        double pa = 0.0, pb = 1.0, sum = 1.0;
        for (int k = 0; k + 1 < m; ++k) {
            const double pc = ((node - d[k]) * pb - (k ? e[k - 1] : 0.0) * pa) / e[k];
            pa = pb;
            pb = pc;
            sum += pc * pc;
        }
        x[j] = 2.0 / (node * (hi - lo) + hi + lo);
        w[j] = len / sum;
    }
}

// The point table: the first n_freq Matsubara frequencies, then the Gauss points (rule) or the
// remaining frequencies; n_pts, pt_w, pt_wt as in LatArgs.  The rule comes as a kernel
// argument, tail points t0 .. t0 + kTailBlock - 1: no device copy that a stream would have to wait
// for.  Every workgroup forms the decision, of 4 n_c^2 entries, and writes its 256 points (one
// workgroup for the whole table took 12 us at 16384 points, a third of preparing a lattice of
// 64 k; 3 to 4 us now).
constexpr int kTailBlock = 64;
struct TailBlock {
    double x[kTailBlock], w[kTailBlock];
};

__global__ __launch_bounds__(256) void k_freq_points(const cd* __restrict__ mom, int nc, int n_freq, int nw_tot,
                                                     int n_tail, TailBlock tail, int t0, double beta,
                                                     int* __restrict__ n_pts, double* __restrict__ pt_w,
                                                     double* __restrict__ pt_wt)
{
    __shared__ double red[4][4];
    const int m2 = nc * nc, t = threadIdx.x;
    double nrm[4] = {0.0, 0.0, 0.0, 0.0};
    for (int e = t; e < m2; e += 256) {
        const cd a = mom[e], b = mom[e / nc + (e % nc) * nc];
        const double ax = 0.5 * (a.x - b.x), ay = 0.5 * (a.y + b.y);  // anti-Hermitian part of m0
        nrm[0] += ax * ax + ay * ay;
        for (int q = 1; q < 4; ++q) {
            const cd m = mom[(size_t)q * m2 + e];
            nrm[q] += m.x * m.x + m.y * m.y;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) nrm[q] += __shfl_xor(nrm[q], o);
        if ((t & 63) == 0) red[q][t >> 6] = nrm[q];
    }
    __syncthreads();
    for (int q = 0; q < 4; ++q) nrm[q] = (red[q][0] + red[q][1]) + (red[q][2] + red[q][3]);
    const double r = 0.746 * matsubara(n_freq, beta), ir = 1.0 / r;
    const double s = sqrt(nrm[0]) + ir * (sqrt(nrm[1]) + ir * (sqrt(nrm[2]) + ir * sqrt(nrm[3])));
    const bool rule = n_tail > 0 && s <= 0.5 * r;  // false for NaN
    const int np = rule ? n_freq + n_tail : nw_tot;
    // t0 = 0: the table from 0, with the first tail points; else tail points alone
    const int i = (t0 ? n_freq + t0 : 0) + blockIdx.x * 256 + t, q = i - n_freq - t0;
    if (t0 == 0 && i == 0) *n_pts = np;
    if (i >= np) return;
    if (rule && i >= n_freq) {
        if (q < kTailBlock) {
            pt_w[i] = kPi * tail.x[q] / beta;
            pt_wt[i] = tail.w[q];
        }
    } else if (t0 == 0) {
        pt_w[i] = matsubara(i, beta);
        pt_wt[i] = 1.0;
    }
}

std::vector<double> form_tail(int n_freq, int nw_tot)
{
    std::vector<double> x, w;
    bool any = false;
    for (int a = n_freq; a < nw_tot;) {
        // w_b <= 2 w_a holds up to n = 2a; runs of at most kGaussMin are listed as they are
        const int b = nw_tot - a <= a ? nw_tot : 2 * a;
        if (b - a > kGaussMin) {
            x.resize(x.size() + kGaussPoints);
            w.resize(w.size() + kGaussPoints);
            gauss_rule(a, b, x.data() + x.size() - kGaussPoints, w.data() + w.size() - kGaussPoints);
            any = true;
        } else {
            for (int n = a; n < b; ++n) {
                x.push_back(2.0 * n + 1.0);
                w.push_back(1.0);
            }
        }
        a = b;
    }
    if (!any) return {};
    x.insert(x.end(), w.begin(), w.end());
    return x;
}

}  // namespace

FreqTail freq_tail(int n_freq, int nw_tot)
{
    // The last kKept rules formed, for every handle of the process: each is some tens of us of
    // host time (12 lattices on one grid formed it 12 times: creating their batch took 2.41 ms, from
    // 2.11 without a rule) and at most a few hundred doubles.
    struct Kept {
        int n_freq, nw_tot;
        FreqTail tail;
    };
    constexpr size_t kKept = 16;
    static std::mutex lock;
    static std::vector<Kept> kept;  // most recent first
    {
        std::lock_guard<std::mutex> lk(lock);
        for (size_t q = 0; q < kept.size(); ++q)
            if (kept[q].n_freq == n_freq && kept[q].nw_tot == nw_tot) {
                std::rotate(kept.begin(), kept.begin() + q, kept.begin() + q + 1);
                return kept[0].tail;
            }
    }
    FreqTail t = std::make_shared<const std::vector<double>>(form_tail(n_freq, nw_tot));
    std::lock_guard<std::mutex> lk(lock);
    if (kept.size() == kKept) kept.pop_back();
    kept.insert(kept.begin(), Kept{n_freq, nw_tot, t});
    return t;
}

hipError_t launch_freq_points(const cd* mom, int nc, int n_freq, int nw_tot, const std::vector<double>& tail,
                              double beta, int* n_pts, double* pt_w, double* pt_wt, hipStream_t s)
{
    const int n_tail = (int)tail.size() / 2;
    for (int t0 = 0; t0 == 0 || t0 < n_tail; t0 += kTailBlock) {
        TailBlock b{};
        const int count = std::min(kTailBlock, n_tail - t0);
        std::copy_n(tail.data() + t0, count, b.x);
        std::copy_n(tail.data() + n_tail + t0, count, b.w);
        hipLaunchKernelGGL(k_freq_points, dim3(t0 ? 1 : (nw_tot + 255) / 256), dim3(256), 0, s, mom, nc, n_freq, nw_tot,
                           n_tail, b, t0, beta, n_pts, pt_w, pt_wt);
    }
    return hipGetLastError();
}

}  // namespace dg
