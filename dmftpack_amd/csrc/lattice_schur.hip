// Schur-complement lattice path, host side: dispatch of the one-matrix-per-lane
// kernels (lattice_schur_lane.hpp, instantiated per n_c in lattice_lane{1..6}.hip)
// and of the column-per-lane kernels (lattice_schur_cols.hpp), the Sigma table,
// and the per-k preparation (W = H_cd V_d, the per-k blocks).
#include "lattice_kernels.hpp"

namespace dg {

// -------------------------------------------------------------------------
// n_c <= 6: one matrix per lane (this file) or, on request, column per lane;
// 7..16: column per lane (lattice_schur_cols.hpp, buckets 4/5/6/8/10/12/16)
bool schur_supported(int n, int nc) { return nc >= 1 && nc <= 16 && n >= nc && n <= 32; }
bool schur_multi_supported(int nc) { return nc >= 1 && nc <= 6; }
static int cols_bucket(int nc)
{
    return nc <= 4 ? 4 : nc <= 6 ? nc : nc <= 8 ? 8 : nc <= 10 ? 10 : nc <= 12 ? 12 : 16;
}
int schur_slots(int nc, bool cols)
{
    if (nc <= 6 && !cols) return 64;
    return 64 / cols_bucket(nc);  // one wavefront of 64/N slots per workgroup
}

static hipError_t dispatch_nc(const LatArgs& a, int mode, const cd* sig_all, hipStream_t s, int wg,
                              const SchurMulti* m)
{
    switch (a.nc) {
        case 1: return launch_lane_1(a, mode, sig_all, s, wg, m);
        case 2: return launch_lane_2(a, mode, sig_all, s, wg, m);
        case 3: return launch_lane_3(a, mode, sig_all, s, wg, m);
        case 4: return launch_lane_4(a, mode, sig_all, s, wg, m);
        case 5: return launch_lane_5(a, mode, sig_all, s, wg, m);
        case 6: return launch_lane_6(a, mode, sig_all, s, wg, m);
        default: return hipErrorInvalidValue;
    }
}

// Sigma at every frequency point of the density sum (moment tail beyond n_freq)
__global__ void k_sigma_all(LatArgs a)
{
    const int m2 = a.nc * a.nc;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nw = t / m2, e = t % m2;
    if (nw < a.n_freq) {  // (n_freq <= *pt_n; on the real axis every point)
        a.pSigAll[t] = a.sigma[t];
        return;
    }
    if (nw >= n_points(a)) return;
    const double w = a.pt_w ? a.pt_w[nw] : matsubara(nw, a.beta);
    a.pSigAll[t] = sigma_elem_at(a.sigma, a.mom, a.nc, a.n_freq, w, nw, e % a.nc, e / a.nc);
}

hipError_t launch_sigma_all(const LatArgs& a, hipStream_t s)
{
    const int m2 = a.nc * a.nc;
    hipLaunchKernelGGL(k_sigma_all, dim3((a.nw_tot * m2 + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

// Launches as wavefronts that split the k walk over the same 64 frequencies, with one
// set of sums in LDS, rather than one wavefront per 64 frequencies.
// Forward (two wavefronts; alone the sums are in registers): half the registers, so at
// n_c = 5 three wavefronts per SIMD instead of two and at n_c = 6 two instead of one,
// against two barriers and n_c^2 LDS updates per k, which a short walk over d does not
// cover.  Measured (8000 k x 1040 points, split / alone, ms): n_c = 6, n_d = 0 0.63 /
// 0.69, 9 1.43 / 2.41; n_c = 5, n_d = 0 0.57 / 0.36, 4 0.62 / 0.58, 6 0.69 / 0.70, 9
// 0.80 / 0.91, 16 1.27 / 1.67; n_c = 4, n_d = 4 0.38 / 0.37, 6 0.44 / 0.45, 16 0.76 /
// 0.87; n_c = 3, n_d = 9 0.33 / 0.35.  Real axis, 32768 k x 1000 points, n_c = 5,
// n_d = 9: 2.84 / 3.35.
// Adjoint (four wavefronts, at n_c = 6 two; gbar and the traces' sums are in LDS and no
// longer in registers): two wavefronts per SIMD at n_c = 4 and 5, no AGPR traffic at
// n_c = 6, against a barrier per column.  n_c = 4, n_d = 0 0.55 / 0.58, 9 1.01 / 1.11, 18
// 1.60 / 1.89; n_c = 5, n_d = 0 1.09 / 1.10, 4 1.36 / 1.41, 9 1.62 / 1.81, 18 2.53 / 3.06;
// n_c = 6, n_d = 0 2.1 / 4.0, 9 3.6 / 5.5, 18 6.5 / 8.2.
// The figures above are for chunks of many k.  A part with no k of its own repeats one, so the
// chunks are multiples of schur_parts (17 k in four parts, adjoint of n = 10, n_c = 4, 4096 k x
// 1040 points: 450 us, 20 k 408; alone 395 to 406), and there must be 256 workgroups of such chunks, one
// to a CU: below that a wavefront for each k ends sooner.  Adjoint of n = 14, n_c = 5, split at four k a
// chunk / alone at one k, us: 64 k x 216 points 27.6 / 25.0, 343 k x 216 39.1 / 49.3, 512 k x 116
// 30.6 / 34.8, 512 k x 272 58 / 64 (one k a chunk, split: 120); forward, two k: 64 k x 80 18.8 / 18.4,
// 64 k x 216 19.9 / 20.1, 512 k x 116 27.7 / 30.0.
bool schur_ksplit(int nc, int nd, int mode, long items)
{
    if (items < 256L * schur_parts(nc, mode)) return false;
    if (mode == MODE_VJP) return nc >= 4 && nc <= 6;
    return mode == MODE_FWD && (nc == 6 || (nc >= 3 && nc <= 5 && nd >= 6));
}

// Real axis, split or else at 128 points per workgroup (the second wavefront finds the k block in
// the scalar cache) unless that pads a tile more than 64 does: n = 14, n_c = 5, 4096 k x 1000
// energies, 128 / 64: 0.454 / 0.474 ms; 1728 k x 400, four tiles of 128 against seven of 64: 0.154 /
// 0.140.  Up to 4096 wavefronts the padding costs nothing (n = 20, n_c = 5, 512 k x 300: 54 / 57 us).
// Summed over k, 64 is no slower at n_c >= 4 (n = 5: 0.217 / 0.212 ms at 4096 k x 1000).
// One k per workgroup (per_k: band spectra): a second part would only repeat it, which cost
// n = 14, n_c = 5, 216 k x 1000 60.6 us against 48.5 at 128; n_c = 6 with few d orbitals alone
// gains from the registers the split form saves (n = 6, 4096 k x 1000: 0.87 ms, 64 0.94, 128 1.00).
int schur_form(int nc, int nd, int mode, bool real_axis, bool per_k, int nk, int n_pts)
{
    const long tiles = (n_pts + 63) / 64, items = nk * tiles;
    if (per_k ? nc == 6 && nd < 2 : schur_ksplit(nc, nd, mode, items)) return SCHUR_WG_KSPLIT;
    if (!real_axis) return 64;
    if (items < 4096) return 128;
    if (tiles % 2) return 64;
    return per_k ? (nc == 6 && nd < 4 ? 64 : 128) : (nc <= 3 ? 128 : 64);
}

hipError_t launch_lattice_schur(const LatArgs& a, int mode, hipStream_t s, int wg, bool cols)
{
    hipError_t e = launch_sigma_all(a, s);
    if (e != hipSuccess) return e;
    if (a.real_axis && mode == MODE_FWD && a.nc <= 6 && !cols)
        return dispatch_nc(a, MODE_FWD_REAL, a.pSigAll, s, wg, nullptr);
    if (a.nc > 6 || cols || a.real_axis) {  // the per-lane kernels take the real axis in the forward only
        switch (cols_bucket(a.nc)) {
            case 4: return launch_cols_4(a, mode, a.pSigAll, s);
            case 5: return launch_cols_5(a, mode, a.pSigAll, s);
            case 6: return launch_cols_6(a, mode, a.pSigAll, s);
            case 8: return launch_cols_8(a, mode, a.pSigAll, s);
            case 10: return launch_cols_10(a, mode, a.pSigAll, s);
            case 12: return launch_cols_12(a, mode, a.pSigAll, s);
            default: return launch_cols_16(a, mode, a.pSigAll, s);
        }
    }
    return dispatch_nc(a, mode, a.pSigAll, s, wg, nullptr);
}

hipError_t launch_lattice_schur_multi(const LatArgs& proto, int mode, hipStream_t s, int wg,
                                      const SchurMulti& m)
{
    return dispatch_nc(proto, mode, nullptr, s, wg, &m);
}

hipError_t launch_lattice_schur_cols_multi(const LatArgs& proto, int mode, hipStream_t s,
                                           const SchurMulti& m)
{
    switch (cols_bucket(proto.nc)) {
        case 8: return launch_cols_multi_8(proto, mode, s, m);
        case 10: return launch_cols_multi_10(proto, mode, s, m);
        case 12: return launch_cols_multi_12(proto, mode, s, m);
        case 16: return launch_cols_multi_16(proto, mode, s, m);
        default: return hipErrorInvalidValue;
    }
}

// W(k) = H_cd(k) V_d(k): W_ad = sum_e H(a, nc+e) V_d(e, d)
__global__ void k_schur_prep(const cd* __restrict__ Hk, const cd* __restrict__ Vd, int n, int nc, int nk,
                             cd* __restrict__ W)
{
    const int nd = n - nc;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nk * nc * nd) return;
    const int k = (int)(t / ((size_t)nc * nd));
    const int r = (int)(t % ((size_t)nc * nd));
    const int aa = r % nc, d = r / nc;
    const cd* H = Hk + (size_t)k * n * n;
    const cd* V = Vd + (size_t)k * nd * nd;
    cd s = cd{0.0, 0.0};
    for (int e = 0; e < nd; ++e) s = cfma(H[aa + (size_t)(nc + e) * n], V[e + (size_t)d * nd], s);
    W[t] = s;
}

// Per-k block of the one-matrix-per-lane kernels, laid out as the LDS
// staging buffer of stage_k: [H_cc nc*nc][P_d(a<=b) nd*np][e_d nd doubles],
// P_d(a, b) = W_ad conj(W_bd), pairs ordered b-major.
__global__ void k_schur_kdata(const cd* __restrict__ Hk, const cd* __restrict__ W, const double* __restrict__ ed, int n,
                              int nc, int nk, int bs, cd* __restrict__ out)
{
    const int nd = n - nc, np = nc * (nc + 1) / 2;
    const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (size_t)nk * bs) return;
    const int k = (int)(gid / bs), t = (int)(gid % bs);
    cd v = cd{0.0, 0.0};
    if (t < nc * nc) {
        v = Hk[(size_t)k * n * n + (t % nc) + (size_t)(t / nc) * n];
    } else if (t < nc * nc + nd * np) {
        const int q = t - nc * nc, d = q / np, p = q % np;
        int ib = 0;
        while ((ib + 1) * (ib + 2) / 2 <= p) ++ib;
        const int ia = p - ib * (ib + 1) / 2;
        const cd* Wk = W + (size_t)k * nc * nd;
        v = cmulc(Wk[ia + d * nc], Wk[ib + d * nc]);
    } else {
        const int q = 2 * (t - nc * nc - nd * np);  // two e_d per cd slot
        const double* e = ed + (size_t)k * nd;
        v.x = q < nd ? e[q] : 0.0;
        v.y = q + 1 < nd ? e[q + 1] : 0.0;
    }
    out[gid] = v;
}

int schur_kdata_size(int n, int nc) { return nc * nc + (n - nc) * (nc * (nc + 1) / 2) + (n - nc + 1) / 2; }

hipError_t launch_schur_kdata(const cd* Hk, const cd* W, const double* ed, int n, int nc, int nk, cd* out,
                              hipStream_t s)
{
    const int bs = schur_kdata_size(n, nc);
    const size_t total = (size_t)nk * bs;
    hipLaunchKernelGGL(k_schur_kdata, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, Hk, W, ed, n, nc, nk, bs,
                       out);
    return hipGetLastError();
}

hipError_t launch_schur_prep(const cd* Hk, const cd* Vd, int n, int nc, int nk, cd* W, hipStream_t s)
{
    const size_t total = (size_t)nk * nc * (n - nc);
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_schur_prep, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, Hk, Vd, n, nc, nk, W);
    return hipGetLastError();
}

}  // namespace dg
