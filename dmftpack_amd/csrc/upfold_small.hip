// upfolding_k (upfolding.cpp:10-35) and the basis changes of upfolding_density (:45-51) for
// n_orb <= 32 in one kernel, and the k -> R sums (:67-86) for R lists that name (nearly) every
// (R, element) pair.
//
// k_upfold_small: two wavefronts per k, three n_orb x n_orb matrices in LDS, so that the
// inputs are read and the results written once (the batched kernels of upfold.hip pass
// every intermediate through memory: 13 launches per chunk of k).
//   * Wavefront 0 inverts T, wavefront 1 S, at the same time, in registers: lane r + 16 g holds
//     rows r and r + 16 of columns 8 g .. 8 g + 7.  Gauss-Jordan with row pivoting (to 15 bits of
//     |a|^2: pivots within 2^-16 of the largest, so entries grow at most as with the largest
//     times 1 + 2^-16 a step), rows not
//     exchanged but marked used (A^-1(j, p_c) is left in row p_j, column c, p_j the pivot row of
//     step j); per step the pivot row and column pass through LDS, and a row entry read
//     there serves two rows' products.
//   * The products E = T^-H K_o, X C, C^H (X C), E K, (E K) E^H, S^-1 D, (S^-1 D) S^-1 on FP64
//     MFMA (v_mfma_f64_16x16x4, complex as four real products), a wavefront taking 16 rows.
// At n_orb = 28, 32^3 k it takes 2.3 ms (the batched kernels: 5.2 ms): 39 KB of LDS per k leave
// two wavefronts per SIMD, whose vector work (7200 instructions each, 0.35 of the SIMD cycles)
// and MFMAs (0.23) share the SIMD, the rest waiting on LDS, barriers and loads.  The
// pivot search by shuffles of (|a|^2, row) pairs and divisions in the copy loops cost 2.7 ms.
#include "upfold_small.hpp"

#include <algorithm>

namespace dg {

namespace {

typedef double dv4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ unsigned dpp_row(unsigned x)
{
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}

// 0 for rows out of the search; otherwise > 0, ordered by |a|^2 (NaN as 0)
__device__ __forceinline__ unsigned pivot_key(cd a, int row, bool in)
{
    const double m = fma(a.x, a.x, a.y * a.y);
    const unsigned hi = m >= 0.0 ? (unsigned)__double2hiint(m) : 0u;
    return in ? ((hi >> 5) << 6) | 32u | (31u - row) : 0u;
}

// In-register inverse of the n x n matrix in a[s][c] = A(r + 16 s, 8 g + c) (zero outside), lane
// r + 16 g.  buf: 64 cd + 32 int of this wavefront's LDS.  On return row s of the lane is row
// jr[s] of the inverse and column 8 g + c is its column pc[c].
__device__ void gj_wave(cd (&a)[2][8], int n, cd* buf, int* pbuf, int lane, int (&jr)[2], int (&pc)[8],
                        int* __restrict__ singular)
{
    const int r = lane & 15, g = lane >> 4;
    cd* row = buf;
    cd* col = buf + 32;
    jr[0] = jr[1] = -1;
    for (int jg = 0; 8 * jg < n; ++jg) {
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            const int j = 8 * jg + jj;
            if (j < n) {
                // pivot: the row with the largest modulus of column j among those not used yet, to
                // 15 bits (the high word of |a|^2 with the row number in its low bits), so that the
                // search is four DPP maxima; the lanes of group jg hold column j
                unsigned key = pivot_key(a[0][jj], r, jr[0] < 0 && r < n);
                key = max(key, pivot_key(a[1][jj], r + 16, jr[1] < 0 && r + 16 < n));
                key = max(key, dpp_row<0xB1>(key));   // quad_perm 1 0 3 2
                key = max(key, dpp_row<0x4E>(key));   // quad_perm 2 3 0 1
                key = max(key, dpp_row<0x141>(key));  // row_half_mirror
                key = max(key, dpp_row<0x140>(key));  // row_mirror
                const int p = 31 - (__builtin_amdgcn_readlane((int)key, 16 * jg) & 31);
                if (lane == 0) pbuf[j] = p;
                const bool mine = r == (p & 15);
                if (mine) {
                    if (p < 16) {
#pragma unroll
                        for (int c = 0; c < 8; ++c) row[8 * g + c] = a[0][c];
                    } else {
#pragma unroll
                        for (int c = 0; c < 8; ++c) row[8 * g + c] = a[1][c];
                    }
                }
                if (g == jg) {
                    col[r] = a[0][jj];
                    col[r + 16] = a[1][jj];
                }
                wave_sync();
                const cd d = row[j];
                cd f0 = col[r], f1 = col[r + 16];
                cd t[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) t[c] = row[8 * g + c];
                const double q = fma(d.x, d.x, d.y * d.y);
                const bool okp = q > 0.0;  // false for NaN
                if (lane == 0 && !okp) *singular = 1;
                cd rp = cd{0.0, 0.0};
                if (okp) {
                    const double iq = q > 1e-280 && q < 1e280 ? rcp_pos(q) : 1.0 / q;
                    rp = cd{d.x * iq, -d.y * iq};
                }
#pragma unroll
                for (int c = 0; c < 8; ++c) t[c] = cmul(t[c], rp);
                if (g == jg) {  // column j of the inverse takes the place of column j
                    t[jj] = rp;
                    a[0][jj] = cd{0.0, 0.0};
                    a[1][jj] = cd{0.0, 0.0};
                }
                if (mine) {  // the pivot row becomes t: 0 - (-1) t
                    if (p < 16) {
                        jr[0] = j;
                        f0 = cd{-1.0, 0.0};
#pragma unroll
                        for (int c = 0; c < 8; ++c) a[0][c] = cd{0.0, 0.0};
                    } else {
                        jr[1] = j;
                        f1 = cd{-1.0, 0.0};
#pragma unroll
                        for (int c = 0; c < 8; ++c) a[1][c] = cd{0.0, 0.0};
                    }
                }
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    a[0][c] = cfms(f0, t[c], a[0][c]);
                    a[1][c] = cfms(f1, t[c], a[1][c]);
                }
                wave_sync();  // row and col are read before the next step writes them
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) pc[c] = 8 * g + c < n ? pbuf[8 * g + c] : 0;
}

__device__ __forceinline__ void gj_load(cd (&a)[2][8], const cd* __restrict__ M, int n, int lane)
{
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int i = r + 16 * s, j = 8 * g + c;
            a[s][c] = (i < n && j < n) ? M[i + (size_t)j * n] : cd{0.0, 0.0};
        }
}

__device__ __forceinline__ void gj_store(const cd (&a)[2][8], int n, cd* M, int ld, int lane, const int (&jr)[2],
                                         const int (&pc)[8])
{
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int s = 0; s < 2; ++s)
        if (r + 16 * s < n && jr[s] >= 0)
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (8 * g + c < n) M[jr[s] + pc[c] * ld] = a[s][c];
}

// Rows 16 wave .. 16 wave + 15 of op(A) op(B), n x n, leading dimension ld, both in LDS.
// Operand layout of the MFMA: A(i, q) on lane i + 16 q, B(q, j) on lane j + 16 q; result
// register v of lane j + 16 q is row 4 v + q.  Out-of-range rows and columns repeat the last
// one (their results are not stored); summed indices past n give zero operands.
struct Prod {
    dv4 re[2], im[2];
};

template <bool HA, bool HB>
__device__ __forceinline__ void zprod(Prod& p, const cd* A, const cd* B, int n, int ld, int wave, int lane)
{
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        p.re[t] = dv4{0.0, 0.0, 0.0, 0.0};
        p.im[t] = p.re[t];
    }
    if (16 * wave >= n) return;
    const bool two = n > 16;
    const int i = min(16 * wave + r, n - 1), j0 = min(r, n - 1), j1 = min(16 + r, n - 1);
    // operands of summed index l at pa + l * sa, pb0 + l * sb, pb1 + l * sb
    const int sa = HA ? 1 : ld, sb = HB ? ld : 1;
    const cd* pa = A + (HA ? i * ld : i);
    const cd* pb0 = B + (HB ? j0 : j0 * ld);
    const cd* pb1 = B + (HB ? j1 : j1 * ld);
    auto step = [&](cd a, cd b0, cd b1) {
        if (HA) a.y = -a.y;
        if (HB) {
            b0.y = -b0.y;
            b1.y = -b1.y;
        }
        p.re[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b0.x, p.re[0], 0, 0, 0);
        p.im[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b0.y, p.im[0], 0, 0, 0);
        if (two) {
            p.re[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b1.x, p.re[1], 0, 0, 0);
            p.im[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b1.y, p.im[1], 0, 0, 0);
        }
        p.re[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b0.y, p.re[0], 0, 0, 0);
        p.im[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b0.x, p.im[0], 0, 0, 0);
        if (two) {
            p.re[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b1.y, p.re[1], 0, 0, 0);
            p.im[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b1.x, p.im[1], 0, 0, 0);
        }
    };
    int l0 = 0;
#pragma unroll 2
    for (; l0 + 4 <= n; l0 += 4) {
        const int l = l0 + q;
        step(pa[l * sa], pb0[l * sb], pb1[l * sb]);
    }
    if (l0 < n) {
        const int l = min(l0 + q, n - 1);
        cd a = pa[l * sa];
        if (l0 + q >= n) a = cd{0.0, 0.0};
        step(a, pb0[l * sb], pb1[l * sb]);
    }
}

// f(i, j, value) for the entries of a product this lane holds
template <class F>
__device__ __forceinline__ void each(const Prod& p, int n, int wave, int lane, F f)
{
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * wave + 4 * v + q, j = 16 * t + r;
            if (i < n && j < n) f(i, j, cd{p.re[t][v], p.im[t][v]});
        }
}

// n x n matrix between global memory and LDS: lane = row, four columns at a time
__device__ __forceinline__ void load_lds(cd* M, int ld, const cd* __restrict__ g, int n, int tid)
{
    const int i = tid & 31;
    if (i < n)
        for (int c = tid >> 5; c < n; c += 4) M[i + c * ld] = g[i + c * n];
}
__device__ __forceinline__ void store_lds(const cd* M, int ld, cd* __restrict__ g, int n, int tid)
{
    const int i = tid & 31;
    if (i < n)
        for (int c = tid >> 5; c < n; c += 4) g[i + c * n] = M[i + c * ld];
}

__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2))) void k_upfold_small(UpfoldArgs u)
{
    extern __shared__ cd sm[];
    __shared__ int sv[kUpfoldSmall], sinv[kUpfoldSmall], spiv[2][kUpfoldSmall];
    const int N = u.n_orb, n = u.n, ld = N | 1, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const size_t k = blockIdx.x, oo = (size_t)N * N;
    const int bs = max(N * ld, 128);
    cd *B1 = sm, *B2 = sm + bs, *B3 = sm + 2 * bs;
    if (tid < kUpfoldSmall) {
        sv[tid] = tid < n ? u.v2k[k * n + tid] : -1;
        sinv[tid] = -1;
    }
    load_lds(B2, ld, u.Ko + k * oo, N, tid);
    // T^-1 (wavefront 0) and S^-1 (wavefront 1); B3 holds the exchange buffers
    cd a[2][8];
    int jr[2], pc[8];
    const bool inv = wave == 0 || u.S;
    if (inv) {
        gj_load(a, (wave == 0 ? u.T : u.S) + k * oo, N, lane);
        gj_wave(a, N, B3 + 64 * wave, spiv[wave], lane, jr, pc, u.singular);
        if (wave == 0) gj_store(a, N, B1, ld, lane, jr, pc);
    }
    __syncthreads();
    if (tid < n && sv[tid] >= 0) sinv[sv[tid]] = tid;
    Prod p;
    zprod<true, false>(p, B1, B2, N, ld, wave, lane);  // E = T^-H K_o
    __syncthreads();
    each(p, N, wave, lane, [&](int i, int j, cd v) { B3[i + j * ld] = v; });
    load_lds(B1, ld, u.X + k * n * n, n, tid);
    load_lds(B2, ld, u.C + k * n * n, n, tid);
    __syncthreads();
    zprod<false, false>(p, B1, B2, n, ld, wave, lane);  // X C
    __syncthreads();
    each(p, n, wave, lane, [&](int i, int j, cd v) { B1[i + j * ld] = v; });
    __syncthreads();
    zprod<true, false>(p, B2, B1, n, ld, wave, lane);  // M = C^H (X C)
    __syncthreads();
    // K: M at the window's bands, the clamped Fermi factor on the other diagonal entries
    for (int e = tid; e < N * ld; e += 128) B2[e] = cd{0.0, 0.0};
    __syncthreads();
    each(p, n, wave, lane, [&](int i, int j, cd v) {
        if (sv[i] >= 0 && sv[j] >= 0) B2[sv[i] + sv[j] * ld] = v;
    });
    if (tid < N && sinv[tid] < 0) {
        const double x = u.beta * (u.eps[k * N + tid] - u.mu);
        B2[tid + tid * ld] = cd{x > 100.0 ? 0.0 : x < -100.0 ? 1.0 : 1.0 / (1.0 + exp(x)), 0.0};
    }
    __syncthreads();
    zprod<false, false>(p, B3, B2, N, ld, wave, lane);  // E K
    each(p, N, wave, lane, [&](int i, int j, cd v) { B1[i + j * ld] = v; });
    __syncthreads();
    zprod<false, true>(p, B1, B3, N, ld, wave, lane);  // D = (E K) E^H
    each(p, N, wave, lane, [&](int i, int j, cd v) { B2[i + j * ld] = v; });
    __syncthreads();
    store_lds(B2, ld, u.D + k * oo, N, tid);
    if (!u.S) return;
    if (wave == 1) gj_store(a, N, B3, ld, lane, jr, pc);
    __syncthreads();
    zprod<false, false>(p, B3, B2, N, ld, wave, lane);  // S^-1 D
    each(p, N, wave, lane, [&](int i, int j, cd v) { B1[i + j * ld] = v; });
    __syncthreads();
    store_lds(B1, ld, u.DDir + k * oo, N, tid);
    zprod<false, false>(p, B1, B3, N, ld, wave, lane);  // (S^-1 D) S^-1
    each(p, N, wave, lane, [&](int i, int j, cd v) { B2[i + j * ld] = v; });
    __syncthreads();
    store_lds(B2, ld, u.DD + k * oo, N, tid);
}

// ph [k][n_r padded]: exp(+i kphase.R), the three axes' factors multiplied; zero in the pad
__global__ __launch_bounds__(256) void k_r_phases(const int4* __restrict__ R, int n_r, int n_pad,
                                                  const double* __restrict__ kphase, int nk, cd* __restrict__ ph)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (size_t)nk * n_pad) return;
    const size_t k = t / n_pad;
    const int r = (int)(t % n_pad);
    cd p = cd{r < n_r ? 1.0 : 0.0, 0.0};
    if (r < n_r) {
        const int4 v = R[r];
        const int c[3] = {v.x, v.y, v.z};
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            if (c[ax] == 0) continue;
            double sn, cs;
            sincos(kphase[3 * k + ax] * c[ax], &sn, &cs);
            p = cmul(p, cd{cs, sn});
        }
    }
    ph[t] = p;
}

typedef __attribute__((address_space(4))) double kconst_d;

struct RsMats {
    const cd* Y[3];
};

// A thread sums one matrix element for kRsTile R: per k one load of the element and kRsTile
// phases, wave-uniform, as SGPR operands (4 FMA each).  grid (element blocks of one matrix, R
// tile + tiles * x, k segment).
__global__ __launch_bounds__(64) void k_r_sums(RsMats m, int oo, int nk, int kseg, int n_r, int n_pad,
                                               const cd* __restrict__ ph, cd* __restrict__ part)
{
    const int tiles = n_pad / kRsTile;
    const int rt = blockIdx.y % tiles, x = blockIdx.y / tiles, nx = gridDim.y / tiles;
    const int e = blockIdx.x * 64 + threadIdx.x, ec = min(e, oo - 1);
    const cd* Y = x == 0 ? m.Y[0] : x == 1 ? m.Y[1] : m.Y[2];
    const int k0 = blockIdx.z * kseg, k1 = min(nk, k0 + kseg);
    cd acc[kRsTile];
#pragma unroll
    for (int q = 0; q < kRsTile; ++q) acc[q] = cd{0.0, 0.0};
    if (k0 < k1) {
        cd y = Y[(size_t)k0 * oo + ec];
        for (int k = k0; k < k1; ++k) {
            const cd yn = Y[(size_t)min(k + 1, k1 - 1) * oo + ec];
            const kconst_d* p = (const kconst_d*)(ph + (size_t)k * n_pad + rt * kRsTile);
#pragma unroll
            for (int q = 0; q < kRsTile; ++q) acc[q] = cfma(y, cd{p[2 * q], p[2 * q + 1]}, acc[q]);
            y = yn;
        }
    }
    if (e >= oo) return;
    cd* out = part + (((size_t)blockIdx.z * nx + x) * n_r + rt * kRsTile) * oo + e;
#pragma unroll
    for (int q = 0; q < kRsTile; ++q)
        if (rt * kRsTile + q < n_r) out[(size_t)q * oo] = acc[q];
}

__global__ __launch_bounds__(256) void k_r_scatter(const cd* __restrict__ part, int nseg, int nx, int n_r, int oo,
                                                   const int2* __restrict__ of, int n_entries, double scale,
                                                   cd* __restrict__ dmr)
{
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 3 * (size_t)n_entries) return;
    const int x = (int)(t / n_entries), q = (int)(t % n_entries);
    const int2 o = of[q];
    const size_t seg = (size_t)nx * n_r * oo;
    const cd* p = part + ((size_t)(nx == 3 ? x : 0) * n_r + o.x) * oo + o.y;
    cd a = p[0];
    for (int y = 1; y < nseg; ++y) a = cadd(a, p[y * seg]);
    dmr[t] = cadd(dmr[t], cscale(a, scale));
}

}  // namespace

hipError_t launch_upfold_small(const UpfoldArgs& a, hipStream_t s)
{
    if (a.n_orb > kUpfoldSmall || a.n > a.n_orb) return hipErrorInvalidValue;
    const int bs = std::max(a.n_orb * (a.n_orb | 1), 128);  // B3 also holds 2 x 64 exchange entries
    const int shm = (int)(sizeof(cd) * 3 * bs);
    hipError_t e = hipFuncSetAttribute((const void*)k_upfold_small, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_upfold_small, dim3(a.nk), dim3(128), shm, s, a);
    return hipGetLastError();
}

hipError_t launch_r_phases(const int4* R, int n_r, const double* kphase, int nk, cd* ph, hipStream_t s)
{
    const int n_pad = rs_pad(n_r);
    const size_t total = (size_t)nk * n_pad;
    hipLaunchKernelGGL(k_r_phases, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, R, n_r, n_pad, kphase, nk, ph);
    return hipGetLastError();
}

hipError_t launch_r_sums(const cd* const Y[3], int nx, int oo, int nk, int n_r, const cd* ph, int nseg, cd* part,
                         hipStream_t s)
{
    const int n_pad = rs_pad(n_r), tiles = n_pad / kRsTile;
    const RsMats m{{Y[0], Y[1], Y[2]}};
    hipLaunchKernelGGL(k_r_sums, dim3((oo + 63) / 64, tiles * nx, nseg), dim3(64), 0, s, m, oo, nk, (nk + nseg - 1) / nseg,
                       n_r, n_pad, ph, part);
    return hipGetLastError();
}

hipError_t launch_r_scatter(const cd* part, int nseg, int nx, int n_r, int oo, const int2* of, int n_entries,
                            double scale, cd* dmr, hipStream_t s)
{
    const size_t total = 3 * (size_t)n_entries;
    hipLaunchKernelGGL(k_r_scatter, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, part, nseg, nx, n_r, oo, of,
                       n_entries, scale, dmr);
    return hipGetLastError();
}

}  // namespace dg
