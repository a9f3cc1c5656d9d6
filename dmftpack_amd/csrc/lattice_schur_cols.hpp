// Schur-complement lattice path for larger correlated blocks (7 <= n_c <= 16),
// column per lane.
//
// Same mathematics as lattice_schur.hip (the hot loop of GreenFtn_w,
// GreenFtn.cpp:218-308, and the densities of GiwToNele :513-635, from the
// block structure of A = (z+mu) I - H(k) - P Sigma P^H with the correlated
// orbitals first, downfolding.cpp:69-79):
//   S     = (z+mu) I - H_cc - Sigma - sum_d g_d w_d w_d^H,  g_d = 1/(z+mu-e_d)
//   G_cc  = S^{-1}
//   tr G  = sum_d g_d + tr G_cc + sum_d g_d^2 M_d,        M_d = w_d^H G_cc w_d
//   tr G^2 = sum_d g_d^2 + tr(Z^2) + 2 sum_d g_d^3 M_d,   Z = G_cc (I + Y),
//            Y = sum_d g_d^2 w_d w_d^H
//   (G^2)_cc = Z G_cc
// An n_c x n_c complex matrix no longer fits one lane's registers, so a slot
// of N lanes (N = n_c rounded up to 8/10/12/16) owns one (k, iw) matrix and
// lane c holds column c of S, then of G_cc:
//   * S column c:  S_ic = E_ic - H_cc,ic - sum_d W_id (g_d conj(W_cd)),
//     E = (z+mu) I - Sigma(iw), Sigma read from the cache at each k;
//     the g_d of the slot's frequency are computed once per slot and shared
//     through LDS;
//   * inversion: column-per-lane Gauss-Jordan (gj.hpp), in FP64 for both Schur methods
//     (lattice_schur_lane.hpp; n = 32, n_c = 10, 1728 k x 528 points, forward + adjoint:
//     4.8 ms against 5.5 ms with an FP32 inverse and one FP64-residual step);
//   * FWD accumulates column c of G_cc over the k chunk in registers; the
//     trace terms are per-lane partials summed over the slot at the end;
//   * DENS/VJP exchange G_cc, Z and V = gbar + cn (I + Y)^H through per-slot
//     LDS matrices for the products Z = G + G Y, tr(Z^2) and
//     sigma_bar += G^H V G^H; lane c accumulates column c of sigma_bar.
// The per-k data (H_cc, W = H_cd V_d, e_d) is read from global memory through
// the constant address space (wave-uniform reads become scalar loads).
#pragma once
#include "gj.hpp"
#include "lattice_kernels.hpp"

namespace dg {

// Smallest n_c the bucket of width N serves (lattice_schur.hip, cols_bucket):
// rows i below it are inside every served block, so in the d loops the tests
// i < n_c on them fold away at compile time and the W loads issue
// unconditionally (a load under a uniform branch waits on its own).
__host__ __device__ constexpr int cols_nc_min(int N)
{
    return N <= 4 ? 1 : N <= 6 ? N : N == 8 ? 7 : N == 10 ? 9 : N == 12 ? 11 : 13;
}

// one wavefront per workgroup: the per-k data comes from global memory, so
// wavefronts share nothing but the cache
__host__ __device__ constexpr int cols_wg() { return 64; }

// per-slot LDS (cd units): gsh 32 - nc_min (g_d; in the forward then the elimination's
// broadcast buffer, 2 N), MA N*N and, but for the forward, MB N*N.
// Sigma and gbar are read from the cache at each k and the spare lanes repeat lanes of
// the last slot instead of writing to a slot of their own: the LDS is what decides how
// many wavefronts of the adjoint a CU holds (N = 10: 39.5 KB each with tables of their
// own for all of these, 4 to a CU; 21.4 KB, 7 to a CU.  With cols_waves below, adjoint
// of n = 32, n_c = 10, 1728 k x 528 points: 4.85 -> 3.28 ms, n_c = 16: 21.8 -> 12.3 ms;
// forward 1.81 -> 1.51 ms and 6.0 -> 3.7 ms).
// The size is odd (in 16-byte entries): the slots of a wavefront read the same entry of
// their own matrices at once, and with a multiple of 16 entries (the adjoint at N = 10 or
// 16, every form at N = 8) all of those fell into the same four banks.
__host__ __device__ constexpr int cols_g_size(int N, int mode)
{
    const int g = 32 - cols_nc_min(N);  // n_d at most
    return mode == MODE_FWD && g < 2 * N ? 2 * N : g;
}
__host__ __device__ constexpr int cols_slot_size(int N, int mode)
{
    return (cols_g_size(N, mode) + (mode == MODE_FWD ? N * N : 2 * N * N)) | 1;
}

__host__ __device__ constexpr int cols_slots(int N) { return 64 / N; }

inline size_t cols_lds_bytes(int N, int mode)
{
    return sizeof(cd) * ((size_t)cols_slots(N) * cols_slot_size(N, mode));
}

// Wavefronts per SIMD the register allocator is held to: as many as fit without spilling
// column-sized values (three in the forward up to N = 10; the adjoint at N = 16
// needs 356 registers, and its LDS admits four wavefronts to a CU anyway).
__host__ __device__ constexpr int cols_waves(int N, int mode)
{
    return mode == MODE_FWD ? (N <= 10 ? 3 : 2) : N <= 12 ? 2 : 1;
}

__device__ __forceinline__ cd ld_off(const cd* base, unsigned bytes) { return *(const cd*)((const char*)base + bytes); }

// out_i += sum_l M_il x_l (ADJ: M^H), M column-major in LDS.  M's entries are read a
// column (row) ahead of their use, four at a time, each into the registers of an entry
// just used: left to itself the compiler reads a column, waits for it and uses it
// (adjoint of n = 32, n_c = 10, 1728 k x 528 points: 3.32 against 2.49 ms; n_c = 16 12.3
// against 8.5; a barrier after every entry instead of every four cost 0.5 ms, the four
// FMAs of an entry being a chain).
// Padding needs no test: entries of M there are finite and meet a zero.
template <int N, bool ADJ, class X>
__device__ __forceinline__ void lds_product(const cd* M, cd (&out)[N], X&& x)
{
    auto at = [M](int i, int l) -> cd { return ADJ ? M[l + i * N] : M[i + l * N]; };
    cd buf[N];
#pragma unroll
    for (int i = 0; i < N; ++i) buf[i] = at(i, 0);
    cd xn = x(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int l = 0; l < N; ++l) {
        const cd xl = xn;
        if (l + 1 < N) xn = x(l + 1);
#pragma unroll
        for (int i0 = 0; i0 < N; i0 += 4) {
#pragma unroll
            for (int i = i0; i < N && i < i0 + 4; ++i) {
                out[i] = ADJ ? cfmac(buf[i], xl, out[i]) : cfma(buf[i], xl, out[i]);
                if (l + 1 < N) buf[i] = at(i, l + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// One (frequency tile, k chunk) work item of one lattice: the body of the
// per-lattice kernel and of the persistent multi-lattice kernel below.
template <int N, int MODE, bool TRACE>
__device__ __forceinline__ void cols_item(const LatArgs& a, const cd* __restrict__ sig_all, int wtile, int chunk,
                                          cd* lds)
{
    constexpr int SPW = 64 / N;
    constexpr int SLOTS = cols_slots(N);
    constexpr int SS = cols_slot_size(N, MODE);
    const int n = a.n, nc = a.nc, nd = a.n - nc, m2 = nc * nc;
    constexpr int NMIN = cols_nc_min(N);
    auto inb = [nc](int i) { return i < NMIN || i < nc; };  // row / column i inside the n_c block
    const int tid = threadIdx.x, lane = tid;  // one wavefront
    // the spare lanes of a wavefront repeat the first lanes of its last slot: the same
    // values to the same LDS entries, and nothing stored at the end
    const bool active = lane < SPW * N;
    const int sl = active ? lane / N : SPW - 1;
    const int c0 = active ? lane - sl * N : lane - SPW * N;
    const int cc = c0 < nc ? c0 : 0;  // clamped column index for loads
    cd* my = lds + (size_t)sl * SS;
    cd* gsh = my;
    cd* MA = gsh + cols_g_size(N, MODE);
    cd* MB = MA + N * N;
    // the elimination's buffer: over g_d, which the forward needs no more by then, or in
    // MA, not yet written; the row values kept across the inversion
    cd* bc = MODE == MODE_FWD ? gsh : MA;
    cd* park = MODE == MODE_FWD ? MA : MB;
    const int npts = n_points(a);
    if (wtile * SLOTS >= npts) return;  // tile past the last frequency point
    const int nw = wtile * SLOTS + sl;
    const bool wvalid = nw < npts;
    const int nwc = nw < npts ? nw : npts - 1;
    const int k0 = chunk * a.k_per_chunk;
    const int k1 = min(a.nk, k0 + a.k_per_chunk);
    double mu, w;
    freq_point(a, nwc, mu, w);
    const bool vjp_here = (MODE == MODE_VJP) && wvalid && nw < a.n_freq;
    const double cn = (MODE == MODE_VJP) ? 2.0 * (a.nbar_dev ? *a.nbar_dev : a.nbar) / a.beta : 0.0;

    // column c of Sigma(iw) and row c of gbar, read at each k: held across the k walk
    // they would take 8 N registers
    // (addresses as a wave-uniform base and a 32-bit offset of the lane: kept across the
    // walk as 64-bit addresses of single entries they spill)
    const cd* sig = sig_all + (size_t)(wtile * SLOTS) * m2;
    const cd* gb = MODE == MODE_VJP ? a.gbar + (size_t)min(wtile * SLOTS, a.n_freq - 1) * m2 : nullptr;
    const unsigned sig_off = ((nwc - wtile * SLOTS) * m2 + cc * nc) * 16;
    const unsigned gb_off = ((min(nw, a.n_freq - 1) - min(wtile * SLOTS, a.n_freq - 1)) * m2 + cc) * 16;
    const unsigned h_off = cc * n * 16;
    cd acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = cd{0.0, 0.0};
    cd trA = cd{0.0, 0.0}, tr2A = cd{0.0, 0.0}, muA = cd{0.0, 0.0};
    __syncthreads();

    for (int k = k0; k < k1; ++k) {
        // (hidden from the compiler at each k: what it derives from these, masks and
        // addresses for every entry, it would hold across the walk, in scratch memory)
        int c = c0, ncs = nc;
        asm volatile("" : "+v"(c), "+s"(ncs)::"memory");
        const bool live = c < nc;  // lanes c >= nc hold identity padding
        // per-k data straight from global memory through the constant address
        // space: the wave-uniform reads (W_id, e_d) become scalar loads
        const cd* Hkk = a.Hk + (size_t)k * n * n;  // H_cc(i, c) at i + c*n
        const kconst_cd* Wk = (const kconst_cd*)(a.W + (size_t)k * nc * nd);
        const kconst_double* ed = (const kconst_double*)(a.ed + (size_t)k * nd);
        // This k's W and e_d into the caches at once: vector loads into L1 for
        // the lane-dependent reads (W_cd, e_d), the scalar-cache fill for the
        // wave-uniform ones (columns of W), one round trip per k instead of
        // one per d
        if (nd > 0) {
            const cd* Wg = a.W + (size_t)k * nc * nd;
            const int wn = nc * nd;  // complex entries of W(k)
            // indices clamped, not branched on: the loads issue together
            double pf = 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = tid + r * 64;
                pf = fma(Wg[e < wn ? e : wn - 1].x, 0.0, pf);
            }
            pf = fma(a.ed[(size_t)k * nd + (tid < nd ? tid : nd - 1)], 0.0, pf);
            kcache_fill64(Wg);
            asm volatile("" ::"v"(pf));
        }
        // g_d = 1/(iw + mu - e_d) of this slot's frequency, shared by its lanes
        cd tg = cd{0.0, 0.0}, t2 = cd{0.0, 0.0};  // lane shares of tr G and tr G^2
        for (int d = c; d < nd; d += N) {
            const double x = mu - ed[d];
            const double r = rcp_pos(fma(x, x, w * w));
            const cd g = cd{x * r, -w * r};
            gsh[d] = g;
            tg = cadd(tg, g);
            if constexpr (MODE != MODE_FWD) t2 = cfma(g, g, t2);
        }
        wave_sync();

        // ---- column c of S (identity column for padding lanes)
        cd col[N];
        cd y[MODE == MODE_FWD ? 1 : N];  // column c of Y = sum_d g_d^2 w_d w_d^H
        // (the loads are unconditional, rows clamped in range, and pinned by an
        // empty asm so that the compiler cannot sink each into a branch of its
        // own: they issue together instead of one round trip per entry)
        {
            cd t[N];
#pragma unroll
            for (int i = 0; i < N; ++i) t[i] = ld_off(Hkk + (inb(i) ? i : 0), h_off);
#pragma unroll
            for (int i = 0; i < N; ++i) asm volatile("" ::"v"(t[i].x), "v"(t[i].y));
#pragma unroll
            for (int i = 0; i < N; ++i) col[i] = csub(i == c ? cd{mu, w} : cd{0.0, 0.0}, t[i]);
#pragma unroll
            for (int i = 0; i < N; ++i) t[i] = ld_off(sig + (inb(i) ? i : 0), sig_off);
#pragma unroll
            for (int i = 0; i < N; ++i) asm volatile("" ::"v"(t[i].x), "v"(t[i].y));
#pragma unroll
            for (int i = 0; i < N; ++i)
                col[i] = live ? (inb(i) ? csub(col[i], t[i]) : cd{0.0, 0.0})
                              : ((i == c) ? cd{1.0, 0.0} : cd{0.0, 0.0});
        }
        // row c of sum_d g_d^p w_d w_d^H, p = 2 (forward) or 3: with column c of G_cc it
        // gives the trace's sum_d g_d^p M_d as sum_i G_ic Y_ci, in this same walk over W
        // (a walk of its own after the inversion, one dot product per d, took 1.51 ms
        // against 1.29, forward of n = 32, n_c = 10, 1728 k x 528 points)
        constexpr bool ROW = MODE != MODE_FWD || TRACE;
        cd yr[ROW ? N : 1];
        if constexpr (ROW) {
#pragma unroll
            for (int i = 0; i < N; ++i) yr[i] = cd{0.0, 0.0};
        }
        if constexpr (MODE != MODE_FWD) {
#pragma unroll
            for (int i = 0; i < N; ++i) y[i] = cd{0.0, 0.0};
        }
        for (int d = 0; d < nd; ++d) {
            const cd g = gsh[d];
            const kconst_cd* Wd = Wk + d * nc;
            const cd wc = live ? ldc(Wd + cc) : cd{0.0, 0.0};
            const cd u = cmulc(g, wc);  // g_d conj(W_cd)
            const cd g2 = cmul(g, g);
            const cd ur = cmul(MODE == MODE_FWD ? g2 : cmul(g2, g), wc);
            const cd u2 = cmul(g, u);
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (inb(i)) {
                    const cd wi = ldc(Wd + i);
                    col[i] = cfms(wi, u, col[i]);
                    if constexpr (MODE != MODE_FWD) y[i] = cfma(wi, u2, y[i]);
                    if constexpr (ROW) yr[i] = cfmac(wi, ur, yr[i]);
                }
        }
        if constexpr (ROW) {  // kept in LDS during the inversion, each lane its own entries
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (nd > 0) park[c + i * N] = yr[i];
        }

        // ---- G_cc = S^{-1}, column c
        gj_columns<N>(col, bc, c, nc);
        if constexpr (ROW) __builtin_amdgcn_sched_barrier(0);
        cd gdiag = cd{0.0, 0.0};  // G_cc(c, c)
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (i == c) gdiag = col[i];

        cd tm = cd{0.0, 0.0};  // lane share of sum_d g_d^p M_d
        if constexpr (ROW) {
            if (nd > 0) {
#pragma unroll
                for (int i = 0; i < N; ++i) tm = cfma(col[i], park[c + i * N], tm);
            }
            // (each stretch between these holds one more column-sized value than fits twice)
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MODE == MODE_FWD) {
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i] = cadd(acc[i], col[i]);
            if constexpr (TRACE) {
                if (live) tg = cadd(tg, cadd(gdiag, tm));
                if (wvalid) trA = cadd(trA, tg);
            }
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) MA[i + c * N] = col[i];
            wave_sync();
            // Z = G (I + Y), column c, over column c of G
            cd(&z)[N] = col;
            lds_product<N, false>(MA, z, [&](int l) { return y[l]; });
            // tr G = sum g + tr G_cc + tr(G Y) = sum g + tr Z,
            // tr G^2 = sum g^2 + tr(Z^2) + 2 sum g^3 M_d
            cd zdiag = cd{0.0, 0.0};
#pragma unroll
            for (int i = 0; i < N; ++i)
                if (i == c) zdiag = z[i];
            if (live) {
                tg = cadd(tg, zdiag);
                t2 = cadd(t2, cscale(tm, 2.0));
            }
            // row c of gbar, on its way during tr(Z^2); earlier, it would not fit beside the product
            cd gv[MODE == MODE_VJP ? N : 1];
            if constexpr (MODE == MODE_VJP) {
#pragma unroll
                for (int j = 0; j < N; ++j) gv[j] = ld_off(gb + (inb(j) ? j : 0) * ncs, gb_off);
            }
#pragma unroll
            for (int i = 0; i < N; ++i) MB[i + c * N] = z[i];
            wave_sync();
            cd zz = cd{0.0, 0.0};  // lane share of tr(Z^2): sum_i Z_ic Z_ci
            if (live) {
#pragma unroll
                for (int i = 0; i < N; ++i)
                    if (i < nc) zz = cfma(z[i], MB[c + i * N], zz);
            }
            t2 = cadd(t2, zz);
            if (wvalid) {
                trA = cadd(trA, tg);
                tr2A = cadd(tr2A, t2);
            }
            if constexpr (MODE == MODE_VJP) {
                // sigma_bar += G^H gbar G^H + cn ((G^2)_cc)^H = C = G^H V G^H with
                // V = gbar + cn S'^H, S' = I + Y ((G^2)_cc = G S' G); lane c forms
                // column c of C.  mu term tr(gbar^H (G^2)_cc) = sum_ij Z_ij conj(L_ij)
                // - cn tr(Z^2) with L = V G^H, as G S' = Z.
                wave_sync();  // every lane has read Z from MB
                if (live) {  // row c of V into MB
#pragma unroll
                    for (int j = 0; j < N; ++j)
                        if (j < nc)
                            MB[c + j * N] = cadd(gv[j], cscale(cadd(cconj(y[j]), cd{j == c ? 1.0 : 0.0, 0.0}), cn));
                }
                wave_sync();
                if (vjp_here && live) {
                    cd l[N];  // column c of L = V G^H: l_i = sum_j V_ij conj(G_cj)
#pragma unroll
                    for (int i = 0; i < N; ++i) l[i] = cd{0.0, 0.0};
                    lds_product<N, false>(MB, l, [&](int j) { return cconj(MA[c + j * N]); });
                    // sum_a S'_ac conj(C_ac) = sum_i Z_ic conj(l_i), as G S' = Z
                    cd ms = cscale(zz, -cn);
#pragma unroll
                    for (int i = 0; i < N; ++i) ms = cfmac(l[i], z[i], ms);
                    // C_ac = sum_i conj(G_ia) l_i
                    lds_product<N, true>(MA, acc, [&](int i) { return l[i]; });
                    muA = cadd(muA, ms);
                }
            }
            wave_sync();
        }
        wave_sync();  // gsh of this k is read by every lane of the slot before it is rewritten
    }

    const int c = c0;
    const bool live = c < nc;
    // ---- sum the trace shares over the lanes of each slot
    my[c] = trA;
    my[N + c] = tr2A;
    my[2 * N + c] = muA;
    wave_sync();
    if (!wvalid || !active) return;
    const size_t ch = chunk;
    if (c == 0) {
        cd s1 = cd{0.0, 0.0}, s2 = cd{0.0, 0.0}, s3 = cd{0.0, 0.0};
        for (int l = 0; l < N; ++l) {
            s1 = cadd(s1, my[l]);
            s2 = cadd(s2, my[N + l]);
            s3 = cadd(s3, my[2 * N + l]);
        }
        a.pTr[ch * a.nw_tot + nw] = s1;
        if (MODE != MODE_FWD) a.pTr2[ch * a.nw_tot + nw] = s2;
        if (MODE == MODE_VJP && nw < a.n_freq) a.pMu[ch * a.n_freq + nw] = s3;
    }
    if (!live) return;
    if constexpr (MODE == MODE_FWD) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (i < nc) a.pG[(ch * a.nw_tot + nw) * m2 + i + c * nc] = acc[i];
    } else if constexpr (MODE == MODE_VJP) {
        if (nw < a.n_freq) {
#pragma unroll
            for (int b = 0; b < N; ++b)
                if (b < nc) a.pSb[(ch * a.n_freq + nw) * m2 + b + c * nc] = acc[b];  // column c
        }
    }
}

template <int N, int MODE, bool TRACE>
__global__ __launch_bounds__(cols_wg()) __attribute__((amdgpu_waves_per_eu(cols_waves(N, MODE)))) void k_lattice_schur_cols(LatArgs a, const cd* __restrict__ sig_all)
{
    extern __shared__ cd lds[];
    cols_item<N, MODE, TRACE>(a, sig_all, lattice_tile(), blockIdx.y, lds);
}

// Persistent form over a work list spanning several lattices with n_c in this
// bucket: workgroup b takes items b, b + gridDim.x, ... ({system, frequency
// tile, k chunk}; static striding, no atomics, so every replay does the same
// work in the same order).  Each system's tables come from its LatArgs.
template <int N, int MODE, bool TRACE>
__global__ __launch_bounds__(cols_wg()) __attribute__((amdgpu_waves_per_eu(cols_waves(N, MODE)))) void k_lattice_schur_cols_multi(const LatArgs* __restrict__ args,
                                                                                 const int4* __restrict__ items,
                                                                                 int n_items)
{
    extern __shared__ cd lds[];
    for (int it = blockIdx.x; it < n_items; it += gridDim.x) {
        const int4 item = items[it];  // {system, wtile, chunk, -}
        const LatArgs a = args[item.x];
        cols_item<N, MODE, TRACE>(a, a.pSigAll, item.y, item.z, lds);
        __syncthreads();
    }
}

template <int N, int MODE, bool TRACE>
hipError_t launch_cols_k(const LatArgs& a, const cd* sig_all, hipStream_t s, const SchurMulti* m)
{
    if (a.nc < cols_nc_min(N) || a.nc > N) return hipErrorInvalidValue;  // the kernels assume this bucket
    const int nd = a.n - a.nc;
    const size_t shm = cols_lds_bytes(N, MODE);
    constexpr int SLOTS = cols_slots(N);
    if (m) {
        hipError_t e = hipFuncSetAttribute((const void*)k_lattice_schur_cols_multi<N, MODE, TRACE>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_lattice_schur_cols_multi<N, MODE, TRACE>), dim3(m->grid),
                           dim3(cols_wg()), shm, s, m->args, m->items, m->n_items);
        return hipGetLastError();
    }
    hipError_t e = hipFuncSetAttribute((const void*)k_lattice_schur_cols<N, MODE, TRACE>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return e;
    const dim3 grid = lattice_grid(a, SLOTS);
    hipLaunchKernelGGL((k_lattice_schur_cols<N, MODE, TRACE>), grid, dim3(cols_wg()), shm, s, a,
                       sig_all);
    return hipGetLastError();
}

// entry of one bucket (one translation unit each); with m, the persistent
// multi-lattice launch over m's work list (a is then only a prototype: n_c, want_trace)
template <int N>
hipError_t launch_cols_bucket(const LatArgs& a, int mode, const cd* sig_all, hipStream_t s,
                              const SchurMulti* m = nullptr)
{
    if (mode == MODE_FWD)
        return a.want_trace ? launch_cols_k<N, MODE_FWD, true>(a, sig_all, s, m)
                            : launch_cols_k<N, MODE_FWD, false>(a, sig_all, s, m);
    if (mode == MODE_DENS) return launch_cols_k<N, MODE_DENS, false>(a, sig_all, s, m);
    return launch_cols_k<N, MODE_VJP, false>(a, sig_all, s, m);
}

}  // namespace dg
