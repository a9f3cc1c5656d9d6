// Schur-complement lattice path: G_cc without the full n x n inverse.
//
// Same outputs as the plain path (the hot loop of GreenFtn_w,
// GreenFtn.cpp:218-308, and the densities of GiwToNele :513-635), computed
// from the block structure of A = (z+mu) I - H(k) - P Sigma P^H with the
// correlated orbitals first (downfolding.cpp:69-79):
//   H_dd(k) = V_d diag(e_d) V_d^H           (once per k, in dmftgpu_prepare)
//   W(k)    = H_cd V_d,  P_d = w_d w_d^H    (w_d = column d of W)
//   g_d     = 1/(z + mu - e_d)
//   S       = (z+mu) I - H_cc - Sigma - sum_d g_d P_d        (Schur complement)
//   G_cc    = S^{-1}
//   tr G    = sum_d g_d + tr G_cc + sum_d g_d^2 M_d,   M_d = w_d^H G_cc w_d
//   tr G^2  = sum_d g_d^2 + tr((G_cc S')^2) + 2 sum_d g_d^3 M_d,
//             S' = I + X, X = sum_d g_d^2 P_d
//   (G^2)_cc = G_cc S' G_cc
// (tr G = d/dz log det A = d/dz[log det A_dd + log det S]; tr G^2 = -d/dz tr G.)
// Per (k, iw) this costs ~ n_c^2 n_d + n_c^3 complex operations instead of n^3.
//
// This header holds the kernel templates; lattice_lane{1..6}.hip instantiate
// one n_c each (launch_lane_<n_c>), lattice_schur.hip dispatches.
//
// Mapping: one (k, iw) matrix per lane, in registers (n_c <= 6):
// a wavefront owns 64 consecutive frequencies and walks a chunk of k points;
// the per-k data (H_cc, e_d, P_d for pairs a <= b; built once by k_schur_kdata)
// is read with wave-uniform scalar loads.  The n_c x n_c inversion is
// Gauss-Jordan without pivoting (the Hermitian part of -iS is >= w_n I for
// causal Sigma, so elimination without pivoting is stable).
//
// Both Schur methods run this FP64 elimination.  An FP32 inverse with one FP64-residual
// step (X0 + X0 (I - S X0)) takes three times the multiply-adds, which pays only where
// FP32 arithmetic is at least that much faster: the FP32 vector rate of gfx950 without
// packed FP32 is the FP64 rate.  Measured in that form and in this one, 8000 k x 1040
// points, forward + adjoint: n = 14, n_c = 5 3.33 against 2.87 ms, n = 14, n_c = 6 9.5
// against 7.3 ms, n_c = 1 and 2 equal.
#pragma once
#include "lattice_kernels.hpp"

namespace dg {

template <int NC>
__device__ __forceinline__ void gj_inverse(cd (&S)[NC][NC])
{
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const cd p = crcp(S[j][j]);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (c != j) S[j][c] = cmul(S[j][c], p);
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if (i == j) continue;
            const cd f = S[i][j];
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (c != j) S[i][c] = cfms(f, S[j][c], S[i][c]);
            S[i][j] = cneg(cmul(f, p));
        }
        S[j][j] = p;
    }
}

// Scalar-cache fill of the next k's block before its d loops need it: one
// dword from each of the first 48 64-byte lines (3 KB; the per-k blocks are
// followed by kKdataPad bytes of padding, so the last block's fill stays in
// the allocation), all into one throw-away SGPR, waited for inside the asm
// block so that no load is in flight when it ends.  Without it every d
// block's scalar loads wait on L2 in turn; with it they hit the scalar cache.
__device__ __forceinline__ void kcache_fill(const void* base)
{
    unsigned t;
    asm volatile(
        "s_load_dword %0, %1, 0x0\n\t"
        "s_load_dword %0, %1, 0x40\n\t"
        "s_load_dword %0, %1, 0x80\n\t"
        "s_load_dword %0, %1, 0xc0\n\t"
        "s_load_dword %0, %1, 0x100\n\t"
        "s_load_dword %0, %1, 0x140\n\t"
        "s_load_dword %0, %1, 0x180\n\t"
        "s_load_dword %0, %1, 0x1c0\n\t"
        "s_load_dword %0, %1, 0x200\n\t"
        "s_load_dword %0, %1, 0x240\n\t"
        "s_load_dword %0, %1, 0x280\n\t"
        "s_load_dword %0, %1, 0x2c0\n\t"
        "s_load_dword %0, %1, 0x300\n\t"
        "s_load_dword %0, %1, 0x340\n\t"
        "s_load_dword %0, %1, 0x380\n\t"
        "s_load_dword %0, %1, 0x3c0\n\t"
        "s_load_dword %0, %1, 0x400\n\t"
        "s_load_dword %0, %1, 0x440\n\t"
        "s_load_dword %0, %1, 0x480\n\t"
        "s_load_dword %0, %1, 0x4c0\n\t"
        "s_load_dword %0, %1, 0x500\n\t"
        "s_load_dword %0, %1, 0x540\n\t"
        "s_load_dword %0, %1, 0x580\n\t"
        "s_load_dword %0, %1, 0x5c0\n\t"
        "s_load_dword %0, %1, 0x600\n\t"
        "s_load_dword %0, %1, 0x640\n\t"
        "s_load_dword %0, %1, 0x680\n\t"
        "s_load_dword %0, %1, 0x6c0\n\t"
        "s_load_dword %0, %1, 0x700\n\t"
        "s_load_dword %0, %1, 0x740\n\t"
        "s_load_dword %0, %1, 0x780\n\t"
        "s_load_dword %0, %1, 0x7c0\n\t"
        "s_load_dword %0, %1, 0x800\n\t"
        "s_load_dword %0, %1, 0x840\n\t"
        "s_load_dword %0, %1, 0x880\n\t"
        "s_load_dword %0, %1, 0x8c0\n\t"
        "s_load_dword %0, %1, 0x900\n\t"
        "s_load_dword %0, %1, 0x940\n\t"
        "s_load_dword %0, %1, 0x980\n\t"
        "s_load_dword %0, %1, 0x9c0\n\t"
        "s_load_dword %0, %1, 0xa00\n\t"
        "s_load_dword %0, %1, 0xa40\n\t"
        "s_load_dword %0, %1, 0xa80\n\t"
        "s_load_dword %0, %1, 0xac0\n\t"
        "s_load_dword %0, %1, 0xb00\n\t"
        "s_load_dword %0, %1, 0xb40\n\t"
        "s_load_dword %0, %1, 0xb80\n\t"
        "s_load_dword %0, %1, 0xbc0\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(t)
        : "s"(base));
    asm volatile("" ::"s"(t));
}

// per-k block (k_schur_kdata): [Hcc: NC*NC cd][P: nd*NP cd][e_d: nd doubles]
template <int NC>
__host__ __device__ __forceinline__ int kblock_size(int nd)
{
    constexpr int NP = NC * (NC + 1) / 2;
    return NC * NC + nd * NP + (nd + 1) / 2;
}

template <int NC>
__host__ __device__ constexpr bool schur_sig_lds() { return NC <= 4; }
template <int NC, int MODE, int KS>
__host__ __device__ constexpr bool schur_sum_lds() { return (MODE == MODE_VJP && KS > 1) || (MODE == MODE_DENS && NC == 5); }

template <int I>
struct ColumnIndex {
    static constexpr int value = I;
};
// f(0), ..., f(NC - 1), or f(b) for a wave-uniform b, with the column as a constant
template <int NC, int B = 0, class F>
__device__ __forceinline__ void for_columns(F&& f)
{
    if constexpr (B < NC) {
        f(ColumnIndex<B>{});
        for_columns<NC, B + 1>(f);
    }
}
template <int NC, int B = 0, class F>
__device__ __forceinline__ void pick_column(int b, F&& f)
{
    if constexpr (B < NC) {
        if (b == B) f(ColumnIndex<B>{});
        else pick_column<NC, B + 1>(b, f);
    }
}

// One (frequency tile, k chunk) work item.  The per-k block is read from
// a.kdata through the constant address space: its addresses are wave-uniform,
// so the loads become scalar loads and the products against it take SGPR
// operands, with no LDS traffic and no barriers in the k loop.
// KS > 1 (schur_ksplit): the WG lanes are KS
// groups of wavefronts over the same WG / KS frequencies, each walking every KS-th k
// of the chunk and adding into one set of LDS accumulators.
template <int NC, int MODE, int WG, bool TRACE, int KS = 1>
__device__ __forceinline__ void schur_item(const LatArgs& a, const cd* __restrict__ sig_all, int wtile, int chunk,
                                           cd* lds)
{
    using BT = kconst_cd;
    using BD = kconst_double;
    constexpr int NP = NC * (NC + 1) / 2;
    constexpr int M2 = NC * NC;
    constexpr bool FWDLIKE = MODE == MODE_FWD || MODE == MODE_FWD_REAL;
    // accumulators that do not fit next to the working matrices live in LDS
    constexpr bool ACC_LDS = MODE == MODE_VJP || KS > 1;
    constexpr int FW = WG / KS;       // frequencies per workgroup
    // adjoint, KS > 1: Sigma in LDS too, where that leaves room for three workgroups to
    // a CU (n_c = 4); at n_c = 5 it would fit twice but gained nothing at n_d = 9 and lost
    // 14 % at n_d = 18
    constexpr bool SIG_LDS = MODE == MODE_VJP && KS > 1 && schur_sig_lds<NC>();
    static_assert(KS == 1 || (FW % 64 == 0 && (FWDLIKE ? KS == 2 : MODE == MODE_VJP)),
                  "split k walk: forward pairs or the adjoint, whole wavefronts per part");
    const int nd = a.n - NC;
    const int bs = kblock_size<NC>(nd);
    cd* sAcc = lds;                   // [M2][FW] complex, frequency-contiguous
    cd* sTr = lds + M2 * FW;          // KS > 1: forward [FW] sums of the tr G shares
    cd* sGb = lds + M2 * FW;          //         adjoint [M2][FW] gbar, [M2][FW] Sigma
    cd* sSig = lds + 2 * M2 * FW;
    // sums of tr G, tr G^2 and the mu term in LDS where registers are short (adjoint with
    // KS > 1: one set a part)
    constexpr bool SUM_LDS = schur_sum_lds<NC, MODE, KS>();
    cd* sSum = nullptr;
    const int lane = KS == 1 ? (int)threadIdx.x : (int)threadIdx.x % FW;  // this lane's frequency in the tile
    // which k of every KS: wave-uniform (FW is a multiple of 64), so that the k
    // walk and the per-k block addresses stay scalar
    const int part = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / FW);
    if constexpr (SUM_LDS) {
        sSum = lds + (MODE == MODE_DENS ? 0 : SIG_LDS ? 3 : 2) * M2 * FW + 3 * part * FW + lane;
        for (int q = 0; q < 3; ++q) sSum[q * FW] = cd{0.0, 0.0};
    }
    const int nw_hi = n_points(a);
    const int nw = wtile * FW + lane;
    // a wavefront past the last point has no work (KS > 1: they meet at barriers, so
    // only a whole workgroup leaves)
    if ((KS > 1 ? wtile * FW : __builtin_amdgcn_readfirstlane(nw)) >= nw_hi) return;
    const bool wvalid = nw < nw_hi;
    const int nwc = wvalid ? nw : nw_hi - 1;  // clamp for loads
    const int k0 = chunk * a.k_per_chunk;
    const int k1 = min(a.nk, k0 + a.k_per_chunk);
    // z + mu = (mu + shift) + i w: the Matsubara point, or on the real axis E + mu + i eta
    double mu, w;
    if constexpr (MODE == MODE_FWD_REAL) {
        freq_point(a, nwc, mu, w);
    } else {
        w = a.pt_w ? a.pt_w[nwc] : matsubara(nwc, a.beta);
        mu = a.mu;
    }
    const bool vjp_here = (MODE == MODE_VJP) && wvalid && nw < a.n_freq;
    const bool tile_vjp = wtile * FW < a.n_freq;  // the same for the whole workgroup
    const cd* sig = sig_all + (size_t)nwc * M2;
    const cd* gb = (MODE == MODE_VJP) ? a.gbar + (size_t)(nw < a.n_freq ? nw : 0) * M2 : nullptr;
    // nbar: host value, or (batched adjoint) a device scalar written by an earlier kernel
    const double cn = 2.0 * (a.nbar_dev ? *a.nbar_dev : a.nbar) / a.beta;

    cd acc[ACC_LDS ? 1 : NC][ACC_LDS ? 1 : NC];
    if (ACC_LDS) {
        // (KS > 1: every part clears the same entries, before the barrier below)
        for (int e = 0; e < M2; ++e) sAcc[e * FW + lane] = cd{0.0, 0.0};
        if constexpr (KS > 1) {
            if constexpr (MODE == MODE_VJP) {
                for (int e = part; e < M2; e += KS) {
                    sGb[e * FW + lane] = gb[e];
                    if constexpr (SIG_LDS) sSig[e * FW + lane] = sig[e];
                }
            } else {
                sTr[lane] = cd{0.0, 0.0};
            }
            __syncthreads();
        }
    } else {
#pragma unroll
        for (int i = 0; i < (ACC_LDS ? 1 : NC); ++i)
#pragma unroll
            for (int j = 0; j < (ACC_LDS ? 1 : NC); ++j) acc[i][j] = cd{0.0, 0.0};
    }
    cd trA = cd{0.0, 0.0}, tr2A = cd{0.0, 0.0}, muA = cd{0.0, 0.0};

    // KS > 1: both parts take the same number of steps (the barriers below); a
    // part past the chunk's end repeats its last k and adds nothing
    for (int kb = k0; kb < k1; kb += KS) {
        const int k = KS == 1 ? kb : min(kb + part, k1 - 1);
        const bool kin = KS == 1 || kb + part < k1;
        // Sigma(iw) is re-read from the cache every k rather than hoisted out
        // of the loop, where it would hold 4*NC*NC registers for its duration.
        // The k block is read through the constant address space, which the
        // compiler treats as invariant: those loads stay scalar despite the
        // clobber.
        __asm__ __volatile__("" ::: "memory");
        // Sigma's loads are issued here, all together, so that they complete under
        // the d loop below instead of waiting in turn where S is combined; not in
        // the FP64 forward kernels, whose G_cc sums already fill the registers
        constexpr bool SIG_EARLY = !FWDLIKE && !SIG_LDS, SIG_REG = SIG_EARLY || SIG_LDS;
        cd sg[SIG_REG ? NC : 1][SIG_REG ? NC : 1];
        if constexpr (SIG_EARLY) {
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia < NC; ++ia) sg[ia][ib] = sig[ia + ib * NC];
        }
        kcache_fill(a.kdata + (size_t)k * bs);
        auto sig_at = [&](int ia, int ib) -> cd {
            if constexpr (SIG_REG) return sg[ia][ib];
            else return sig[ia + ib * NC];
        };
        const BT* B = (const BT*)(a.kdata + (size_t)k * bs);
        const BT* Hcc = B;
        const BT* P = B + M2;
        const BD* ed = (const BD*)(P + nd * NP);
        // ---- Schur complement S = (z+mu) I - H_cc - Sigma - sum_d g_d P_d.
        // sum_d g_d P_d = R + i J with R = sum_d Re(g_d) P_d and
        // J = sum_d Im(g_d) P_d both Hermitian: their upper triangles (real
        // diagonals) are accumulated in place of S, G[a][b] = R_ab,
        // G[b][a] = J_ab (a < b), G[a][a] = (R_aa, J_aa), a real-by-complex
        // update per stored entry (4 FMA per pair instead of 8).
        cd G[NC][NC];
#pragma unroll
        for (int j = 0; j < NC; ++j)
#pragma unroll
            for (int i = 0; i < NC; ++i) G[i][j] = cd{0.0, 0.0};
        // g_d = 1/(z + mu - e_d) one d ahead: its reciprocal chain is independent
        // of the d step's FMAs, so the two interleave instead of the chain
        // stalling the top of every step; e_{d+1} is read one step earlier still,
        // with that step's P_d, so that the chain does not wait for it either
        auto g_of = [&](double e) -> cd {
            const double x = mu - e;
            const double r = rcp_pos(fma(x, x, w * w));
            return cd{x * r, -w * r};
        };
        auto e_at = [&](int d) -> double { return (double)ed[d < nd ? d : nd - 1]; };
        cd g_next = nd > 0 ? g_of(e_at(0)) : cd{0.0, 0.0};
        double e_next = nd > 0 ? e_at(1) : 0.0;
        for (int d = 0; d < nd; ++d) {
            const double gr = g_next.x, gi = g_next.y;
            g_next = g_of(e_next);
            e_next = e_at(d + 2);
            const BT* Pd = P + d * NP;
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia <= ib; ++ia) {
                    const cd p = ldc(Pd + ib * (ib + 1) / 2 + ia);
                    if (ia == ib) {  // P_aa is real
                        G[ia][ia].x = fma(gr, p.x, G[ia][ia].x);
                        G[ia][ia].y = fma(gi, p.x, G[ia][ia].y);
                    } else {
                        G[ia][ib] = cd{fma(gr, p.x, G[ia][ib].x), fma(gr, p.y, G[ia][ib].y)};
                        G[ib][ia] = cd{fma(gi, p.x, G[ib][ia].x), fma(gi, p.y, G[ib][ia].y)};
                    }
                }
        }
        if constexpr (SIG_LDS) {
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia < NC; ++ia) sg[ia][ib] = sSig[(ia + ib * NC) * FW + lane];
            __builtin_amdgcn_sched_barrier(0);  // issued together
        }
#pragma unroll
        for (int ib = 0; ib < NC; ++ib)
#pragma unroll
            for (int ia = 0; ia <= ib; ++ia) {
                cd bab = csub(cneg(ldc(Hcc + ia + ib * NC)), sig_at(ia, ib));
                if (ia == ib) {
                    bab = cadd(bab, cd{mu, w});
                    G[ia][ia] = csub(bab, G[ia][ia]);  // - (R_aa + i J_aa)
                } else {
                    const cd R = G[ia][ib], J = G[ib][ia];
                    const cd bba = csub(cneg(ldc(Hcc + ib + ia * NC)), sig_at(ib, ia));
                    G[ia][ib] = csub(bab, cd{R.x - J.y, R.y + J.x});   // - (R + i J)_ab
                    G[ib][ia] = csub(bba, cd{R.x + J.y, J.x - R.y});   // - (R + i J)_ba
                }
            }
        // ---- G_cc = S^{-1}
        gj_inverse<NC>(G);

        if (FWDLIKE) {
            if constexpr (ACC_LDS) {
                // the parts add in turn, part 0 first, so that every sum has one
                // order and the result is the same on every run
                auto add_g = [&]() {
#pragma unroll
                    for (int j = 0; j < NC; ++j)
#pragma unroll
                        for (int i = 0; i < NC; ++i) lds_add(&sAcc[(i + j * NC) * FW + lane], G[i][j]);
                };
                __syncthreads();
                if (part == 0) add_g();
                __syncthreads();
                if (part == 1 && kin) add_g();
            } else {
#pragma unroll
                for (int i = 0; i < (ACC_LDS ? 1 : NC); ++i)
#pragma unroll
                    for (int j = 0; j < (ACC_LDS ? 1 : NC); ++j) acc[i][j] = cadd(acc[i][j], G[i][j]);
            }
            if (TRACE) {  // tr G = sum_d g_d + tr G_cc + sum_d g_d^2 M_d
                cd t = cd{0.0, 0.0};
#pragma unroll
                for (int i = 0; i < NC; ++i) t = cadd(t, G[i][i]);
                // M_d = sum_ab G_ab P_d(b, a): for a < b the pair contributes
                // Re = (G_ab + G_ba).x p.x + (G_ab - G_ba).y p.y and
                // Im = (G_ab + G_ba).y p.x + (G_ba - G_ab).x p.y (p = P_d(a, b)),
                // so G is folded once into those sums (in place; G is not needed
                // after this) and each pair costs 4 FMA per d.
#pragma unroll
                for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                    for (int ia = 0; ia < ib; ++ia) {
                        const cd x1 = G[ia][ib], x2 = G[ib][ia];
                        G[ia][ib] = cd{x1.x + x2.x, x1.y - x2.y};
                        G[ib][ia] = cd{x1.y + x2.y, x2.x - x1.x};
                    }
                g_next = nd > 0 ? g_of(e_at(0)) : cd{0.0, 0.0};
                e_next = nd > 0 ? e_at(1) : 0.0;
                for (int d = 0; d < nd; ++d) {
                    const cd g = g_next;
                    g_next = g_of(e_next);
                    e_next = e_at(d + 2);
                    const BT* Pd = P + d * NP;
                    cd Md = cd{0.0, 0.0};
#pragma unroll
                    for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                        for (int ia = 0; ia <= ib; ++ia) {
                            const cd p = ldc(Pd + ib * (ib + 1) / 2 + ia);
                            if (ia == ib) {
                                Md.x = fma(G[ia][ia].x, p.x, Md.x);
                                Md.y = fma(G[ia][ia].y, p.x, Md.y);
                            } else {
                                const cd sd = G[ia][ib], sm = G[ib][ia];
                                Md.x = fma(sd.x, p.x, fma(sd.y, p.y, Md.x));
                                Md.y = fma(sm.x, p.x, fma(sm.y, p.y, Md.y));
                            }
                        }
                    t = cadd(t, cadd(g, cmul(cmul(g, g), Md)));
                }
                if (wvalid && kin) trA = cadd(trA, t);
            }
        } else {
            // the adjoint's cotangent (KS > 1: in LDS), on its way during the d loop below
            // (it is k-invariant; kept across k it would hold 4 NC^2 registers)
            constexpr bool GB_REG = MODE == MODE_VJP && KS == 1;
            cd gbv[GB_REG ? NC : 1][GB_REG ? NC : 1];
            if constexpr (GB_REG) {
#pragma unroll
                for (int j = 0; j < NC; ++j)
#pragma unroll
                    for (int i = 0; i < NC; ++i) gbv[i][j] = gb[i + j * NC];
            }
            // ---- Y = sum_d g_d^2 P_d (X of the header), trace terms via M_d = w_d^H G w_d
            cd Y[NC][NC];
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int j = 0; j < NC; ++j) Y[i][j] = cd{0.0, 0.0};
            cd trG = cd{0.0, 0.0}, tz = cd{0.0, 0.0};  // sum_d g + g^2 M_d, sum_d g^2 + 2 g^3 M_d
            // Y is accumulated as R + i J (R = sum Re(g^2) P_d, J = sum Im(g^2) P_d,
            // upper triangles in place: Y[a][b] = R_ab, Y[b][a] = J_ab), as S is
            // M_d = sum_ab conj(w_a) G_ab w_b = sum_ab G_ab P_{ba} with G folded
            // into pair sums for the loop (as in the forward trace) and
            // unfolded after it: for a < b, G[a][b] <- (G_ab + G_ba).x, (G_ab - G_ba).y
            // and G[b][a] <- (G_ab + G_ba).y, (G_ba - G_ab).x
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia < ib; ++ia) {
                    const cd x1 = G[ia][ib], x2 = G[ib][ia];
                    G[ia][ib] = cd{x1.x + x2.x, x1.y - x2.y};
                    G[ib][ia] = cd{x1.y + x2.y, x2.x - x1.x};
                }
            g_next = nd > 0 ? g_of(e_at(0)) : cd{0.0, 0.0};
            e_next = nd > 0 ? e_at(1) : 0.0;
            for (int d = 0; d < nd; ++d) {
                const cd g = g_next;
                g_next = g_of(e_next);
                e_next = e_at(d + 2);
                const cd g2 = cmul(g, g);
                const BT* Pd = P + d * NP;
                cd Md = cd{0.0, 0.0};
#pragma unroll
                for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                    for (int ia = 0; ia <= ib; ++ia) {
                        const cd p = ldc(Pd + ib * (ib + 1) / 2 + ia);  // P_{ia ib} = w_a conj(w_b)
                        if (ia == ib) {
                            Y[ia][ia].x = fma(g2.x, p.x, Y[ia][ia].x);
                            Y[ia][ia].y = fma(g2.y, p.x, Y[ia][ia].y);
                            Md.x = fma(G[ia][ia].x, p.x, Md.x);
                            Md.y = fma(G[ia][ia].y, p.x, Md.y);
                        } else {
                            Y[ia][ib] = cd{fma(g2.x, p.x, Y[ia][ib].x), fma(g2.x, p.y, Y[ia][ib].y)};
                            Y[ib][ia] = cd{fma(g2.y, p.x, Y[ib][ia].x), fma(g2.y, p.y, Y[ib][ia].y)};
                            const cd sd = G[ia][ib], sm = G[ib][ia];
                            Md.x = fma(sd.x, p.x, fma(sd.y, p.y, Md.x));
                            Md.y = fma(sm.x, p.x, fma(sm.y, p.y, Md.y));
                        }
                    }
                trG = cfma(g2, Md, cadd(trG, g));
                tz = cfma(cscale(cmul(g2, g), 2.0), Md, cadd(tz, g2));
            }
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia < ib; ++ia) {
                    const cd a1 = G[ia][ib], a2 = G[ib][ia];
                    G[ia][ib] = cd{0.5 * (a1.x - a2.y), 0.5 * (a2.x + a1.y)};
                    G[ib][ia] = cd{0.5 * (a1.x + a2.y), 0.5 * (a2.x - a1.y)};
                }
#pragma unroll
            for (int ib = 0; ib < NC; ++ib)
#pragma unroll
                for (int ia = 0; ia < ib; ++ia) {
                    const cd R = Y[ia][ib], J = Y[ib][ia];
                    Y[ia][ib] = cd{R.x - J.y, R.y + J.x};
                    Y[ib][ia] = cd{R.x + J.y, J.x - R.y};
                }
#pragma unroll
            for (int i = 0; i < NC; ++i) trG = cadd(trG, G[i][i]);
            if constexpr (SUM_LDS) {  // out of the registers before the product
                if (kin) {
                    lds_add(&sSum[0], trG);
                    lds_add(&sSum[FW], tz);
                }
                tz = cd{0.0, 0.0};
            }
            // Z = G S' = G + G Y, column by column in place of Y
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                cd t[NC];
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    cd s = G[i][j];
#pragma unroll
                    for (int l = 0; l < NC; ++l) s = cfma(G[i][l], Y[l][j], s);
                    t[i] = s;
                }
#pragma unroll
                for (int i = 0; i < NC; ++i) Y[i][j] = t[i];
            }
            cd(&Z)[NC][NC] = Y;
            // tr(Z^2) = sum_i Z_ii^2 + 2 sum_{i<j} Z_ij Z_ji
            {
                cd off = cd{0.0, 0.0};
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    tz = cfma(Z[i][i], Z[i][i], tz);
#pragma unroll
                    for (int j = i + 1; j < NC; ++j) off = cfma(Z[i][j], Z[j][i], off);
                }
                tz = cadd(tz, cscale(off, 2.0));
            }
            if constexpr (SUM_LDS) {
                if (kin) lds_add(&sSum[FW], tz);
            } else if (wvalid && kin) {
                trA = cadd(trA, trG);
                tr2A = cadd(tr2A, tz);
            }
            if (MODE == MODE_VJP && tile_vjp) {
                // sigma_bar += G^H gbar G^H + cn ((G^2)_cc)^H with (G^2)_cc = Z G: column b
                // of both is G^H t, t_i = s_i + cn conj(Z_bi), s_i = sum_l gbar_il conj(G_bl).
                // mu term tr(gbar^H (G^2)_cc) = tr(Z G gbar^H) = sum_bi Z_ib conj(s_i), as
                // (G gbar^H)_bi = conj(s_i).  G and Z are all that lives here; with
                // V = gbar + cn S'^H as a third matrix n_c = 6 spilled 0.6 KB per lane.
                cd ms = cd{0.0, 0.0};
                auto gbar_at = [&](int i, int l) -> cd {
                    if constexpr (GB_REG) return gbv[i][l];
                    else return sGb[(i + l * NC) * FW + lane];
                };
                auto barrier = [] {
                    if constexpr (KS > 1) __builtin_amdgcn_sched_barrier(0);
                };
                auto column = [&](auto bc) {
                    constexpr int b = decltype(bc)::value;
                    // gbar (rows in turn, then the column's sums) comes AHEAD entries early, an
                    // entry's registers loaded again as soon as it is used: left to itself the
                    // compiler reads one entry, waits and uses it, an LDS round trip per entry
                    constexpr int AHEAD = 3;
                    auto fetch = [&](int q) -> cd {
                        if (q >= M2 + NC) return cd{0.0, 0.0};  // past the last (n_c < AHEAD), not used
                        return q < M2 ? gbar_at(q / NC, q % NC) : sAcc[(q - M2 + b * NC) * FW + lane];
                    };
                    cd buf[AHEAD], t[NC];
#pragma unroll
                    for (int q = 0; q < AHEAD; ++q) buf[q] = fetch(q);
                    barrier();
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        cd s = cd{0.0, 0.0};
#pragma unroll
                        for (int l = 0; l < NC; ++l) {
                            const int q = i * NC + l;
                            s = cfma(buf[q % AHEAD], cconj(G[b][l]), s);
                            buf[q % AHEAD] = fetch(q + AHEAD);
                            barrier();
                        }
                        ms = cfmac(s, Z[i][b], ms);
                        t[i] = cd{fma(cn, Z[b][i].x, s.x), fma(-cn, Z[b][i].y, s.y)};
                    }
#pragma unroll
                    for (int aa = 0; aa < NC; ++aa) {  // C_ab = sum_i conj(G_ia) t_i
                        cd s = buf[(M2 + aa) % AHEAD];
                        if (aa + AHEAD < NC) buf[(M2 + aa) % AHEAD] = fetch(M2 + aa + AHEAD);
#pragma unroll
                        for (int i = 0; i < NC; ++i) s = cfmac(G[i][aa], t[i], s);
                        sAcc[(aa + b * NC) * FW + lane] = s;
                    }
                };
                if constexpr (KS == 1) {
                    for_columns<NC>(column);
                } else {
                    // part p takes column p + step (mod the number of steps): at each step the
                    // parts add to different columns, and every sum has one order
                    constexpr int STEPS = NC > KS ? NC : KS;
                    int b = part;
#pragma unroll 1
                    for (int st = 0; st < STEPS; ++st) {
                        if (kin) pick_column<NC>(b, column);
                        b = b + 1 == STEPS ? 0 : b + 1;
                        __syncthreads();
                    }
                }
                if constexpr (SUM_LDS) lds_add(&sSum[2 * FW], ms);
                else if (vjp_here) muA = cadd(muA, ms);
            }
        }
    }

    if constexpr (KS > 1) {  // the parts' tr G shares and G_cc sums meet in LDS; part 0 writes them
        if constexpr (FWDLIKE) {
            lds_add(&sTr[lane], trA);
            __syncthreads();
            if (part != 0) return;
            trA = sTr[lane];
        } else {
            __syncthreads();
            if (part == 0)
                for (int p = 0; p < KS; ++p) {
                    trA = cadd(trA, sSum[3 * p * FW]);
                    tr2A = cadd(tr2A, sSum[(3 * p + 1) * FW]);
                    muA = cadd(muA, sSum[(3 * p + 2) * FW]);
                }
        }
    }
    if constexpr (SUM_LDS && KS == 1) {
        trA = sSum[0];
        tr2A = sSum[FW];
    }
    if (!wvalid) return;
    const size_t ch = chunk;
    if (MODE == MODE_FWD || MODE == MODE_FWD_REAL) {
        a.pTr[ch * a.nw_tot + nw] = trA;
        if (ACC_LDS) {
            for (int e = 0; e < M2; ++e) a.pG[(ch * a.nw_tot + nw) * M2 + e] = sAcc[e * FW + lane];
        } else {
#pragma unroll
            for (int i = 0; i < (ACC_LDS ? 1 : NC); ++i)
#pragma unroll
                for (int j = 0; j < (ACC_LDS ? 1 : NC); ++j)
                    a.pG[(ch * a.nw_tot + nw) * M2 + i + j * NC] = acc[i][j];
        }
    } else {
        if (part == 0) {
            a.pTr[ch * a.nw_tot + nw] = trA;
            a.pTr2[ch * a.nw_tot + nw] = tr2A;
            if (MODE == MODE_VJP && vjp_here) a.pMu[ch * a.n_freq + nw] = muA;
        }
        if (MODE == MODE_VJP && vjp_here)
            for (int e = part; e < M2; e += KS) a.pSb[(ch * a.n_freq + nw) * M2 + e] = sAcc[e * FW + lane];
    }
}

// Waves per SIMD the register allocator is held to: as many as fit without values
// spilled in the k walk (at these rates a spilled value a lane is gigabytes of writes:
// with 136 B of scratch the adjoint at n_c = 5 wrote 8 GB a launch, and the loss and
// gradient of 32^3 k x 2048 frequencies took 20.5 ms against 18.4).
template <int NC, int MODE, int KS>
constexpr int schur_waves()
{
    if (MODE == MODE_VJP) return NC == 4 || (NC == 5 && KS > 1) ? 2 : 1;
    if (KS > 1) return NC <= 4 ? 4 : NC == 5 ? 3 : 2;
    return NC == 5 ? 2 : 1;
}

template <int NC, int MODE, int WG, bool TRACE, int KS = 1>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(schur_waves<NC, MODE, KS>())))
void k_lattice_schur(LatArgs a, const cd* __restrict__ sig_all)
{
    extern __shared__ cd lds[];
    schur_item<NC, MODE, WG, TRACE, KS>(a, sig_all, lattice_tile(), blockIdx.y, lds);
}

// Persistent form over a work list spanning several lattices of the same n_c:
// workgroup b takes items b, b + gridDim.x, ... (static striding, no atomics,
// so every replay does the same work in the same order).  Each system's per-k
// blocks come from its LatArgs (kdata), read through the constant address space.
template <int NC, int MODE, int WG, bool TRACE, int KS = 1>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(schur_waves<NC, MODE, KS>())))
void k_lattice_schur_multi(const LatArgs* __restrict__ args,
                                                            const int4* __restrict__ items, int n_items)
{
    extern __shared__ cd lds[];
    for (int it = blockIdx.x; it < n_items; it += gridDim.x) {
        const int4 item = items[it];  // {system, wtile, chunk, -}
        const LatArgs a = args[item.x];
        schur_item<NC, MODE, WG, TRACE, KS>(a, a.pSigAll, item.y, item.z, lds);
        __syncthreads();
    }
}

template <int NC, int MODE, int WG, int KS = 1>
constexpr size_t schur_shm()
{
    if (MODE == MODE_DENS) return schur_sum_lds<NC, MODE, KS>() ? sizeof(cd) * 3 * (size_t)WG : 0;
    constexpr bool ACC_LDS = MODE == MODE_VJP || KS > 1;
    // KS > 1: one accumulator set per frequency, plus the tr G sums (forward) or gbar,
    // Sigma and the parts' three sums (adjoint)
    constexpr int extra = KS == 1 ? 0 : MODE != MODE_VJP ? 1 : (schur_sig_lds<NC>() ? 2 : 1) * NC * NC + 3 * KS;
    return ACC_LDS ? sizeof(cd) * (size_t)(NC * NC + extra) * (WG / KS) : 0;
}

template <int NC, int MODE, bool TRACE, int WG, int KS = 1>
hipError_t launch_nc_w(const LatArgs& a, const cd* sig_all, hipStream_t s, const SchurMulti* multi)
{
    constexpr size_t shm = schur_shm<NC, MODE, WG, KS>();
    if (multi) {
        hipError_t e = hipFuncSetAttribute((const void*)k_lattice_schur_multi<NC, MODE, WG, TRACE, KS>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_lattice_schur_multi<NC, MODE, WG, TRACE, KS>), dim3(multi->grid), dim3(WG),
                           shm, s, multi->args, multi->items, multi->n_items);
        return hipGetLastError();
    }
    constexpr int FW = WG / KS;  // frequencies per workgroup
    const dim3 grid = lattice_grid(a, FW);
    hipError_t e = hipFuncSetAttribute((const void*)k_lattice_schur<NC, MODE, WG, TRACE, KS>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_lattice_schur<NC, MODE, WG, TRACE, KS>), grid, dim3(WG), shm, s, a, sig_all);
    return hipGetLastError();
}

template <int NC, int MODE, bool TRACE>
hipError_t launch_nc(const LatArgs& a, const cd* sig_all, hipStream_t s, int wg, const SchurMulti* m)
{
    if constexpr (NC >= 3 && (MODE == MODE_FWD || MODE == MODE_FWD_REAL)) {  // two wavefronts over 64 frequencies
        if (wg == SCHUR_WG_KSPLIT) return launch_nc_w<NC, MODE, TRACE, 128, 2>(a, sig_all, s, m);
    }
    if constexpr (NC >= 4 && MODE == MODE_VJP) {  // four, or at n_c = 6 two
        constexpr int KS = schur_parts(NC, MODE_VJP);
        if (wg == SCHUR_WG_KSPLIT) return launch_nc_w<NC, MODE, TRACE, 64 * KS, KS>(a, sig_all, s, m);
    }
    if (wg == 128) return launch_nc_w<NC, MODE, TRACE, 128>(a, sig_all, s, m);
    return launch_nc_w<NC, MODE, TRACE, 64>(a, sig_all, s, m);
}

// All variants of one n_c: mode, trace.
template <int NC>
hipError_t launch_lane_nc(const LatArgs& a, int mode, const cd* sig_all, hipStream_t s, int wg, const SchurMulti* m)
{
    if (mode == MODE_FWD)
        return a.want_trace ? launch_nc<NC, MODE_FWD, true>(a, sig_all, s, wg, m)
                            : launch_nc<NC, MODE_FWD, false>(a, sig_all, s, wg, m);
    if (mode == MODE_FWD_REAL)
        return a.want_trace ? launch_nc<NC, MODE_FWD_REAL, true>(a, sig_all, s, wg, m)
                            : launch_nc<NC, MODE_FWD_REAL, false>(a, sig_all, s, wg, m);
    if (mode == MODE_DENS) return launch_nc<NC, MODE_DENS, false>(a, sig_all, s, wg, m);
    return launch_nc<NC, MODE_VJP, false>(a, sig_all, s, wg, m);
}

}  // namespace dg
