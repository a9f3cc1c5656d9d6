// The sums of FourierTransform_tau (FourierTransform.cpp:46-90) and FT_t_to_w (:531-547)
// on the uniform tau grid as chirp-z transforms.
//
// With tau_j = j beta/N and w_n = pi (2n+1)/beta the phase w_n tau_j is pi (2n+1) j / N,
// an integer multiple of pi/N: both sums are transforms by e^{-+ 2 pi i n j/N} with an
// extra factor e^{-+ i pi j/N}, for any N and any number of frequencies.  Writing
// 2ab = a^2 + b^2 - (b-a)^2 turns a tile of 2048 inputs x 2048 outputs into a
// convolution with the chirp e^{i pi k^2/N}, done by FFTs of length 4096; the tile's
// offsets only add phases that are linear in a or in b.  The phases are exact: integer
// multiples reduced mod 2N, looked up in one table of e^{i pi m/N}.
//
// Cost: 2 FFTs per tile and matrix element instead of 2048^2 products.  At d = 10, N_freq =
// 4096, N_tau = 8192 the kernel takes 64 us (iw -> tau) and 67 us (tau -> iw) where the dense sums
// on FP64 MFMA took 739 and 1197 us; down to one tile (N_freq = 64) the whole call is no slower
// either, so there is no dense form on the uniform grid.  Errors against 64-bit sums with
// exact phases fall too (2.6e-14 -> 4e-15 at that size): the dense form rounded w tau.
//
// The FFT: 256 threads hold 16 elements each (element t + 256 r in register r), three
// radix-16 passes with two exchanges through LDS (68 KB with one pad element in 16, so
// that the strided stores of the first pass spread over the banks; two workgroups per
// CU).  Input and output order are the same, so the product with the chirp's spectrum and
// the second FFT follow in registers.
#include "ft_czt.hpp"

#include <algorithm>

namespace dg {

namespace {

__device__ __forceinline__ cd mul_mi(cd a) { return cd{a.y, -a.x}; }  // -i a

// x[0..3] -> DFT of length 4, e^{-2 pi i jk/4}
__device__ __forceinline__ void dft4(cd& a, cd& b, cd& c, cd& d)
{
    const cd s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = mul_mi(csub(b, d));
    a = cadd(s0, s2);
    b = cadd(s1, s3);
    c = csub(s0, s2);
    d = csub(s1, s3);
}

// v -> DFT of length 16, natural order
__device__ __forceinline__ void dft16(cd (&v)[16])
{
    constexpr double C1 = 0.92387953251128675613, S1 = 0.38268343236508977173, R = 0.70710678118654752440;
#pragma unroll
    for (int i = 0; i < 4; ++i) dft4(v[i], v[i + 4], v[i + 8], v[i + 12]);
    // twiddles e^{-2 pi i i k/16}, row k = element i + 4k
    v[5] = cmul(v[5], cd{C1, -S1});
    v[6] = cmul(v[6], cd{R, -R});
    v[7] = cmul(v[7], cd{S1, -C1});
    v[9] = cmul(v[9], cd{R, -R});
    v[10] = mul_mi(v[10]);
    v[11] = cmul(v[11], cd{-R, -R});
    v[13] = cmul(v[13], cd{S1, -C1});
    v[14] = cmul(v[14], cd{-R, -R});
    v[15] = cmul(v[15], cd{-C1, S1});
    cd o[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        cd a = v[4 * k], b = v[4 * k + 1], c = v[4 * k + 2], d = v[4 * k + 3];
        dft4(a, b, c, d);
        o[k] = a;
        o[k + 4] = b;
        o[k + 8] = c;
        o[k + 12] = d;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = o[r];
}

__device__ __forceinline__ int pad(int i) { return i + (i >> 4); }
constexpr int kFftLds = kCztM + kCztM / 16;

// FFT of length 4096 of the elements t + 256 r (thread t, register r), same order out
__device__ void fft4096(cd (&v)[16], cd* sm, const cd* __restrict__ tw, int t)
{
    dft16(v);
    __syncthreads();  // sm is free again
#pragma unroll
    for (int r = 0; r < 16; ++r) sm[pad(16 * t + r)] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = sm[pad(t + 256 * r)];
    const int k1 = t & 15;
#pragma unroll
    for (int r = 1; r < 16; ++r) v[r] = cmul(v[r], tw[16 * r * k1]);
    dft16(v);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) sm[pad((t >> 4) * 256 + k1 + 16 * r)] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = sm[pad(t + 256 * r)];
#pragma unroll
    for (int r = 1; r < 16; ++r) v[r] = cmul(v[r], tw[r * t]);
    dft16(v);
}

// m mod 2N for 0 <= m < 2^52
__device__ __forceinline__ int mod2n(long long m, int n2, double inv)
{
    int r = (int)(m - (long long)n2 * (long long)((double)m * inv));
    if (r < 0) r += n2;
    return r >= n2 ? r - n2 : r;
}

__global__ __launch_bounds__(256) void k_czt_phases(int n_tau, cd* __restrict__ tab)
{
    const int t = blockIdx.x * 256 + threadIdx.x, n2 = 2 * n_tau;
    double s, c;
    if (t < n2) {
        sincospi((double)t / n_tau, &s, &c);
        tab[t] = cd{c, s};
    } else if (t < n2 + kCztM) {
        sincospi((double)(t - n2) / (kCztM / 2), &s, &c);
        tab[t] = cd{c, -s};
    }
}

// spectrum of the chirp e^{i pi k^2/N}, k = -2048..2047 at k mod 4096, with the 1/4096 of
// the inverse FFT
__global__ __launch_bounds__(256) void k_czt_filter(int n_tau, cd* __restrict__ tab)
{
    extern __shared__ cd sm[];
    const int t = threadIdx.x, n2 = 2 * n_tau;
    const cd* tw = tab + n2;
    const double inv = 1.0 / n2;
    cd v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = t + 256 * r, k = i < kCztM / 2 ? i : kCztM - i;
        v[r] = tab[mod2n((long long)k * k, n2, inv)];
    }
    fft4096(v, sm, tw, t);
#pragma unroll
    for (int r = 0; r < 16; ++r) tab[n2 + kCztM + t + 256 * r] = cscale(v[r], 1.0 / kCztM);
}

// One output tile, b0..b0+2047, of element e: the sum of this group's input tiles a0..a0+2047
// (grid: element, output tile, group).  Phase -+ pi (2f+1) t/N with (f, t) = (input, output) for
// iw -> tau and (output, input) for tau -> iw; the + sign by conjugating input and output.
// ONE: a group is one tile, whose results go straight out (with the sums in registers d = 10, 4096 x
// 8192 took 20 us more either way).
template <bool TO_W, bool ONE>
__global__ __launch_bounds__(256) void k_czt(CztPlan p, int m2, const cd* __restrict__ tab, const cd* __restrict__ in,
                                             cd* __restrict__ parts)
{
    extern __shared__ cd sm[];
    const int t = threadIdx.x, e = blockIdx.x, n2 = 2 * p.n_tau;
    const long long b0 = (long long)blockIdx.y * kCztTile;
    const cd *tw = tab + n2, *filt = tw + kCztM;
    const double inv = 1.0 / n2;
    const int nb = min(kCztTile, p.n_out - (int)b0);
    cd* out = parts + ((size_t)blockIdx.z * m2 + e) * p.ld_out + b0;
    cd y[ONE ? 1 : 8];
#pragma unroll
    for (int r = 0; r < (ONE ? 1 : 8); ++r) y[r] = cd{0.0, 0.0};
    for (int tile = blockIdx.z; tile < p.in_tiles; tile += p.in_groups) {
        const long long a0 = (long long)tile * kCztTile;
        const cd* x = in + (size_t)e * p.ld_in + a0;
        const int na = min(kCztTile, p.n_in - (int)a0);
        cd v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int a = t + 256 * r;
            v[r] = cd{0.0, 0.0};
            if (r < 8 && a < na) {
                cd g = x[a];
                if (TO_W) g.y = -g.y;
                // 2 a b0 + a^2, and the half step (2f+1) t: + t for the tau index on the input side
                const long long m = 2 * (long long)a * b0 + (long long)a * a + (TO_W ? a0 + a : 0);
                v[r] = cmulc(g, tab[mod2n(m, n2, inv)]);
            }
        }
        fft4096(v, sm, tw, t);
        // inverse FFT as conj(FFT(conj(.)))
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = cconj(cmul(v[r], filt[t + 256 * r]));
        fft4096(v, sm, tw, t);
        const long long ab = mod2n(2 * a0 * b0, n2, inv);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int b = t + 256 * r;
            if (b < nb) {
                const long long m = ab + 2 * (long long)b * a0 + (long long)b * b + (TO_W ? 0 : b0 + b);
                const cd w = cmulc(cconj(v[r]), tab[mod2n(m, n2, inv)]);
                if constexpr (ONE) out[b] = TO_W ? cconj(w) : w;
                else y[r] = cadd(y[r], w);
            }
        }
        if constexpr (ONE) return;
    }
    if constexpr (!ONE) {
#pragma unroll
        for (int r = 0; r < 8; ++r)
            if (t + 256 * r < nb) out[t + 256 * r] = TO_W ? cconj(y[r]) : y[r];
    }
}

// Definiteness of M_b = -X_b, or of -(X_b - X_b^H)/2i (ANTI), by the pivots of its elimination: a
// slot of N lanes (a power of two, N >= d) per matrix, lane c holds column c in LDS.
// M_b counts as positive definite only by a margin of 1e-13 of its trace (>= its largest
// eigenvalue), a hundred times the rounding of an eigenvalue.  ANTI: the others are eliminated
// again with 1e-12 of the largest entry added to the diagonal; a pivot below zero after positive
// ones shows a negative eigenvalue of that matrix up to the rounding of the elimination
// (Higham, Accuracy and Stability of Numerical Algorithms, sec. 10.1: some N^2 eps of the
// diagonal, 1e-13 at N = 32), hence one of M_b.
// A matrix is read once and its elimination is a chain, so the loops are rolled: with the columns
// in registers the straight-line code of the steps ran once per launch, and fetching it
// (12 KB at d = 16, 24 with the second elimination) was most of the time.  A call with every matrix
// below, d = 10, 64 frequencies: 76 us in registers, 42 so; with every matrix sent to the eigensolver 202.
template <bool ANTI>
__global__ __launch_bounds__(64) void k_not_posdef(const cd* __restrict__ X, int d, int N, int count,
                                                   int* __restrict__ bad)
{
    extern __shared__ cd sm[];
    const int lane = threadIdx.x, c = lane & (N - 1), slots = 64 / N, sl = lane / N, ld = N + 1;
    const int b = blockIdx.x * slots + sl;
    const bool mine = b < count, live = mine && c < d;
    const cd* M = X + (size_t)(mine ? b : count - 1) * d * d;
    cd *A = sm + sl * N * ld, *col = A + c * ld;  // columns of this slot's matrix, this lane's
    // one addition a wavefront, of its matrices for which `which` holds
    auto add = [&](int* to, bool which) {
        const int n = __popcll(__ballot(live && c == 0 && which));
        if (lane == 0 && n) atomicAdd(to, n);
    };
    bool ok = true;
    for (int pass = 0; pass < (ANTI ? 2 : 1); ++pass) {
        double diag = 0.0, top = 0.0;
        if (c < d) {
#pragma unroll 4
            for (int i = 0; i < d; ++i) {
                cd v;
                if (ANTI) {  // -(x - conj(y))/2i
                    const cd x = M[i + c * d], y = M[c + i * d];
                    v = cd{-0.5 * (x.y + y.y), 0.5 * (x.x - y.x)};
                } else {  // Hermitian to the last bit: the lower triangle
                    const cd m = i >= c ? M[i + c * d] : cconj(M[c + i * d]);
                    v = cd{-m.x, i == c ? 0.0 : -m.y};
                }
                col[i] = v;
                if (i == c) diag = v.x;
                top = fmax(top, fmax(fabs(v.x), fabs(v.y)));
            }
        }
        double tr = diag;
        for (int o = N / 2; o > 0; o >>= 1) {
            tr += __shfl_xor(tr, o);
            top = fmax(top, __shfl_xor(top, o));
        }
        if (c < d) col[c].x = diag + (pass ? 1e-12 * top : -1e-13 * tr);
        wave_sync();
        int sign = 1;  // 1: every pivot positive and finite; -1: a negative one after such; 0: neither
        for (int j = 0; j < d; ++j) {
            const double p = A[j * ld + j].x;
            if (sign == 1 && !(p > 0.0 && p < 1e300)) sign = p < 0.0 && p > -1e300 ? -1 : 0;  // (NaN: 0)
            if (c > j && c < d) {
                const cd f = cscale(col[j], 1.0 / p);  // A_jc / p
#pragma unroll 4
                for (int i = j + 1; i < d; ++i) col[i] = cfms(A[j * ld + i], f, col[i]);
            }
            wave_sync();
        }
        if (pass == 0) {
            ok = sign == 1;
            if (!ANTI) add(bad, !ok);
            if (!__any(live && !ok)) return;
        } else {
            add(bad, !ok && sign >= 0);
            add(bad + 1, !ok && sign < 0);
        }
    }
}

}  // namespace

hipError_t launch_czt_tables(int n_tau, cd* tab, hipStream_t s)
{
    const int total = 2 * n_tau + kCztM;
    hipLaunchKernelGGL(k_czt_phases, dim3((total + 255) / 256), dim3(256), 0, s, n_tau, tab);
    const int shm = (int)(sizeof(cd) * kFftLds);
    hipError_t e = hipFuncSetAttribute((const void*)k_czt_filter, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_czt_filter, dim3(1), dim3(256), shm, s, n_tau, tab);
    return hipGetLastError();
}

CztPlan czt_plan(int n_tau, int n_in, int n_out, int m2)
{
    CztPlan p;
    p.n_tau = n_tau;
    p.n_in = n_in;
    p.n_out = n_out;
    p.in_tiles = (n_in + kCztTile - 1) / kCztTile;
    const size_t fit = kCztPartBytes / ((size_t)m2 * n_out * sizeof(cd));
    p.in_groups = (int)std::max<size_t>(1, std::min<size_t>(p.in_tiles, fit));
    p.out_tiles = (n_out + kCztTile - 1) / kCztTile;
    p.ld_in = n_in;
    p.ld_out = n_out;
    return p;
}

hipError_t launch_czt(const CztPlan& p, bool to_w, int m2, const cd* tab, const cd* in, cd* parts, hipStream_t s)
{
    const int shm = (int)(sizeof(cd) * kFftLds);
    const dim3 grid(m2, p.out_tiles, p.in_groups);
    const bool one = p.in_groups == p.in_tiles;
    auto kernel = to_w ? one ? k_czt<true, true> : k_czt<true, false> : one ? k_czt<false, true> : k_czt<false, false>;
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(256), shm, s, p, m2, tab, in, parts);
    return hipGetLastError();
}

hipError_t launch_not_posdef(const cd* X, int d, int count, bool anti, int* bad, hipStream_t s)
{
    const int N = d <= 4 ? 4 : d <= 8 ? 8 : d <= 16 ? 16 : 32, slots = 64 / N;
    const dim3 grid((count + slots - 1) / slots);
    const size_t shm = sizeof(cd) * 64 * (N + 1);
    if (anti) hipLaunchKernelGGL((k_not_posdef<true>), grid, dim3(64), shm, s, X, d, N, count, bad);
    else hipLaunchKernelGGL((k_not_posdef<false>), grid, dim3(64), shm, s, X, d, N, count, bad);
    return hipGetLastError();
}

}  // namespace dg
