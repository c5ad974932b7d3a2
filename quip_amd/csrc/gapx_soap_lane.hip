// SOAP forward of the calls that form the GAP variance, specialised on (n_max, l_max).
//
// The variance k(x,x) - k^T (K_MM + reg I)^-1 k is a difference of nearly equal numbers: it carries
// the descriptor's last bits magnified a hundred million times (it is 1.5e-7 relative off at 216
// Si atoms with 500 sparse points), so its digits beyond that belong to the order in which the
// descriptor is summed.  These calls keep the summation order of this kernel, whose digits
// callers have seen; another order moves them by 8e-8, neither nearer nor further by any
// measurement here.  Every other call takes the matrix-core forward of gapx_soap.hip, at less
// than half the time (31 us here against 9 of 216 atoms).
//
// Per l, lanes = neighbours stage fc F_l(a) and Y_l,m in LDS, lanes = (a, m) accumulate c' in
// the primitive radial basis; c = T^T c' once per centre; lanes = power-spectrum entries form
// p, a wave reduction gives |p|.  The radial transform T lives in LDS; an empty asm with a memory
// clobber closes every step so that T is re-read instead of pinned in VGPRs.
#include "gapx_kernels.h"

#include <algorithm>

namespace gapx {

#define GAPX_PI_S 3.14159265358979323846264338327950288

// N_lm of the real spherical harmonics (x sqrt 2 for m > 0) and (2m-1)!!
static __constant__ double c_ynorm[(kMaxL + 1) * (kMaxL + 2) / 2];
static __constant__ double c_dfact[kMaxL + 2];
static __constant__ double c_rinv[2 * kMaxL + 4];   // 1/k (k = 0 unused)
// place and factor of coefficient l*l + l + m in the buffer the adjoint reads (l <= 8)
static __constant__ int c_place[81];
static __constant__ double c_factor[81];

static bool g_soap_const_ready[64] = {};   // per device
static hipError_t ensure_soap_constants() {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (g_soap_const_ready[dev]) return hipSuccess;
    double yn[(kMaxL + 1) * (kMaxL + 2) / 2], df[kMaxL + 2];
    for (int l = 0; l <= kMaxL; l++)
        for (int m = 0; m <= l; m++) {
            double r = 1.0;   // (l-m)!/(l+m)!
            for (int k = l - m + 1; k <= l + m; k++) r /= (double)k;
            double v = sqrt((2.0 * l + 1.0) / (4.0 * GAPX_PI_S) * r);
            if (m > 0) v *= sqrt(2.0);
            yn[l * (l + 1) / 2 + m] = v;
        }
    df[0] = 1.0;
    for (int m = 1; m < kMaxL + 2; m++) df[m] = df[m - 1] * (2.0 * m - 1.0);
    double ri[2 * kMaxL + 4];
    ri[0] = 0.0;
    for (int k = 1; k < 2 * kMaxL + 4; k++) ri[k] = 1.0 / (double)k;
    int place[81];
    double factor[81];
    for (int l = 0; l <= 8; l++)
        for (int m = -l; m <= l; m++) soap_coefficient_order(l, m, place + l * l + l + m, factor + l * l + l + m);
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_place), place, sizeof(place))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_factor), factor, sizeof(factor))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_rinv), ri, sizeof(ri))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_ynorm), yn, sizeof(yn))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_dfact), df, sizeof(df))) != hipSuccess) return e;
    g_soap_const_ready[dev] = true;
    return hipSuccess;
}

hipError_t soap_lane_constants_init() { return ensure_soap_constants(); }

#define RELOAD_BARRIER() __asm__ volatile("" ::: "memory")

// neighbours staged per pass of the forward kernel (one lane each)
constexpr int kSoapChunk = 32;

__device__ __forceinline__ double fc_s(double r, double rc, double w) {
    if (r > rc) return 0.0;
    if (r > rc - w) return 0.5 * (cos(GAPX_PI_S * (r - rc + w) / w) + 1.0);
    return 1.0;
}
__device__ __forceinline__ double wave_sum_s(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ int species_s(const SoapDev &sp, int z) {
    for (int s = 0; s < sp.S; s++)
        if (sp.species_Z[s] == z || sp.species_Z[s] == 0) return s;
    return -1;
}

// Associated Legendre values P_l^m (m = 0..l) of one neighbour, level by level,
// in two LDS rows: on entry cur holds P_(l-2), prev P_(l-1); on exit cur holds P_l.
__device__ __forceinline__ void legendre_level(int l, double uz, const double *prev, double *cur) {
    for (int m = 0; m <= l; m++) {
        double pc;
        if (m == l) pc = c_dfact[m];
        else if (m == l - 1) pc = (2.0 * l - 1.0) * uz * prev[m];
        else pc = ((2.0 * l - 1.0) * uz * prev[m] - (double)(l + m - 1) * cur[m]) * c_rinv[l - m];
        cur[m] = pc;
    }
}

// i_l recursion state for all grid points: F0 = f_l, F1 = f_(l+1).  The
// recursion factor 1/x_a = 1/(2 alpha r r_a) is ixq / a with ixq = 1/(2 alpha r dr)
// (r_a = a dr), formed from ixq when used (no per-point array: fewer registers).
// rbs: grid r_a = a * dr; gA[a] = exp(-alpha r_a^2); iA[a] = 1/a.
// exp(-alpha (r -+ r_a)^2) = exp(-alpha r^2) gA[a] q^(+-a) with q = exp(2 alpha r dr):
// two exponentials and one division per neighbour.  Outside the range where the
// powers stay finite, every point is direct.
template <int N>
struct Rad {
    double F0[N], F1[N], ixq;
    __device__ __forceinline__ void init(const double *rbs, const double *gA, const double *iA, double alpha,
                                         double r) {
        const double xq = N > 1 ? 2.0 * alpha * r * rbs[1] : 0.0;
        const double rmax = rbs[N - 1];
        ixq = 1.0 / xq;
        if (xq > 0.0 && xq * (N - 1) < 600.0 && alpha * (r * r + rmax * rmax) < 600.0) {
            const double e0 = exp(-alpha * r * r);
            const double q = exp(xq), qi = 1.0 / q;
            double qa = 1.0, qia = 1.0;
            F0[0] = e0;
            F1[0] = 0.0;
#pragma unroll
            for (int a = 1; a < N; a++) {
                qa *= q;
                qia *= qi;
                const double eg = e0 * gA[a];
                const double em = eg * qa, ep = eg * qia;
                const double iv = ixq * iA[a];
                F0[a] = 0.5 * (em - ep) * iv;
                F1[a] = 0.5 * (em + ep) * iv - F0[a] * iv;
            }
            return;
        }
#pragma unroll
        for (int a = 0; a < N; a++) {
            const double ra = rbs[a];
            if (a == 0) {
                F0[a] = exp(-alpha * (ra * ra + r * r));
                F1[a] = 0.0;
            } else {
                const double ep = exp(-alpha * (r + ra) * (r + ra)), em = exp(-alpha * (r - ra) * (r - ra));
                const double iv = ixq * (1.0 / (double)a);
                F0[a] = 0.5 * (em - ep) * iv;
                F1[a] = 0.5 * (em + ep) * iv - F0[a] * iv;
            }
            __builtin_amdgcn_sched_barrier(0);   // one grid point's exponentials at a time
        }
    }
    __device__ __forceinline__ void step(int l) {
        F0[0] = F1[0];   // grid point 0 (r_a = 0): f_(l+1) = 0 for every l
        F1[0] = 0.0;
#pragma unroll
        for (int a = 1; a < N; a++) {
            const double n2 = F0[a] - (2.0 * l + 3.0) * (ixq * (1.0 / (double)a)) * F1[a];
            F0[a] = F1[a];
            F1[a] = n2;
        }
    }
};

// Forward.  With g_b(r) = fc(r) sum_a F_l(a, r) T[a][b] (F = the i_l recursion
// values of grid point a), c[b][lm] = sum_a T[a][b] c'[a][lm] where
// c'[a][lm] = sum_k fc F_l(a, r_k) Y_lm(k) is accumulated in the primitive
// (Gaussian) radial basis and transformed once per centre.
// Per neighbour chunk: the chunk's neighbours are listed per species (wave
// ballot); per l, lanes = neighbours stage fc F_l(a) and Y_l,m in LDS and
// lanes = (a, m) accumulate c' of each species over that species' list only.
// One level of a chunk: stage fc F_l and Y_l of the neighbours, then accumulate
// c' of level l.  A macro so that both level loops (rolled and unrolled) inline it.
#define SOAP_FWD_LEVEL(l, cur, prv)                                                                                  \
            __syncthreads();   /* the previous level's reads of Rl / Yl are done */                                  \
            if (lane < 32 * CPW) {   /* rows of neighbours outside every list stay zero for the dense loop */        \
_Pragma("unroll")                                                                                                    \
                for (int a = 0; a < N; a++) Rh[a * RT + kl] = s >= 0 ? fc * rs.F0[a] : 0.0;                          \
            }                                                                                                        \
            if (s >= 0) {                                                                                            \
                rs.step(l);                                                                                          \
                legendre_level(l, uz, prv, cur);                                                                     \
                double A = 1.0, B = 0.0;                                                                             \
                double *Yr = Yh + kl;   /* slot m of this neighbour at Yr[m * RT] */                                 \
                for (int m = 0; m <= l; m++) {                                                                       \
                    if (m > 0) {                                                                                     \
                        const double An = A * ux - B * uy;                                                           \
                        B = A * uy + B * ux;                                                                         \
                        A = An;                                                                                      \
                    }                                                                                                \
                    const double Nn = c_ynorm[l * (l + 1) / 2 + m] * cur[m];                                         \
                    if (m == 0) Yr[l * RT] = Nn;                                                                     \
                    else {                                                                                           \
                        Yr[(l + m) * RT] = Nn * A;                                                                   \
                        Yr[(l - m) * RT] = Nn * B;                                                                   \
                    }                                                                                                \
                }                                                                                                    \
            } else if (lane < 32 * CPW) {                                                                            \
                for (int m = 0; m < 2 * l + 1; m++) Yh[m * RT + kl] = 0.0;                                           \
            }                                                                                                        \
            __syncthreads();                                                                                         \
            const int W = 2 * l + 1;                                                                                 \
            for (int it = lane; it < CPW * N * W; it += 64) {                                                        \
                const int hh = CPW == 1 ? 0 : it / (N * W), r_ = it - hh * (N * W);                                 \
                const int a = r_ / W, mi = r_ - a * W;                                                               \
                const double *Rc = Rl + hh * (N * RT), *Yc = Yl + hh * (YW * RT);                                   \
                double *cPc = cP + hh * KLMp;                                                                        \
                if (S == 1) {   /* one species: every row of the chunk in pairs, zero rows included */            \
                    const double2 *R2 = (const double2 *)(Rc + a * RT), *Y2 = (const double2 *)(Yc + mi * RT);      \
                    double acc0 = 0.0, acc1 = 0.0;                                                                   \
_Pragma("unroll 4")                                                                                                  \
                    for (int k2 = 0; k2 < NB / 2; k2++) {                                                            \
                        const double2 rv = R2[k2], yv = Y2[k2];                                                      \
                        acc0 += rv.x * yv.x;                                                                         \
                        acc1 += rv.y * yv.y;                                                                         \
                    }                                                                                                \
                    cPc[a * LM + l * l + mi] += acc0 + acc1;                                                         \
                    continue;                                                                                        \
                }                                                                                                    \
                for (int si = 0; si < S; si++) {                                                                     \
                    const int n = ns[hh * S + si];                                                                   \
                    const int *ki = kidx + (hh * S + si) * NB;                                                       \
                    double acc0 = 0.0, acc1 = 0.0;                                                                   \
                    int q = 0;                                                                                       \
_Pragma("unroll 2")                                                                                                  \
                    for (; q + 1 < n; q += 2) {                                                                      \
                        const int k0 = ki[q], k1 = ki[q + 1];                                                        \
                        acc0 += Rc[a * RT + k0] * Yc[mi * RT + k0];                                                  \
                        acc1 += Rc[a * RT + k1] * Yc[mi * RT + k1];                                                  \
                    }                                                                                                \
                    if (q < n) {                                                                                     \
                        const int k0 = ki[q];                                                                        \
                        acc0 += Rc[a * RT + k0] * Yc[mi * RT + k0];                                                  \
                    }                                                                                                \
                    cPc[(si * N + a) * LM + l * l + mi] += acc0 + acc1;                                              \
                }                                                                                                    \
            }

// Each lane keeps its Legendre levels in registers, with the level loop unrolled.
// CPW: centres per wavefront.  A centre's chunk of 32 neighbours occupies 32 lanes,
// so with two centres lanes 0-31 and 32-63 stage the neighbours of one centre each
// and every staging instruction serves two centres.
template <int N, int L, int CPW>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_soap_fwd_lane(
    SoapDev sp, int nc, const int *__restrict__ centres, const int *__restrict__ Z, const int *__restrict__ nb_off,
    const int *__restrict__ nb_j, const double *__restrict__ nb_r, const double *__restrict__ nb_d, double *X,
    double *norm_out, double *cbuf) {
    extern __shared__ double lds[];
    constexpr int LM = (L + 1) * (L + 1);
    constexpr int YW = 2 * L + 1;
    constexpr int NB = kSoapChunk;
    const int K = sp.K, KLM = K * LM, S = sp.S;
    const int KLMp = (KLM + 1) & ~1;   // per-centre c' rows, 16-byte aligned
    double *Ts = lds;              // N*N
    double *rbs = Ts + N * N;      // N grid points, then exp(-alpha r_a^2) and 1/a (N each)
    double *gA = rbs + N, *iA = gA + N;
    double *cP = rbs + 3 * N;      // CPW x K*LM: c' during accumulation, c after the transform
    // The staged levels are stored one row per radial point a (Rl) and per m slot (Yl),
    // neighbours along the row: the writes of 32 lanes are consecutive, and the dense
    // accumulation reads two neighbours per 16-byte access.  The row stride RT = NB + 2
    // keeps rows 16-byte aligned (N (N + 3) and KLMp are even) and puts successive rows
    // 16 bytes apart in the bank cycle.
    constexpr int RT = NB + 2;     // row stride of Rl and Yl
    double *Rl = cP + CPW * KLMp;  // CPW x N x RT: fc F_l(a) of neighbour k of centre h at Rl[(h N + a) RT + k]
    double *Yl = Rl + CPW * N * RT;   // CPW x YW x RT: Y_l,m of neighbour k at Yl[(h YW + slot) RT + k]
    int *kidx = (int *)(Yl + CPW * YW * RT);   // CPW x S x NB: the chunk's neighbours of each species
    int *ns = kidx + CPW * S * NB; // their counts
    const int lane = threadIdx.x;
    const int h = CPW == 2 ? lane >> 5 : 0, kl = lane & 31;   // this lane's centre and neighbour slot
    const int desc = CPW * blockIdx.x + h;
    const bool valid = desc < nc;   // this lane's centre exists (the same for all lanes with CPW 1)
    const int ci = valid ? centres[desc] : 0;
    double *Rh = Rl + h * (N * RT), *Yh = Yl + h * (YW * RT);
    for (int e = lane; e < N * N; e += 64) Ts[e] = sp.T[e];
    if (lane < N) {
        rbs[lane] = sp.rb[lane];
        gA[lane] = exp(-sp.alpha * sp.rb[lane] * sp.rb[lane]);
        iA[lane] = lane > 0 ? 1.0 / (double)lane : 0.0;
    }
    for (int e = lane; e < CPW * KLMp; e += 64) cP[e] = 0.0;
    __syncthreads();
    const int p0 = valid ? nb_off[ci] : 0, np = valid ? nb_off[ci + 1] - p0 : 0;
    int npmax = np;   // chunks of the wave (uniform): those of its larger centre
    if (CPW == 2) npmax = max(np, __shfl_xor(np, 32, 64));
    for (int c0 = 0; c0 < npmax; c0 += NB) {
        const int nk = max(0, min(NB, np - c0));
        __syncthreads();   // the previous chunk's reads of the lists are done
        int s = -1;
        double fc = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
        Rad<N> rs;
        if (kl < nk && lane < 32 * CPW) {
            const int p = p0 + c0 + kl;
            const double r = nb_r[p];
            s = species_s(sp, Z[nb_j[p]]);
            if (r > sp.rc) s = -1;
            if (s >= 0) {
                fc = fc_s(r, sp.rc, sp.ctw);
                rs.init(rbs, gA, iA, sp.alpha, r);
                const double ir = 1.0 / r;
                ux = nb_d[3 * p] * ir; uy = nb_d[3 * p + 1] * ir; uz = nb_d[3 * p + 2] * ir;
            }
        }
        for (int si = 0; S > 1 && si < S; si++) {   // neighbours beyond the cutoff are in no list
            const bool mine = lane < 32 * CPW && s == si;
            const unsigned long long mk = __ballot(mine);
            const unsigned long long mh = (mk >> (32 * h)) & 0xffffffffull;   // this centre's half
            if (mine) kidx[(h * S + si) * NB + __popcll(mh & ((1ull << kl) - 1ull))] = kl;
            if (kl == 0 && lane < 32 * CPW) ns[h * S + si] = __popcll(mh);
        }
        double P0[L + 2], P1[L + 2];
#pragma unroll
        for (int l = 0; l <= L; l++) {
            double *cur = (l & 1) ? P1 : P0;
            const double *prv = (l & 1) ? P0 : P1;
            SOAP_FWD_LEVEL(l, cur, prv);
        }
    }
    __syncthreads();
    // c = T^T c', one (centre, species, lm) column per lane, in place
    for (int it = lane; it < CPW * S * LM; it += 64) {
        const int hh = CPW == 1 ? 0 : it / (S * LM), r_ = it - hh * (S * LM), si = r_ / LM, lm = r_ - si * LM;
        double *cc = cP + hh * KLMp;
        RELOAD_BARRIER();   // T is re-read from LDS for every column
        double cp[N];
#pragma unroll
        for (int a = 0; a < N; a++) cp[a] = cc[(si * N + a) * LM + lm];
#pragma unroll
        for (int b = 0; b < N; b++) {
            double acc = 0.0;
#pragma unroll
            for (int a = 0; a < N; a++) acc += Ts[a * N + b] * cp[a];
            cc[(si * N + b) * LM + lm] = acc;
            RELOAD_BARRIER();   // one column of T in registers at a time
        }
    }
    __syncthreads();
    if (kl == 0 && valid && lane < 32 * CPW) {   // centre atom term
        const int sc = species_s(sp, Z[ci]);
        if (sc >= 0) cP[h * KLMp + (sc * N) * LM] += sp.cw * sp.u00 * c_ynorm[0];
    }
    __syncthreads();
    // power spectrum, written unnormalised and rescaled in place by the same lanes
    const int d = sp.dim;
    const int d0 = CPW * blockIdx.x;
    double ss[CPW];
#pragma unroll
    for (int hh = 0; hh < CPW; hh++) ss[hh] = 0.0;
    for (int it = lane; it < CPW * (d - 1); it += 64) {
        const int hh = CPW == 1 ? 0 : it / (d - 1), q = it - hh * (d - 1);
        if (d0 + hh >= nc) continue;
        const double *cc = cP + hh * KLMp;
        const int code = sp.qmap[q];
        const int ia = code >> 16, jb = (code >> 8) & 0xff, l = code & 0xff;
        double v = 0.0;
        for (int m = -l; m <= l; m++) v += cc[ia * LM + l * l + l + m] * cc[jb * LM + l * l + l + m];
        v *= (ia != jb ? 1.4142135623730950488 : 1.0) / sqrt(2.0 * l + 1.0);
        X[(size_t)(d0 + hh) * d + q] = v;
#pragma unroll
        for (int g2 = 0; g2 < CPW; g2++)
            if (g2 == hh) ss[g2] += v * v;
    }
    double inv[CPW];
#pragma unroll
    for (int hh = 0; hh < CPW; hh++) {
        const double nrm = sqrt(wave_sum_s(ss[hh]));
        inv[hh] = nrm > 0.0 ? 1.0 / nrm : 0.0;
        if (lane == 0 && d0 + hh < nc) {
            X[(size_t)(d0 + hh) * d + d - 1] = 0.0;
            norm_out[d0 + hh] = nrm;
        }
    }
    for (int it = lane; it < CPW * (d - 1); it += 64) {
        const int hh = CPW == 1 ? 0 : it / (d - 1), q = it - hh * (d - 1);
        if (d0 + hh >= nc) continue;
        double sc = inv[0];
#pragma unroll
        for (int g2 = 1; g2 < CPW; g2++)
            if (g2 == hh) sc = inv[g2];
        X[(size_t)(d0 + hh) * d + q] *= sc;
    }
    // c in the order and with the factors in which the adjoint takes it
    for (int hh = 0; hh < CPW; hh++) {
        if (d0 + hh >= nc) break;
        double *co = cbuf + (size_t)(d0 + hh) * KLM;
        for (int e = lane; e < KLM; e += 64) {
            const int row = e / LM, lm = e - row * LM;
            co[row * LM + c_place[lm]] = cP[hh * KLMp + e] * c_factor[lm];
        }
    }
}

#define SOAP_LANE(X) X(4, 4) X(5, 4) X(6, 4) X(8, 4) X(6, 6) X(8, 6) X(10, 6) X(12, 6) X(8, 8) X(10, 8) X(12, 8)

// Two centres per wave: single-species models with n <= 8, l <= 6 whose register
// state fits without spilling (n l >= 32: 8/4, 6/6, 8/6).
static constexpr bool fwd_pair_ok(int n, int L) { return n <= 8 && L <= 6 && n * L >= 32; }
template <int N, int L>
static void fwd_go(int cpw, int nblk, size_t sh, hipStream_t s, const SoapDev &sp, int nc, const int *centres,
                   const int *Z, const int *nb_off, const int *nb_j, const double *nb_r, const double *nb_d,
                   double *X, double *norm, double *cbuf) {
    if constexpr (fwd_pair_ok(N, L)) {
        if (cpw == 2) {
            hipLaunchKernelGGL((k_soap_fwd_lane<N, L, 2>), dim3(nblk), dim3(64), sh, s, sp, nc, centres, Z, nb_off,
                               nb_j, nb_r, nb_d, X, norm, cbuf);
            return;
        }
    }
    hipLaunchKernelGGL((k_soap_fwd_lane<N, L, 1>), dim3(nblk), dim3(64), sh, s, sp, nc, centres, Z, nb_off, nb_j,
                       nb_r, nb_d, X, norm, cbuf);
}

// LDS bytes of the block: transform, radial grid, c' accumulators, the staged neighbour chunk
size_t soap_lane_lds_bytes(const SoapDev &sp) {
    const int cpw = sp.S == 1 && fwd_pair_ok(sp.n, sp.L) ? 2 : 1;
    const int LM = (sp.L + 1) * (sp.L + 1), KLM = sp.K * LM, NB = kSoapChunk;
    return (size_t)(sp.n * sp.n + 3 * sp.n + cpw * ((KLM + 1) & ~1) + cpw * (NB + 2) * (sp.n + 2 * sp.L + 1)) * 8 +
           (size_t)cpw * sp.S * (NB + 1) * 4;
}

bool launch_soap_fwd_lane(const SoapDev &sp, int nc, const int *centres, const int *Z, const int *nb_off,
                          const int *nb_j, const double *nb_r, const double *nb_d, double *X, double *norm,
                          double *cbuf, hipStream_t s) {
    if (!soap_fast_supported(sp.n, sp.L)) return false;
    ensure_soap_constants();
    if (nc <= 0) return true;
    // two centres per wave with the Legendre levels in registers for single-species models up
    // to n 8, l 6; one centre per wave otherwise
    const int cpw = sp.S == 1 && fwd_pair_ok(sp.n, sp.L) ? 2 : 1;
    const size_t sh = soap_lane_lds_bytes(sp);
    const int nblk = (nc + cpw - 1) / cpw;
#define LAUNCH(NN, LL)                                                                                          \
    if (sp.n == NN && sp.L == LL) {                                                                             \
        fwd_go<NN, LL>(cpw, nblk, sh, s, sp, nc, centres, Z, nb_off, nb_j, nb_r, nb_d, X, norm, cbuf);          \
        return true;                                                                                            \
    }
    SOAP_LANE(LAUNCH)
#undef LAUNCH
    return false;
}

}  // namespace gapx
