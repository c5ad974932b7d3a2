// SOAP descriptor kernels specialised on (n_max, l_max), on the FP64 matrix cores.
//
// Every contraction of the descriptor is a batch of small products: the density
// coefficients c'_l = sum_k F_l(a, k) Y_lm(k) over the neighbours k, the radial
// transform T, the power spectrum c_l c_l^T, and in the adjoint dE/dc_l = P_l c_l and the
// products of dE/dc' with the neighbours' radial functions.  They run on
// v_mfma_f64_4x4x4: four independent 4x4 blocks of a k of 4, at the same rate per
// operation as 16x16x4 (measured 16 and 64 cycles), so levels of 1 to 17 harmonics waste
// little.  The recursions and the products' operands meet in registers: the lane that
// holds an operand element computes it, so neighbour data never pass through LDS except
// for a small table of per-neighbour scalars.
//
// Lane roles of the 4x4x4 product (lane = 16 k + 4 b + i): A holds row i, inner index k
// of block b; B holds inner index k, column i of block b; D holds row k, column i of block b.
//
// Harmonics of a level come in groups of four: group v = 0 holds cos(m phi) terms of
// m = 0..3, v = 1 sin terms of m = 0..3 (m = 0 is empty), v = 2, 3 the same for m = 4..7 and
// v = 4, 5 for m = 8 (empty beyond it).  Empty slots meet zeros.
#include "gapx_kernels.h"

#include <algorithm>
#include <type_traits>

namespace gapx {

#define GAPX_PI_S 3.14159265358979323846264338327950288

__host__ __device__ constexpr int lev_groups(int l) { return l == 0 ? 1 : l < 4 ? 2 : l < 8 ? 4 : 6; }
__host__ __device__ constexpr int lev_base(int l) { return l == 0 ? 0 : l <= 4 ? 2 * l - 1 : l <= 8 ? 4 * l - 9 : 29; }
__host__ __device__ constexpr int soap_groups(int L) { return lev_base(L) + lev_groups(L); }

constexpr int kSoapMaxL = 8;                             // of the specialised shapes
constexpr int kSoapGroups = soap_groups(kSoapMaxL);      // 29

// per group: its level; per (group, slot): the place of the harmonic within the (L+1)^2
// coefficients of a radial row (-1: empty) and the factor between the monic Legendre
// recursion used here and the real harmonic
static __constant__ int c_glev[kSoapGroups + 3];
static __constant__ int c_gpos[4 * kSoapGroups + 12];
static __constant__ double c_gnorm[4 * kSoapGroups + 12];
static __constant__ double c_ginv[4 * kSoapGroups + 12];   // 1 / c_gnorm (0: empty)
static __constant__ double c_isq[kSoapMaxL + 1];         // 1/sqrt(2l+1)

static bool g_soap_const_ready[64] = {};   // per device
static hipError_t ensure_soap_constants() {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (g_soap_const_ready[dev]) return hipSuccess;
    int lev[kSoapGroups + 3] = {}, pos[4 * kSoapGroups + 12];
    double nrm[4 * kSoapGroups + 12] = {}, inv[4 * kSoapGroups + 12] = {}, isq[kSoapMaxL + 1];
    std::fill(pos, pos + 4 * kSoapGroups + 12, -1);
    for (int l = 0; l <= kSoapMaxL; l++) {
        isq[l] = 1.0 / sqrt(2.0 * l + 1.0);
        for (int v = 0; v < lev_groups(l); v++) {
            const int g = lev_base(l) + v;
            lev[g] = l;
            for (int j = 0; j < 4; j++) {
                const int m = 4 * (v / 2) + j;
                if (m > l || (m == 0 && (v & 1))) continue;
                soap_coefficient_order(l, v & 1 ? -m : m, pos + 4 * g + j, nrm + 4 * g + j);
                inv[4 * g + j] = 1.0 / nrm[4 * g + j];
            }
        }
    }
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_glev), lev, sizeof(lev))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_gpos), pos, sizeof(pos))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_gnorm), nrm, sizeof(nrm))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_ginv), inv, sizeof(inv))) != hipSuccess) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_isq), isq, sizeof(isq))) != hipSuccess) return e;
    g_soap_const_ready[dev] = true;
    return hipSuccess;
}

hipError_t soap_fast_constants_init() { return ensure_soap_constants(); }

// The real harmonic (l, m) (m < 0: sin) in a radial row of the coefficient buffer: its place
// and the factor it is stored with.
void soap_coefficient_order(int l, int m, int *place, double *factor) {
    const int a = m < 0 ? -m : m, v = 2 * (a / 4) + (m < 0);
    int next = l * l;   // of group v's first slot
    for (int u = 0; u < v; u++) next += std::min(l + 1 - 4 * (u / 2), 4) - (u == 1);
    *place = next + a % 4 - (v == 1);
    double r = 1.0, lead = 1.0;   // (l-a)!/(l+a)!; the a-th derivative of P_l over its monic form
    for (int k = l - a + 1; k <= l + a; k++) r /= (double)k;
    for (int k = 1; k <= l; k++) lead *= 2.0 * k - 1.0;
    for (int k = 2; k <= l - a; k++) lead /= (double)k;
    *factor = sqrt((2.0 * l + 1.0) / (4.0 * GAPX_PI_S) * r) * (a > 0 ? sqrt(2.0) : 1.0) * lead;
}

__device__ __forceinline__ double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
// orders this wavefront's LDS writes before its reads of other lanes' data
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// orders the block's LDS accesses: a barrier that waits for LDS only (memory accesses stay
// in flight), or within a lone wavefront the fence only
template <int NW>
__device__ __forceinline__ void block_lds_sync() {
    if constexpr (NW > 1) __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else wave_lds_sync();
}
// the lane number anew: what follows from it is recomputed here instead of being kept in
// registers across a loop over centres
__device__ __forceinline__ int fresh_lane() {
    int l = threadIdx.x & 63;
    __asm__ volatile("" : "+v"(l));
    return l;
}
__device__ __forceinline__ double wave_sum_s(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ int species_s(const SoapDev &sp, int S, int z) {
    for (int s = 0; s < S; s++)
        if (sp.species_Z[s] == z || sp.species_Z[s] == 0) return s;
    return -1;
}

// The neighbour table in LDS: one row per field, one slot per neighbour.  A pass covers
// kSoapPass neighbours (one per lane); the slots of each species start at a multiple of
// 16, the neighbours of one tile.
constexpr int kSoapPass = 64;
enum { kUx, kUy, kUz, kIxq, kE0, kQ, kQi, kFwdFields, kFc = kFwdFields, kDfc, kIr, kR, kBwdFields };

// A wavefront's neighbours of one pass, one per lane, on their way from memory.
struct SoapNb {
    int j, z;
    double r, dx, dy, dz;
    __device__ __forceinline__ void load(int p0, int nk, const int *__restrict__ nb_j, const double *__restrict__ nb_r,
                                         const double *__restrict__ nb_d) {
        const int lane = threadIdx.x & 63;
        if (lane < nk) {
            const int p = p0 + lane;
            j = nb_j[p];
            r = nb_r[p];
            dx = nb_d[3 * p]; dy = nb_d[3 * p + 1]; dz = nb_d[3 * p + 2];
        }
    }
    __device__ __forceinline__ void species(int nk, const int *__restrict__ Z) {
        if ((int)(threadIdx.x & 63) < nk) z = Z[j];
    }
};

// One wavefront writes the table of nk <= 64 neighbours from pair p0 on, the first slot
// (sb) and the number (sc) of each species' slots, and (adjoint) the pair of each slot.
// Radial functions of grid point r_a = a dr: exp(-alpha (r -+ r_a)^2) = e0 gA[a] q^(+-a)
// with e0 = exp(-alpha r^2), gA = exp(-alpha r_a^2), q = exp(2 alpha r dr).  Outside the range
// where these stay finite q = 0 marks the slot and its exponentials are formed directly (r in the
// place of 1/q).  The forward's e0 carries the cutoff function.
template <int N, bool BWD>
__device__ __forceinline__ void soap_stage(const SoapDev &sp, int S, const SoapNb &nb, int p0, int nk, double *tab,
                                           int slots, int *sb, int *sc, int *pair) {
    const int lane = threadIdx.x & 63;
    const double r = nb.r;
    int s = -1;
    if (lane < nk && !(r > sp.rc)) s = species_s(sp, S, nb.z);
    int slot = 0, base = 0;
    for (int si = 0; si < S; si++) {
        const unsigned long long mk = __ballot(s == si);
        const int n = __popcll(mk);
        if (s == si) slot = base + __popcll(mk & ((1ull << lane) - 1ull));
        if (lane == 0) { sb[si] = base; sc[si] = n; }
        base += (n + 15) & ~15;
    }
    if (s < 0) return;
    double fc = 1.0, dfc = 0.0;
    if (r > sp.rc - sp.ctw) {
        double sn, cs;
        sincospi((r - sp.rc + sp.ctw) * sp.ictw, &sn, &cs);
        fc = 0.5 * (cs + 1.0);
        dfc = -0.5 * GAPX_PI_S * sp.ictw * sn;
    }
    const double ir = 1.0 / r, xq = sp.a2dr * r, rmax = (N - 1) * sp.dr;
    double e0 = 1.0, q = 0.0, qi = r;
    if (xq > 0.0 && xq * (4 * ((N + 3) / 4) - 1) < 600.0 && sp.alpha * (r * r + rmax * rmax) < 600.0) {
        e0 = exp(-sp.alpha * r * r);
        q = exp(xq);
        qi = 1.0 / q;
    }
    if (!BWD) e0 *= fc;
    tab[kUx * slots + slot] = nb.dx * ir;
    tab[kUy * slots + slot] = nb.dy * ir;
    tab[kUz * slots + slot] = nb.dz * ir;
    tab[kIxq * slots + slot] = ir * sp.ia2dr;
    tab[kE0 * slots + slot] = e0;
    tab[kQ * slots + slot] = q;
    tab[kQi * slots + slot] = qi;
    if constexpr (BWD) {
        tab[kFc * slots + slot] = fc;
        tab[kDfc * slots + slot] = dfc;
        tab[kIr * slots + slot] = ir;
        tab[kR * slots + slot] = r;
        pair[slot] = p0 + lane;
    }
}

// The constant tables of a block in LDS (a table in memory would queue behind the neighbour
// data on their way): the transform, the radial tables, per (group, slot) the harmonics' factor
// and the place and level of the harmonic, per level 1/sqrt(2l+1).
template <int N, int L>
struct SoapTables {
    static constexpr int NA = (N + 3) / 4, NQ4 = (soap_groups(L) + 3) / 4 * 4;
    double *T, *rt, *gn, *isq;
    int *pos;   // place (0xffff: an empty slot) | level << 16
    __device__ __forceinline__ SoapTables(double *p) : T(p), rt(T + N * N), gn(rt + 24), isq(gn + 4 * NQ4), pos((int *)(isq + L + 1)) {}
    __device__ __forceinline__ void fill(const SoapDev &sp, int nthr) {
        for (int e = threadIdx.x; e < N * N; e += nthr) T[e] = sp.T[e];
        for (int e = threadIdx.x; e < 24; e += nthr) rt[e] = sp.rt[e];
        for (int e = threadIdx.x; e < L + 1; e += nthr) isq[e] = c_isq[e];
        for (int e = threadIdx.x; e < 4 * NQ4; e += nthr) {
            const bool in = e < 4 * soap_groups(L);
            gn[e] = in ? c_gnorm[e] : 0.0;
            pos[e] = in ? (c_gpos[e] & 0xffff) | c_glev[e / 4] << 16 : 0xffff;
        }
    }
    // T[a][b], zero beyond the basis
    __device__ __forceinline__ double t(int a, int b) const {
        return N % 4 == 0 || (a < N && b < N) ? T[min(a, N - 1) * N + min(b, N - 1)] : 0.0;
    }
};

// recursion coefficient of the monic m-th derivatives of P_l: p_l = z p_(l-1) - beta p_(l-2),
// beta = ((l-1)^2 - m^2) / ((2l-1)(2l-3)); zero states below l = m keep p_(m+1) = z p_m
__device__ __forceinline__ double leg_beta(int l, double m2) {
    const double rl = 1.0 / ((2.0 * l - 1.0) * (2.0 * l - 3.0));
    return fma(-m2, rl, (l - 1.0) * (l - 1.0) * rl);
}

// One lane's share of a neighbour: the radial functions of grid points a = g + 4u and the
// harmonics of m = g and g + 4 (and m = 8 in lane group 0).
template <int N>
struct SoapLane {
    static constexpr int NA = (N + 3) / 4;
    // per lane group: exp(-alpha r_a^2) / 2 and 1/a (0 for a = 0 and a >= N)
    double hg[NA], ia[NA];
    // recursion state F_l, F_(l+1), 1/x_a; the a = 0 value of l = 0
    double F0[NA], F1[NA], iv[NA], z0;
    double z, mA2, mB2, pA, pA1, pB, pB1;   // monic Legendre values of levels l, l - 1
    double start[4];                        // 1 in the group whose m starts at this level

    __device__ __forceinline__ void setup(const double *rt, int g) {
#pragma unroll
        for (int u = 0; u < NA; u++) {
            hg[u] = rt[g + 4 * u];
            ia[u] = rt[12 + g + 4 * u];
        }
        mA2 = (double)(g * g);
        mB2 = (double)((g + 4) * (g + 4));
#pragma unroll
        for (int l = 0; l < 4; l++) start[l] = g == l ? 1.0 : 0.0;
    }
    // monic m-th derivative of P_l, m = g + m0 (zero below l = m), from the states of l-1 and l-2
    __device__ __forceinline__ double legendre(int l, int m0, double m2, double p1, double p2) const {
        const int k = l - m0;
        if (k == 0) return start[0];
        const double t = k < 4 ? fma(z, p1, start[k < 4 ? k : 0]) : z * p1;
        return k == 1 ? t : t - leg_beta(l, m2) * p2;
    }
    // i_l recursion from i_(-1) = cosh(x)/x, i_0 = sinh(x)/x, x_a = 2 alpha r r_a; ixq = 1/x_1
    __device__ __forceinline__ void radial(const SoapDev &sp, int g, double ixq, double e0, double q,
                                           double qi) {
        const double q2 = q * q, i2 = qi * qi;
        double ep = g == 0 ? 1.0 : g == 1 ? q : g == 2 ? q2 : q2 * q;
        double em = g == 0 ? 1.0 : g == 1 ? qi : g == 2 ? i2 : i2 * qi;
        const double q4 = q2 * q2, i4 = i2 * i2;
        const bool direct = q == 0.0;
        z0 = g == 0 ? e0 : 0.0;
        if (__any(direct)) {
            const double r = qi;
            if (direct && g == 0) z0 = e0 * exp(-sp.alpha * r * r);
#pragma unroll
            for (int u = 0; u < NA; u++) {
                const int a = g + 4 * u;
                const double ra = a * sp.dr;
                iv[u] = ixq * ia[u];
                double m_ = e0 * hg[u] * ep, p_ = e0 * hg[u] * em;
                if (direct) {
                    m_ = a < N ? 0.5 * e0 * exp(-sp.alpha * (r - ra) * (r - ra)) : 0.0;
                    p_ = a < N ? 0.5 * e0 * exp(-sp.alpha * (r + ra) * (r + ra)) : 0.0;
                    if (a == 0 || a >= N) iv[u] = 0.0;
                }
                F0[u] = (m_ - p_) * iv[u];
                F1[u] = (m_ + p_) * iv[u] - F0[u] * iv[u];
                ep *= q4;
                em *= i4;
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < NA; u++) {
            iv[u] = ixq * ia[u];
            const double eg = e0 * hg[u];
            const double m_ = eg * ep, p_ = eg * em;
            F0[u] = (m_ - p_) * iv[u];
            F1[u] = (m_ + p_) * iv[u] - F0[u] * iv[u];
            if (u + 1 < NA) {
                ep *= q4;
                em *= i4;
            }
        }
    }
    __device__ __forceinline__ double f(int l, int u) const { return l == 0 && u == 0 ? F0[0] + z0 : F0[u]; }
    __device__ __forceinline__ void step(int l) {
#pragma unroll
        for (int u = 0; u < NA; u++) {
            const double n2 = F0[u] - ((2.0 * l + 3.0) * iv[u]) * F1[u];
            F0[u] = F1[u];
            F1[u] = n2;
        }
    }
};

// Which groups a forward wavefront accumulates: 1 the groups of m < 4, 2 those of m >= 4, 3 all.
template <int L, int SETS>
struct FwdGroups {
    static constexpr int count = SETS == 1 ? 2 * L + 1 : SETS == 2 ? 2 * (L - 3) + (L >= 8 ? 2 : 0) : soap_groups(L);
    __host__ __device__ static constexpr int index(int l, int v) {   // place of (level, group) in this wavefront's list
        return SETS == 1 ? (l == 0 ? 0 : 2 * l - 1 + v) : SETS == 2 ? 2 * (l - 4) + v - 2 : lev_base(l) + v;
    }
    __device__ static __forceinline__ int group(int idx) {           // and back, to the group number
        if (SETS == 3) return idx;
        if (SETS == 1) {
            const int l = (idx + 1) >> 1;
            return idx == 0 ? 0 : lev_base(l) + ((idx + 1) & 1);
        }
        const int l = 4 + (idx >> 1);
        return l > 8 ? lev_base(8) + 4 + (idx & 1) : lev_base(l) + 2 + (idx & 1);
    }
};

// LDS layout of the forward kernel, in doubles (shared by the kernel and its launcher)
struct FwdLds {
    int slots, gs, rs, cs, p_off, c_off, tab_off, tail, total;   // total in bytes
    __host__ __device__ FwdLds(int NA, int L, int S, int nw, int dim, bool p_lds, bool c_lds) {
        slots = kSoapPass + 16 * (S - 1);
        gs = 64 * NA + 4;                       // partial sums of one group; 4 apart so that groups fall on distinct banks
        rs = 4 * gs;                            // four groups at a time per wavefront
        cs = 4 * soap_groups(L) + 1;            // odd: rows on distinct banks
        const int tab = kFwdFields * slots;
        // a single wavefront is done with the table before it reduces: they share their place
        const int red = nw * rs, front = nw == 1 && S == 1 ? (tab > red ? tab : red) : tab + red;
        tab_off = 0;
        p_off = nw == 1 && S == 1 ? 0 : tab;    // the reduction area, later the power spectrum
        const int p_need = p_lds ? dim : 0;
        const int room = front - p_off;
        c_off = p_off + (p_need > room ? p_need : room);
        c_off = (c_off + 1) & ~1;
        tail = c_off + (c_lds ? S * NA * 4 * cs : 0);
        total = (tail + nw) * 8 + 2 * S * 4;   // followed by the constant tables
        total = (total + 7) & ~7;
    }
};

// Forward: a block of NW wavefronts takes cpb centres in turn; a centre's neighbours are
// fetched while the one before is worked on.  A wavefront takes the neighbours of one
// species (and, SPLIT, the harmonics of m < 4 or m >= 4) in tiles of 16: lane 4 n + g
// evaluates neighbour n's radial functions of a = g, g+4, .. and its harmonics of m = g, g+4,
// which are the operands of 4x4x4 products whose four blocks are four quarters of the tile.
// The quarters are summed through LDS once per centre, T and the power spectrum follow as
// further 4x4x4 products.  135612 Si centres at 8/6: 1.10 -> 0.46 ms against lanes accumulating
// c' from levels staged in LDS (945 MB moved at 2.0 TB/s; VALU issue 50% and the matrix pipe 22%
// of it); 32768 SiC centres at 12/8: 3.19 -> 0.77 ms.  SP: the number of species where it is fixed at compile time, else 0.
template <int N, int L, int NW, bool SPLIT, int SP>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(N <= 8 && L <= 6 ? 3 : 2, 8))) void k_soap_fwd_x(
    SoapDev sp, int nc, int cpb, const int *__restrict__ centres, const int *__restrict__ Z,
    const int *__restrict__ nb_off, const int *__restrict__ nb_j, const double *__restrict__ nb_r,
    const double *__restrict__ nb_d, double *X, double *norm_out, double *cbuf, int p_lds_, int c_lds_) {
    extern __shared__ double lds[];
    constexpr int NA = (N + 3) / 4, LM = (L + 1) * (L + 1);
    const int S = SP ? SP : sp.S, K = S * N, KLM = K * LM, d = K * (K + 1) / 2 * (L + 1) + 1;
    const bool p_lds = SP || p_lds_, c_lds = SP || c_lds_;
    const FwdLds lo(NA, L, S, NW, d, p_lds, c_lds);
    double *tab = lds + lo.tab_off, *red = lds + lo.p_off, *pL = red, *cL = lds + lo.c_off, *ssw = lds + lo.tail;
    int *sb = (int *)(ssw + NW), *sc = sb + S;
    SoapTables<N, L> tb(lds + lo.total / 8);
    tb.fill(sp, 64 * NW);
    const int lane = threadIdx.x & 63;
    const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int d0 = blockIdx.x * cpb, dn = min(d0 + cpb, nc);
    int ci = centres[d0], cn = centres[min(d0 + 1, dn - 1)];
    int p0 = nb_off[ci], np = nb_off[ci + 1] - p0;
    SoapNb nb;
    if (w == NW - 1) {
        nb.load(p0, min(kSoapPass, np), nb_j, nb_r, nb_d);
        nb.species(min(kSoapPass, np), Z);
    }
    __syncthreads();
    for (int desc = d0; desc < dn; desc++) {
        // the next centre's pairs and the index of the one after it
        const int pn = nb_off[cn], nn = nb_off[cn + 1] - pn;
        const int c2 = centres[min(desc + 2, dn - 1)];
        const int csp = species_s(sp, S, Z[ci]);
        double *co = cbuf + (size_t)desc * KLM;

        auto unit = [&](auto sets_tag, int s, bool first_pass, bool last_pass) {
            constexpr int SETS = decltype(sets_tag)::value;
            using FG = FwdGroups<L, SETS>;
            constexpr int NGS = FG::count;
            const int ln0 = fresh_lane(), i4 = ln0 & 3;
            SoapLane<N> rl;
            rl.setup(tb.rt, i4);
            double acc[NGS][NA];
#pragma unroll
            for (int i = 0; i < NGS; i++)
#pragma unroll
                for (int u = 0; u < NA; u++) acc[i][u] = 0.0;
            for (int c0 = 0; c0 < np; c0 += kSoapPass) {
                const int nk = min(kSoapPass, np - c0);
                if (first_pass || np > kSoapPass) {   // a single pass of neighbours stays staged for every unit
                    block_lds_sync<NW>();
                    if (w == NW - 1) {
                        if (!first_pass || c0 > 0) {
                            nb.load(p0 + c0, nk, nb_j, nb_r, nb_d);
                            nb.species(nk, Z);
                        }
                        soap_stage<N, false>(sp, S, nb, p0 + c0, nk, tab, lo.slots, sb, sc, nullptr);
                    }
                    block_lds_sync<NW>();
                }
                if (s < 0) continue;
                const int base = sb[s], cnt = sc[s];
                for (int t = 0; t < cnt; t += 16) {
                    const int off = t + (lane >> 2);
                    const int sl = base + min(off, cnt - 1);
                    const double x = tab[kUx * lo.slots + sl], y = tab[kUy * lo.slots + sl];
                    rl.z = tab[kUz * lo.slots + sl];
                    const double e0 = off < cnt ? tab[kE0 * lo.slots + sl] : 0.0;
                    rl.radial(sp, i4, tab[kIxq * lo.slots + sl], e0, tab[kQ * lo.slots + sl], tab[kQi * lo.slots + sl]);
                    // (x + i y)^m of m = i4 and i4 + 4
                    const double x2 = x * x - y * y, y2 = 2.0 * x * y;
                    const double x3 = x2 * x - y2 * y, y3 = x2 * y + y2 * x;
                    const double Aa = i4 == 0 ? 1.0 : i4 == 1 ? x : i4 == 2 ? x2 : x3;
                    const double Ba = i4 == 0 ? 0.0 : i4 == 1 ? y : i4 == 2 ? y2 : y3;
                    const double x4 = x2 * x2 - y2 * y2, y4 = 2.0 * x2 * y2;
                    const double Ab = Aa * x4 - Ba * y4, Bb = Aa * y4 + Ba * x4;
                    rl.pA = rl.pA1 = rl.pB = rl.pB1 = 0.0;
#pragma unroll
                    for (int l = 0; l <= L; l++) {
                        double F[NA];
#pragma unroll
                        for (int u = 0; u < NA; u++) F[u] = rl.f(l, u);
                        if constexpr (SETS & 1) {
                            const double p = rl.legendre(l, 0, rl.mA2, rl.pA, rl.pA1);
                            rl.pA1 = rl.pA;
                            rl.pA = p;
                            const double ya = p * Aa, yb = p * Ba;
#pragma unroll
                            for (int u = 0; u < NA; u++) {
                                acc[FG::index(l, 0)][u] = mfma4(F[u], ya, acc[FG::index(l, 0)][u]);
                                if (l > 0) acc[FG::index(l, 1)][u] = mfma4(F[u], yb, acc[FG::index(l, 1)][u]);
                            }
                        }
                        if constexpr (SETS & 2) {
                            if (l >= 4) {
                                const double p = rl.legendre(l, 4, rl.mB2, rl.pB, rl.pB1);
                                rl.pB1 = rl.pB;
                                rl.pB = p;
                                const double ya = p * Ab, yb = p * Bb;
#pragma unroll
                                for (int u = 0; u < NA; u++) {
                                    acc[FG::index(l, 2)][u] = mfma4(F[u], ya, acc[FG::index(l, 2)][u]);
                                    acc[FG::index(l, 3)][u] = mfma4(F[u], yb, acc[FG::index(l, 3)][u]);
                                }
                            }
                            if (l >= 8) {   // m = 8 in slot 0; the other slots' factor is zero
                                const double ya = x4 * x4 - y4 * y4, yb = 2.0 * x4 * y4;
                                constexpr int v4 = L >= 8 ? 4 : 2, v5 = L >= 8 ? 5 : 3;
#pragma unroll
                                for (int u = 0; u < NA; u++) {
                                    acc[FG::index(l, v4)][u] = mfma4(F[u], ya, acc[FG::index(l, v4)][u]);
                                    acc[FG::index(l, v5)][u] = mfma4(F[u], yb, acc[FG::index(l, v5)][u]);
                                }
                            }
                        }
                        if (l < L) rl.step(l);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            if (last_pass && desc + 1 < dn && w == NW - 1)   // the next centre's neighbours set out
                nb.load(pn, min(kSoapPass, nn), nb_j, nb_r, nb_d);
            if (s < 0) return;
            // sum the four quarters, four groups at a time, transform, and store c (times the
            // harmonics' factor, as the adjoint takes it)
            const int ln = fresh_lane(), k4 = ln >> 4, b4 = (ln >> 2) & 3;
            double TA[NA][NA];   // T[a = 4u + k][b = 4v + i] of the transform's operand
#pragma unroll
            for (int u = 0; u < NA; u++)
#pragma unroll
                for (int v = 0; v < NA; v++) {
                    const int a = 4 * u + k4, b = 4 * v + i4;
                    TA[v][u] = tb.t(a, b);
                }
            double *rw = red + w * lo.rs;
            constexpr int NQ = (NGS + 3) / 4;
#pragma unroll
            for (int t = 0; t < NQ; t++) {
                wave_lds_sync();
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * t + i < NGS)
#pragma unroll
                        for (int u = 0; u < NA; u++)
                            rw[i * lo.gs + 64 * u + lane] = acc[4 * t + i < NGS ? 4 * t + i : 0][u];
                wave_lds_sync();
                const bool ok = 4 * t + 3 < NGS || 4 * t + b4 < NGS;
                const int g = FG::group(ok ? 4 * t + b4 : 0);
                const double nk = ok ? tb.gn[4 * g + i4] : 0.0;
                const int pos = ok ? tb.pos[4 * g + i4] & 0xffff : 0xffff;
                double Bv[NA];
#pragma unroll
                for (int u = 0; u < NA; u++) {
                    const double *q = rw + (ok ? b4 : 0) * lo.gs + 64 * u + 16 * k4 + i4;
                    Bv[u] = ((q[0] + q[4]) + (q[8] + q[12])) * nk;
                }
#pragma unroll
                for (int v = 0; v < NA; v++) {
                    double D = 0.0;
#pragma unroll
                    for (int u = 0; u < NA; u++) D = mfma4(TA[v][u], Bv[u], D);
                    const int row = 4 * v + k4;
                    if (v == 0 && k4 == 0 && i4 == 0 && ok && g == 0 && s == csp) D += sp.cw * sp.u00 * nk;
                    if (c_lds && ok) cL[(s * NA * 4 + row) * lo.cs + 4 * g + i4] = D;
                    if (pos != 0xffff && (N % 4 == 0 || row < N)) co[(s * N + row) * LM + pos] = D * nk;
                }
            }
        };
        const int nunits = SPLIT ? 2 * S : S;
        for (int u0 = 0; u0 < nunits; u0 += NW) {
            const int un = u0 + w;
            const int s = un < nunits ? (SPLIT ? un >> 1 : un) : -1;
            if constexpr (SPLIT) {
                if (un & 1) unit(std::integral_constant<int, 2>{}, s, u0 == 0, u0 + NW >= nunits);
                else unit(std::integral_constant<int, 1>{}, s, u0 == 0, u0 + NW >= nunits);
            } else {
                unit(std::integral_constant<int, 3>{}, s, u0 == 0, u0 + NW >= nunits);
            }
        }
        if (c_lds) block_lds_sync<NW>();
        else __syncthreads();
        // power spectrum: blocks of 4 x 4 row pairs (gi >= gj), four pairs per product
        const int R = S * NA, npair = R * (R + 1) / 2;
        double *xo = X + (size_t)desc * d;
        double ss = 0.0;
        for (int q0 = 4 * w; q0 < npair; q0 += 4 * NW) {
            const int ln = fresh_lane(), k4 = ln >> 4, b4 = (ln >> 2) & 3, i4 = ln & 3;
            const int pi = min(q0 + b4, npair - 1);
            int gi = (int)((sqrtf(8.0f * (float)pi + 1.0f) - 1.0f) * 0.5f);
            while ((gi + 1) * (gi + 2) / 2 <= pi) gi++;
            while (gi * (gi + 1) / 2 > pi) gi--;
            const int gj = pi - gi * (gi + 1) / 2;
            const int ri = 4 * gi + k4, rj = 4 * gj + i4;   // rows of this lane's result
            const int ai = ri % (4 * NA), aj = rj % (4 * NA);
            const int ia = ri / (4 * NA) * N + ai, jb = rj / (4 * NA) * N + aj;
            const bool ok = q0 + b4 < npair && ai < N && aj < N && ia >= jb;
            const double f = ia != jb ? 1.4142135623730950488 : 1.0;
            const int q = (ia * (ia + 1) / 2 + jb) * (L + 1);
            if (c_lds) {
                const double *ca = cL + (4 * gi + i4) * lo.cs + k4, *cb = cL + (4 * gj + i4) * lo.cs + k4;
#pragma unroll
                for (int l = 0; l <= L; l++) {
                    double D = 0.0;
#pragma unroll
                    for (int v = 0; v < lev_groups(l); v++)
                        D = mfma4(ca[4 * (lev_base(l) + v)], cb[4 * (lev_base(l) + v)], D);
                    const double p = D * (f * tb.isq[l]);
                    if (ok) {
                        if (p_lds) pL[q + l] = p;
                        else xo[q + l] = p;
                        ss += p * p;
                    }
                }
            } else {   // many species: c is read back from memory
                const int ra = 4 * gi + i4, rb = 4 * gj + i4;
                const bool oa = ra % (4 * NA) < N, ob = rb % (4 * NA) < N;
                const double *ca = co + (size_t)(ra / (4 * NA) * N + ra % (4 * NA)) * LM;
                const double *cb = co + (size_t)(rb / (4 * NA) * N + rb % (4 * NA)) * LM;
                for (int l = 0; l <= L; l++) {
                    double D = 0.0;
                    for (int v = 0; v < lev_groups(l); v++) {
                        const int pos = c_gpos[4 * (lev_base(l) + v) + k4];
                        const double f1 = c_ginv[4 * (lev_base(l) + v) + k4];
                        D = mfma4(oa && pos >= 0 ? ca[pos] * f1 : 0.0, ob && pos >= 0 ? cb[pos] * f1 : 0.0, D);
                    }
                    const double p = D * (f * tb.isq[l]);
                    if (ok) {
                        if (p_lds) pL[q + l] = p;
                        else xo[q + l] = p;
                        ss += p * p;
                    }
                }
            }
        }
        if (desc + 1 < dn && w == NW - 1) nb.species(min(kSoapPass, nn), Z);
        ss = wave_sum_s(ss);
        if (NW > 1 && lane == 0) ssw[w] = ss;
        if (p_lds) block_lds_sync<NW>();
        else __syncthreads();
        if (NW > 1) {
            ss = ssw[0];
#pragma unroll
            for (int i = 1; i < NW; i++) ss += ssw[i];
        }
        const double nrm = sqrt(ss);
        const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
        for (int q = threadIdx.x; q < d - 1; q += 64 * NW) xo[q] = (p_lds ? pL[q] : xo[q]) * inv;
        if (threadIdx.x == 0) {
            xo[d - 1] = 0.0;
            norm_out[desc] = nrm;
        }
        ci = cn;
        cn = c2;
        p0 = pn;
        np = nn;
        if (NW > 1) block_lds_sync<NW>();   // the power spectrum's place is free again
    }
}

// LDS layout of the adjoint kernel, in doubles: the neighbour table, dE/dc' of SB species as
// operands, dE/dp (p_lds), a wave sum per wavefront, then the slot tables
struct BwdLds {
    int slots, a_off, p_off, w_off, total;
    __host__ __device__ BwdLds(int NA, int L, int S, int SB, int nw, int dim, bool p_lds) {
        slots = kSoapPass + 16 * (S - 1);
        a_off = kBwdFields * slots;
        p_off = a_off + SB * soap_groups(L) * NA * 16;
        w_off = p_off + (p_lds ? dim : 0);
        total = (w_off + nw) * 8 + (2 * S + slots) * 4;   // followed by the constant tables
        total = (total + 7) & ~7;
    }
};

// Adjoint: a block of NW wavefronts takes cpb centres in turn; a centre's neighbours (and
// where they fit the registers X and G) are fetched while the one before is worked on.
// dE/dp = (G - x (x.G)) / |p| is staged in LDS; dE/dc_l = P_l c_l and dE/dc' = T dE/dc follow as
// chained 4x4x4 products, four harmonic groups at a time, the result of the first being the
// operand of the second as it stands.  Then tiles of 16 neighbours: lane 16 g + n holds
// neighbour n's radial functions of a = g, g+4, .. and their r derivatives, which multiply
// dE/dc' from LDS; the products come out in the lanes that hold the harmonics they belong
// to (m = g, g+4).  With S0_lm = sum_a F_l(a) dc'[a][lm] and S1_lm = sum_a F_l'(a) dc'[a][lm]
// the pair's force is (fc sum S1 Y + dfc sum S0 Y) u + fc (V - u (u.V)) / r, V = sum S0 gradY.
// The sums over l are kept per m with the Legendre factors only; (x + i y)^m enters once at
// the end, and a last product with unit rows sums the lanes of a neighbour.  135612 Si
// centres at 8/6: 1.09 -> 0.63 ms against a lane per neighbour reading dE/dc' from LDS (VALU issue
// 47%, matrix pipe 27% of it); 32768 SiC centres at 12/8: 3.80 -> 0.90 ms.  A wavefront per centre and
// 2 wavefronts per SIMD: with spills at 3 the reloads queue behind the data on their way (1.07 ms).
// Up to l = 4, two species (183 to 190 registers cut to 168: 55296 centres at 5/4 868 -> 798 us)
// and those not fixed at compile time (13440 centres of five at 5/4 1240 -> 928 us) take 3.
// SP: the number of species where it is fixed at compile time, else 0; then X, G and c are
// fetched several at a time, c a species ahead of its product (22400 centres of three
// species at 12/6: 3346 -> 2347 us).
constexpr int bwd_waves(int L, int SP) { return L <= 4 && (SP == 0 || SP == 2) ? 3 : 2; }
template <int N, int L, int NW, int SP>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(bwd_waves(L, SP), 8))) void k_soap_bwd_x(
    SoapDev sp, int nc, int cpb, const int *__restrict__ centres, const int *__restrict__ Z,
    const int *__restrict__ nb_off, const int *__restrict__ nb_j, const double *__restrict__ nb_r,
    const double *__restrict__ nb_d, const double *__restrict__ X, const double *__restrict__ G,
    const double *__restrict__ norm, const double *__restrict__ cbuf, double *pairF, int p_lds_, int SB_, int add) {
    extern __shared__ double lds[];
    constexpr int NA = (N + 3) / 4, LM = (L + 1) * (L + 1), NG = soap_groups(L), NQ = (NG + 3) / 4;
    constexpr int DC = SP * N * (SP * N + 1) / 2 * (L + 1);            // components (less the last, zero one)
    constexpr int QR = SP ? (DC + 64 * NW - 1) / (64 * NW) : 1;        // of them per lane
    constexpr bool AHEAD = SP && QR <= 4;                              // X and G of the next centre in registers
    constexpr int UN = SP ? (NQ * SP + NW - 1) / NW : 1;               // quads of groups per wavefront (one species each)
    constexpr bool CAHEAD = SP && UN * SP * NA <= 12;                  // the next centre's c likewise
    static_assert(SP <= 1 || NW % SP == 0, "wavefronts are dealt evenly to the species");
    const int S = SP ? SP : sp.S, KLM = S * N * LM, d = SP ? DC + 1 : sp.dim;
    const int SB = SP ? SP : SB_;
    const bool p_lds = SP || p_lds_;
    const BwdLds lo(NA, L, S, SB, NW, d, p_lds);
    double *tab = lds, *Aop = lds + lo.a_off, *P = lds + lo.p_off, *ws = lds + lo.w_off;
    int *sb = (int *)(ws + NW), *sc = sb + S, *pair = sc + S;
    SoapTables<N, L> tb(lds + lo.total / 8);
    tb.fill(sp, 64 * NW);
    const int lane = threadIdx.x & 63;
    const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int d0 = blockIdx.x * cpb, dn = min(d0 + cpb, nc);
    double xr[QR], gr[QR];   // X and G of this lane's components
    auto load_xg = [&](int desc) {
        const double *x = X + (size_t)desc * d, *gg = G + (size_t)desc * d;
#pragma unroll
        for (int i = 0; i < QR; i++) {
            const int q = threadIdx.x + 64 * NW * i;
            xr[i] = q < d - 1 ? x[q] : 0.0;
            gr[i] = q < d - 1 ? gg[q] : 0.0;
        }
    };
    if (SP) load_xg(d0);
    int ci = centres[d0], cn = centres[min(d0 + 1, dn - 1)];
    int p0 = nb_off[ci], np = nb_off[ci + 1] - p0;
    SoapNb nb;
    if (w == NW - 1) {
        nb.load(p0, min(kSoapPass, np), nb_j, nb_r, nb_d);
        nb.species(min(kSoapPass, np), Z);
    }
    __syncthreads();
    // columns of c of this wavefront's quads of groups (times the harmonics' factor)
    const int ws_ = SP > 1 ? w / (NW / SP) : 0, tw = SP > 1 ? w % (NW / SP) : w;
    constexpr int TS = SP > 1 ? NW / SP : NW;
    double cB[UN][SP ? SP * NA : 1];
    auto load_c = [&](int desc) {
        const double *cg = cbuf + (size_t)desc * KLM;
        const int ln = fresh_lane(), k4 = ln >> 4;
#pragma unroll
        for (int i = 0; i < UN; i++) {
            const int g4 = 16 * (tw + TS * i) + (ln & 15);   // 4 group + slot
            const int pos = g4 < 4 * NG ? tb.pos[g4] & 0xffff : 0xffff;
#pragma unroll
            for (int k = 0; k < SP * NA; k++) {
                const int aj = 4 * (k % NA) + k4;
                cB[i][k] = pos != 0xffff && (N % 4 == 0 || aj < N) ? cg[(k / NA * N + aj) * LM + pos] : 0.0;
            }
        }
    };
    if (CAHEAD) load_c(d0);
    for (int desc = d0; desc < dn; desc++) {
        const int pn = nb_off[cn], nn = nb_off[cn + 1] - pn;
        const int c2 = centres[min(desc + 2, dn - 1)];
        const double *x = X + (size_t)desc * d, *gg = G + (size_t)desc * d, *cg = cbuf + (size_t)desc * KLM;
        const double nrm = norm[desc];
        const int ln = fresh_lane(), k4 = ln >> 4, b4 = (ln >> 2) & 3, i4 = ln & 3;
        double dot = 0.0;
        if (SP) {
            if (!AHEAD && desc > d0) load_xg(desc);
            if (!CAHEAD) load_c(desc);
#pragma unroll
            for (int i = 0; i < QR; i++) dot += xr[i] * gr[i];
        } else {
#pragma unroll 4
            for (int q = threadIdx.x; q < d; q += 64 * NW) dot += x[q] * gg[q];
        }
        dot = wave_sum_s(dot);
        if (NW > 1) {
            if (lane == 0) ws[w] = dot;
            block_lds_sync<NW>();
            dot = ws[0];
#pragma unroll
            for (int i = 1; i < NW; i++) dot += ws[i];
        }
        const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
        if (SP) {
#pragma unroll
            for (int i = 0; i < QR; i++) {
                const int q = threadIdx.x + 64 * NW * i;
                if (q < d - 1) P[q] = gr[i] - xr[i] * dot;
            }
        } else if (p_lds) {
#pragma unroll 4
            for (int q = threadIdx.x; q < d - 1; q += 64 * NW) P[q] = gg[q] - x[q] * dot;
        }
        block_lds_sync<NW>();
        // dE/dc = P_l c with P_l[ia][jb] = (G - x (x.G))_(ia,jb),l / |p| x (2 if ia = jb else sqrt 2) / sqrt(2l+1):
        // the diagonal's factor enters with the operand, the columns' factor with the result
        const double dg = i4 == k4 ? 1.4142135623730950488 : 1.0;
        const double invs = 1.4142135623730950488 * inv;
        double TA[NA][NA];   // T[a = 4v + i][b = 4u + k]
#pragma unroll
        for (int u = 0; u < NA; u++)
#pragma unroll
            for (int v = 0; v < NA; v++) TA[v][u] = tb.t(4 * v + i4, 4 * u + k4);
        bool staged_first = false;
        for (int s0 = 0; s0 < S; s0 += SB) {
            const int ns = min(SB, S - s0);
            if (s0 > 0) block_lds_sync<NW>();   // the previous species' operands are done with
            if constexpr (SP > 0) {
                int qi[SP * NA][NA];   // place of P_0[ia = (s, 4u + i)][jb = (sj, 4kk + k)], -1: none
#pragma unroll
                for (int k = 0; k < SP * NA; k++)
#pragma unroll
                    for (int u = 0; u < NA; u++) {
                        const int ai = 4 * u + i4, aj = 4 * (k % NA) + k4;
                        const int ia = ws_ * N + ai, jb = k / NA * N + aj;
                        const int hi = max(ia, jb), lw = min(ia, jb);
                        qi[k][u] = N % 4 == 0 || (ai < N && aj < N) ? (__umul24(hi, hi + 1) / 2 + lw) * (L + 1) : -1;
                    }
#pragma unroll
                for (int i = 0; i < UN; i++) {
                    const int g = 4 * (tw + TS * i) + b4;
                    if (4 * (tw + TS * i) >= NG) continue;
                    const int l = tb.pos[4 * g + i4] >> 16;
                    const double cf = invs * tb.isq[l];
                    double D1[NA];
#pragma unroll
                    for (int u = 0; u < NA; u++) D1[u] = 0.0;
#pragma unroll
                    for (int k = 0; k < SP * NA; k++)
#pragma unroll
                        for (int u = 0; u < NA; u++) {
                            double a = N % 4 == 0 || qi[k][u] >= 0 ? P[qi[k][u] + l] : 0.0;
                            if (k == ws_ * NA + u) a *= dg;
                            D1[u] = mfma4(a, cB[i][k], D1[u]);
                        }
                    double *ao = Aop + ((ws_ * NG + g) * NA) * 16 + 4 * k4 + i4;
#pragma unroll
                    for (int v = 0; v < NA; v++) {
                        double D = 0.0;
#pragma unroll
                        for (int u = 0; u < NA; u++) D = mfma4(TA[v][u], D1[u], D);
                        if (g < NG) ao[16 * v] = D * cf;
                    }
                }
            } else {
                for (int un = w; un < NQ * ns; un += NW) {
                    const int sr = un / NQ, t = un - sr * NQ, s = s0 + sr;
                    const int g = min(4 * t + b4, NG - 1);
                    const int pos = tb.pos[4 * g + i4] & 0xffff, l = tb.pos[4 * g + i4] >> 16;
                    double D1[NA];
#pragma unroll
                    for (int u = 0; u < NA; u++) D1[u] = 0.0;
                    double cn[NA];   // a column of c ahead of its product
                    auto load_col = [&](int sj) {
#pragma unroll
                        for (int kk = 0; kk < NA; kk++) {
                            const int aj = 4 * kk + k4;
                            cn[kk] = sj < S && (N % 4 == 0 || aj < N) && pos != 0xffff ? cg[(sj * N + aj) * LM + pos] : 0.0;
                        }
                    };
                    load_col(0);
                    for (int sj = 0; sj < S; sj++) {
                        double cc[NA];
#pragma unroll
                        for (int kk = 0; kk < NA; kk++) cc[kk] = cn[kk];
                        load_col(sj + 1);
#pragma unroll
                        for (int kk = 0; kk < NA; kk++) {
                            const int aj = 4 * kk + k4, jb = sj * N + aj;
                            const bool okj = N % 4 == 0 || aj < N;
                            const double cb = cc[kk];
#pragma unroll
                            for (int u = 0; u < NA; u++) {
                                const int ai = 4 * u + i4, ia = s * N + ai;
                                const int hi = max(ia, jb), lw = min(ia, jb);
                                const int q = (hi * (hi + 1) / 2 + lw) * (L + 1) + l;
                                double a = 0.0;
                                if (okj && (N % 4 == 0 || ai < N)) {
                                    a = p_lds ? P[q] : gg[q] - x[q] * dot;
                                    if (ia == jb) a *= 1.4142135623730950488;
                                }
                                D1[u] = mfma4(a, cb, D1[u]);
                            }
                        }
                    }
                    double *ao = Aop + ((sr * NG + g) * NA) * 16 + 4 * k4 + i4;
#pragma unroll
                    for (int v = 0; v < NA; v++) {
                        double D = 0.0;
#pragma unroll
                        for (int u = 0; u < NA; u++) D = mfma4(TA[v][u], D1[u], D);
                        if (4 * t + b4 < NG) ao[16 * v] = D * (invs * tb.isq[l]);
                    }
                }
            }
            for (int c0 = 0; c0 < np; c0 += kSoapPass) {
                const int nk = min(kSoapPass, np - c0);
                if (!staged_first || np > kSoapPass) {   // a single pass of neighbours stays staged
                    if (staged_first) block_lds_sync<NW>();
                    if (w == NW - 1) {
                        if (staged_first) {
                            nb.load(p0 + c0, nk, nb_j, nb_r, nb_d);
                            nb.species(nk, Z);
                        }
                        soap_stage<N, true>(sp, S, nb, p0 + c0, nk, tab, lo.slots, sb, sc, pair);
                    }
                    staged_first = true;
                }
                block_lds_sync<NW>();
                if (s0 + SB >= S && c0 + kSoapPass >= np && desc + 1 < dn) {   // the next centre's data set out
                    if (w == NW - 1) nb.load(pn, min(kSoapPass, nn), nb_j, nb_r, nb_d);
                    if (AHEAD) load_xg(desc + 1);
                    if (CAHEAD) load_c(desc + 1);
                }
                const int lt = fresh_lane(), k4 = lt >> 4, i4 = lt & 3;
                SoapLane<N> rl;
                rl.setup(tb.rt, k4);
                int tile = 0;   // tiles are dealt to the wavefronts in turn
                for (int sr = 0; sr < ns; sr++) {
                    const int base = sb[s0 + sr], cnt = sc[s0 + sr];
                    const double *as = Aop + sr * NG * NA * 16 + 4 * k4 + i4;
                    for (int t = 0; t < cnt; t += 16, tile++) {
                        if (NW > 1 && tile % NW != w) continue;
                        const int off = t + (lane & 15);
                        const int sl = base + min(off, cnt - 1);
                        // an earlier descriptor's force on the pair (add), fetched before it is needed
                        const double old = add && k4 < 3 ? pairF[3 * (size_t)pair[sl] + k4] : 0.0;
                        const double ux = tab[kUx * lo.slots + sl], uy = tab[kUy * lo.slots + sl];
                        const double uz = tab[kUz * lo.slots + sl];
                        rl.radial(sp, k4, tab[kIxq * lo.slots + sl], tab[kE0 * lo.slots + sl], tab[kQ * lo.slots + sl],
                                  tab[kQi * lo.slots + sl]);
                        rl.z = uz;
                        double ca[NA];   // 2 alpha r_a
#pragma unroll
                        for (int u = 0; u < NA; u++) ca[u] = (k4 + 4 * u) * sp.a2dr;
                        const double ir = tab[kIr * lo.slots + sl];
                        const double m2ar = -2.0 * sp.alpha * tab[kR * lo.slots + sl];
                        double pA = 0.0, pA1 = 0.0, dA = 0.0, dA1 = 0.0, pB = 0.0, pB1 = 0.0, dB = 0.0, dB1 = 0.0;
                        // per m: sums over l of S0 p, S1 p, S0 p' for the cos (a) and sin (b) harmonics
                        double a0 = 0.0, a1 = 0.0, az = 0.0, b0 = 0.0, b1 = 0.0, bz = 0.0;
                        double e0 = 0.0, e1 = 0.0, ez = 0.0, f0 = 0.0, f1 = 0.0, fz = 0.0;
                        double h0 = 0.0, h1 = 0.0, i0 = 0.0, i1 = 0.0;
#pragma unroll
                        for (int l = 0; l <= L; l++) {
                            double F[NA], Fd[NA];
                            const double cl = fma((double)l, ir, m2ar);
#pragma unroll
                            for (int u = 0; u < NA; u++) {
                                F[u] = rl.f(l, u);
                                Fd[u] = fma(cl, F[u], ca[u] * rl.F1[u]);
                            }
                            double S0[6], S1[6];
#pragma unroll
                            for (int v = 0; v < lev_groups(l); v++) {
                                S0[v] = S1[v] = 0.0;
#pragma unroll
                                for (int u = 0; u < NA; u++) {
                                    const double a = as[((lev_base(l) + v) * NA + u) * 16];
                                    S0[v] = mfma4(a, F[u], S0[v]);
                                    S1[v] = mfma4(a, Fd[u], S1[v]);
                                }
                            }
                            {
                                const double p = rl.legendre(l, 0, rl.mA2, pA, pA1);
                                double dp = 0.0;
                                if (l == 1) dp = pA;
                                if (l > 1) dp = pA + (uz * dA - leg_beta(l, rl.mA2) * dA1);
                                pA1 = pA; pA = p;
                                dA1 = dA; dA = dp;
                                a0 += S0[0] * p; a1 += S1[0] * p; az += S0[0] * dp;
                                if (l > 0) { b0 += S0[1] * p; b1 += S1[1] * p; bz += S0[1] * dp; }
                            }
                            if (l >= 4) {
                                const double p = rl.legendre(l, 4, rl.mB2, pB, pB1);
                                double dp = 0.0;
                                if (l == 5) dp = pB;
                                if (l > 5) dp = pB + (uz * dB - leg_beta(l, rl.mB2) * dB1);
                                pB1 = pB; pB = p;
                                dB1 = dB; dB = dp;
                                constexpr int va = 2, vb = 3;
                                e0 += S0[va] * p; e1 += S1[va] * p; ez += S0[va] * dp;
                                f0 += S0[vb] * p; f1 += S1[vb] * p; fz += S0[vb] * dp;
                            }
                            if (l >= 8) { h0 = S0[4]; h1 = S1[4]; i0 = S0[5]; i1 = S1[5]; }
                            if (l < L) rl.step(l);
                            __builtin_amdgcn_sched_barrier(0);
                        __builtin_amdgcn_sched_barrier(0);
                        }
                        const double x2 = ux * ux - uy * uy, y2 = 2.0 * ux * uy;
                        const double x3 = x2 * ux - y2 * uy, y3 = x2 * uy + y2 * ux;
                        const double x4 = x2 * x2 - y2 * y2, y4 = 2.0 * x2 * y2;
                        // (x + i y)^g and ^(g-1) (which meets the factor m = 0 in group 0)
                        const double Aa = k4 == 0 ? 1.0 : k4 == 1 ? ux : k4 == 2 ? x2 : x3;
                        const double Ba = k4 == 0 ? 0.0 : k4 == 1 ? uy : k4 == 2 ? y2 : y3;
                        const double Am = k4 <= 1 ? 1.0 : k4 == 2 ? ux : x2;
                        const double Bm = k4 <= 1 ? 0.0 : k4 == 2 ? uy : y2;
                        const double m = (double)k4;
                        double T0 = Aa * a0 + Ba * b0, T1 = Aa * a1 + Ba * b1, Vz = Aa * az + Ba * bz;
                        double Vx = m * (a0 * Am + b0 * Bm), Vy = m * (b0 * Am - a0 * Bm);
                        {
                            const double Ab = Aa * x4 - Ba * y4, Bb = Aa * y4 + Ba * x4;
                            const double An = Aa * x3 - Ba * y3, Bn = Aa * y3 + Ba * x3, mm = m + 4.0;
                            T0 += Ab * e0 + Bb * f0;
                            T1 += Ab * e1 + Bb * f1;
                            Vz += Ab * ez + Bb * fz;
                            Vx += mm * (e0 * An + f0 * Bn);
                            Vy += mm * (f0 * An - e0 * Bn);
                        }
                        if constexpr (L >= 8) {   // group 0 only: the others' operands are zero
                            const double A8 = x4 * x4 - y4 * y4, B8 = 2.0 * x4 * y4;
                            const double A7 = x4 * x3 - y4 * y3, B7 = x4 * y3 + y4 * x3;
                            T0 += A8 * h0 + B8 * i0;
                            T1 += A8 * h1 + B8 * i1;
                            Vx += 8.0 * (h0 * A7 + i0 * B7);
                            Vy += 8.0 * (i0 * A7 - h0 * B7);
                        }
                        const double fc = tab[kFc * lo.slots + sl], dfc = tab[kDfc * lo.slots + sl];
                        Vx *= fc; Vy *= fc; Vz *= fc;
                        const double rad = (fc * T1 + dfc * T0) - (ux * Vx + uy * Vy + uz * Vz) * ir;
                        // row c of the product: component c summed over the neighbour's four lanes
                        double D = mfma4(i4 == 0 ? 1.0 : 0.0, rad * ux + Vx * ir, 0.0);
                        D = mfma4(i4 == 1 ? 1.0 : 0.0, rad * uy + Vy * ir, D);
                        D = mfma4(i4 == 2 ? 1.0 : 0.0, rad * uz + Vz * ir, D);
                        if (k4 < 3 && off < cnt) pairF[3 * (size_t)pair[sl] + k4] = add ? old + D : D;
                    }
                }
            }
        }
        if (np == 0 && desc + 1 < dn) {
            if (w == NW - 1) nb.load(pn, min(kSoapPass, nn), nb_j, nb_r, nb_d);
            if (AHEAD) load_xg(desc + 1);
            if (CAHEAD) load_c(desc + 1);
        }
        if (desc + 1 < dn && w == NW - 1) nb.species(min(kSoapPass, nn), Z);
        ci = cn;
        cn = c2;
        p0 = pn;
        np = nn;
        block_lds_sync<NW>();   // the table and the operands are free again
    }
}

#define SOAP_FAST(X) X(4, 4) X(5, 4) X(6, 4) X(8, 4) X(6, 6) X(8, 6) X(10, 6) X(12, 6) X(8, 8) X(10, 8) X(12, 8)

int soap_fast_supported(int n, int L) {
#define CHK(NN, LL) if (n == NN && L == LL) return 1;
    SOAP_FAST(CHK)
#undef CHK
    return 0;
}

// What a block may take: within it the power spectrum, c and dE/dp are kept in LDS where
// they fit, so that two blocks of four wavefronts, what the registers of bases past l = 4 allow,
// share a CU (160 KB; the constant tables take up to 3 KB more); the rest goes through memory.
// 22400 centres of five species at 6/6: the adjoint 3326 us with dE/dp in memory.
constexpr int kSoapLdsCap = 76 * 1024;

struct FwdPlan {
    bool own, split, p_lds, c_lds;
    int nw;
    size_t lds;
};
static size_t table_lds(const SoapDev &sp) {
    const int nq4 = (soap_groups(sp.L) + 3) / 4 * 4;
    return (size_t)(sp.n * sp.n + 24 + 4 * nq4 + sp.L + 1) * 8 + 4 * nq4 * 4;
}
// A wavefront per species: its own neighbours with all harmonics, and its own rows of dE/dc
// (bases up to 8/6, two to four species).  Otherwise four wavefronts share a centre, m < 4 and
// m >= 4 apart.  A small basis leaves those little to do between their barriers, and species
// that are not fixed at compile time have c and dE/dp read where they are needed.  Forward
// + adjoint of 55296 centres at 5/4: two species 868 + 1237 -> 541 + 868 us, four 938 + 1528 ->
// 626 + 875; of 8/6, four species: 1646 + 3510 -> 1196 + 1549.  Two species have half as many
// wavefronts this way: up to 512 centres, whose four wavefronts the card holds at once, these
// are faster (500 centres at 8/6 53 us against 61, 600 centres 67 against 63).
static bool wave_per_species(const SoapDev &sp, int nc) {
    return sp.n <= 8 && sp.L <= 6 && sp.S >= (nc > 512 ? 2 : 3) && sp.S <= 4;
}
static FwdPlan fwd_plan(const SoapDev &sp, bool own, bool split) {
    FwdPlan f;
    const int NA = (sp.n + 3) / 4;
    f.own = own;
    f.split = split || (sp.S > 1 && !own);
    f.nw = own ? sp.S : sp.S > 1 ? 4 : split ? 2 : 1;
    f.p_lds = f.c_lds = true;
    if (FwdLds(NA, sp.L, sp.S, f.nw, sp.dim, true, true).total > kSoapLdsCap) f.p_lds = false;
    if (FwdLds(NA, sp.L, sp.S, f.nw, sp.dim, f.p_lds, true).total > kSoapLdsCap) f.c_lds = false;
    f.lds = FwdLds(NA, sp.L, sp.S, f.nw, sp.dim, f.p_lds, f.c_lds).total + table_lds(sp);
    // the form of fixed species keeps both in LDS
    return own && !(f.p_lds && f.c_lds) ? fwd_plan(sp, false, split) : f;
}
struct BwdPlan {
    bool own, p_lds;
    int nw, SB;
    size_t lds;
};
static BwdPlan bwd_plan(const SoapDev &sp, bool own, bool split) {
    BwdPlan b;
    const int NA = (sp.n + 3) / 4;
    b.own = own;
    b.nw = own ? sp.S : sp.S > 1 ? 4 : split ? 2 : 1;
    b.p_lds = true;
    b.SB = sp.S;
    if (BwdLds(NA, sp.L, sp.S, sp.S, b.nw, sp.dim, true).total > kSoapLdsCap) b.p_lds = false;
    while (b.SB > 1 && BwdLds(NA, sp.L, sp.S, b.SB, b.nw, sp.dim, b.p_lds).total > kSoapLdsCap) b.SB--;
    b.lds = BwdLds(NA, sp.L, sp.S, b.SB, b.nw, sp.dim, b.p_lds).total + table_lds(sp);
    return own && !(b.p_lds && b.SB == sp.S) ? bwd_plan(sp, false, split) : b;
}

// What a model's descriptors are admitted by (the size a level-by-level adjoint with its
// coefficients and one K x K level in LDS would take, and the variance's forward); the kernels
// here stay within kSoapLdsCap and their tables for every shape admitted.
size_t soap_fast_lds_bytes(const SoapDev &sp) {
    if (!soap_fast_supported(sp.n, sp.L)) return 0;
    const size_t KLM = (size_t)sp.K * (sp.L + 1) * (sp.L + 1), level = (size_t)sp.K * sp.K + (size_t)sp.K * (2 * sp.L + 1);
    const size_t adjoint = sp.n * sp.n + 3 * sp.n + KLM + 2 + std::max(level, (size_t)64 * ((2 * (sp.L + 2)) | 1));
    return std::max(soap_lane_lds_bytes(sp), adjoint * 8);
}

// Centres a block takes in turn: several once the launch has many more blocks than the GPU
// holds (2048 to 3072 wavefronts), so that a centre's data arrive while the one before is
// worked on and the tables are filled once; fewer blocks leave a longer last round.  Forward +
// adjoint in us with 1, 2, 4 and 8: 8/6 of one species 53, 52, 65, 108 (4096 centres), 136, 132,
// 147, 165 (13824), 292, 281, 277, 287 (32768), 580, 557, 543, 543 (64000), 1218, 1151, 1114, 1112
// (135200); 12/8 of two 718, 712, 744, 811 (6912), 1623, 1621, 1613, 1669 (16384).  2 from 4096
// centres on would gain 1 to 4% there in one species and lose as much in two.
static int centres_per_block(int nc) { return nc >= 65536 ? 8 : nc >= 16384 ? 4 : 1; }

bool launch_soap_fwd_fast(const SoapDev &sp, int nc, const int *centres, const int *Z, const int *nb_off,
                          const int *nb_j, const double *nb_r, const double *nb_d, double *X, double *norm,
                          double *cbuf, hipStream_t s) {
    if (!soap_fast_supported(sp.n, sp.L)) return false;
    ensure_soap_constants();
    if (nc <= 0) return true;
    // More species than two keep the harmonics together up to l = 4, where m >= 4 is one pair of
    // groups and would run the recursions again (22118 centres of five species at 6/4: 1007 -> 886
    // us; at 6/6, four species: 1259 together, 1190 apart).
    // Two wavefronts per centre (m < 4, m >= 4) while a wavefront per centre would not fill the
    // GPU (si4055: 44 -> 30 us), and where the accumulators of all groups (2 x 29 x 3 registers
    // at 12/8) leave too few registers; one otherwise (no recursion is run twice).
    const FwdPlan f = fwd_plan(sp, wave_per_species(sp, nc), sp.n > 8 || sp.L > 6 || nc < 4096);
    const int cpb = centres_per_block(nc), nblk = (nc + cpb - 1) / cpb;
#define GO(NN, LL, NW, SPLIT, SP)                                                                                  \
    hipLaunchKernelGGL((k_soap_fwd_x<NN, LL, NW, SPLIT, SP>), dim3(nblk), dim3(64 * NW), f.lds, s, sp, nc, cpb,    \
                       centres, Z, nb_off, nb_j, nb_r, nb_d, X, norm, cbuf, (int)f.p_lds, (int)f.c_lds)
#define LAUNCH(NN, LL)                                                                                             \
    if (sp.n == NN && sp.L == LL) {                                                                                \
        if constexpr (NN <= 8 && LL <= 6)                                                                          \
            if (f.own) {                                                                                           \
                if (sp.S == 2) GO(NN, LL, 2, false, 2);                                                            \
                else if (sp.S == 3) GO(NN, LL, 3, false, 3);                                                       \
                else GO(NN, LL, 4, false, 4);                                                                      \
                return true;                                                                                       \
            }                                                                                                      \
        if (sp.S > 2 || !f.p_lds || !f.c_lds) GO(NN, LL, 4, (LL > 4), 0);                                          \
        else if (sp.S == 2) GO(NN, LL, 4, true, 2);                                                                \
        else if (f.split) GO(NN, LL, 2, true, 1);                                                                  \
        else if constexpr (NN <= 8 && LL <= 6) GO(NN, LL, 1, false, 1);                                            \
        return true;                                                                                               \
    }
    SOAP_FAST(LAUNCH)
#undef LAUNCH
#undef GO
    return false;
}

bool launch_soap_bwd_fast(const SoapDev &sp, int nc, const int *centres, const int *Z, const int *nb_off,
                          const int *nb_j, const double *nb_r, const double *nb_d, const double *X, const double *G,
                          const double *norm, const double *cbuf, double *pairF, bool add, hipStream_t s) {
    if (!soap_fast_supported(sp.n, sp.L)) return false;
    ensure_soap_constants();
    if (nc <= 0) return true;
    const BwdPlan b = bwd_plan(sp, wave_per_species(sp, nc), sp.n > 8 || sp.L > 6 || nc < 4096);
    const int cpb = centres_per_block(nc), nblk = (nc + cpb - 1) / cpb;
#define GO(NN, LL, NW, SP)                                                                                         \
    hipLaunchKernelGGL((k_soap_bwd_x<NN, LL, NW, SP>), dim3(nblk), dim3(64 * NW), b.lds, s, sp, nc, cpb, centres,  \
                       Z, nb_off, nb_j, nb_r, nb_d, X, G, norm, cbuf, pairF, (int)b.p_lds, b.SB, (int)add)
#define LAUNCH(NN, LL)                                                                                             \
    if (sp.n == NN && sp.L == LL) {                                                                                \
        if constexpr (NN <= 8 && LL <= 6)                                                                          \
            if (b.own) {                                                                                           \
                if (sp.S == 2) GO(NN, LL, 2, 2);                                                                   \
                else if (sp.S == 3) GO(NN, LL, 3, 3);                                                              \
                else GO(NN, LL, 4, 4);                                                                             \
                return true;                                                                                       \
            }                                                                                                      \
        if (sp.S > 2 || !b.p_lds || b.SB < sp.S) GO(NN, LL, 4, 0);                                                 \
        else if (sp.S == 2) GO(NN, LL, 4, 2);                                                                      \
        else if (b.nw == 2) GO(NN, LL, 2, 1);                                                                      \
        else if constexpr (NN <= 8 && LL <= 6) GO(NN, LL, 1, 1);                                                   \
        return true;                                                                                               \
    }
    SOAP_FAST(LAUNCH)
#undef LAUNCH
#undef GO
    return false;
}

}  // namespace gapx
