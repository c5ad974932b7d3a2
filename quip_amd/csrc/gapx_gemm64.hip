// FP64 GEMMs of the GP contraction on large tiles, streamed straight into LDS.
//
// Block = 8 wavefronts (2 x 4) over a tile of 32 TM x 64 TN of C = A . B^T (BT, both
// k-contiguous: K = X Xs^T with the GP epilogue) or A . B (G = W Xs), k tiles of 16.  The slices of a
// k tile go from memory to one of two LDS buffers by buffer loads with the lds flag, 16 bytes
// a lane from offsets computed once, while the other buffer is used: one wait and one
// barrier per k tile, and no vector instruction between memory and LDS.  That is the point: a FP64
// matrix instruction and vector instructions of the same SIMD do not overlap (a wavefront of
// FMAs beside one of matrix instructions costs two thirds of its own time), and the tiles
// staged through registers issue 3.2 vector instructions per matrix instruction.
//
// k-contiguous slices: a row is 8 chunks of 16 bytes, chunk c of row r at c ^ (r % 8), so
// that 16-byte reads of 8 rows fall on distinct bank groups.  Lane group g = lane / 16 reads
// chunks g and g + 4: its operands of four k steps, k = 2g, 2g+1, 2g+8, 2g+9.  The slices of the
// plain B are rows of k, read 8 bytes a lane.  Rows and columns past the matrices are clamped
// to the last ones (their results are not stored); a last k tile of fewer than 16 is staged
// through registers with zeros, so that no product crosses from one row into the next.
//
// Measured against the best of six tiles staged through registers: 2048 x 2000 x 2701 (K, 22.1
// GFLOP) 402 -> 334 us, 66 TFLOP/s (the library's product of that shape: 419), and 2048 x 2701 x
// 2000 (G) 394 -> 338 us; 17553 x 2000 x 253 366 -> 316 us; 997 x 2000 x 253 31 -> 26 us;
// 64 x 500 x 253 17 -> 11 us.  Matrix pipe 88% busy at the first (75% before).
//
// v_mfma_f64_16x16x4f64: A lane l = A[l%16][k = l/16], B lane l = B[k = l/16][l%16],
// C lane l element v = C[l/16 + 4v][l%16].
#include "gapx_kernels.h"

#include <algorithm>

namespace gapx {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));

__host__ __device__ static inline int cdivg(long a, long b) { return (int)((a + b - 1) / b); }

constexpr int kGK = 16;   // k tile

template <bool BT, int TM, int TN>
struct StreamTile {
    static constexpr int BM = 32 * TM, BN = 64 * TN;
    static constexpr int AI = BM / 64, BI = BN / 64;   // 1 KB loads per wavefront: BM x 128 bytes of A over 8
    static constexpr int AS = BM * kGK, BS = BN * kGK, BUF = AS + BS;
    __amdgpu_buffer_rsrc_t ra, rb;
    unsigned ao[AI], bo[BI], bstep;   // this lane's byte offsets; bytes per k row of the plain B
    int wv, fa, fb, kb;               // kb: the row of the plain B where its resource starts

    __device__ __forceinline__ static __amdgpu_buffer_rsrc_t rsrc(const double *p, size_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)(unsigned)bytes, 0x00020000);
    }
    __device__ __forceinline__ void init(const double *A, const double *B, int Mr, int Nc, int Kd, int m0, int n0,
                                         int kbeg, int kend) {
        const int t = threadIdx.x, lane = t & 63, g = lane >> 4, l16 = lane & 15;
        wv = __builtin_amdgcn_readfirstlane(t >> 6);
        const int ar = min(BM, Mr - m0), br = min(BN, Nc - n0);
        ra = rsrc(A + (size_t)m0 * Kd, (size_t)ar * Kd * 8);
        // of the plain B the rows of this block's k range; the last pair of an odd row length
        // ends 8 bytes past the last row
        kb = kbeg;
        rb = BT ? rsrc(B + (size_t)n0 * Kd, (size_t)br * Kd * 8)
                : rsrc(B + (size_t)kbeg * Nc, (size_t)(kend - kbeg) * Nc * 8 + 8);
        bstep = (unsigned)Nc * 8;
#pragma unroll
        for (int i = 0; i < AI; i++) {
            const int row = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ (row & 7);
            ao[i] = (unsigned)(min(row, ar - 1) * Kd + 2 * c) * 8;
        }
#pragma unroll
        for (int i = 0; i < BI; i++) {
            if (BT) {
                const int row = 8 * (wv + 8 * i) + (lane >> 3), c = (lane & 7) ^ (row & 7);
                bo[i] = (unsigned)(min(row, br - 1) * Kd + 2 * c) * 8;
            } else {
                const int vi = 64 * (wv + 8 * i) + lane, row = vi / (BN / 2), col = n0 + 2 * (vi % (BN / 2));
                bo[i] = (unsigned)row * bstep + (unsigned)min(col, (Nc - 1) & ~1) * 8;
            }
        }
        fa = ((wv >> 2) * 16 * TM + l16) * kGK;
        fb = BT ? ((wv & 3) * 16 * TN + l16) * kGK : (wv & 3) * 16 * TN + l16;
    }
    __device__ __forceinline__ void stage(int k0, double *buf) const {
#pragma unroll
        for (int i = 0; i < AI; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void *)(buf + 128 * (wv + 8 * i)),
                                                     16, (int)ao[i], k0 * 8, 0, 0);
#pragma unroll
        for (int i = 0; i < BI; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void *)(buf + AS + 128 * (wv + 8 * i)),
                                                     16, (int)bo[i], BT ? k0 * 8 : (int)((unsigned)(k0 - kb) * bstep), 0, 0);
    }
    // a last k tile of kt < 16, zeros beyond it
    __device__ __forceinline__ void stage_tail(const double *A, const double *B, int Mr, int Nc, int Kd, int m0, int n0,
                                               int k0, int kt, double *buf) const {
        for (int e = threadIdx.x; e < AS; e += 512) {
            const int row = e / kGK, k = e % kGK, c = (k >> 1) ^ (row & 7);
            buf[row * kGK + 2 * c + (k & 1)] = k < kt && m0 + row < Mr ? A[(size_t)(m0 + row) * Kd + k0 + k] : 0.0;
        }
        for (int e = threadIdx.x; e < BS; e += 512) {
            if (BT) {
                const int row = e / kGK, k = e % kGK, c = (k >> 1) ^ (row & 7);
                buf[AS + row * kGK + 2 * c + (k & 1)] = k < kt && n0 + row < Nc ? B[(size_t)(n0 + row) * Kd + k0 + k] : 0.0;
            } else {
                const int k = e / BN, col = e % BN;
                buf[AS + e] = k < kt && n0 + col < Nc ? B[(size_t)(k0 + k) * Nc + n0 + col] : 0.0;
            }
        }
    }
    __device__ __forceinline__ void compute(const double *__restrict__ cur, double4_t (&acc)[TM][TN]) const {
        const int lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int c2 = ((g + 4 * h) ^ (l16 & 7)) * 2;
            double2_t a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) a[i] = *(const double2_t *)(cur + fa + 16 * i * kGK + c2);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if (BT) b[j] = *(const double2_t *)(cur + AS + fb + 16 * j * kGK + c2);
                else {
                    b[j][0] = cur[AS + (2 * g + 8 * h) * BN + fb + 16 * j];
                    b[j][1] = cur[AS + (2 * g + 8 * h + 1) * BN + fb + 16 * j];
                }
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
        }
    }
    // one k tile while the next streams into the other buffer (distinct restrict-qualified
    // buffers: the reads here do not wait for those loads)
    __device__ __forceinline__ void step(bool more, int knext, const double *__restrict__ cur,
                                         double *__restrict__ next, double4_t (&acc)[TM][TN]) const {
        if (more) stage(knext, next);
        compute(cur, acc);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
    __device__ __forceinline__ void run(const double *A, const double *B, int Mr, int Nc, int Kd, int m0, int n0,
                                        int kbeg, int kend, double *buf0, double *buf1, double4_t (&acc)[TM][TN]) const {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};
        const int nf = (kend - kbeg) / kGK, kt = kend - kbeg - nf * kGK;
        if (nf > 0) {
            stage(kbeg, buf0);
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            for (int f = 0; f < nf; f += 2) {
                step(f + 1 < nf, kbeg + (f + 1) * kGK, buf0, buf1, acc);
                if (f + 1 < nf) step(f + 2 < nf, kbeg + (f + 2) * kGK, buf1, buf0, acc);
            }
        }
        if (kt > 0) {   // every wavefront has left both buffers
            stage_tail(A, B, Mr, Nc, Kd, m0, n0, kbeg + nf * kGK, kt, buf0);
            __syncthreads();
            compute(buf0, acc);
        }
    }
};

template <bool BT, bool EPI, int ZI, int TM, int TN>
__global__ __launch_bounds__(512) void k_gemm_f64_stream(int Mr, int Nc, int Kd, int kchunk,
                                                         const double *__restrict__ A, const double *__restrict__ B,
                                                         double *__restrict__ C, const double *__restrict__ wvec,
                                                         double zeta, int izeta, double *__restrict__ e_part) {
    typedef StreamTile<BT, TM, TN> ST;
    __shared__ __attribute__((aligned(16))) double buf0[ST::BUF], buf1[ST::BUF];
    // blocks are dealt to the 8 XCDs in turn: each takes a contiguous range of tiles, row by row
    const int nb = gridDim.x, bx = blockIdx.x, ntn = cdivg(Nc, ST::BN);
    const int tile = nb % 8 == 0 ? (bx % 8) * (nb / 8) + bx / 8 : bx, tm = tile / ntn, tn = tile - tm * ntn;
    const int m0 = tm * ST::BM, n0 = tn * ST::BN;
    const int kbeg = blockIdx.z * kchunk, kend = max(kbeg, min(Kd, kbeg + kchunk));
    const bool store = C != nullptr;   // energies alone need no W
    C += (size_t)blockIdx.z * Mr * Nc;
    double4_t acc[TM][TN];
    ST st;
    st.init(A, B, Mr, Nc, Kd, m0, n0, kbeg, kend);
    st.run(A, B, Mr, Nc, Kd, m0, n0, kbeg, kend, buf0, buf1, acc);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 2, wn = w & 3;
    double *red = buf1;   // [4][BM]; the tail left it free
    if constexpr (EPI) __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; i++) {
        double rowsum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = n0 + wn * 16 * TN + j * 16 + (lane & 15);
            double wv = 0.0;
            if constexpr (EPI) wv = col < Nc ? wvec[col] : 0.0;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = m0 + wm * 16 * TM + i * 16 + (lane >> 4) + 4 * v;
                double kv = acc[i][j][v];
                if constexpr (EPI) {
                    double kz1, kz;
                    if constexpr (ZI > 0) {
                        kz1 = 1.0;
#pragma unroll
                        for (int q = 1; q < ZI; q++) kz1 *= kv;
                        kz = kz1 * kv;
                    } else if (izeta > 0) {
                        kz1 = 1.0;
                        for (int q = 1; q < izeta; q++) kz1 *= kv;
                        kz = kz1 * kv;
                    } else {
                        kz1 = pow(kv, zeta - 1.0);
                        kz = pow(kv, zeta);
                    }
                    rowsum[v] += col < Nc ? wv * kz : 0.0;
                    kv = wv * zeta * kz1;
                }
                if ((!EPI || store) && row < Mr && col < Nc) C[(size_t)row * Nc + col] = kv;
            }
        }
        if constexpr (EPI) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                double x = rowsum[v];
                for (int off = 8; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
                if ((lane & 15) == 0) red[wn * ST::BM + wm * 16 * TM + i * 16 + (lane >> 4) + 4 * v] = x;
            }
        }
    }
    if constexpr (EPI) {
        __syncthreads();
        if ((int)threadIdx.x < ST::BM) {
            const int r = threadIdx.x;
            if (m0 + r < Mr)
                e_part[(size_t)(m0 + r) * ntn + tn] = (red[r] + red[ST::BM + r]) + (red[2 * ST::BM + r] + red[3 * ST::BM + r]);
        }
    }
}

static int int_zeta_g(double z) {
    double r = floor(z + 0.5);
    return (fabs(z - r) == 0.0 && r >= 1.0 && r <= 16.0) ? (int)r : 0;
}

static const int kTile[kGemmTiles][2] = {{4, 2}, {2, 2}, {2, 1}};   // (TM, TN): 128 x 128, 64 x 128, 64 x 64

// Byte offsets stay within 31 bits: those of a tile's rows of both matrices (K), those of its
// rows of W and of a part's rows of the plain Xs (G).  64-bit addresses of the tiles staged
// through registers reach further, at 394 us against 338 (2048 x 2701 x 2000).
constexpr size_t kReach = (size_t)1 << 31;
static int part_rows(int parts, int M) { return (cdivg(M, parts) + kGK - 1) / kGK * kGK; }
bool gemm1_stream_ok(int d) { return (size_t)128 * d * 8 < kReach; }
bool gemm2_stream_ok(int parts, int M, int d) {
    return (size_t)128 * M * 8 < kReach && (size_t)part_rows(parts, M) * d * 8 + 8 < kReach;
}
int gemm_stream_ntile(int t, int M) { return cdivg(M, 64 * kTile[t][1]); }

template <int TM, int TN>
static void stream1_go(int nc, int M, int d, const double *X, const double *Xs, const double *wvec, double zeta,
                       double *W, double *e_part, hipStream_t s) {
    const dim3 grid(cdivg(nc, 32 * TM) * cdivg(M, 64 * TN));
    const int iz = int_zeta_g(zeta);
    if (iz == 4)
        hipLaunchKernelGGL((k_gemm_f64_stream<true, true, 4, TM, TN>), grid, dim3(512), 0, s, nc, M, d, d, X, Xs, W, wvec,
                           zeta, iz, e_part);
    else
        hipLaunchKernelGGL((k_gemm_f64_stream<true, true, 0, TM, TN>), grid, dim3(512), 0, s, nc, M, d, d, X, Xs, W, wvec,
                           zeta, iz, e_part);
}
void launch_gemm1_f64_stream(int t, int nc, int M, int d, const double *X, const double *Xs, const double *wvec,
                             double zeta, double *W, double *e_part, hipStream_t s) {
    switch (t) {
        case 0: stream1_go<4, 2>(nc, M, d, X, Xs, wvec, zeta, W, e_part, s); break;
        case 1: stream1_go<2, 2>(nc, M, d, X, Xs, wvec, zeta, W, e_part, s); break;
        default: stream1_go<2, 1>(nc, M, d, X, Xs, wvec, zeta, W, e_part, s); break;
    }
}
template <int TM, int TN>
static void stream2_go(int nc, int M, int d, int parts, const double *W, const double *Xs, double *out, hipStream_t s) {
    const int kchunk = part_rows(parts, M);
    hipLaunchKernelGGL((k_gemm_f64_stream<false, false, 0, TM, TN>), dim3(cdivg(nc, 32 * TM) * cdivg(d, 64 * TN), 1, parts),
                       dim3(512), 0, s, nc, d, M, kchunk, W, Xs, out, (const double *)nullptr, 0.0, 0, (double *)nullptr);
}
void launch_gemm2_f64_stream(int t, int parts, int nc, int M, int d, const double *W, const double *Xs, double *out,
                             hipStream_t s) {
    switch (t) {
        case 0: stream2_go<4, 2>(nc, M, d, parts, W, Xs, out, s); break;
        case 1: stream2_go<2, 2>(nc, M, d, parts, W, Xs, out, s); break;
        default: stream2_go<2, 1>(nc, M, d, parts, W, Xs, out, s); break;
    }
}

}  // namespace gapx
