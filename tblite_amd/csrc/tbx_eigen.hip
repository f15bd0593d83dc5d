// tbx_eigen.hip -- gfx950 kernels of the generalized symmetric eigenproblem
// H C = S C diag(e) (lapack/sygvd.f90, scf/diag.f90:84) of all molecules of a
// batch at once, up to TBX_EIG_MAXN orbitals each.  A library call per
// molecule leaves the chip idle: one molecule is a chain of thousands of small
// dependent launches.  Here every launch serves all molecules of the list:
//
//   k_eig_symm    upper triangles of S and H -> full symmetric copies
//   k_eig_chol    S = L L^T, one launch per 64 columns; the diagonal blocks of
//                 L are kept as their inverses
//   k_eig_trsm    Y = L^-1 H, then A = L^-1 Y^T: strips of 16 columns in LDS,
//                 FP64 MFMA products with the 64 x 64 blocks of L
//   k_trd_step    one Householder column of A per launch (n > TBX_TRD_TAIL)
//   k_trd_tail    the last TBX_TRD_TAIL columns, the whole rest of A in registers
//   k_dc_leaf     eigenpairs of tridiagonal blocks of at most 64 rows by divide
//                 and conquer from single rows, in LDS; triangular factors of
//                 blocks of 16 reflectors beside them
//   k_dc_prep, k_dc_secular, k_dc_zhat, k_dc_norm, k_dc_gemm
//                 the merges above that (Cuppen's rank-one update; deflation
//                 and the recomputed vector z of M. Gu and S. Eisenstat, SIAM J.
//                 Matrix Anal. Appl. 16, 172 (1995)), products on MFMA
//   k_eig_back    the blocks of reflectors of the tridiagonal form applied to
//                 16 eigenvectors in registers, then C = L^-T Z in LDS
//
// Matrices are column-major n x n at EigMol::w0 of the workspace buffers,
// vectors at the molecule's first orbital a0.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tbx_eigen.h"

namespace {

typedef double dbl4 __attribute__((ext_vector_type(4)));

constexpr double kEps = 1.1102230246251565e-16;  // unit roundoff

// v_mfma_f64_16x16x4_f64: lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator register r holds D[l / 16 + 4 r][l % 16].
__device__ __forceinline__ dbl4 mfma(double a, double b, dbl4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWMASK, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ double lane63(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, 63);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// sum over the wavefront, on every lane: row shifts, row broadcasts, lane 63
__device__ __forceinline__ double wsum(double v)
{
    v += dpp<0x111, 0xf>(v);
    v += dpp<0x112, 0xf>(v);
    v += dpp<0x114, 0xf>(v);
    v += dpp<0x118, 0xf>(v);
    v += dpp<0x142, 0xa>(v);
    v += dpp<0x143, 0xc>(v);
    return lane63(v);
}

// a and b folded into one register: lanes 0..31 hold the sum of the two halves
// of a, lanes 32..63 that of b (fold32); rows 0 / 1 and 2 / 3 of 16 lanes
// likewise (fold16)
__device__ __forceinline__ double fold32(double a, double b)
{
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32),
                                                     false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}
__device__ __forceinline__ double fold16(double a, double b)
{
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32),
                                                     false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

__device__ __forceinline__ double lane_of(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// the four sums over the wavefront at once (a third of the instructions of
// four wsum): after the folds each row of 16 lanes belongs to one of them
__device__ __forceinline__ void wsum4(double s[4])
{
    double v = fold16(fold32(s[0], s[1]), fold32(s[2], s[3]));  // rows: s0, s2, s1, s3
    v += dpp<0x128, 0xf>(v);  // rotations within the row
    v += dpp<0x124, 0xf>(v);
    v += dpp<0x122, 0xf>(v);
    v += dpp<0x121, 0xf>(v);
    s[0] = lane_of(v, 0);
    s[2] = lane_of(v, 16);
    s[1] = lane_of(v, 32);
    s[3] = lane_of(v, 48);
}

// sums and a product over the four lanes of a quad, on all of them
__device__ __forceinline__ double qsum(double v)
{
    v += dpp<0xB1, 0xf>(v);
    return v + dpp<0x4E, 0xf>(v);
}
__device__ __forceinline__ double qprod(double v)
{
    v *= dpp<0xB1, 0xf>(v);
    return v * dpp<0x4E, 0xf>(v);
}
__device__ __forceinline__ double qmax(double v)
{
    v = fmax(v, dpp<0xB1, 0xf>(v));
    return fmax(v, dpp<0x4E, 0xf>(v));
}

// reciprocal to about one unit in the last place (finite, nonzero arguments)
__device__ __forceinline__ double fast_rcp(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// ---------------------------------------------------------------------------
// full symmetric copies of the upper triangles: 32 x 32 tiles through LDS

__global__ void __launch_bounds__(256) k_eig_symm(const EigMol *mols, const double *S,
                                                  const double *H, double *wS, double *wH,
                                                  int *info)
{
    __shared__ double t[32][33];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n, nt = (n + 31) / 32;
    if (blockIdx.x == 0 && blockIdx.z == 0 && threadIdx.x == 0) info[M.mol] = 0;
    // tile pair of the upper triangle: bi <= bj
    int bj = (int)((sqrtf(8.0f * blockIdx.x + 1.0f) - 1.0f) * 0.5f);
    while ((bj + 1) * (bj + 2) / 2 <= (int)blockIdx.x) ++bj;
    while (bj * (bj + 1) / 2 > (int)blockIdx.x) --bj;
    const int bi = blockIdx.x - bj * (bj + 1) / 2;
    if (bj >= nt) return;
    const double *src = (blockIdx.z ? H : S) + M.d0;
    double *dst = (blockIdx.z ? wH : wS) + M.w0;
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    for (int c = y; c < 32; c += 8) {
        const int r = 32 * bi + x, k = 32 * bj + c;
        t[c][x] = (r < n && k < n && r <= k) ? src[r + (long long)k * n] : 0.0;
    }
    __syncthreads();
    for (int c = y; c < 32; c += 8) {
        const int r = 32 * bi + x, k = 32 * bj + c;  // element (r, k) and its mirror
        if (r < n && k < n && (bi != bj || r <= k)) dst[r + (long long)k * n] = t[c][x];
        const int r2 = 32 * bj + x, k2 = 32 * bi + c;
        if (r2 < n && k2 < n && (bi != bj || r2 > k2)) dst[r2 + (long long)k2 * n] = t[x][c];
    }
}

// ---------------------------------------------------------------------------
// Cholesky by blocks of 64

constexpr int NB = 64;
constexpr int PR = NB + 16;  // LDS row length (doubles), as in the density kernel

// element (r, c) of an n x n matrix, zero outside
__device__ __forceinline__ double ldg(const double *M, int n, int r, int c)
{
    return (r < n && c < n) ? M[r + (long long)c * n] : 0.0;
}

// Tile T[k][r] = M(r0 + r, c0 + k), zero outside n
__device__ __forceinline__ void tile_load(double (*T)[PR], const double *M, int n, int r0, int c0)
{
    const int r = threadIdx.x & (NB - 1), k = threadIdx.x / NB;
    double v[NB / 4];  // every load is under way before the first is stored
#pragma unroll
    for (int q = 0; q < NB / 4; ++q) v[q] = ldg(M, n, r0 + r, c0 + k + 4 * q);
#pragma unroll
    for (int q = 0; q < NB / 4; ++q) T[k + 4 * q][r] = v[q];
}

// D(r, c) = sum_k A(r, k) B(c, k) of 64 x 64 tiles T[k][row]: each of the four
// wavefronts a 32 x 32 quarter (rows sr, columns sc)
__device__ __forceinline__ void tile_nt(const double (*A)[PR], const double (*B)[PR], int sr,
                                        int sc, dbl4 acc[2][2])
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[s][u] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int ks = 0; ks < NB; ks += 4) {
        double a[2], b[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            a[s] = A[ks + lk][sr + 16 * s + li];
            b[s] = B[ks + lk][sc + 16 * s + li];
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u) acc[s][u] = mfma(a[s], b[u], acc[s][u]);
    }
}

// quarter (sr, sc) of D into T[c][r] (the k-major form of the next product)
__device__ __forceinline__ void tile_put(double (*T)[PR], int sr, int sc, const dbl4 acc[2][2])
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                T[sc + 16 * u + li][sr + 16 * s + lk + 4 * r] = acc[s][u][r];
}

// Cholesky factor of the symmetric tile T (nv valid rows) and the inverse of
// the factor, by elimination without square roots on [T | I]: thread (ty, tx)
// holds the elements (ty + 16 a, tx + 16 b) of both in registers, so a step is
// one broadcast of the pivot's column and row through LDS and one barrier.
// Writes inv(L) (zero above the diagonal) to Linv (column-major, ld n) and
// returns false if a pivot is not positive.
__device__ bool factor_inverse(double (*T)[PR], double (*buf)[2 * NB], double *pivot, int nv,
                               double *Linv, int n)
{
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    double t[4][4], x[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = ty + 16 * a, j = tx + 16 * b;
            t[a][b] = (i < nv && j < nv) ? T[j][i] : (i == j ? 1.0 : 0.0);
            x[a][b] = i == j ? 1.0 : 0.0;
        }
    bool ok = true;
    if (tid < NB) pivot[tid] = 1.0;
    // step k = 16 kb + kk changes the rows below k only: the columns from the
    // block kb on in T (those before k are no longer used), up to it in X
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
        for (int kk = 0; kk < 16; ++kk) {
            const int k = 16 * kb + kk;
            if (k >= nv) break;  // uniform
            double *col = buf[k & 1], *row = buf[k & 1] + NB;
            if (tx == kk) {
#pragma unroll
                for (int a = kb; a < 4; ++a) col[ty + 16 * a] = t[a][kb];
            }
            if (ty == kk) {
#pragma unroll
                for (int b = 0; b <= kb; ++b) row[tx + 16 * b] = x[kb][b];
            }
            __syncthreads();
            const double piv = col[k];
            if (tid == 0) pivot[k] = piv;
            ok = ok && piv > 0.0;
            const double inv = fast_rcp(piv);
            double cj[4], rj[4];
#pragma unroll
            for (int b = kb; b < 4; ++b) cj[b] = col[tx + 16 * b];
#pragma unroll
            for (int b = 0; b <= kb; ++b) rj[b] = row[tx + 16 * b];
#pragma unroll
            for (int a = kb; a < 4; ++a) {
                const int i = ty + 16 * a;
                const double m = i > k ? col[i] * inv : 0.0;
#pragma unroll
                for (int b = kb; b < 4; ++b) t[a][b] -= m * cj[b];
#pragma unroll
                for (int b = 0; b <= kb; ++b) x[a][b] -= m * rj[b];
            }
        }
    if (!ok) return false;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int i = ty + 16 * a;
        const double s = 1.0 / sqrt(pivot[i]);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int j = tx + 16 * b;
            if (i < nv && j < nv) Linv[i + (long long)j * n] = j <= i ? x[a][b] * s : 0.0;
        }
    }
    return true;
}

// Block column kb of the factor, for the tiles (bi, bj) with bi >= bj > kb:
// P_i = A_ik inv(L_kk)^T (the block of L, stored by the tiles of column
// kb + 1), A_ij -= P_i P_j^T; the tile (kb + 1, kb + 1) goes on to its own
// factor and inverse, so a block column is one launch.  kb = -1: the first
// diagonal block only.  768 orbitals: 33 us a launch, about half of it the
// chain of 64 eliminations (60 us with loads one at a time and unmasked rows).
// A molecule whose S has failed goes on, into values that nobody reads: one
// workgroup of the launch writes its info, so a look at it here could send the
// wavefronts of another to different sides of a barrier.
__global__ void __launch_bounds__(256) k_eig_chol(const EigMol *mols, double *A, double *L,
                                                  int kb, int *info)
{
    __shared__ __align__(16) double T0[NB][PR], T1[NB][PR], T2[NB][PR];
    __shared__ double buf[2][2 * NB], pivot[NB];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n, nblk = (n + NB - 1) / NB, left = nblk - 1 - kb;
    if (left <= 0) return;
    int tj = 0, rest = blockIdx.x;  // tile column tj: left - tj tiles
    while (tj < left && rest >= left - tj) rest -= left - tj++;
    if (tj >= left || (kb < 0 && blockIdx.x > 0)) return;
    const int bj = kb + 1 + tj, bi = bj + rest;
    double *Am = A + M.w0, *Lm = L + M.w0;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int sr = 32 * (wv >> 1), sc = 32 * (wv & 1);
    if (kb < 0) {
        tile_load(T0, Am, n, 0, 0);
        __syncthreads();
    } else {
        tile_load(T0, Am, n, NB * bi, NB * kb);
        if (bi != bj) tile_load(T1, Am, n, NB * bj, NB * kb);
        tile_load(T2, Lm, n, NB * kb, NB * kb);  // inv(L_kk)
        __syncthreads();
        dbl4 pi[2][2], pj[2][2];
        tile_nt(T0, T2, sr, sc, pi);
        if (bi != bj) tile_nt(T1, T2, sr, sc, pj);
        __syncthreads();
        tile_put(T0, sr, sc, pi);
        if (bi != bj) tile_put(T1, sr, sc, pj);
        __syncthreads();
        if (tj == 0) {  // the block (bi, kb) of L
            for (int e = threadIdx.x; e < NB * NB; e += 256) {
                const int r = e & (NB - 1), k = e / NB;
                if (NB * bi + r < n) Lm[NB * bi + r + (long long)(NB * kb + k) * n] = T0[k][r];
            }
        }
        dbl4 d[2][2];
        tile_nt(T0, bi != bj ? T1 : T0, sr, sc, d);
        const bool next = bi == kb + 1;  // bi == bj == kb + 1
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = NB * bi + sr + 16 * s + lk + 4 * r, j = NB * bj + sc + 16 * u + li;
                    double v = 0.0;
                    if (i < n && j < n) {
                        v = Am[i + (long long)j * n] - d[s][u][r];
                        if (!next) Am[i + (long long)j * n] = v;
                    }
                    if (next) T2[sc + 16 * u + li][sr + 16 * s + lk + 4 * r] = v;
                }
        if (!next) return;
        __syncthreads();
    }
    const int b0 = NB * (kb + 1);
    const bool ok = factor_inverse(kb < 0 ? T0 : T2, buf, pivot, min(NB, n - b0),
                                   Lm + b0 + (long long)b0 * n, n);
    if (!ok && threadIdx.x == 0) info[M.mol] = 1;
}

// ---------------------------------------------------------------------------
// triangular solves of 16-column strips in LDS: X[r][c], rows padded to 64

constexpr int XS = 17;  // row length of the strip (doubles)

// X <- L^-1 X (forward) or L^-T X (backward) for the strip, block row by block
// row: the four wavefronts take 16 rows each; the products with the earlier
// (later) blocks run on MFMA with L read from L2, then the block is multiplied
// by the inverse of its diagonal block.
template <bool FWD>
__device__ void strip_solve(const double *Lm, int n, double *X)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    const int nblk = (n + NB - 1) / NB;
    for (int q = 0; q < nblk; ++q) {
        const int b = FWD ? q : nblk - 1 - q;
        const int r0 = NB * b + 16 * wv;  // this wavefront's rows
        dbl4 acc = dbl4{0.0, 0.0, 0.0, 0.0};
        for (int kb = FWD ? 0 : b + 1; kb < (FWD ? b : nblk); ++kb) {
            double a[16];
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const int k = NB * kb + 4 * s + lk;
                a[s] = FWD ? ldg(Lm, n, r0 + li, k) : ldg(Lm, n, k, r0 + li);
            }
#pragma unroll
            for (int s = 0; s < 16; ++s)
                acc = mfma(a[s], X[(NB * kb + 4 * s + lk) * XS + li], acc);
        }
        double a[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const int k = NB * b + 4 * s + lk;
            a[s] = FWD ? ldg(Lm, n, r0 + li, k) : ldg(Lm, n, k, r0 + li);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) X[(r0 + lk + 4 * r) * XS + li] -= acc[r];
        __syncthreads();
        acc = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 16; ++s) acc = mfma(a[s], X[(NB * b + 4 * s + lk) * XS + li], acc);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) X[(r0 + lk + 4 * r) * XS + li] = acc[r];
        __syncthreads();
    }
}

// out = L^-1 in (TRANS = false) or L^-1 in^T
template <bool TRANS>
__global__ void __launch_bounds__(256) k_eig_trsm(const EigMol *mols, const double *L,
                                                  const double *in, double *out, const int *info)
{
    extern __shared__ double X[];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n, c0 = 16 * blockIdx.x;
    if (c0 >= n || info[M.mol] != 0) return;
    const int rows = (n + NB - 1) / NB * NB;
    const double *src = in + M.w0;
    // batches of 64 rows: four loads per thread under way at a time, sixteen
    // with the unrolling
#pragma unroll 4
    for (int r0 = 0; r0 < rows; r0 += NB) {
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = threadIdx.x + 256 * q;
            v[q] = TRANS ? ldg(src, n, c0 + (e & 15), r0 + (e >> 4))
                         : ldg(src, n, r0 + (e & 63), c0 + (e >> 6));
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = threadIdx.x + 256 * q;
            X[(r0 + (TRANS ? e >> 4 : e & 63)) * XS + (TRANS ? e & 15 : e >> 6)] = v[q];
        }
    }
    __syncthreads();
    strip_solve<true>(L + M.w0, n, X);
    double *dst = out + M.w0;
    for (int c = 0; c < 16 && c0 + c < n; ++c)
        for (int r = threadIdx.x; r < n; r += 256) dst[r + (long long)(c0 + c) * n] = X[r * XS + c];
}

// ---------------------------------------------------------------------------
// tridiagonal form.  Column k: with the pending rank-two update of column
// k - 1 (A -= v w^T + w v^T, w from v and p = A v), x = A(k:, k) gives d_k,
// the reflector v_k, tau_k and e_k; the update of the trailing columns and
// the product p_k = A v_k then are one pass over them.  A is symmetric, so
// row i is read as column i.

struct TrdPtr {
    double *A;            // [n * n] destroyed
    double *V;            // [n * n] reflectors, column k
    double *d, *e, *tau;  // [n] at a0
    double *p;            // [2][nao]: A v of the even and odd columns
    long long pstride;
};

// reflector of x = (alpha, rest of squared norm xx): beta, tau and the scale of
// the rest of v
__device__ __forceinline__ void reflector(double alpha, double xx, double &beta, double &tau,
                                          double &scale)
{
    if (xx == 0.0) {
        beta = alpha;
        tau = 0.0;
        scale = 0.0;
    } else {
        beta = -copysign(sqrt(alpha * alpha + xx), alpha);
        tau = (beta - alpha) / beta;
        scale = 1.0 / (alpha - beta);
    }
}

constexpr int TRD_THREADS = 256;
constexpr int TRD_COLS = 8;  // trailing columns per workgroup

__device__ __forceinline__ double block_sum4(double v, double *red)
{
    const double s = wsum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// One column k of every molecule with n > TBX_TRD_TAIL + k (and n - k at most
// 256 Q): workgroup blockIdx.x takes the trailing columns k + 1 + TRD_COLS
// blockIdx.x ...; every workgroup forms w, x and v_k itself (O(n) work), which
// saves a launch.  The launch is bound by its chain of dependent steps, so
// the trailing columns are loaded before it begins: 4.3 / 5.1 / 6.0 us a column
// at up to 256 / 512 / 768 rows, 7.3 us with the loads after the reflector.
template <int Q>
__global__ void __launch_bounds__(TRD_THREADS) k_trd_step(const EigMol *mols, TrdPtr T, int k)
{
    constexpr int LEN = TRD_THREADS * Q;
    __shared__ double v[LEN], w[LEN], vn[LEN];  // rows k ..
    __shared__ double red[2][4];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n, len = n - k;
    const int i0 = 1 + TRD_COLS * blockIdx.x;  // columns and rows count from k
    if (n <= TBX_TRD_TAIL + k || i0 >= len) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double *A = T.A + M.w0 + (long long)k * n + k, *V = T.V + M.w0 + (long long)k * n + k;
    const double *pold = T.p + ((k + 1) & 1) * T.pstride + M.a0 + k;
    double *pnew = T.p + (k & 1) * T.pstride + M.a0 + k;
    // the pending update of column k - 1: rows k.. of v and w
    double vr[Q], pr[Q], xr[Q];
    double s = 0.0, tau0 = 0.0;
    if (k > 0) tau0 = T.tau[M.a0 + k - 1];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + TRD_THREADS * q;
        vr[q] = (i < len && k > 0) ? V[i - n] : 0.0;
        pr[q] = (i < len && k > 0) ? pold[i] : 0.0;
        xr[q] = i < len ? A[i] : 0.0;
    }
    double a[TRD_COLS / 4][4 * Q];
#pragma unroll
    for (int c = 0; c < TRD_COLS / 4; ++c) {
        const int i = i0 + wv + 4 * c;
#pragma unroll
        for (int q = 0; q < 4 * Q; ++q) {
            const int j = 1 + lane + 64 * q;
            a[c][q] = (i < len && j < len) ? A[(long long)i * n + j] : 0.0;
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) s += vr[q] * pr[q];
    s = block_sum4(s, red[0]);
    const double h = 0.5 * tau0 * s;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + TRD_THREADS * q;
        pr[q] = tau0 * (pr[q] - h * vr[q]);  // w
        v[i] = vr[q];
        w[i] = pr[q];
    }
    __syncthreads();
    const double vk = v[0], wk = w[0];
    double xx = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + TRD_THREADS * q;
        xr[q] -= vr[q] * wk + pr[q] * vk;
        vn[i] = xr[q];
        if (i >= 2) xx += xr[q] * xr[q];
    }
    xx = block_sum4(xx, red[1]);
    const double dk = vn[0], alpha = vn[1];
    double beta, tau, scale;
    reflector(alpha, xx, beta, tau, scale);
    __syncthreads();  // vn[1] is read before it is replaced
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = tid + TRD_THREADS * q;
        const double x = i == 1 ? 1.0 : xr[q] * scale;
        vn[i] = x;
        if (blockIdx.x == 0 && i > 0 && i < len) V[i] = x;
    }
    if (blockIdx.x == 0 && tid == 0) {
        T.d[M.a0 + k] = dk;
        T.e[M.a0 + k] = beta;
        T.tau[M.a0 + k] = tau;
    }
    __syncthreads();
    // update and product of this workgroup's trailing columns, two per wavefront
    double acc[TRD_COLS / 4];
#pragma unroll
    for (int c = 0; c < TRD_COLS / 4; ++c) {
        const int i = i0 + wv + 4 * c;
        const bool in = i < len;
        const double vi = in ? v[i] : 0.0, wi = in ? w[i] : 0.0;
        acc[c] = 0.0;
#pragma unroll
        for (int q = 0; q < 4 * Q; ++q) {
            const int j = 1 + lane + 64 * q;
            if (in && j < len) {
                const double x = a[c][q] - (vi * w[j] + wi * v[j]);
                A[(long long)i * n + j] = x;
                acc[c] += x * vn[j];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < TRD_COLS / 4; ++c) {
        const double t = wsum(acc[c]);
        const int i = i0 + wv + 4 * c;
        if (lane == 0 && i < len) pnew[i] = t;
    }
}

// The remaining (at most TBX_TRD_TAIL) columns, one workgroup of four
// wavefronts per molecule, with the whole rest of A in registers: lane and
// lane + 64 are a thread's rows, the columns j = wave + 4 t are in a[.][t].
// Each wavefront forms v, w and the new reflector redundantly, so a column
// costs one barrier: before it the wavefronts leave their share of p = A v and
// the next column (by symmetry the row of the lane that holds it) in LDS.  The
// factors of column j are read from their lane (v_readlane).  Columns that are
// done are still updated, eight at a time: their reflector entries are zero.
// 1.7 us a column at 128 rows, 215 us in all; with A in LDS, eight wavefronts
// and a reduction per row 378 us; in registers with a branch per column 375 us.
constexpr int TL_THREADS = 256;
constexpr int TL = TBX_TRD_TAIL;
constexpr int TLT = TL / 4;  // columns per thread

__global__ void __launch_bounds__(TL_THREADS) k_trd_tail(const EigMol *mols, TrdPtr T,
                                                         double *anorm, int *info)
{
    __shared__ double part[2][4][TL];  // p by wavefront
    __shared__ double xcol[2][TL];     // the next column, pending update not applied
    const EigMol M = mols[blockIdx.x];
    const int n = M.n;
    if (info[M.mol] != 0) return;
    const int k0 = n > TL ? n - TL : 0, nt = n - k0;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double *Ag = T.A + M.w0 + (long long)k0 * n + k0;
    double *V = T.V + M.w0 + (long long)k0 * n + k0;
    double a[2][TLT];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t = 0; t < TLT; ++t) {
            const int j = wv + 4 * t, r = lane + 64 * q;
            a[q][t] = (r < nt && j < nt) ? Ag[r + (long long)j * n] : 0.0;
        }
    double v[2] = {0.0, 0.0}, p[2] = {0.0, 0.0}, w[2], x[2];
    double tau = 0.0, mx = 0.0;
    bool bad = false;
    if (k0 > 0) {
        const double *pold = T.p + ((k0 + 1) & 1) * T.pstride + M.a0 + k0;
        tau = T.tau[M.a0 + k0 - 1];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = lane + 64 * q;
            if (r < nt) {
                v[q] = V[r - n];
                p[q] = pold[r];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) x[q] = lane + 64 * q < nt ? Ag[lane + 64 * q] : 0.0;
    for (int k = 0; k < nt; ++k) {
        // w of the pending update, then the column itself
        const double s = wsum(v[0] * p[0] + v[1] * p[1]);
        const double h = 0.5 * tau * s;
#pragma unroll
        for (int q = 0; q < 2; ++q) w[q] = tau * (p[q] - h * v[q]);
        const double vk = lane_of(k < 64 ? v[0] : v[1], k & 63);
        const double wk = lane_of(k < 64 ? w[0] : w[1], k & 63);
        double xx = 0.0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = lane + 64 * q;
            x[q] = r >= k && r < nt ? x[q] - (v[q] * wk + w[q] * vk) : 0.0;
            if (r >= k + 2) xx += x[q] * x[q];
        }
        const double dk = lane_of(k < 64 ? x[0] : x[1], k & 63);
        const double alpha = lane_of(k + 1 < 64 ? x[0] : x[1], (k + 1) & 63);
        xx = wsum(xx);
        double beta = 0.0, scale = 0.0;
        tau = 0.0;
        if (k + 1 < nt) reflector(alpha, xx, beta, tau, scale);
        double vn[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = lane + 64 * q;
            vn[q] = r <= k || r >= nt ? 0.0 : (r == k + 1 ? 1.0 : x[q] * scale);
        }
        if (wv == 0) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int r = lane + 64 * q;
                if (r > k && r < nt) V[r + (long long)k * n] = vn[q];
            }
            bad = bad || !(fabs(dk) < 1e300) || !(fabs(beta) < 1e300);
            mx = fmax(mx, fmax(fabs(dk), fabs(beta)));
            if (lane == 0) {
                T.d[M.a0 + k0 + k] = dk;
                T.e[M.a0 + k0 + k] = beta;
                T.tau[M.a0 + k0 + k] = tau;
            }
        }
        double acc[2] = {0.0, 0.0};
#pragma unroll
        for (int b = 0; b < TLT / 8; ++b)
            if (32 * b + 31 > k && 32 * b < nt) {  // uniform
#pragma unroll
                for (int t = 8 * b; t < 8 * b + 8; ++t) {
                    const int j = (wv + 4 * t) & 63;
                    const double vj = lane_of(v[t / 16], j), wj = lane_of(w[t / 16], j);
                    const double nj = lane_of(vn[t / 16], j);
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        a[q][t] -= v[q] * wj;
                        a[q][t] -= w[q] * vj;
                        acc[q] += a[q][t] * nj;
                    }
                }
            }
#pragma unroll
        for (int q = 0; q < 2; ++q) part[k & 1][wv][lane + 64 * q] = acc[q];
        if (k + 1 < nt && lane == ((k + 1) & 63)) {  // row k + 1 of this wavefront's columns
            double *xc = xcol[k & 1] + wv;
            if (k + 1 < 64) {
#pragma unroll
                for (int t = 0; t < TLT; ++t) xc[4 * t] = a[0][t];
            } else {
#pragma unroll
                for (int t = 16; t < TLT; ++t) xc[4 * t] = a[1][t];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = lane + 64 * q;
            v[q] = vn[q];
            p[q] = x[q] = 0.0;
            if (r > k && r < nt) {
                p[q] = (part[k & 1][0][r] + part[k & 1][1][r]) +
                       (part[k & 1][2][r] + part[k & 1][3][r]);
                x[q] = xcol[k & 1][r];
            }
        }
    }
    // scale of the tridiagonal matrix (largest |d|, |e|); a matrix with a
    // non-finite entry is marked: its results are NaN
    if (wv == 0) {
        for (int i = lane; i < k0; i += 64) {
            const double di = T.d[M.a0 + i], ei = T.e[M.a0 + i];
            bad = bad || !(fabs(di) < 1e300) || !(fabs(ei) < 1e300);
            mx = fmax(mx, fmax(fabs(di), fabs(ei)));
        }
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) mx = fmax(mx, __shfl_xor(mx, s, 64));
        const bool any = __any(bad);
        if (lane == 0) {
            anorm[M.mol] = mx;
            if (any) info[M.mol] = TBX_EIG_NONFINITE;
        }
    }
}

// ---------------------------------------------------------------------------
// divide and conquer of the tridiagonal matrix

// split of n rows into 2^lev segments
__device__ __forceinline__ int seg_at(int n, int lev, int s) { return (int)(((long long)n * s) >> lev); }

// levels of merges above the leaves (segments of at most TBX_DC_LEAF rows)
__device__ __forceinline__ int dc_levels(int n)
{
    int l = 0;
    while (((n + (1 << l) - 1) >> l) > TBX_DC_LEAF) ++l;
    return l;
}

// Root j of 1/rho + sum_i z_i^2 / (d_i - x) = 0, the j-th of K ascending
// poles, by LPR lanes together (a quad, or the wavefront): x = d[org] + tau.
// Rational interpolation at the two poles next to the root with the weight of
// the nearer one fixed (R.-C. Li, LAPACK working note 89), kept inside a bracket
// by bisection: 4 evaluations on average, about 10 for the slowest root.  The
// loop ends in at most 100 steps.
template <int LPR>
__device__ __forceinline__ void secular_root(int K, const double *d, const double *z, double rho,
                                             int j, int sub, double &tau, int &org)
{
    if (K == 1) {
        org = 0;
        tau = rho * z[0] * z[0];
        return;
    }
    const double rhoinv = fast_rcp(rho);
    const bool last = j == K - 1;
    const int jl = last ? K - 2 : j;  // interpolation poles jl, jl + 1
    double psi, phi, dpsi, dphi, lo, hi;
    auto eval = [&](double dorg, double t) {
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int i = sub; i < K; i += LPR) {
            const double zi = z[i];
            const double q = zi * fast_rcp((d[i] - dorg) - t);
            const double q0 = i <= jl ? q : 0.0, q1 = q - q0;
            s[0] += zi * q0;
            s[1] += zi * q1;
            s[2] += q0 * q0;
            s[3] += q1 * q1;
        }
        if (LPR == 64) {
            wsum4(s);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) s[k] = qsum(s[k]);
        }
        psi = s[0];
        phi = s[1];
        dpsi = s[2];
        dphi = s[3];
    };
    const double gap = d[jl + 1] - d[jl], za = z[jl] * z[jl], zb = z[jl + 1] * z[jl + 1];
    // first guess from the value in the middle of the interval: the two poles
    // next to the root kept, the others as a constant
    if (last) {
        org = K - 1;
        double zz = 0.0;
        for (int i = sub; i < K; i += LPR) zz += z[i] * z[i];
        lo = 0.0;
        hi = rho * (LPR == 64 ? wsum(zz) : qsum(zz)) * (1.0 + 4.0 * kEps);
        const double mid = 0.5 * hi;
        eval(d[org], mid);
        const double w = rhoinv + psi + phi;
        if (w < 0.0) lo = mid; else hi = mid;
        const double c = w + za * fast_rcp(gap + mid) + zb * fast_rcp(mid);
        const double a = za + zb - c * gap, b = zb * gap, q = sqrt(fabs(a * a + 4.0 * b * c));
        tau = (a < 0.0 ? 2.0 * b : a + q) * fast_rcp(a < 0.0 ? q - a : 2.0 * c);
    } else {
        const double half = 0.5 * gap;
        eval(d[j], half);
        const double w = rhoinv + psi + phi, c = w + (za - zb) * fast_rcp(half);
        const bool left = w >= 0.0;
        org = left ? j : j + 1;
        lo = left ? 0.0 : -half;
        hi = left ? half : 0.0;
        // c tau^2 - a tau + b = 0 with the signs of the side
        const double a = c * gap + (left ? za + zb : -za - zb), b = left ? za * gap : -zb * gap;
        const double q = sqrt(fabs(a * a - 4.0 * b * c));
        const bool small = left ? a > 0.0 : a < 0.0;  // the root without cancellation
        const double num = small ? 2.0 * b : (left ? a - q : a + q);
        const double den = small ? (left ? a + q : a - q) : 2.0 * c;
        tau = num * fast_rcp(den);
    }
    if (!(tau > lo && tau < hi)) tau = 0.5 * (lo + hi);
    const double dorg = d[org];
    const double p1 = d[jl] - dorg, p2 = d[jl + 1] - dorg;
    for (int it = 0; it < 100; ++it) {
        eval(dorg, tau);
        const double w = rhoinv + psi + phi, dw = dpsi + dphi;
        const double err = 8.0 * (fabs(psi) + fabs(phi)) + rhoinv + fabs(tau) * dw;
        if (!(fabs(w) > kEps * err)) break;
        if (w < 0.0) lo = tau; else hi = tau;
        const double D1 = p1 - tau, D2 = p2 - tau;
        const double a = (D1 + D2) * w - D1 * D2 * dw, b = D1 * D2 * w;
        double c;
        if (last) {
            c = fabs(w - D1 * dpsi - D2 * dphi);
        } else {
            const bool left = org == j;
            const double r = fast_rcp(left ? D1 : D2);
            c = left ? w - D2 * dw + gap * za * r * r : w - D1 * dw - gap * zb * r * r;
        }
        const double q = sqrt(fabs(a * a - 4.0 * b * c));
        const bool small = last ? a < 0.0 : a > 0.0;
        const double num = small ? 2.0 * b : (last ? a + q : a - q);
        const double den = small ? (last ? a - q : a + q) : 2.0 * c;
        double eta = num * fast_rcp(den);
        if (!(w * eta < 0.0)) eta = -w * fast_rcp(dw);
        double t = tau + eta;
        if (!(t > lo && t < hi)) t = 0.5 * (lo + hi);
        if (t == tau || !(t > lo && t < hi)) break;
        tau = t;
    }
}

// Deflation of the sorted pairs (ds, zs) of one merge, serial: entries with a
// negligible z, and of two nearly equal d one after a rotation that zeroes its
// z (recorded: columns src[a], src[b], c, s).  nd: the K kept entries
// (ascending), df: the others.
struct Rot {
    int a, b;
    double c, s;
};
__device__ int deflate(int N, double *ds, double *zs, const int *src, double rho, double tol,
                       int *nd, int *df, Rot *rot, int &nrot)
{
    int K = 0, ndf = 0, pj = -1;
    double dp = 0.0, zp = 0.0;
    nrot = 0;
    double dn = ds[0], zn = zs[0];
    for (int t = 0; t < N; ++t) {
        const double dt = dn, zt = zn;
        if (t + 1 < N) {  // the next entry, loaded one step ahead
            dn = ds[t + 1];
            zn = zs[t + 1];
        }
        if (!(rho * fabs(zt) > tol)) {
            df[ndf++] = t;
            continue;
        }
        if (pj < 0) {
            pj = t;
            dp = dt;
            zp = zt;
            continue;
        }
        const double h2 = zp * zp + zt * zt;
        if (fabs((dt - dp) * zp * zt) <= tol * h2) {
            const double h = sqrt(h2), c = zt / h, s = -zp / h;
            rot[nrot++] = Rot{src[pj], src[t], c, s};
            zs[pj] = 0.0;
            zs[t] = h;
            ds[pj] = dp * c * c + dt * s * s;
            dp = dp * s * s + dt * c * c;
            ds[t] = dp;
            zp = h;
            df[ndf++] = pj;
            pj = t;
        } else {
            nd[K++] = pj;
            pj = t;
            dp = dt;
            zp = zt;
        }
    }
    if (pj >= 0) nd[K++] = pj;
    return K;
}

// Zeros in the rows of the sibling of segment s of level lev, in its columns
// c0 .. c1 - 1 (the merge above reads both children's rows): the rows at
// r = lane, lane + 64, ...
__device__ __forceinline__ void sibling_zero(double *Q, int n, int lev, int s, int c0, int c1,
                                             int lane)
{
    const int g0 = seg_at(n, lev, s), h0 = seg_at(n, lev, s ^ 1), h1 = seg_at(n, lev, (s ^ 1) + 1);
    for (int c = c0 + (threadIdx.x >> 6); c < c1; c += 4)
        for (int r = h0 + lane; r < h1; r += 64) Q[r + (long long)(g0 + c) * n] = 0.0;
}

// Leaves: one workgroup solves a segment of at most 64 rows by merges from
// single rows, everything in LDS.  Four lanes per entry; at each level all
// merges of the segment run together.  Bound by the chain of its phases, the
// roots first: 91 us for 50 rows (222 us with a serial deflation pass and the
// vectors' products on the vector unit).
constexpr int LN = TBX_DC_LEAF;
constexpr int LQ = LN + 1;

struct LeafShared {
    double Q[2][LN * LQ];  // eigenvectors of the children / merged, [column][row]
    double U[LN * LQ];     // [root][entry] of the secular vectors, zero outside the segment
    double d[LN], z[LN], ds[LN], zs[LN], dk[LN], zk[LN], zh[LN], tau[LN], lam[LN], e[LN], zmax[LN],
        rho[LN];
    int src[LN], nd[LN], df[LN], org[LN], idx[LN], K[LN], nrot[LN], pos[LN], lo[LN], hi[LN];
    Rot rot[LN];
};

// Triangular factor M of block g of 16 reflectors (k_eig_back), column c from
// reflector c on, into the part of V above the reflector (column kmax - c, which
// holds nothing else).  Workgroups of the leaves' launch, which is longer: as a
// launch of its own 5 us for 26 orbitals, 10 for 768.
constexpr int WB = 16;
__device__ void wy_block(const EigMol &M, double *V, const double *tau, int g,
                         double (*red)[WB][WB + 1])
{
    const int n = M.n, kmax = n - 3 - WB * g;
    if (kmax < 0) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    double *Vm = V + M.w0;
    const int k = kmax - li;
    const double *col = Vm + (long long)max(k, 0) * n;
    dbl4 acc = dbl4{0.0, 0.0, 0.0, 0.0};
    for (int r0 = (max(kmax - WB + 2, 0) & ~15) + 16 * wv; r0 < n; r0 += 64) {
        double v[4];
        const double *src = col + min(r0 + 4 * lk, n - 1);  // at most 3 past the column: in V
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = src[r];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 4 * lk + r;
            v[r] = (k >= 0 && row > k && row < n) ? v[r] : 0.0;
            acc = mfma(v[r], v[r], acc);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][lk + 4 * r][li] = acc[r];
    __syncthreads();
    const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
    red[0][i][j] += red[1][i][j] + red[2][i][j] + red[3][i][j];
    __syncthreads();
    if (threadIdx.x >= WB) return;
    const int c = threadIdx.x, m = min(WB, kmax + 1);  // column of M; reflectors
    double t[WB], s[WB];
#pragma unroll
    for (int q = 0; q < WB; ++q) t[q] = tau[M.a0 + max(kmax - q, 0)];
#pragma unroll
    for (int q = 0; q < WB; ++q) {
        double x = q == c ? 1.0 : 0.0;
#pragma unroll
        for (int e = 0; e < q; ++e) x -= red[0][q][e] * s[e];
        s[q] = q < m ? t[q] * x : 0.0;
    }
    if (c < m) {
        double *out = Vm + (long long)(kmax - c) * n;
#pragma unroll
        for (int q = 0; q < WB; ++q)
            if (q >= c && q < m) out[q - c] = s[q];
    }
}

__global__ void __launch_bounds__(256) k_dc_leaf(const EigMol *mols, const double *dg,
                                                 const double *eg, double *dout, double *q0,
                                                 double *q1, const double *anorm, int leaves,
                                                 double *V, const double *tau, const int *info)
{
    extern __shared__ double sh[];
    LeafShared &W = *reinterpret_cast<LeafShared *>(sh);
    const EigMol M = mols[blockIdx.y];
    const int n = M.n;
    if (info[M.mol] != 0) return;
    if ((int)blockIdx.x >= leaves) {
        wy_block(M, V, tau, (int)blockIdx.x - leaves,
                 reinterpret_cast<double (*)[WB][WB + 1]>(sh));
        return;
    }
    const int L = dc_levels(n);
    if ((int)blockIdx.x >= (1 << L)) return;
    const int g0 = seg_at(n, L, blockIdx.x), g1 = seg_at(n, L, blockIdx.x + 1), N = g1 - g0;
    if (N <= 0) return;
    const int tid = threadIdx.x, el = tid >> 2, sub = tid & 3;
    const double scale = anorm[M.mol];
    if (tid < LN) {
        // every boundary between rows is a split: d loses |e| on both sides
        double d = 0.0, e = 0.0;
        if (tid < N) {
            const int i = g0 + tid;
            d = dg[M.a0 + i];
            if (i > 0) d -= fabs(eg[M.a0 + i - 1]);
            if (i + 1 < n) {
                e = eg[M.a0 + i];
                d -= fabs(e);
            }
        }
        W.d[tid] = d;
        W.e[tid] = e;
    }
    for (int k = tid; k < LN * LQ; k += 256) {
        const int c = k / LQ, r = k - c * LQ;
        W.Q[0][k] = c == r ? 1.0 : 0.0;
    }
    int cur = 0, top = 0;
    while ((1 << top) < N) ++top;  // 2^top single rows (or none)
    __syncthreads();
    for (int lev = top - 1; lev >= 0; --lev) {
        double *Q = W.Q[cur], *Qn = W.Q[cur ^ 1];
        // this entry's segment and its split
        int lo = 0, hi = 0, mid = 0;
        if (el < N) {
            int s = ((el << lev) + N - 1) / N;
            while ((N * (s + 1)) >> lev <= el) ++s;
            while ((N * s) >> lev > el) --s;
            lo = (N * s) >> lev;
            hi = (N * (s + 1)) >> lev;
            mid = (N * (2 * s + 1)) >> (lev + 1);
        }
        const int len = hi - lo;
        const bool act = el < N, merge = act && mid > lo && mid < hi;
        const double ecut = merge ? W.e[mid - 1] : 0.0;
        const double rho = 2.0 * fabs(ecut);
        if (act && sub == 0) {
            double z = 0.0;
            if (merge) {
                z = el < mid ? Q[el * LQ + mid - 1] : Q[el * LQ + mid];
                z *= (el >= mid && ecut < 0.0) ? -0.70710678118654752440 : 0.70710678118654752440;
            }
            W.z[el] = z;
            W.lo[el] = lo;
            W.hi[el] = hi;
            W.rho[el] = rho;
            W.src[el] = el;  // every slot holds a column, whatever the order below makes of them
        }
        __syncthreads();
        if (act) {  // rank sort within the segment
            int r = 0;
            double zm = 0.0;
            const double de = W.d[el];
#pragma unroll 4
            for (int f = lo + sub; f < hi; f += 4) {
                const double df = W.d[f];
                r += (df < de || (df == de && f < el)) ? 1 : 0;
                zm = fmax(zm, fabs(W.z[f]));
            }
            zm = qmax(zm);
            if (el == lo && sub == 0) W.zmax[lo] = zm;
            r += __builtin_amdgcn_update_dpp(0, r, 0xB1, 0xf, 0xf, false);
            r += __builtin_amdgcn_update_dpp(0, r, 0x4E, 0xf, 0xf, false);
            if (sub == 0) {
                W.ds[lo + r] = de;
                W.zs[lo + r] = W.z[el];
                W.src[lo + r] = el;
            }
        }
        __syncthreads();
        if (tid < LN) {  // one lane per sorted entry
            int slo = 0, shi = 0;
            double srho = 0.0, tol = 0.0;
            if (tid < N) {
                slo = W.lo[tid];
                shi = W.hi[tid];
                srho = W.rho[tid];
                tol = 16.0 * kEps * fmax(fmax(fabs(W.ds[slo]), fabs(W.ds[shi - 1])),
                                         scale * W.zmax[slo]);
            }
            const double dt = W.ds[tid], zt = W.zs[tid];
            const bool keep = tid < N && srho * fabs(zt) > tol;
            const unsigned long long below = (1ull << tid) - 1ull, from = ~((1ull << slo) - 1ull);
            const unsigned long long mask = __ballot(keep) & from, prev = mask & below;
            bool close = false;
            if (keep && prev) {
                const int a = 63 - __clzll((long long)prev);
                const double zp = W.zs[a];
                close = fabs((dt - W.ds[a]) * zp * zt) <= tol * (zp * zp + zt * zt);
            }
            const unsigned long long in = shi < 64 ? (1ull << shi) - 1ull : ~0ull;
            const bool serial = (__ballot(close) & from & in) != 0;
            const int before = __popcll(prev);
            if (tid < N) {
                if (!serial) {  // no two neighbours are close: what the serial pass would keep
                    if (keep) W.nd[slo + before] = tid - slo;
                    else W.df[slo + (tid - slo - before)] = tid - slo;
                }
                if (tid == slo) {
                    int nr = 0;
                    W.K[slo] = serial ? deflate(shi - slo, W.ds + slo, W.zs + slo, W.src + slo, srho,
                                                tol, W.nd + slo, W.df + slo, W.rot + slo, nr)
                                      : __popcll(mask & in);
                    W.nrot[slo] = nr;
                }
            }
        }
        __syncthreads();
        const int K = act ? W.K[lo] : 0;
        for (int i = tid; i < LN * LQ; i += 256) W.U[i] = 0.0;
        // rotations (each row on its own), then the kept entries compacted
        if (act && sub == 0) {
            for (int t = 0; t < W.nrot[lo]; ++t) {
                const Rot R = W.rot[lo + t];
                const double x = Q[R.a * LQ + el], y = Q[R.b * LQ + el];
                Q[R.a * LQ + el] = R.c * x + R.s * y;
                Q[R.b * LQ + el] = R.c * y - R.s * x;
            }
            const int t = el - lo;
            if (t < K) {
                const int q = lo + W.nd[el];
                W.dk[el] = W.ds[q];
                W.zk[el] = W.zs[q];
                W.idx[el] = W.src[q];
            } else {
                const int q = lo + W.df[el - K];
                W.lam[el] = W.ds[q];
                W.idx[el] = W.src[q];
            }
        }
        __syncthreads();
        const int t = el - lo;
        if (act && t < K) {
            double tau;
            int org;
            secular_root<4>(K, W.dk + lo, W.zk + lo, rho, t, sub, tau, org);
            if (sub == 0) {
                W.tau[el] = tau;
                W.org[el] = org;
                W.lam[el] = W.dk[lo + org] + tau;
            }
        }
        __syncthreads();
        if (act && t < K) {  // z that the computed roots belong to exactly
            const double di = W.dk[el];
            double pr = 1.0;
            for (int j = sub; j < K; j += 4) {
                const double del = (di - W.dk[lo + W.org[lo + j]]) - W.tau[lo + j];
                pr *= j == t ? -del : del * fast_rcp(di - W.dk[lo + j]);
            }
            pr = qprod(pr);
            if (sub == 0) W.zh[el] = copysign(sqrt(fabs(pr)), W.zk[el]);
        }
        __syncthreads();
        if (act) {
            if (t < K) {  // normalised secular vectors
                const double dorg = W.dk[lo + W.org[el]], tau = W.tau[el];
                double nn = 0.0;
#pragma unroll 4
                for (int i = sub; i < K; i += 4) {
                    const double u = W.zh[lo + i] * fast_rcp((W.dk[lo + i] - dorg) - tau);
                    W.U[el * LQ + lo + i] = u;
                    nn += u * u;
                }
                const double inv = 1.0 / sqrt(qsum(nn));
                for (int i = sub; i < K; i += 4) W.U[el * LQ + lo + i] *= inv;
            } else if (sub == 0) {
                W.U[el * LQ + el] = 1.0;  // deflated: the vector itself
            }
            int r = 0;  // place among the segment's new eigenvalues
            const double le = W.lam[el];
            for (int f = lo + sub; f < hi; f += 4) {
                const double lf = W.lam[f];
                r += (lf < le || (lf == le && f < el)) ? 1 : 0;
            }
            r += __builtin_amdgcn_update_dpp(0, r, 0xB1, 0xf, 0xf, false);
            r += __builtin_amdgcn_update_dpp(0, r, 0x4E, 0xf, 0xf, false);
            if (sub == 0) {
                W.pos[el] = lo + r;
                W.d[lo + r] = le;
            }
        }
        __syncthreads();
        // new vectors: Q (columns idx) times the block-diagonal U on MFMA, a
        // 32 x 32 quarter per wavefront
        const int lane = tid & 63, li = lane & 15, lk = lane >> 4, wv = tid >> 6;
        const int sr = 32 * (wv >> 1), sc = 32 * (wv & 1);
        dbl4 acc[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[u][q] = dbl4{0.0, 0.0, 0.0, 0.0};
        if (sr < N && sc < N) {
            // the entries of the columns' segments, which are also their rows
            const int klo = W.lo[sc], khi = W.hi[min(sc + 31, N - 1)];
            const int kend = sr < khi && sr + 32 > klo ? khi : klo;
            // sixteen entries at a time, their columns' indices, then their
            // operands under way together (U is zero outside the segment): 39
            // against 59 thousand cycles over the six merges of 50 rows with an
            // index, its operands and its products at a time
            for (int ks = klo & ~15; ks < kend; ks += 16) {
                int col[4];
                double x[4][2], y[4][2];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int kk = ks + 4 * p + lk;
                    col[p] = W.idx[min(kk, N - 1)];
#pragma unroll
                    for (int u = 0; u < 2; ++u) y[p][u] = W.U[(sc + 16 * u + li) * LQ + kk];
                }
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int u = 0; u < 2; ++u) x[p][u] = Q[col[p] * LQ + sr + 16 * u + li];
#pragma unroll
                for (int p = 0; p < 4; ++p)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
                            acc[u][q] = mfma(x[p][u], y[p][q], acc[u][q]);
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int c = sc + 16 * q + li;
                if (c < N) {
#pragma unroll
                    for (int u = 0; u < 2; ++u)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            Qn[W.pos[c] * LQ + sr + 16 * u + lk + 4 * r] = acc[u][q][r];
                }
            }
        }
        __syncthreads();
        cur ^= 1;
    }
    // after L merges the result is in q0
    double *qo = ((L & 1) ? q1 : q0) + M.w0;
    if (tid < N) dout[((L & 1) ? M.astride : 0) + M.a0 + g0 + tid] = W.d[tid];
    for (int c = tid >> 6; c < N; c += 4)
        if ((tid & 63) < N)
            qo[g0 + (tid & 63) + (long long)(g0 + c) * n] = W.Q[cur][c * LQ + (tid & 63)];
    if (L > 0) sibling_zero(qo, n, L, blockIdx.x, 0, N, tid & 63);
}

// One merge: the parts of its state in global memory, all at a0 + lo
struct DcPtr {
    double *q[2];              // eigenvectors, by parity
    double *d;                 // [2][nao] eigenvalues, by parity
    double *dk, *zk, *zh, *tau, *lam, *inv;  // [nao]
    int *idx, *org, *pos;      // [nao]
    int *K;                    // [nao] at the segment's first row
    double *rho;               // [nao]
    const double *e;           // off-diagonals
    const double *anorm;       // [nmol] scale of the matrix
};

struct Seg {
    int lo, mid, hi, par;
};
// segment blockIdx.z of level lev of a molecule of n rows; false: none there
__device__ __forceinline__ bool dc_seg(int n, int lev, int s, Seg &g)
{
    const int L = dc_levels(n);
    if (lev >= L || s >= (1 << lev)) return false;
    g.lo = seg_at(n, lev, s);
    g.hi = seg_at(n, lev, s + 1);
    g.mid = seg_at(n, lev + 1, 2 * s + 1);
    g.par = (lev + 1) & 1;  // parity of the children's buffers
    return true;
}

// sort, deflation and rotations of one merge
constexpr int PREP_THREADS = 512;
__global__ void __launch_bounds__(PREP_THREADS) k_dc_prep(const EigMol *mols, DcPtr D, int lev,
                                                          const int *info)
{
    extern __shared__ double sh[];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n;
    Seg g;
    if (!dc_seg(n, lev, blockIdx.z, g) || info[M.mol] != 0) return;
    const int N = g.hi - g.lo, N1 = g.mid - g.lo, tid = threadIdx.x;
    double *d = sh, *z = d + N, *ds = z + N, *zs = ds + N;
    Rot *rot = reinterpret_cast<Rot *>(zs + N);
    int *src = reinterpret_cast<int *>(rot + N), *nd = src + N, *df = nd + N;
    __shared__ int sK, snrot, wcnt[PREP_THREADS / 64];
    __shared__ double zred[PREP_THREADS / 64];
    const double *dc = D.d + g.par * M.astride + M.a0 + g.lo;
    double *Q = D.q[g.par] + M.w0;
    const double ecut = D.e[M.a0 + g.mid - 1];
    const double rho = 2.0 * fabs(ecut);
    double zm = 0.0;
    for (int i = tid; i < N; i += PREP_THREADS) {
        d[i] = dc[i];
        double x = Q[(i < N1 ? g.mid - 1 : g.mid) + (long long)(g.lo + i) * n];
        x *= (i >= N1 && ecut < 0.0) ? -0.70710678118654752440 : 0.70710678118654752440;
        z[i] = x;
        src[i] = i;  // every slot holds a column, whatever the order below makes of them
        zm = fmax(zm, fabs(x));
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) zm = fmax(zm, __shfl_xor(zm, s, 64));
    if ((tid & 63) == 0) zred[tid >> 6] = zm;
    __syncthreads();
    // merge of the two ascending halves by binary search
    for (int i = tid; i < N; i += PREP_THREADS) {
        const double x = d[i];
        int a = i < N1 ? N1 : 0, b = i < N1 ? N : N1;  // the other half
        const int base = a;
        while (a < b) {
            const int m = (a + b) >> 1;
            if (d[m] < x || (i >= N1 && d[m] == x)) a = m + 1; else b = m;
        }
        const int r = (i < N1 ? i : i - N1) + (a - base);
        ds[r] = x;
        zs[r] = z[i];
        src[r] = i;
    }
    __syncthreads();
    double zmax = 0.0;
    for (int q = 0; q < PREP_THREADS / 64; ++q) zmax = fmax(zmax, zred[q]);
    const double dmax = fmax(fabs(ds[0]), fabs(ds[N - 1]));
    const double tol = 16.0 * kEps * fmax(dmax, D.anorm[M.mol] * zmax);
    // the entries with a z that counts, in order; where no two neighbours among
    // them are close the serial pass would keep just these
    const int per = (N + PREP_THREADS - 1) / PREP_THREADS, i0 = tid * per, i1 = min(i0 + per, N);
    int cnt = 0;
    for (int i = i0; i < i1; ++i) cnt += rho * fabs(zs[i]) > tol ? 1 : 0;
    int inc = cnt;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int y = __shfl_up(inc, s, 64);
        if ((tid & 63) >= s) inc += y;
    }
    if ((tid & 63) == 63) wcnt[tid >> 6] = inc;
    __syncthreads();
    int kept = inc - cnt, total = 0;
    for (int q = 0; q < PREP_THREADS / 64; ++q) {
        if (q < (tid >> 6)) kept += wcnt[q];
        total += wcnt[q];
    }
    for (int i = i0; i < i1; ++i) {
        if (rho * fabs(zs[i]) > tol) nd[kept++] = i;
        else df[i - kept] = i;
    }
    __syncthreads();
    bool close = false;
    for (int i = tid + 1; i < total; i += PREP_THREADS) {
        const int a = nd[i - 1], b = nd[i];
        const double za = zs[a], zb = zs[b];
        close = close || fabs((ds[b] - ds[a]) * za * zb) <= tol * (za * za + zb * zb);
    }
    const bool serial = __syncthreads_or(close) != 0;
    if (tid == 0) {
        int nr = 0;
        sK = serial ? deflate(N, ds, zs, src, rho, tol, nd, df, rot, nr) : total;
        snrot = nr;
        D.K[M.a0 + g.lo] = sK;
        D.rho[M.a0 + g.lo] = rho;
    }
    __syncthreads();
    const int K = sK, nrot = snrot;
    // rotations, a row per thread, eight loaded at a time (a column that the
    // rotation before has just changed is taken from its register)
    constexpr int RB = 8;
    for (int r = tid; r < N; r += PREP_THREADS) {
        double *q = Q + g.lo + r + (long long)g.lo * n;
        for (int t0 = 0; t0 < nrot; t0 += RB) {
            double x[RB], y[RB], last = 0.0;
#pragma unroll
            for (int u = 0; u < RB; ++u) {
                x[u] = t0 + u < nrot ? q[(long long)rot[t0 + u].a * n] : 0.0;
                y[u] = t0 + u < nrot ? q[(long long)rot[t0 + u].b * n] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < RB; ++u)
                if (t0 + u < nrot) {
                    const Rot R = rot[t0 + u];
                    const double xa = u > 0 && R.a == rot[t0 + u - 1].b ? last : x[u];
                    q[(long long)R.a * n] = R.c * xa + R.s * y[u];
                    last = R.c * y[u] - R.s * xa;
                    q[(long long)R.b * n] = last;
                }
        }
    }
    const int o = M.a0 + g.lo;
    for (int i = tid; i < N; i += PREP_THREADS) {
        if (i < K) {
            const int q = nd[i];
            D.dk[o + i] = ds[q];
            D.zk[o + i] = zs[q];
            D.idx[o + i] = src[q];
        } else {
            const int q = df[i - K];
            D.lam[o + i] = ds[q];
            D.idx[o + i] = src[q];
        }
    }
}

// roots: one wavefront each, the poles in LDS
__global__ void __launch_bounds__(256) k_dc_secular(const EigMol *mols, DcPtr D, int lev,
                                                    const int *info)
{
    __shared__ double d[TBX_EIG_MAXN], z[TBX_EIG_MAXN];
    const EigMol M = mols[blockIdx.y];
    Seg g;
    if (!dc_seg(M.n, lev, blockIdx.z, g) || info[M.mol] != 0) return;
    const int o = M.a0 + g.lo, K = D.K[o];
    if (4 * (int)blockIdx.x >= K) return;
    for (int i = threadIdx.x; i < K; i += 256) {
        d[i] = D.dk[o + i];
        z[i] = D.zk[o + i];
    }
    __syncthreads();
    const int j = 4 * blockIdx.x + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= K) return;
    double tau;
    int org;
    secular_root<64>(K, d, z, D.rho[o], j, lane, tau, org);
    if (lane == 0) {
        D.tau[o + j] = tau;
        D.org[o + j] = org;
        D.lam[o + j] = d[org] + tau;
    }
}

// the recomputed z: one wavefront per entry
__global__ void __launch_bounds__(256) k_dc_zhat(const EigMol *mols, DcPtr D, int lev,
                                                 const int *info)
{
    const EigMol M = mols[blockIdx.y];
    Seg g;
    if (!dc_seg(M.n, lev, blockIdx.z, g) || info[M.mol] != 0) return;
    const int o = M.a0 + g.lo, K = D.K[o];
    const int i = 4 * blockIdx.x + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= K) return;
    const double di = D.dk[o + i];
    double pr = 1.0;
    for (int j = lane; j < K; j += 64) {
        const double del = (di - D.dk[o + D.org[o + j]]) - D.tau[o + j];
        pr *= j == i ? -del : del * fast_rcp(di - D.dk[o + j]);
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) pr *= __shfl_xor(pr, s, 64);
    if (lane == 0) D.zh[o + i] = copysign(sqrt(fabs(pr)), D.zk[o + i]);
}

// 1 / norm of each secular vector and the place of each eigenvalue: one
// wavefront per entry
__global__ void __launch_bounds__(256) k_dc_norm(const EigMol *mols, DcPtr D, int lev,
                                                 const int *info)
{
    const EigMol M = mols[blockIdx.y];
    Seg g;
    if (!dc_seg(M.n, lev, blockIdx.z, g) || info[M.mol] != 0) return;
    const int o = M.a0 + g.lo, K = D.K[o], N = g.hi - g.lo;
    const int j = 4 * blockIdx.x + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= N) return;
    const double lj = D.lam[o + j];
    int r = 0;
    for (int f = lane; f < N; f += 64) {
        const double lf = D.lam[o + f];
        r += (lf < lj || (lf == lj && f < j)) ? 1 : 0;
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) r += __shfl_xor(r, s, 64);
    if (j < K) {
        const double dorg = D.dk[o + D.org[o + j]], tau = D.tau[o + j];
        double nn = 0.0;
        for (int i = lane; i < K; i += 64) {
            const double u = D.zh[o + i] * fast_rcp((D.dk[o + i] - dorg) - tau);
            nn += u * u;
        }
        nn = wsum(nn);
        if (lane == 0) D.inv[o + j] = 1.0 / sqrt(nn);
    }
    if (lane == 0) {
        D.pos[o + j] = r;
        D.d[(g.par ^ 1) * M.astride + o + r] = lj;
    }
}

// New vectors of one merge, a 64 x 64 tile (rows, roots) per workgroup: the
// products of the children's vectors (columns idx) with the secular vectors,
// which are formed while their panel is staged (one reciprocal each).
// Deflated columns are copied to their place.
__global__ void __launch_bounds__(256) k_dc_gemm(const EigMol *mols, DcPtr D, int lev,
                                                 const int *info)
{
    constexpr int KB = 16;
    __shared__ double As[KB][PR], Bs[KB][PR];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n;
    Seg g;
    if (!dc_seg(n, lev, blockIdx.z, g) || info[M.mol] != 0) return;
    const int o = M.a0 + g.lo, K = D.K[o], N = g.hi - g.lo, nt = (N + 63) / 64;
    if ((int)blockIdx.x >= nt * nt) return;
    const int R0 = 64 * (blockIdx.x % nt), C0 = 64 * (blockIdx.x / nt);
    const double *Q = D.q[g.par] + M.w0 + g.lo;
    double *Qn = D.q[g.par ^ 1] + M.w0 + g.lo;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int sr = 32 * (wv >> 1), sc = 32 * (wv & 1);
    const int kk = tid >> 4, rr = tid & 15;
    if (lev > 0 && R0 == 0)
        sibling_zero(D.q[g.par ^ 1] + M.w0, n, lev, blockIdx.z, C0, min(C0 + 64, N), lane);
    if (C0 + 63 >= K) {  // deflated columns of the tile
        for (int c = max(C0, K) + wv; c < min(C0 + 64, N); c += 4) {
            const int r = R0 + lane;
            if (r < N) Qn[r + (long long)(g.lo + D.pos[o + c]) * n] =
                Q[r + (long long)(g.lo + D.idx[o + c]) * n];
        }
        if (C0 >= K) return;
    }
    double dorg[4], tau[4], inv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = C0 + rr + 16 * q;
        dorg[q] = tau[q] = inv[q] = 0.0;
        if (c < K) {
            dorg[q] = D.dk[o + D.org[o + c]];
            tau[q] = D.tau[o + c];
            inv[q] = D.inv[o + c];
        }
    }
    double pa[4], dk = 0.0, zh = 0.0;
    auto load = [&](int k0) {
        const int k = k0 + kk;
        const bool kin = k < K;
        dk = kin ? D.dk[o + k] : 0.0;
        zh = kin ? D.zh[o + k] : 0.0;
        const double *col = Q + (long long)(g.lo + (kin ? D.idx[o + k] : 0)) * n;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = R0 + rr + 16 * q;
            pa[q] = (kin && i < N) ? col[i] : 0.0;
        }
    };
    dbl4 acc[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[s][u] = dbl4{0.0, 0.0, 0.0, 0.0};
    load(0);
    for (int k0 = 0; k0 < K; k0 += KB) {
        __syncthreads();
        const bool kin = k0 + kk < K;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            As[kk][rr + 16 * q] = pa[q];
            Bs[kk][rr + 16 * q] = (kin && C0 + rr + 16 * q < K)
                                      ? zh * inv[q] * fast_rcp((dk - dorg[q]) - tau[q])
                                      : 0.0;
        }
        __syncthreads();
        if (k0 + KB < K) load(k0 + KB);
#pragma unroll
        for (int ks = 0; ks < KB; ks += 4) {
            double a[2], b[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                a[s] = As[ks + lk][sr + 16 * s + li];
                b[s] = Bs[ks + lk][sc + 16 * s + li];
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[s][u] = mfma(a[s], b[u], acc[s][u]);
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int c = C0 + sc + 16 * u + li;
        if (c >= K) continue;
        double *col = Qn + (long long)(g.lo + D.pos[o + c]) * n;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = R0 + sr + 16 * s + lk + 4 * r;
                if (i < N) col[i] = acc[s][u][r];
            }
    }
}

// ---------------------------------------------------------------------------
// Back-transformation of 16 eigenvectors per workgroup, by blocks of 16 reflectors
// from the last to the first: H_15 .. H_0 = I - V M V^T with M the transpose of the
// triangular factor of the compact WY form (R. Schreiber and C. Van Loan, SIAM J.
// Sci. Stat. Comput. 10, 53 (1989)), H_0 the block's last column.  Each wavefront
// holds a quarter of the rows, in tiles of 16 dealt in turn, as accumulators of
// the matrix instruction, whose registers are also the right operand of V^T Z;
// V comes from global memory in the layout of that product (the next block
// meanwhile: two ahead are no faster) and goes through LDS to the layout of the
// update.  Then the strip is solved with L^T in LDS.  768 orbitals, us: 556 with
// the reflectors applied one by one (a sum across the wavefront each; 535 four at
// a time), 412 now, of which the solve is 160, reads of V not hidden 90; 26
// orbitals 20 and 11.
constexpr int WP = 18;   // row length of a staged tile of V (doubles; banks)

template <int R>
__global__ void __launch_bounds__(256) k_eig_back(const EigMol *mols, const double *Z,
                                                  const double *V, const double *L,
                                                  const double *eval, double *C, double *ev,
                                                  const int *info)
{
    extern __shared__ double X[];
    const EigMol M = mols[blockIdx.y];
    const int n = M.n, c0 = 16 * blockIdx.x;
    if (c0 >= n || info[M.mol] == 1) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lk = lane >> 4;
    if (info[M.mol] != 0) {  // non-finite input
        const double nan = __longlong_as_double(0x7ff8000000000000LL);
        for (int c = 0; c < 16 && c0 + c < n; ++c)
            for (int r = tid; r < n; r += 256) C[M.d0 + r + (long long)(c0 + c) * n] = nan;
        if (tid < 16 && c0 + tid < n) ev[M.a0 + c0 + tid] = nan;
        return;
    }
    if (tid < 16 && c0 + tid < n) ev[M.a0 + c0 + tid] = eval[M.a0 + c0 + tid];
    const double *Zm = Z + M.w0, *Vm = V + M.w0;
    const int rows = (n + NB - 1) / NB * NB;  // <= 64 R
    // tile t: rows 64 t + 16 wv ..; register r of lane (lk, li): row 4 lk + r, column li
    const int row0 = 16 * wv + 4 * lk;
    dbl4 z[R];
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) z[t][r] = ldg(Zm, n, row0 + 64 * t + r, c0 + li);
    double *stage = X + wv * (R * WB * WP), *red = X + 4 * (R * WB * WP);
    double px[R][4], pm[4];
    // block g: V of reflector kmax - li in the tile's rows, -M[li][4 s + lk]
    auto fetch = [&](int g) {
        const int kmax = n - 3 - WB * g, k = kmax - li;
        const double *col = Vm + (long long)max(k, 0) * n;
#pragma unroll
        for (int t = 0; t < R; ++t)
            if (64 * t + 64 > kmax - WB + 2) {  // uniform: V is zero in the rows above
                const double *src = col + min(row0 + 64 * t, n - 1);  // at most 3 past: in V
#pragma unroll
                for (int r = 0; r < 4; ++r) px[t][r] = src[r];
            }
        const int m = min(WB, kmax + 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = 4 * s + lk;
            const double x = Vm[max(li - c, 0) + (long long)max(kmax - c, 0) * n];
            pm[s] = (li >= c && li < m) ? -x : 0.0;
        }
    };
    const int nblk = n > 2 ? (n - 2 + WB - 1) / WB : 0;
    if (nblk > 0) fetch(0);
    for (int g = 0; g < nblk; ++g) {
        const int kmax = n - 3 - WB * g, k = kmax - li, low = kmax - WB + 2;
        dbl4 w0 = dbl4{0.0, 0.0, 0.0, 0.0}, w1 = w0;
#pragma unroll
        for (int t = 0; t < R; ++t)
            if (64 * t + 64 > low) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = row0 + 64 * t + r;
                    px[t][r] = (k >= 0 && row > k && row < n) ? px[t][r] : 0.0;
                }
                double2 *st = reinterpret_cast<double2 *>(stage + (t * WB + li) * WP + 4 * lk);
                st[0] = make_double2(px[t][0], px[t][1]);
                st[1] = make_double2(px[t][2], px[t][3]);
                w0 = mfma(px[t][0], z[t][0], w0);
                w1 = mfma(px[t][1], z[t][1], w1);
                w0 = mfma(px[t][2], z[t][2], w0);
                w1 = mfma(px[t][3], z[t][3], w1);
            }
        double a[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) a[s] = pm[s];
        if (g + 1 < nblk) fetch(g + 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wv * 4 + r) * 64 + lane] = w0[r] + w1[r];
        __syncthreads();
        dbl4 w, y = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < 4; ++r)
            w[r] = red[r * 64 + lane] + red[(4 + r) * 64 + lane] + red[(8 + r) * 64 + lane] +
                   red[(12 + r) * 64 + lane];
        __syncthreads();  // red is read before the next block's
#pragma unroll
        for (int s = 0; s < 4; ++s) y = mfma(a[s], w[s], y);
        // rows of the update's accumulators are 4 lk + r: row of operand lane li
        const double *sv = stage + lk * WP + 4 * (li & 3) + (li >> 2);
#pragma unroll
        for (int t = 0; t < R; ++t)
            if (64 * t + 64 > low) {
#pragma unroll
                for (int s = 0; s < 4; ++s) z[t] = mfma(sv[(t * WB + 4 * s) * WP], y[s], z[t]);
            }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < R; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (row0 + 64 * t + r < rows) X[(row0 + 64 * t + r) * XS + li] = z[t][r];
    __syncthreads();
    strip_solve<false>(L + M.w0, n, X);
    for (int c = 0; c < 16 && c0 + c < n; ++c)
        for (int r = tid; r < n; r += 256) C[M.d0 + r + (long long)(c0 + c) * n] = X[r * XS + c];
}

// LDS of k_eig_back<R>: the strip (64 R rows), or the block of reflectors and the
// partial products before it
constexpr size_t back_lds(size_t R)
{
    return sizeof(double) * std::max(XS * 64 * R, 4 * R * WB * WP + 16 * 64);
}
static_assert(back_lds(TBX_EIG_MAXN / 64) <= 160 * 1024, "LDS of a CU");

template <class F>
hipError_t allow_lds(F f, size_t bytes)
{
    return hipFuncSetAttribute(reinterpret_cast<const void *>(f),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Molecules of the library route: info = TBX_EIG_NONFINITE for an infinity or
// NaN in the upper triangle of H, a wavefront per column
__global__ void __launch_bounds__(256) k_eig_finite(int n, const double *H, int *info)
{
    const int c = 4 * blockIdx.x + (threadIdx.x >> 6);
    if (c >= n) return;
    bool bad = false;
    for (int r = threadIdx.x & 63; r <= c; r += 64) {
        const int hi = __double2hiint(H[r + (long long)c * n]) & 0x7fffffff;
        bad = bad || hi >= 0x7ff00000;
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) *info = TBX_EIG_NONFINITE;
}

__global__ void __launch_bounds__(256) k_eig_set(int n, double *H, double *ev, double v)
{
    for (int r = threadIdx.x; r < n; r += 256) H[r + (long long)blockIdx.x * n] = v;
    if (threadIdx.x == 0) ev[blockIdx.x] = v;
}

} // namespace

// info[0] <- TBX_EIG_NONFINITE for an infinity or NaN in the upper triangle of H, else 0
extern "C" hipError_t tbx_launch_eigen_finite(int n, const double *H, int *info, hipStream_t s)
{
    const hipError_t e = hipMemsetAsync(info, 0, sizeof(int), s);  // the solver waits: no capture
    if (e != hipSuccess) return e;
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_eig_finite, dim3((n + 3) / 4), dim3(256), 0, s, n, H, info);
    return hipGetLastError();
}

// every element of H [n * n] and ev [n] <- v
extern "C" hipError_t tbx_launch_eigen_set(int n, double *H, double *ev, double v, hipStream_t s)
{
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_eig_set, dim3(n), dim3(256), 0, s, n, H, ev, v);
    return hipGetLastError();
}

// The molecules mols[0 .. nmol) (device; nmax .. nmin orbitals, descending):
// H, S and ev are the batch's dense and orbital arrays, wk the workspace.
extern "C" hipError_t tbx_launch_eigen(const EigMol *mols, const int *n_host, int nmol,
                                       const EigWork *wk, double *H, const double *S, double *ev,
                                       int *info, hipStream_t s)
{
    if (nmol <= 0) return hipSuccess;
    const int nmax = n_host[0];
    if (nmax > TBX_EIG_MAXN) return hipErrorInvalidValue;
    const size_t strip = sizeof(double) * XS * (size_t)((nmax + NB - 1) / NB * NB);
    const size_t lds_leaf = sizeof(LeafShared);
    const size_t lds_prep = (4 * sizeof(double) + sizeof(Rot) + 3 * sizeof(int)) * (size_t)nmax;
    const size_t lds_max = sizeof(double) * XS * TBX_EIG_MAXN;
    const size_t prep_max = (4 * sizeof(double) + sizeof(Rot) + 3 * sizeof(int)) * TBX_EIG_MAXN;
    hipError_t e = hipSuccess;
    if ((e = allow_lds(k_eig_trsm<false>, lds_max)) || (e = allow_lds(k_eig_trsm<true>, lds_max)) ||
        (e = allow_lds(k_dc_leaf, lds_leaf)) ||
        (e = allow_lds(k_dc_prep, prep_max)) || (e = allow_lds(k_eig_back<2>, back_lds(2))) ||
        (e = allow_lds(k_eig_back<4>, back_lds(4))) || (e = allow_lds(k_eig_back<8>, back_lds(8))) ||
        (e = allow_lds(k_eig_back<12>, back_lds(12))) ||
        (e = allow_lds(k_eig_back<16>, back_lds(16))))
        return e;
    (void)hipGetLastError();
    double *B0 = wk->m[0], *B1 = wk->m[1], *B2 = wk->m[2], *B3 = wk->m[3];
    const unsigned nm = nmol;
    const int nt32 = (nmax + 31) / 32, nblk = (nmax + NB - 1) / NB, ns = (nmax + 15) / 16;
    // first molecule with at most `n` orbitals (the list is descending)
    auto above = [&](int n) {
        int k = 0;
        while (k < nmol && n_host[k] > n) ++k;
        return k;
    };
    hipLaunchKernelGGL(k_eig_symm, dim3(nt32 * (nt32 + 1) / 2, nm, 2), dim3(256), 0, s, mols, S, H,
                       B0, B2, info);
    for (int kb = -1; kb < nblk - 1; ++kb) {
        const int left = nblk - 1 - kb, cnt = above(NB * (kb + 1));
        hipLaunchKernelGGL(k_eig_chol, dim3(kb < 0 ? 1 : left * (left + 1) / 2, cnt), dim3(256), 0,
                           s, mols, B0, B1, kb, info);
    }
    hipLaunchKernelGGL(k_eig_trsm<false>, dim3(ns, nm), dim3(256), strip, s, mols, B1, B2, B0, info);
    hipLaunchKernelGGL(k_eig_trsm<true>, dim3(ns, nm), dim3(256), strip, s, mols, B1, B0, B2, info);
    // A in B2, the reflectors go to B0
    const TrdPtr T{B2, B0, wk->d, wk->e, wk->tau, wk->p, wk->stride};
    for (int k = 0; nmax > TBX_TRD_TAIL + k; ++k) {
        const int cnt = above(TBX_TRD_TAIL + k);
        const dim3 grid((nmax - k - 1 + TRD_COLS - 1) / TRD_COLS, cnt), blk(TRD_THREADS);
        switch ((nmax - k + 255) / 256) {
        case 1: hipLaunchKernelGGL(k_trd_step<1>, grid, blk, 0, s, mols, T, k); break;
        case 2: hipLaunchKernelGGL(k_trd_step<2>, grid, blk, 0, s, mols, T, k); break;
        case 3: hipLaunchKernelGGL(k_trd_step<3>, grid, blk, 0, s, mols, T, k); break;
        default: hipLaunchKernelGGL(k_trd_step<4>, grid, blk, 0, s, mols, T, k); break;
        }
    }
    hipLaunchKernelGGL(k_trd_tail, dim3(nm), dim3(TL_THREADS), 0, s, mols, T, wk->anorm, info);
    // eigenvectors by parity in B2, B3
    int levels = 0;
    while (((nmax + (1 << levels) - 1) >> levels) > TBX_DC_LEAF) ++levels;
    const int leaves = 1 << levels, wy = nmax > 2 ? (nmax - 2 + WB - 1) / WB : 0;
    hipLaunchKernelGGL(k_dc_leaf, dim3(leaves + wy, nm), dim3(256), lds_leaf, s, mols, wk->d,
                       wk->e, wk->ev, B2, B3, wk->anorm, leaves, B0, wk->tau, info);
    DcPtr D{};
    D.q[0] = B2;
    D.q[1] = B3;
    D.d = wk->ev;
    D.dk = wk->v[0];
    D.zk = wk->v[1];
    D.zh = wk->v[2];
    D.tau = wk->v[3];
    D.lam = wk->v[4];
    D.inv = wk->v[5];
    D.rho = wk->v[6];
    D.idx = wk->iv[0];
    D.org = wk->iv[1];
    D.pos = wk->iv[2];
    D.K = wk->iv[3];
    D.e = wk->e;
    D.anorm = wk->anorm;
    for (int lev = levels - 1; lev >= 0; --lev) {
        const int cnt = above(TBX_DC_LEAF << lev);  // more than lev levels
        const int seg = ((nmax + (1 << lev) - 1) >> lev), tiles = (seg + 63) / 64;
        const unsigned ms = 1u << lev;
        hipLaunchKernelGGL(k_dc_prep, dim3(1, cnt, ms), dim3(PREP_THREADS), lds_prep, s, mols, D,
                           lev, info);
        hipLaunchKernelGGL(k_dc_secular, dim3((seg + 3) / 4, cnt, ms), dim3(256), 0, s, mols, D,
                           lev, info);
        hipLaunchKernelGGL(k_dc_zhat, dim3((seg + 3) / 4, cnt, ms), dim3(256), 0, s, mols, D, lev,
                           info);
        hipLaunchKernelGGL(k_dc_norm, dim3((seg + 3) / 4, cnt, ms), dim3(256), 0, s, mols, D, lev,
                           info);
        hipLaunchKernelGGL(k_dc_gemm, dim3(tiles * tiles, cnt, ms), dim3(256), 0, s, mols, D, lev,
                           info);
    }
    // back-transformation, by the register rows the molecules need
    const int cap[5] = {16, 12, 8, 4, 2};
    int m0 = 0;
    for (int q = 0; q < 5 && m0 < nmol; ++q) {
        const int m1 = q == 4 ? nmol : above(64 * cap[q + 1]);
        if (m1 <= m0) continue;
        const int nx = n_host[m0];
        const dim3 grid((nx + 15) / 16, m1 - m0);
        const size_t lds = back_lds(cap[q]);
        const EigMol *mm = mols + m0;
        switch (cap[q]) {
        case 16: hipLaunchKernelGGL(k_eig_back<16>, grid, dim3(256), lds, s, mm, B2, B0, B1, wk->ev, H, ev, info); break;
        case 12: hipLaunchKernelGGL(k_eig_back<12>, grid, dim3(256), lds, s, mm, B2, B0, B1, wk->ev, H, ev, info); break;
        case 8: hipLaunchKernelGGL(k_eig_back<8>, grid, dim3(256), lds, s, mm, B2, B0, B1, wk->ev, H, ev, info); break;
        case 4: hipLaunchKernelGGL(k_eig_back<4>, grid, dim3(256), lds, s, mm, B2, B0, B1, wk->ev, H, ev, info); break;
        default: hipLaunchKernelGGL(k_eig_back<2>, grid, dim3(256), lds, s, mm, B2, B0, B1, wk->ev, H, ev, info); break;
        }
        m0 = m1;
    }
    return hipGetLastError();
}
