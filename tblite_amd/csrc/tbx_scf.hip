// tbx_scf.hip -- SCF-loop consumers of the device-resident integrals of a
// batch (gfx950, FP64):
//
//   add_vao_to_h1                  scf/potential.f90:192-219
//   add_vmp_to_h1                  scf/potential.f90:221-255
//   get_mulliken_shell_charges     wavefunction/mulliken.f90:37-62
//   get_mulliken_atomic_multipoles wavefunction/mulliken.f90:65-98
//   updown_to_magnet               wavefunction/spin.f90 (applied to the sums)
//
// Dense arrays use the batch layout: element (r, c) of molecule m at
// mol_dense[m] + c * nao_m + r, components innermost for the multipole
// integrals (D: 3, Q: 6 per element), spin outermost with stride ndense.
// Every kernel is one pass over the dense blocks: HBM-bound.
#include <hip/hip_runtime.h>

#include "tbx_tables.h"

#define SCF_THREADS 256
#define SCF_TILE 32

struct ScfArgs {
    TbxMols mt;
    int nspin;
    long long dstride;   // spin stride of dense spin arrays (P, h1): ndense
    int mpdim, vdim;     // leading dimensions of the multipole integrals / potential
    int nmp;             // components used: min(mpdim, vdim) (add_vmp_to_h1) or mpdim
    const double *S;     // [ndense]
    const double *mp;    // [mpdim * ndense]
    const double *P;     // [ndense * nspin]
    const double *vao;   // [nao_tot * nspin]
    const double *vmp;   // [vdim * nat * nspin]
    const double *n0sh;  // [nsh_tot]
    double *h1;          // [ndense * nspin], accumulated into
    double *out;         // qsh [nsh_tot * nspin] or mpat [mpdim * nat * nspin]
};

// the first NMP components of an element; 16-byte loads when mpdim is even
// (every element then starts on a 16-byte boundary)
template <int NMP>
__device__ __forceinline__ void mp_load(const double *e, int mpdim, double x[NMP])
{
    if ((mpdim & 1) == 0) {
        const double2 *e2 = reinterpret_cast<const double2 *>(e);
#pragma unroll
        for (int q = 0; q + 1 < NMP; q += 2) {
            const double2 y = e2[q >> 1];
            x[q] = y.x;
            x[q + 1] = y.y;
        }
        if (NMP & 1) x[NMP - 1] = e[NMP - 1];
    } else {
#pragma unroll
        for (int q = 0; q < NMP; ++q) x[q] = e[q];
    }
}

template <int NMP>
__device__ __forceinline__ double mp_dot(const double *x, const double *v)
{
    double b = 0.0;
#pragma unroll
    for (int q = 0; q + 1 < NMP; q += 2) b += x[q] * v[q] + x[q + 1] * v[q + 1];
    if (NMP & 1) b += x[NMP - 1] * v[NMP - 1];
    return b;
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// Both spins of a call are served by one pass over the integrals: every
// kernel below is a template on the number of spins and reads S, D or Q once
// (a pass per spin read them twice, and the caches do not hold a batch).  Two
// spins, 256 molecules of 8..256 atoms (1.7e7 dense elements), us before and
// after: add_vao 155, 142; add_vmp with D 255, 217 and Q 349, 300; shell charges
// 122, 102; multipoles with D and Q together 650, 374 (about 4.5..5 TB/s of the
// bytes each needs, what a streaming copy reaches).

// add_vao_to_h1: h1(r, c, s) -= S(r, c) (vao(r, s) + vao(c, s)) / 2, one
// wavefront per column (global AO) of every molecule.
template <int NS>
__global__ void __launch_bounds__(SCF_THREADS) k_add_vao(ScfArgs A)
{
    const TbxMols &mt = A.mt;
    const int g = blockIdx.x * (SCF_THREADS / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int nao_tot = mt.nao_tot;
    if (g >= nao_tot) return;
    const int m = mt.at_mol[mt.ao_atom[g]];
    const int a0 = mt.mol_ao[m], n = mt.mol_nao[m];
    const long long col = mt.mol_dense[m] + (long long)(g - a0) * n;
    double vc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) vc[s] = A.vao[(long long)s * nao_tot + g];
    for (int r = lane; r < n; r += 64) {
        const double x = A.S[col + r] * 0.5;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double *h = A.h1 + s * A.dstride + col + r;
            *h -= x * (A.vao[(long long)s * nao_tot + a0 + r] + vc[s]);
        }
    }
}

// add_vmp_to_h1: h1(r, c, s) -= (B(r, c) + B(c, r)) / 2 with
// B(r, c) = sum_k mp(k, r, c) vmp(k, atom(c), s): the operator of mp sits on
// the column atom.  One workgroup per pair of 32 x 32 tiles (bi, bj), bi <= bj,
// and its transpose, so that both reads are coalesced; B goes through LDS.
// NMP = min(mpdim, vdim) components.
template <int NMP, int NS>
__global__ void __launch_bounds__(SCF_THREADS) k_add_vmp(ScfArgs A)
{
    constexpr int KS = SCF_TILE / (SCF_THREADS / SCF_TILE);  // columns per thread and tile
    __shared__ double B1[NS][SCF_TILE][SCF_TILE + 1];  // tile (bi, bj): [col][row]
    __shared__ double B2[NS][SCF_TILE][SCF_TILE + 1];  // tile (bj, bi): [col][row]
    __shared__ double vc[2][NS][SCF_TILE][NMP];  // potential of the column atoms of both tiles
    const TbxMols &mt = A.mt;
    const int4 tile = reinterpret_cast<const int4 *>(mt.tiles)[blockIdx.x];
    const int m = tile.x, bi = tile.y, bj = tile.z;
    const int n = mt.mol_nao[m], a0 = mt.mol_ao[m], nat = mt.nat;
    const long long dense0 = mt.mol_dense[m];
    const int rl = threadIdx.x & (SCF_TILE - 1), cl0 = threadIdx.x / SCF_TILE;
    const bool diag = bi == bj;
    const int r1 = bi * SCF_TILE + rl, r2 = bj * SCF_TILE + rl;
    if (threadIdx.x < 2 * SCF_TILE) {  // columns bj*32.. (tile 1) and bi*32.. (tile 2)
        const int t = threadIdx.x / SCF_TILE, cl = threadIdx.x % SCF_TILE;
        const int c = (t == 0 ? bj : bi) * SCF_TILE + cl;
        if (c < n) {
            const int at = mt.ao_atom[a0 + c];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const double *v = A.vmp + (long long)A.vdim * ((long long)s * nat + at);
#pragma unroll
                for (int q = 0; q < NMP; ++q) vc[t][s][cl][q] = v[q];
            }
        }
    }
    __syncthreads();
    double h1a[NS][KS], h1b[NS][KS];  // current h1 of the two tiles, loaded with the integrals
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const int cl = cl0 + k * (SCF_THREADS / SCF_TILE);
        const int c1 = bj * SCF_TILE + cl, c2 = bi * SCF_TILE + cl;
        double b1[NS], b2[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) b1[s] = b2[s] = h1a[s][k] = h1b[s][k] = 0.0;
        if (r1 < n && c1 < n) {
            const long long e = dense0 + (long long)c1 * n + r1;
            double x[NMP];
            mp_load<NMP>(A.mp + (long long)A.mpdim * e, A.mpdim, x);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                h1a[s][k] = A.h1[s * A.dstride + e];
                b1[s] = mp_dot<NMP>(x, vc[0][s][cl]);
            }
        }
        if (!diag && r2 < n && c2 < n) {
            const long long e = dense0 + (long long)c2 * n + r2;
            double x[NMP];
            mp_load<NMP>(A.mp + (long long)A.mpdim * e, A.mpdim, x);
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                h1b[s][k] = A.h1[s * A.dstride + e];
                b2[s] = mp_dot<NMP>(x, vc[1][s][cl]);
            }
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            B1[s][cl][rl] = b1[s];
            B2[s][cl][rl] = b2[s];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const int cl = cl0 + k * (SCF_THREADS / SCF_TILE);
        const int c1 = bj * SCF_TILE + cl, c2 = bi * SCF_TILE + cl;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double *h = A.h1 + s * A.dstride + dense0;
            if (r1 < n && c1 < n)
                h[(long long)c1 * n + r1] =
                    h1a[s][k] - 0.5 * (B1[s][cl][rl] + (diag ? B1[s][rl][cl] : B2[s][rl][cl]));
            if (!diag && r2 < n && c2 < n)
                h[(long long)c2 * n + r2] = h1b[s][k] - 0.5 * (B2[s][cl][rl] + B1[s][rl][cl]);
        }
    }
}

// get_mulliken_shell_charges: qsh(sh, s) = -sum_{c in sh} sum_r P(r, c, s)
// S(r, c), then updown_to_magnet and + n0sh.  One wavefront per shell.
template <int NS>
__global__ void __launch_bounds__(SCF_THREADS) k_mulliken_shell(ScfArgs A)
{
    const TbxMols &mt = A.mt;
    const int sh = blockIdx.x * (SCF_THREADS / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int nsh_tot = mt.nsh_tot;
    if (sh >= nsh_tot) return;
    const int g0 = mt.sh_aog[sh], g1 = mt.sh_aog[sh + 1];
    const int m = mt.at_mol[mt.ao_atom[g0]];
    const int a0 = mt.mol_ao[m], n = mt.mol_nao[m];
    // the shell's columns are one contiguous run of (g1 - g0) * n elements
    const long long e0 = mt.mol_dense[m] + (long long)(g0 - a0) * n;
    const int len = (g1 - g0) * n;
    double q[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) q[s] = 0.0;
    for (int k = lane; k < len; k += 64) {
        const double x = A.S[e0 + k];
#pragma unroll
        for (int s = 0; s < NS; ++s) q[s] += A.P[s * A.dstride + e0 + k] * x;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) q[s] = -wave_sum(q[s]);
    if (lane == 0) {
        if (NS == 2) {
            A.out[sh] = q[0] + q[NS - 1] + A.n0sh[sh];
            A.out[sh + nsh_tot] = q[0] - q[NS - 1];
        } else {
            A.out[sh] = q[0] + A.n0sh[sh];
        }
    }
}

// get_mulliken_atomic_multipoles: mpat(k, at, s) = -sum_{c in at} sum_r
// P(r, c, s) mp(k, r, c), then updown_to_magnet.  One wavefront per atom; NMP =
// mpdim components.
template <int NMP, int NS>
__global__ void __launch_bounds__(SCF_THREADS) k_mulliken_atom(ScfArgs A)
{
    const TbxMols &mt = A.mt;
    const int at = blockIdx.x * (SCF_THREADS / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (at >= mt.nat) return;
    const int m = mt.at_mol[at];
    const int a0 = mt.mol_ao[m], n = mt.mol_nao[m];
    const int g0 = a0 + mt.at_ao[at];
    const int g1 = (at + 1 < mt.nat && mt.at_mol[at + 1] == m) ? a0 + mt.at_ao[at + 1] : a0 + n;
    // the atom's columns are one contiguous run of (g1 - g0) * n elements
    const long long e0 = mt.mol_dense[m] + (long long)(g0 - a0) * n;
    const int len = (g1 - g0) * n;
    double q[NS][NMP];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int c = 0; c < NMP; ++c) q[s][c] = 0.0;
    for (int k = lane; k < len; k += 64) {
        double x[NMP];
        mp_load<NMP>(A.mp + (long long)NMP * (e0 + k), NMP, x);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const double pv = A.P[s * A.dstride + e0 + k];
#pragma unroll
            for (int c = 0; c < NMP; ++c) q[s][c] += pv * x[c];
        }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int c = 0; c < NMP; ++c) q[s][c] = -wave_sum(q[s][c]);
    if (lane < NMP) {
        double v0 = 0.0, v1 = 0.0;
#pragma unroll
        for (int k = 0; k < NMP; ++k)
            if (k == lane) {
                v0 = q[0][k];
                v1 = q[NS - 1][k];
            }
        const long long o = (long long)NMP * at + lane;
        if (NS == 2) {
            A.out[o] = v0 + v1;
            A.out[o + (long long)NMP * mt.nat] = v0 - v1;
        } else {
            A.out[o] = v0;
        }
    }
}

template <int NMP>
void launch_vmp(const ScfArgs &a, hipStream_t stream)
{
    const dim3 g(a.mt.ntile), t(SCF_THREADS);
    if (a.nspin == 2) hipLaunchKernelGGL((k_add_vmp<NMP, 2>), g, t, 0, stream, a);
    else hipLaunchKernelGGL((k_add_vmp<NMP, 1>), g, t, 0, stream, a);
}

template <int NMP>
void launch_mulliken_atom(const ScfArgs &a, hipStream_t stream)
{
    const int wpb = SCF_THREADS / 64;
    const dim3 g((a.mt.nat + wpb - 1) / wpb), t(SCF_THREADS);
    if (a.nspin == 2) hipLaunchKernelGGL((k_mulliken_atom<NMP, 2>), g, t, 0, stream, a);
    else hipLaunchKernelGGL((k_mulliken_atom<NMP, 1>), g, t, 0, stream, a);
}

extern "C" hipError_t tbx_launch_scf(int what, const TbxMols *mol, int nspin, long long dstride,
                                     int mpdim, int vdim, const double *S, const double *mp,
                                     const double *P, const double *vao, const double *vmp,
                                     const double *n0sh, double *h1, double *out,
                                     hipStream_t stream)
{
    ScfArgs a;
    a.mt = *mol;
    a.nspin = nspin;
    a.dstride = dstride;
    a.mpdim = mpdim;
    a.vdim = vdim;
    a.nmp = what == 1 ? (mpdim < vdim ? mpdim : vdim) : mpdim;
    a.S = S;
    a.mp = mp;
    a.P = P;
    a.vao = vao;
    a.vmp = vmp;
    a.n0sh = n0sh;
    a.h1 = h1;
    a.out = out;
    const int wpb = SCF_THREADS / 64;
    const dim3 t(SCF_THREADS);
    switch (what) {
    case 0:  // add_vao_to_h1
        if (mol->nao_tot > 0) {
            const dim3 g((mol->nao_tot + wpb - 1) / wpb);
            if (nspin == 2) hipLaunchKernelGGL(k_add_vao<2>, g, t, 0, stream, a);
            else hipLaunchKernelGGL(k_add_vao<1>, g, t, 0, stream, a);
        }
        break;
    case 1:  // add_vmp_to_h1
        if (mol->ntile > 0) {
            switch (a.nmp) {
            case 1: launch_vmp<1>(a, stream); break;
            case 2: launch_vmp<2>(a, stream); break;
            case 3: launch_vmp<3>(a, stream); break;
            case 4: launch_vmp<4>(a, stream); break;
            case 5: launch_vmp<5>(a, stream); break;
            default: launch_vmp<6>(a, stream); break;
            }
        }
        break;
    case 2:  // Mulliken shell charges
        if (mol->nsh_tot > 0) {
            const dim3 g((mol->nsh_tot + wpb - 1) / wpb);
            if (nspin == 2) hipLaunchKernelGGL(k_mulliken_shell<2>, g, t, 0, stream, a);
            else hipLaunchKernelGGL(k_mulliken_shell<1>, g, t, 0, stream, a);
        }
        break;
    case 3:  // Mulliken atomic multipoles
        if (mol->nat > 0) {
            switch (mpdim) {
            case 1: launch_mulliken_atom<1>(a, stream); break;
            case 2: launch_mulliken_atom<2>(a, stream); break;
            case 3: launch_mulliken_atom<3>(a, stream); break;
            case 4: launch_mulliken_atom<4>(a, stream); break;
            case 5: launch_mulliken_atom<5>(a, stream); break;
            default: launch_mulliken_atom<6>(a, stream); break;
            }
        }
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
