// tbx_ncoord.hip -- gfx950 kernels of the GFN2 coordination number and of
// its chain rule into the nuclear gradient.
//
// cn(i) = sum_{j, T; 0 < r <= cutoff} f(r),  r = |R_i - R_j - T|,
// f(r) = 1/(1+exp(-ka (r0/r - 1))) * 1/(1+exp(-kb ((r0+rshift)/r - 1))),
// r0 = rcov(i) + rcov(j): the double-exponential counting function GFN2 uses
// (mctc-lib ncoord "dexp", created at xtb/gfn2.f90:640 and evaluated at
// xtb/singlepoint.f90:224).  The derivative kernel applies what the
// reference does with dcndr(3,nat,nat) and dcndL(3,3,nat) after
// get_hamiltonian_gradient (xtb/singlepoint.f90:375-378, two gemv calls),
// without forming either array:
//   dE/dR_i  += sum_{j,T} (dEdcn_i + dEdcn_j) f'(r) v / r,   v = R_i - R_j - T
//   sigma_m  += sum_{i in m} dEdcn_i sum_{j,T} f'(r) v v^T / r.
// One, two or four wavefronts per atom i; their lanes walk the atoms j of i's
// molecule and the molecule's translations.  Every sum over j is a reduction
// within the workgroup, so cn and dE/dR need no atomics; sigma is summed per
// molecule with FP64 atomics (nine per workgroup and molecule).
#include <hip/hip_runtime.h>

#include "tbx_tables.h"

namespace {

constexpr double kEpsR2 = 2.220446049250313e-16;

struct CnPar {
    const double *rcov;  // [nsp] covalent radii (bohr)
    double ka, kb, rshift, cutoff2;
};

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// Counting function of the pair vector v, r2 = |v|^2, and with GRAD its
// r-derivative over r.  One division gives 1/r; the two others are the factors'.
template <bool GRAD>
__device__ __forceinline__ void dexp_count(const CnPar &c, double r2, double r0, double &f,
                                           double &dfr)
{
    const double ir = 1.0 / sqrt(r2);
    const double a0 = r0, a1 = r0 + c.rshift;
    const double e1 = exp(-c.ka * (a0 * ir - 1.0)), e2 = exp(-c.kb * (a1 * ir - 1.0));
    const double s1 = 1.0 / (1.0 + e1), s2 = 1.0 / (1.0 + e2);
    f = s1 * s2;
    if (GRAD) {
        // d/dr 1/(1+exp(-k (a/r - 1))) = -k a e s^2 / r^2
        const double d1 = -c.ka * a0 * (e1 * s1) * s1, d2 = -c.kb * a1 * (e2 * s2) * s2;
        dfr = (d1 * s2 + s1 * d2) * (ir * ir * ir);
    }
}

// Sums of one atom i over the atoms j of its molecule and the translations,
// by W wavefronts: the pairs (T, j) are dealt to the lanes in one flat range.
// Molecules (one translation) take them as they come, nearly all lie within
// the cutoff.  With lattice images most do not: each wavefront queues those
// that do in LDS and takes them 64 at a time, so the exponentials run on full
// wavefronts.  One wavefront per atom and a loop over the translations left
// the lanes beyond the cell's atoms idle and ran the exponentials for each
// translation: 6 crystals of 6..96 atoms 127 us (cn) and 145 us (gradient), now
// 13 and 15; 1536 atoms 21 and 43 us, now 15 and 22.  W > 1 where an atom has
// enough pairs to share (tbx_launch_ncoord).
constexpr int QN = 128;  // queue entries per wavefront
struct Queue {
    double v[3][QN];
    int j[QN];
};

// sums: GRAD false: cn; true: dE/dR (3) and the strain sums (6)
template <bool GRAD, int W>
__device__ __forceinline__ void atom_sums(const TbxMols &mt, const CnPar &c, const double *xyz,
                                          const double *dEdcn, int i, int wv, Queue &q,
                                          double (&sum)[GRAD ? 9 : 1])
{
    const int lane = threadIdx.x & 63;
    const int m = mt.at_mol[i];
    const int a0 = mt.mol_atom[m], nj = mt.mol_atom[m + 1] - a0;
    const int2 tr = mt.mol_tr[m];
    const double xi = xyz[3 * i], yi = xyz[3 * i + 1], zi = xyz[3 * i + 2];
    const double ri = c.rcov[mt.at_sp[i]], ei = GRAD ? dEdcn[i] : 0.0;
    auto add = [&](double vx, double vy, double vz, int j) {
        double f, dfr;
        dexp_count<GRAD>(c, vx * vx + vy * vy + vz * vz, ri + c.rcov[mt.at_sp[j]], f, dfr);
        if (!GRAD) {
            sum[0] += f;
        } else {
            const double w = (ei + dEdcn[j]) * dfr, ws = ei * dfr;
            sum[0] += w * vx;
            sum[1] += w * vy;
            sum[2] += w * vz;
            const double sx = ws * vx, sy = ws * vy;
            sum[3] += sx * vx;  // xx xy yy xz yz zz
            sum[4] += sx * vy;
            sum[5] += sy * vy;
            sum[6] += sx * vz;
            sum[7] += sy * vz;
            sum[8] += ws * vz * vz;
        }
    };
    if (tr.y == 1) {
        const double tx = mt.trans[3 * tr.x], ty = mt.trans[3 * tr.x + 1],
                     tz = mt.trans[3 * tr.x + 2];
        for (int j = a0 + lane + 64 * wv; j < a0 + nj; j += 64 * W) {
            const double vx = xi - xyz[3 * j] - tx, vy = yi - xyz[3 * j + 1] - ty,
                         vz = zi - xyz[3 * j + 2] - tz;
            const double r2 = vx * vx + vy * vy + vz * vz;
            if (r2 < kEpsR2 || r2 > c.cutoff2) continue;
            add(vx, vy, vz, j);
        }
        return;
    }
    // (t, jj) of this lane, advanced by 64 W pairs a step
    const int st = 64 * W / nj, sj = 64 * W - st * nj, p0 = lane + 64 * wv;
    int t = p0 / nj, jj = p0 - t * nj, nq = 0;
    const long long steps = ((long long)nj * tr.y + 64 * W - 1) / (64 * W);
    for (long long s = 0; s < steps; ++s) {
        bool in = t < tr.y;
        double vx = 0.0, vy = 0.0, vz = 0.0;
        const int j = a0 + jj;
        if (in) {
            const double *T = mt.trans + 3 * (tr.x + t);
            vx = xi - xyz[3 * j] - T[0];
            vy = yi - xyz[3 * j + 1] - T[1];
            vz = zi - xyz[3 * j + 2] - T[2];
            const double r2 = vx * vx + vy * vy + vz * vz;
            in = !(r2 < kEpsR2 || r2 > c.cutoff2);
        }
        const unsigned long long mask = __ballot(in);
        if (in) {
            const int o = nq + __popcll(mask & ((1ull << lane) - 1ull));
            q.v[0][o] = vx;
            q.v[1][o] = vy;
            q.v[2][o] = vz;
            q.j[o] = j;
        }
        nq += __popcll(mask);
        __builtin_amdgcn_wave_barrier();
        if (nq >= 64) {  // the last 64 of the queue
            nq -= 64;
            add(q.v[0][nq + lane], q.v[1][nq + lane], q.v[2][nq + lane], q.j[nq + lane]);
        }
        __builtin_amdgcn_wave_barrier();
        t += st;
        jj += sj;
        if (jj >= nj) {
            jj -= nj;
            ++t;
        }
    }
    if (lane < nq) add(q.v[0][lane], q.v[1][lane], q.v[2][lane], q.j[lane]);
}

template <int W>
__global__ void __launch_bounds__(256) k_ncoord(TbxMols mt, CnPar c, const double *xyz,
                                                double *cn)
{
    __shared__ Queue q[4];
    __shared__ double part[4];
    const int i = W == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
    const int wv = W == 1 ? 0 : threadIdx.x >> 6;
    if (i >= mt.nat) return;  // whole atoms leave together
    double sum[1] = {0.0};
    atom_sums<false, W>(mt, c, xyz, nullptr, i, wv, q[threadIdx.x >> 6], sum);
    sum[0] = wave_sum(sum[0]);
    if (W > 1) {
        if ((threadIdx.x & 63) == 0) part[wv] = sum[0];
        __syncthreads();
        sum[0] = (part[0] + part[1]) + (part[2] + part[3]);
    }
    if ((threadIdx.x & 63) == 0 && wv == 0) cn[i] = sum[0];
}

// dE/dR (accumulated into grad) and sigma (accumulated, per molecule) from
// dE/dcn, A atoms of W wavefronts a workgroup.  The workgroup's atoms of one
// molecule add to its sigma together: nine atomics an atom to the same nine
// addresses were 10 of 29 us for 1536 atoms of one molecule, 11 of 25 us for 8
// clusters of 200 to 500 (now 14.6).
template <int W, int A>
__global__ void __launch_bounds__(64 * W * A) k_ncoord_grad(TbxMols mt, CnPar c, const double *xyz,
                                                            const double *dEdcn, double *grad,
                                                            double *sigma)
{
    __shared__ Queue q[W * A];
    __shared__ double part[W * A][9];
    __shared__ int mol[A];
    const int wave = threadIdx.x >> 6, slot = wave / W, i0 = blockIdx.x * A, i = i0 + slot;
    double sum[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (i < mt.nat) atom_sums<true, W>(mt, c, xyz, dEdcn, i, wave - slot * W, q[wave], sum);
#pragma unroll
    for (int k = 0; k < 9; ++k) sum[k] = wave_sum(sum[k]);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 9; ++k) part[wave][k] = sum[k];
        if (wave == slot * W) mol[slot] = i < mt.nat ? mt.at_mol[i] : -1;
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < 3 * A && i0 + t / 3 < mt.nat) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) v += part[t / 3 * W + w][t % 3];
        grad[3 * i0 + t] += v;
    }
    // sigma (3, 3) column-major from the packed symmetric sums, by the first
    // atom of each molecule
    if (t >= 64 && t < 64 + 9 * A) {
        const int a = (t - 64) / 9, e = (t - 64) % 9, m = mol[a];
        if (m >= 0 && (a == 0 || mol[a - 1] != m)) {
            const int r = e % 3, col = e / 3, lo = min(r, col), hi = max(r, col);
            const int k = 3 + hi * (hi + 1) / 2 + lo;  // xx xy yy xz yz zz
            double v = 0.0;
            for (int b = a; b < A && mol[b] == m; ++b)
#pragma unroll
                for (int w = 0; w < W; ++w) v += part[b * W + w][k];
            if (v != 0.0) unsafeAtomicAdd(&sigma[9 * m + e], v);
        }
    }
}

} // namespace

// Four wavefronts per atom from 384 pairs (atoms times translations) an atom
// on average, so that each has more than one step to share; one for the small
// molecules of a batch, where a step already covers the molecule.
static bool share_atoms(const TbxMols *mol) { return mol->atom_pairs >= 384; }

extern "C" hipError_t tbx_launch_ncoord(const TbxMols *mol, const double *rcov, double ka,
                                        double kb, double rshift, double cutoff,
                                        const double *xyz, double *cn, hipStream_t stream)
{
    if (mol->nat <= 0) return hipSuccess;
    const CnPar c{rcov, ka, kb, rshift, cutoff * cutoff};
    (void)hipGetLastError();
    if (share_atoms(mol))
        hipLaunchKernelGGL(k_ncoord<4>, dim3(mol->nat), dim3(256), 0, stream, *mol, c, xyz, cn);
    else
        hipLaunchKernelGGL(k_ncoord<1>, dim3((mol->nat + 3) / 4), dim3(256), 0, stream, *mol, c,
                           xyz, cn);
    return hipGetLastError();
}

extern "C" hipError_t tbx_launch_ncoord_grad(const TbxMols *mol, const double *rcov, double ka,
                                             double kb, double rshift, double cutoff,
                                             const double *xyz, const double *dEdcn,
                                             double *grad, double *sigma, hipStream_t stream)
{
    if (mol->nat <= 0) return hipSuccess;
    const CnPar c{rcov, ka, kb, rshift, cutoff * cutoff};
    (void)hipGetLastError();
    // From 1024 atoms with many pairs two atoms of two wavefronts fill the chip and
    // halve the atomics: 1536 atoms 21.8 us, one atom of four wavefronts 29.0, two
    // 22.7, four 28.5.  Below, one atom of four: 6 crystals of 6 to 96 atoms 15.1 us
    // (four atoms a workgroup 26).
    const unsigned nat = mol->nat;
    if (!share_atoms(mol))
        hipLaunchKernelGGL((k_ncoord_grad<1, 4>), dim3((nat + 3) / 4), dim3(256), 0, stream, *mol,
                           c, xyz, dEdcn, grad, sigma);
    else if (nat >= 1024)
        hipLaunchKernelGGL((k_ncoord_grad<2, 2>), dim3((nat + 1) / 2), dim3(256), 0, stream, *mol,
                           c, xyz, dEdcn, grad, sigma);
    else
        hipLaunchKernelGGL((k_ncoord_grad<4, 1>), dim3(nat), dim3(256), 0, stream, *mol, c, xyz,
                           dEdcn, grad, sigma);
    return hipGetLastError();
}
