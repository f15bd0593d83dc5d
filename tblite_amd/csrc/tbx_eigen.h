// tbx_eigen.h -- interface of the batched generalized eigensolver
// (tbx_eigen.hip) to the host side (tbx_capi.hip).  Internal.
#pragma once
#include <hip/hip_runtime.h>

#define TBX_EIG_MAXN 1024  /* most orbitals: a 16-column strip of the matrix fits LDS */
#define TBX_TRD_TAIL 128   /* trailing columns of the tridiagonal form held in registers */
#define TBX_EIG_NONFINITE (-1) /* info: H holds an infinity or NaN, the results are NaN */
#define TBX_DC_LEAF 64     /* rows of a divide-and-conquer leaf */

// One molecule of a launch: its order, where its blocks are
struct EigMol {
    int n, mol;    // orbitals; index in the batch
    int a0;        // first orbital (vectors)
    int astride;   // length of a vector over the batch
    long long w0;  // first element in the workspace matrices
    long long d0;  // first element in the batch's dense arrays
};

// Workspace: four matrices of the molecules of a launch, vectors over the batch
struct EigWork {
    double *m[4];
    double *d, *e, *tau;  // tridiagonal form and the reflectors' factors
    double *p, *ev;       // two of each
    double *v[7], *anorm;
    int *iv[4];
    long long stride;     // = EigMol::astride
};
