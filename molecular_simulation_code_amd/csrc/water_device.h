// The bonded terms of the rigid waters that the engine's constraint kernel evaluates itself.
#pragma once

#include "sofia_device.h"

namespace sofia {

struct ShakeArgs {
    const int32_t *atoms;
    const double *bond;
    const int4 *water;        // per cluster: bond types (O-H1, O-H2), angle type, fused flag
    const float4 *pos4;
    const double *xd, *vd, *fnb;
    long long *fix;
    const double4 *mtab;
    const int32_t *rep;
    const RepInfo *reps;
    const double *bond_k, *bond_r0, *angle_k, *angle_th0;
    int32_t n;
    double dt, dtsq, tol;
    int maxiter;
    int32_t *err;
};

// The two O-H bonds and the H-O-H angle of a rigid water (atoms idx = O, H1, H2), added to
// the atoms' fixed-point sums with the quanta the bond and angle kernels would add.
__device__ inline void water_bonded(const int4 w, const ShakeArgs &A, const int *idx, double box,
                                    double ibox, long long (*own)[3], long long &eb, long long &ea) {
    long long f[3], f1[3], f3[3];
    eb += bond_term(A.xd, A.n, idx[0], idx[1], box, ibox, A.bond_k[w.x - 1], A.bond_r0[w.x - 1], f);
#pragma unroll
    for (int c = 0; c < 3; ++c) { own[0][c] += f[c]; own[1][c] -= f[c]; }
    eb += bond_term(A.xd, A.n, idx[0], idx[2], box, ibox, A.bond_k[w.y - 1], A.bond_r0[w.y - 1], f);
#pragma unroll
    for (int c = 0; c < 3; ++c) { own[0][c] += f[c]; own[2][c] -= f[c]; }
    ea += angle_term(A.xd, A.n, idx[1], idx[0], idx[2], box, ibox, A.angle_k[w.z - 1],
                     A.angle_th0[w.z - 1], f1, f3);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        own[1][c] += f1[c];
        own[0][c] -= f1[c] + f3[c];
        own[2][c] += f3[c];
    }
}

// Cluster m's own terms added to its atoms' sums, their energies left to the closing force
// evaluation: for steps that run no SHAKE (the minimiser).
__device__ inline void water_terms(int32_t ns, const int32_t *num, const ShakeArgs &A, int m) {
    if (m >= ns || num[m] == 1 || num[m] == 3 || num[m] == 4 || A.water[m].w == 0) return;
    int idx[3];
    for (int k = 0; k < 3; ++k) idx[k] = A.atoms[4 * (size_t)m + k];
    const int rr = A.rep[idx[0]];
    long long own[3][3], eb = 0, ea = 0;
    for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 3; ++c) own[a][c] = A.fix[(size_t)c * A.n + idx[a]];
    water_bonded(A.water[m], A, idx, A.reps[rr].box, A.reps[rr].ibox, own, eb, ea);
    for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 3; ++c) A.fix[(size_t)c * A.n + idx[a]] = own[a][c];
}

ShakeArgs shake_args(sofia_ctx *c);

}  // namespace sofia
