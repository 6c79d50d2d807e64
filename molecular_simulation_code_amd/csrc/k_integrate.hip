// Integration, wrapping, Langevin and SHAKE kernels.
//
// Two flavours:
//  * drop-in ("32"): the reference's real*4 state (ainfo positions, coords velocities and
//    forces) with its FP64 temporaries -- nve_v/nve_x (Source/mod_ensemble.f90:11-87),
//    pbc (Source/mod_pbc.f90:6-39), shake (Source/mod_shake.f90:8-913),
//    langevin_debug_intel (Source/mod_langevin.f90:15-43);
//  * engine ("64"): the same algorithms on FP64 positions and velocities, with forces read
//    as FP64 nonbond sums + int64 fixed-point sums of every other term.
#include <type_traits>

#include "water_device.h"

namespace sofia {
namespace {

__global__ void k_zero(int32_t n3, long long *__restrict__ f, int32_t ne, long long *__restrict__ e) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n3) f[i] = 0;
    if (e && i < ne) e[i] = 0;
}

// What the force wrapper's terms start from: two force sums at zero, and the real*4 positions
// promoted to the FP64 copy that the bonded kernels read.
__global__ void k_start_forces(int32_t n, long long *__restrict__ a, long long *__restrict__ b,
                               const float4 *__restrict__ pos4, double *__restrict__ xd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos4[i];
    const float x[3] = {p.x, p.y, p.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        a[o] = 0;
        b[o] = 0;
        xd[o] = x[c];
    }
}

// The ESPREAD copies of every energy slot summed (16 lanes a slot) and the device's flags, all
// written to the host's page-locked words; the copies (and the solver's flags, whose engine
// form stays up until the lists are set up again, on request) are cleared on the way.
// A drop-in call used to copy the raw copies (26 KB) and each flag on their own.
struct ReportArgs {
    int32_t slots;
    long long *eacc;
    int32_t *shake_err, *shake_iters;
    const int32_t *maxcnt;
    HostWords *hw;
    long long *hw_e;
    bool clear_shake;
};
__device__ inline void report_words(const ReportArgs &A, int t) {
    static_assert(ESPREAD == 16, "one lane per copy");
    const int slot = t / ESPREAD;
    long long v = 0;
    if (slot < A.slots) {
        long long *p = &A.eacc[(size_t)t * ECOPY];
        v = *p;
        *p = 0;
    }
#pragma unroll
    for (int off = ESPREAD / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (slot < A.slots && t % ESPREAD == 0) A.hw_e[slot] = v;
    if (t == 0) {
        A.hw->shake_err = *A.shake_err;
        A.hw->shake_iters = *A.shake_iters;
        A.hw->maxcnt = *A.maxcnt;
        if (A.clear_shake) {
            *A.shake_err = 0;
            *A.shake_iters = 0;
        }
    }
}
__global__ void k_report(ReportArgs A) { report_words(A, blockIdx.x * blockDim.x + threadIdx.x); }

// x | y | z of src (and FIX_INV fix) as x, y, z rows; with gid, the row of an atom is its global
// id's place within its replica (ids a permutation of 1..natom).
__global__ void k_soa_to_aos(int32_t n, const double *__restrict__ src, const long long *__restrict__ fix,
                             const int32_t *__restrict__ gid, const int32_t *__restrict__ rep,
                             const RepInfo *__restrict__ reps, double *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t row = gid ? (size_t)(reps[rep[i]].atom0 + gid[i] - 1) : (size_t)i;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        // FIX_INV is a power of two: the product is exact, the sum the one k_nve_v64 forms
        dst[3 * row + c] = fix ? src[o] + (double)fix[o] * FIX_INV : src[o];
    }
}

__global__ void k_aos_to_soa(int32_t n, const double *__restrict__ src, double *__restrict__ dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) dst[(size_t)c * n + i] = src[3 * (size_t)i + c];
}

__global__ void k_fix_to_aos(int32_t n, const long long *__restrict__ f, float *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) out[3 * (size_t)i + c] = (float)((double)f[(size_t)c * n + i] * FIX_INV);
}

// ------------------------------------------------------------------ drop-in (real*4 state)
__global__ void k_nve_v32(int32_t n, float dt_partial, const float4 *__restrict__ pos4,
                          const double *__restrict__ mass, float *__restrict__ v,
                          const float *__restrict__ ff, const int32_t *__restrict__ rep,
                          double amu2e, long long *__restrict__ eacc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    double k = 0.0;
    int r = 0;
    if (live) {
        r = rep[i];
        const double m = mass[__float_as_int(pos4[i].w) - 1];
        const double dtm = (double)dt_partial / m;
        float vv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            vv[c] = (float)((double)v[3 * (size_t)i + c] + dtm * (double)ff[3 * (size_t)i + c]);
            v[3 * (size_t)i + c] = vv[c];
        }
        k = 0.5 * amu2e * m * (double)((vv[0] * vv[0] + vv[1] * vv[1]) + vv[2] * vv[2]);
    }
    wave_add(to_efix(k), live, r, eacc, E_KE);
}

__global__ void k_nve_x32(int32_t n, float dt, const float *__restrict__ v, float4 *__restrict__ pos4,
                          float *__restrict__ dr) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pos4[i];
    const float dx = dt * v[3 * (size_t)i], dy = dt * v[3 * (size_t)i + 1], dz = dt * v[3 * (size_t)i + 2];
    dr[i] += dx;
    dr[(size_t)n + i] += dy;
    dr[2 * (size_t)n + i] += dz;
    p.x += dx;
    p.y += dy;
    p.z += dz;
    pos4[i] = p;
}

// while-loop wrap into (0, box]; bounded so a non-finite coordinate cannot spin forever
__device__ inline float wrap32(float x, float box) {
    for (int it = 0; it < 64 && x > box; ++it) x = x - box;
    for (int it = 0; it < 64 && (double)x <= 0.0; ++it) x = x + box;
    return x;
}

__global__ void k_pbc32(int32_t n, float4 *__restrict__ pos4, const int32_t *__restrict__ rep,
                        const RepInfo *__restrict__ reps) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float box = reps[rep[i]].box;
    float4 p = pos4[i];
    p.x = wrap32(p.x, box);
    p.y = wrap32(p.y, box);
    p.z = wrap32(p.z, box);
    pos4[i] = p;
}

// berendsen, Source/mod_ensemble.f90:167-205: position = position*mu (real*4 * real*8, stored
// real*4); dx = new - dble(old); drx = drx + dx (real*8 sum stored real*4).
__global__ void k_berendsen32(int32_t n, float4 *__restrict__ pos4, float *__restrict__ dr,
                              const int32_t *__restrict__ rep, const double *__restrict__ mu) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = mu[rep[i]];
    float4 p = pos4[i];
    float *c[3] = {&p.x, &p.y, &p.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double old = (double)*c[d];
        const float nw = (float)(old * m);
        *c[d] = nw;
        float *r = dr + (size_t)d * n + i;
        *r = (float)((double)*r + ((double)nw - old));
    }
    pos4[i] = p;
}

__global__ void k_langevin32(int32_t n, const float4 *__restrict__ pos4, const float *__restrict__ v,
                             const int32_t *__restrict__ gid, const double *__restrict__ mass,
                             float fric, float gconst, uint64_t seed, uint64_t step,
                             float *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = mass[__float_as_int(pos4[i].w) - 1];
    const double g1 = -(double)fric * m, g2 = (double)gconst * sqrt(m);
    float u[3];
    uniform3(seed, step, (uint32_t)gid[i], u);
#pragma unroll
    for (int c = 0; c < 3; ++c)
        out[3 * (size_t)i + c] = (float)(g1 * (double)v[3 * (size_t)i + c] + g2 * (double)u[c]);
}

// ------------------------------------------------------------------ SHAKE
// Constraint k joins atoms (P[k], Q[k]) of the cluster: shake2 one bond, shake3 (0,1),(0,2),
// shake4 (0,1),(0,2),(0,3), shake3angle (0,1),(0,2),(1,2).  The Lagrange multipliers solve
// |s_k + sum_l cpl[k][l] lambda_l r_l|^2 = d_k^2 by the reference's iteration: linear
// system with the quadratic terms lagged, stopped when every |delta lambda| <= tol.
// The solver is instantiated per cluster kind, so that the constraint topology is known at
// compile time and the arrays stay in registers.  Cluster atoms are exclusive to their cluster.
template <int KIND> __device__ constexpr int topo_nc() { return KIND == 1 ? 1 : (KIND == 3 ? 2 : 3); }
template <int KIND> __device__ constexpr int topo_na() { return KIND == 1 ? 2 : (KIND == 4 ? 4 : 3); }
template <int KIND> __device__ constexpr int topo_p(int k) { return (KIND == -3 && k == 2) ? 1 : 0; }
template <int KIND> __device__ constexpr int topo_q(int k) { return (KIND == -3 && k == 2) ? 2 : k + 1; }

template <int KIND>
__device__ inline bool shake_solve_t(const double *im, const double *bl, const double (*r)[3],
                                     const double (*s)[3], double tol, int maxiter, double *lam,
                                     int *iters) {
    constexpr int NC = topo_nc<KIND>();
    if constexpr (NC == 1) {   // closed-form root of the quadratic (Source/mod_shake.f90:133-168)
        const double r01sq = r[0][0] * r[0][0] + r[0][1] * r[0][1] + r[0][2] * r[0][2];
        const double s01sq = s[0][0] * s[0][0] + s[0][1] * s[0][1] + s[0][2] * s[0][2];
        const double ims = im[0] + im[1];
        const double a = ims * ims * r01sq;
        const double b = 2.0 * ims * (s[0][0] * r[0][0] + s[0][1] * r[0][1] + s[0][2] * r[0][2]);
        const double cc = s01sq - bl[0] * bl[0];
        const double det = b * b - 4.0 * a * cc;
        if (det < 0.0) return false;
        const double l1 = (-b + sqrt(det)) / (2.0 * a), l2 = (-b - sqrt(det)) / (2.0 * a);
        lam[0] = (fabs(l1) <= fabs(l2)) ? l1 : l2;
        *iters = 1;
        return true;
    } else {
        double cpl[NC][NC], A[NC][NC], G[NC][NC], ssq[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            ssq[k] = s[k][0] * s[k][0] + s[k][1] * s[k][1] + s[k][2] * s[k][2];
#pragma unroll
            for (int l = 0; l < NC; ++l) {
                double c = 0.0;
                if (topo_p<KIND>(k) == topo_p<KIND>(l)) c += im[topo_p<KIND>(k)];
                if (topo_p<KIND>(k) == topo_q<KIND>(l)) c -= im[topo_p<KIND>(k)];
                if (topo_q<KIND>(k) == topo_p<KIND>(l)) c -= im[topo_q<KIND>(k)];
                if (topo_q<KIND>(k) == topo_q<KIND>(l)) c += im[topo_q<KIND>(k)];
                cpl[k][l] = c;
                A[k][l] = 2.0 * c * (s[k][0] * r[l][0] + s[k][1] * r[l][1] + s[k][2] * r[l][2]);
                G[k][l] = r[k][0] * r[l][0] + r[k][1] * r[l][1] + r[k][2] * r[l][2];
            }
        }
        double Ai[NC][NC];
        if constexpr (NC == 2) {
            const double det = A[0][0] * A[1][1] - A[0][1] * A[1][0];
            if (det == 0.0) return false;
            const double di = 1.0 / det;
            Ai[0][0] = A[1][1] * di; Ai[0][1] = -A[0][1] * di;
            Ai[1][0] = -A[1][0] * di; Ai[1][1] = A[0][0] * di;
        } else {
            const double det = A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0] +
                               A[0][2] * A[1][0] * A[2][1] - A[0][0] * A[1][2] * A[2][1] -
                               A[0][1] * A[1][0] * A[2][2] - A[0][2] * A[1][1] * A[2][0];
            if (det == 0.0) return false;
            const double di = 1.0 / det;
            Ai[0][0] = di * (A[1][1] * A[2][2] - A[1][2] * A[2][1]);
            Ai[0][1] = -di * (A[0][1] * A[2][2] - A[0][2] * A[2][1]);
            Ai[0][2] = di * (A[0][1] * A[1][2] - A[0][2] * A[1][1]);
            Ai[1][0] = -di * (A[1][0] * A[2][2] - A[1][2] * A[2][0]);
            Ai[1][1] = di * (A[0][0] * A[2][2] - A[0][2] * A[2][0]);
            Ai[1][2] = -di * (A[0][0] * A[1][2] - A[0][2] * A[1][0]);
            Ai[2][0] = di * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
            Ai[2][1] = -di * (A[0][0] * A[2][1] - A[0][1] * A[2][0]);
            Ai[2][2] = di * (A[0][0] * A[1][1] - A[0][1] * A[1][0]);
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) lam[k] = 0.0;
        int it = 0;
        bool done = false;
        while (!done && it < maxiter) {
            double bb[NC], nl[NC];
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                double qd = 0.0;
#pragma unroll
                for (int l = 0; l < NC; ++l)
#pragma unroll
                    for (int m = 0; m < NC; ++m) qd += cpl[k][l] * cpl[k][m] * G[l][m] * lam[l] * lam[m];
                bb[k] = bl[k] * bl[k] - ssq[k] - qd;
            }
            done = true;
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                double v = 0.0;
#pragma unroll
                for (int l = 0; l < NC; ++l) v += Ai[k][l] * bb[l];
                nl[k] = v;
            }
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                if (fabs(nl[k] - lam[k]) > tol) done = false;
                lam[k] = nl[k];
            }
            ++it;
        }
        *iters = it;
        return true;
    }
}

// One cluster of the drop-in SHAKE.  Returns the iterations, or -1 where the system has no
// solution; adds to the virial.
template <int KIND>
__device__ inline int shake32_cluster(const int4 at, const double *__restrict__ bond,
                                      const float4 *__restrict__ pos4, const float *__restrict__ v,
                                      float *__restrict__ ff, const double4 *__restrict__ mtab,
                                      float box, float ibox, float dt, double dtsq, double tol,
                                      int maxiter, double vir[3]) {
    constexpr int NA = topo_na<KIND>(), NC = topo_nc<KIND>();
    const int all[4] = {at.x, at.y, at.z, at.w};
    double im[NA], bl[3], xs[NA][3];
    float pp[NA][3], f[NA][3];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        const size_t i = (size_t)all[a];
        const float4 p = pos4[i];
        im[a] = mtab[__float_as_int(p.w) - 1].w;
        pp[a][0] = p.x; pp[a][1] = p.y; pp[a][2] = p.z;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            f[a][c] = ff[3 * i + c];
            xs[a][c] = (double)(pp[a][c] + dt * v[3 * i + c]) + dtsq * im[a] * (double)f[a][c];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) bl[k] = bond[k];
    double r[NC][3], s[NC][3], lam[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int a = topo_p<KIND>(k), b = topo_q<KIND>(k);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double d = (double)(pp[a][c] - pp[b][c]);
            r[k][c] = d - (double)(box * (float)(int)round((double)ibox * d));
            const double e = xs[a][c] - xs[b][c];
            s[k][c] = e - (double)(box * (float)(int)round((double)ibox * e));
        }
    }
    int its = 0;
    if (!shake_solve_t<KIND>(im, bl, r, s, tol, maxiter, lam, &its)) return -1;
    // the force is real*4 after every constraint, as in the reference
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const double l = lam[k] / dtsq;
        const int a = topo_p<KIND>(k), b = topo_q<KIND>(k);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            f[a][c] = (float)((double)f[a][c] + l * r[k][c]);
            f[b][c] = (float)((double)f[b][c] - l * r[k][c]);
            vir[c] += r[k][c] * r[k][c] * l;
        }
    }
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) ff[3 * (size_t)all[a] + c] = f[a][c];
    return its;
}

// drop-in: real*4 positions/velocities/forces, FP64 solve (Source/mod_shake.f90:8-85, 888-913).
// Few wavefronts (one per SIMD at 204,000 atoms) walk a chain of FP64 steps, so the time is that
// chain's: with the solver's arrays indexed by the cluster's kind at run time, in scratch, it
// took 54 us at 13,500 atoms and 83 at 204,000; with one instance per kind and one iteration
// count per wavefront 10 and 21.
__global__ void __launch_bounds__(64)
k_shake32(int32_t ns, const int32_t *__restrict__ num, const int4 *__restrict__ atoms,
          const double *__restrict__ bond, const float4 *__restrict__ pos4,
          const float *__restrict__ v, float *__restrict__ ff, const double4 *__restrict__ mtab,
          const int32_t *__restrict__ rep, const RepInfo *__restrict__ reps, float dt, double dtsq,
          double tol, int maxiter, int32_t *__restrict__ err, int32_t *__restrict__ iters_max,
          long long *__restrict__ eacc) {
    const int m = blockIdx.x * 64 + threadIdx.x;
    const bool live = m < ns;
    double vir[3] = {0.0, 0.0, 0.0};
    int rr = 0, its = 0;
    if (live) {
        const int kind = num[m];
        const int4 at = atoms[m];
        rr = rep[at.x];
        const float box = reps[rr].box, ibox = reps[rr].ibox;
        auto solve = [&](auto k) {
            its = shake32_cluster<decltype(k)::value>(at, bond + 3 * (size_t)m, pos4, v, ff, mtab, box,
                                                      ibox, dt, dtsq, tol, maxiter, vir);
        };
        if (kind == 1) solve(std::integral_constant<int, 1>{});
        else if (kind == 3) solve(std::integral_constant<int, 3>{});
        else if (kind == 4) solve(std::integral_constant<int, 4>{});
        else solve(std::integral_constant<int, -3>{});   // rigid triangle
        if (its < 0) atomicOr(err, 1);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) its = max(its, __shfl_xor(its, off, 64));
    if (threadIdx.x == 0 && its > 0) atomicMax(iters_max, its);
    wave_add(to_efix(vir[0]), live, rr, eacc, V_X);
    wave_add(to_efix(vir[1]), live, rr, eacc, V_Y);
    wave_add(to_efix(vir[2]), live, rr, eacc, V_Z);
}

// ------------------------------------------------------------------ engine (FP64 state)
__global__ void k_from32(int32_t n, const float4 *__restrict__ pos4, const float *__restrict__ v32,
                         double *__restrict__ xd, double *__restrict__ vd, double *__restrict__ drd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos4[i];
    xd[i] = p.x; xd[(size_t)n + i] = p.y; xd[2 * (size_t)n + i] = p.z;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        vd[(size_t)c * n + i] = v32[3 * (size_t)i + c];
        drd[(size_t)c * n + i] = 0.0;
    }
}

__global__ void k_to32(int32_t n, const double *__restrict__ xd, const double *__restrict__ vd,
                       float4 *__restrict__ pos4, float *__restrict__ v32) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pos4[i];
    p.x = (float)xd[i]; p.y = (float)xd[(size_t)n + i]; p.z = (float)xd[2 * (size_t)n + i];
    pos4[i] = p;
#pragma unroll
    for (int c = 0; c < 3; ++c) v32[3 * (size_t)i + c] = (float)vd[(size_t)c * n + i];
}

// v += (dt/2 kcal2amu / m) F with F = nonbond + fixed-point rest; optional kinetic energy
__global__ void k_nve_v64(int32_t n, double dthalf, const float4 *__restrict__ pos4,
                          const double *__restrict__ mass, double *__restrict__ vd,
                          const double *__restrict__ fnb, const long long *__restrict__ fix,
                          const int32_t *__restrict__ rep, double amu2e, int ke,
                          long long *__restrict__ eacc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    double k = 0.0;
    int r = 0;
    if (live) {
        r = rep[i];
        const double m = mass[__float_as_int(pos4[i].w) - 1];
        const double dtm = dthalf / m;
        double v2 = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const size_t o = (size_t)c * n + i;
            const double f = fnb[o] + (double)fix[o] * FIX_INV;
            const double vv = vd[o] + dtm * f;
            vd[o] = vv;
            v2 += vv * vv;
        }
        k = 0.5 * amu2e * m * v2;
    }
    if (ke) wave_add(to_efix(k), live, r, eacc, E_KE);
}

__device__ inline double wrap64(double x, double box) {
    for (int it = 0; it < 64 && x > box; ++it) x -= box;
    for (int it = 0; it < 64 && x <= 0.0; ++it) x += box;
    return x;
}

// Where an integration launch leaves what the rest of the step starts from: the rebuild flags
// (an atom displaced by half the usable skin flags its replica; the first to do so raises
// `any`), the fixed-point force sum (zero, or the Langevin term) and the mixed pair kernel's
// position record (pf; q as in write_record).
struct StepOut {
    int32_t *rebuild, *any;
    long long *fix;
    int4 *pf;
    const float *q;
};

__device__ inline void flag_rebuild(const StepOut &O, int r, const double dr[3], double chk2) {
    if ((dr[0] * dr[0] + dr[1] * dr[1]) + dr[2] * dr[2] >= chk2 && atomicOr(&O.rebuild[r], 1) == 0)
        atomicOr(O.any, 1);
}

// Everything between two force evaluations that one atom can do alone, in one pass over the
// state: the previous step's second half kick (KICK2; the first step of a segment has none
// left), this step's first half kick, the drift (wrapped into (0, box], the float4 copy
// refreshed), the rebuild check, the Langevin force at the half-step velocity as the force
// sum's first term, and the pair kernel's record.  These were seven launches of 1.5 to 4.5 us, a
// quarter of a 5,000-atom step (138 us); the one takes 4.3 us there, 12.5 at 204,000 atoms (HBM).
template <bool KICK2>
__global__ void __launch_bounds__(256)
k_advance(int32_t n, double dt, const double4 *__restrict__ mtab, double *__restrict__ xd,
          double *__restrict__ vd, double *__restrict__ drd, float4 *__restrict__ pos4,
          const double *__restrict__ fnb, const int32_t *__restrict__ gid,
          const int32_t *__restrict__ rep, const RepInfo *__restrict__ reps,
          const uint64_t *__restrict__ step, int thermostat, StepOut O) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = rep[i];
    const RepInfo &R = reps[r];
    const double box = R.box;
    float4 p = pos4[i];
    const uint32_t type = (uint32_t)__float_as_int(p.w);
    const double4 mt = mtab[type - 1];
    double v[3], x[3], dr[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        const double f = fnb[o] + (double)O.fix[o] * FIX_INV;
        v[c] = vd[o];
        if (KICK2) v[c] += mt.y * f;
        v[c] += mt.y * f;
        vd[o] = v[c];
        const double d = dt * v[c];
        dr[c] = drd[o] + d;
        drd[o] = dr[c];
        x[c] = wrap64(xd[o] + d, box);
        xd[o] = x[c];
    }
    p.x = (float)x[0]; p.y = (float)x[1]; p.z = (float)x[2];
    pos4[i] = p;
    flag_rebuild(O, r, dr, R.chk2);
    long long q[3] = {0, 0, 0};
    if (thermostat && !(R.fric == 0.0 && R.gconst == 0.0)) {
        float u[3];
        uniform3(R.seed, step[r], (uint32_t)gid[i], u);
#pragma unroll
        for (int c = 0; c < 3; ++c) q[c] = to_fix(-R.fric * mt.x * v[c] + R.gconst * mt.z * (double)u[c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) O.fix[(size_t)c * n + i] = q[c];
    if (O.pf) write_record(O.pf, i, x[0], x[1], x[2], R.fscale, type, O.q);
}

// Langevin force -fric m v + gconst sqrt(m) U(-1/2,1/2) added to the fixed-point sum
__global__ void k_langevin64(int32_t n, const float4 *__restrict__ pos4, const double *__restrict__ vd,
                             const int32_t *__restrict__ gid, const int32_t *__restrict__ rep,
                             const RepInfo *__restrict__ reps, const double *__restrict__ mass,
                             const uint64_t *__restrict__ step, long long *__restrict__ fix) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const RepInfo &R = reps[rep[i]];
    if (R.fric == 0.0 && R.gconst == 0.0) return;
    const double m = mass[__float_as_int(pos4[i].w) - 1];
    float u[3];
    uniform3(R.seed, step[rep[i]], (uint32_t)gid[i], u);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        fix[o] += to_fix(-R.fric * m * vd[o] + R.gconst * sqrt(m) * (double)u[c]);
    }
}

// One cluster of kind KIND.  A fused rigid water (KIND -3, water flag set) also evaluates its
// two O-H bonds and its H-O-H angle here -- with the same fixed-point quanta the bond and
// angle kernels would add -- and owns its three atoms, so it writes their force sums without
// atomics.  Returns the cluster's replica; adds to the virial and energy partial sums.
template <int KIND>
__device__ inline int shake_cluster(int m, const ShakeArgs &A, double vir[3], long long &eb,
                                    long long &ea) {
    constexpr int NA = topo_na<KIND>(), NC = topo_nc<KIND>();
    int idx[NA];
    double im[NA], bl[3];
#pragma unroll
    for (int k = 0; k < NA; ++k) {
        idx[k] = A.atoms[4 * (size_t)m + k];
        im[k] = A.mtab[__float_as_int(A.pos4[idx[k]].w) - 1].w;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) bl[k] = A.bond[3 * (size_t)m + k];
    const int rr = A.rep[idx[0]];
    const double box = A.reps[rr].box, ibox = A.reps[rr].ibox;
    const int n = A.n;
    long long own[NA][3];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) own[a][c] = A.fix[(size_t)c * n + idx[a]];
    bool fused = false;
    if constexpr (KIND == -3) {
        const int4 w = A.water[m];
        fused = w.w != 0;
        if (fused) water_bonded(w, A, idx, box, ibox, own, eb, ea);
    }
    double xs[NA][3];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const size_t o = (size_t)c * n + idx[a];
            const double f = A.fnb[o] + (double)own[a][c] * FIX_INV;
            xs[a][c] = A.xd[o] + A.dt * A.vd[o] + A.dtsq * im[a] * f;
        }
    double r[NC][3], s[NC][3];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int pa = topo_p<KIND>(k), qa = topo_q<KIND>(k);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double d = A.xd[(size_t)c * n + idx[pa]] - A.xd[(size_t)c * n + idx[qa]];
            r[k][c] = d - box * rint(d * ibox);
            const double e = xs[pa][c] - xs[qa][c];
            s[k][c] = e - box * rint(e * ibox);
        }
    }
    double lam[NC];
    int its = 0;
    if (!shake_solve_t<KIND>(im, bl, r, s, A.tol, A.maxiter, lam, &its)) {
        atomicOr(A.err, 1);
        return rr;
    }
    long long add[NA][3];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) add[a][c] = 0;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const double l = lam[k] / A.dtsq;
        const int pa = topo_p<KIND>(k), qa = topo_q<KIND>(k);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const long long q = to_fix(l * r[k][c]);
            add[pa][c] += q;
            add[qa][c] -= q;
            vir[c] += r[k][c] * r[k][c] * l;
        }
    }
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            long long *p = &A.fix[(size_t)c * n + idx[a]];
            if (fused) *p = own[a][c] + add[a][c];
            else atomicAdd((unsigned long long *)p, (unsigned long long)add[a][c]);
        }
    return rr;
}

// Rigid symmetric 3-site water (a -3 cluster with |O-H1| = |O-H2| and equal H masses) by
// SETTLE (Miyamoto & Kollman, J. Comput. Chem. 13, 952, 1992): the closed-form solution of
// the constraint equations that the iterative triangle SHAKE converges to.  Positions are
// taken relative to the old O with the minimum image; the constraint force of an atom is
// m (x_settled - x_unconstrained) / dtsq, the O force is minus the sum of the H forces in
// fixed point (exact momentum), and the virial is sum_k lambda_k r_k^2, written through the
// H forces and the old O-H vectors.  The fused water bond/angle terms are evaluated first,
// as in shake_cluster<-3>.
__device__ inline int settle_water(int m, const ShakeArgs &A, double vir[3], long long &eb,
                                   long long &ea) {
    int rr;
    {
        int idx[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) idx[k] = A.atoms[4 * (size_t)m + k];
        const double4 to4 = A.mtab[__float_as_int(A.pos4[idx[0]].w) - 1];
        const double4 th4 = A.mtab[__float_as_int(A.pos4[idx[1]].w) - 1];
        const double mo = to4.x, mh = th4.x;
        const double doh = A.bond[3 * (size_t)m], dhh = A.bond[3 * (size_t)m + 2];
        rr = A.rep[idx[0]];
        const double box = A.reps[rr].box, ibox = A.reps[rr].ibox;
        const int n = A.n;
        long long own[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c) own[a][c] = A.fix[(size_t)c * n + idx[a]];
        const int4 w = A.water[m];
        const bool fused = w.w != 0;
        if (fused) water_bonded(w, A, idx, box, ibox, own, eb, ea);
        // old (b0, c0) and unconstrained new (x1) positions relative to the old O
        const double im[3] = {to4.w, th4.w, th4.w};
        double b0[3], c0[3], x1[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const size_t oo = (size_t)c * n + idx[0];
            const double xo = A.xd[oo];
            double d = A.xd[(size_t)c * n + idx[1]] - xo;
            b0[c] = d - box * rint(d * ibox);
            d = A.xd[(size_t)c * n + idx[2]] - xo;
            c0[c] = d - box * rint(d * ibox);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const size_t o = (size_t)c * n + idx[a];
                const double f = A.fnb[o] + (double)own[a][c] * FIX_INV;
                const double step = A.dt * A.vd[o] + A.dtsq * im[a] * f;
                const double base = a == 0 ? 0.0 : (a == 1 ? b0[c] : c0[c]);
                x1[a][c] = base + step;
            }
        }
        // canonical triangle: O at ra above the centre of mass, the H-H midpoint rb below
        const double wt = mo + 2.0 * mh, rc = 0.5 * dhh;
        const double hgt = sqrt(doh * doh - rc * rc);
        const double ra = 2.0 * mh * hgt / wt, rb = hgt - ra;
        double com[3], a1[3], b1[3], c1[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            com[c] = (mo * x1[0][c] + mh * (x1[1][c] + x1[2][c])) / wt;
            a1[c] = x1[0][c] - com[c];
            b1[c] = x1[1][c] - com[c];
            c1[c] = x1[2][c] - com[c];
        }
        auto cross = [](const double *u, const double *v, double *o) {
            o[0] = u[1] * v[2] - u[2] * v[1];
            o[1] = u[2] * v[0] - u[0] * v[2];
            o[2] = u[0] * v[1] - u[1] * v[0];
        };
        double T[3][3];   // rows: the frame axes x', y', z'
        cross(b0, c0, T[2]);
        cross(a1, T[2], T[0]);
        cross(T[2], T[0], T[1]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double inv = 1.0 / sqrt(T[k][0] * T[k][0] + T[k][1] * T[k][1] + T[k][2] * T[k][2]);
            T[k][0] *= inv; T[k][1] *= inv; T[k][2] *= inv;
        }
        auto to = [&](const double *v, int k) { return T[k][0] * v[0] + T[k][1] * v[1] + T[k][2] * v[2]; };
        const double xb0 = to(b0, 0), yb0 = to(b0, 1), xc0 = to(c0, 0), yc0 = to(c0, 1);
        const double za1 = to(a1, 2);
        const double xb1 = to(b1, 0), yb1 = to(b1, 1), zb1 = to(b1, 2);
        const double xc1 = to(c1, 0), yc1 = to(c1, 1), zc1 = to(c1, 2);
        // The closed form exists only while the unconstrained step leaves the water within
        // reach of the rigid triangle: each radicand below must be non-negative (and every
        // value finite).  Otherwise the step is rejected as a failed constraint solve, as the
        // iterative solver rejects a singular one, instead of writing NaN into the state.
        const double sinphi = za1 / ra;
        const double rad_phi = 1.0 - sinphi * sinphi;
        const double cosphi = sqrt(fmax(rad_phi, 0.0));
        const double sinpsi = (zb1 - zc1) / (2.0 * rc * cosphi);
        const double rad_psi = 1.0 - sinpsi * sinpsi;
        const double cospsi = sqrt(fmax(rad_psi, 0.0));
        const double ya2 = ra * cosphi, xb2 = -rc * cospsi;
        const double t1 = -rb * cosphi, t2 = rc * sinpsi * sinphi;
        const double yb2 = t1 - t2, yc2 = t1 + t2;
        const double alpha = xb2 * (xb0 - xc0) + yb0 * yb2 + yc0 * yc2;
        const double beta = xb2 * (yc0 - yb0) + xb0 * yb2 + xc0 * yc2;
        const double gamma = xb0 * yb1 - xb1 * yb0 + xc0 * yc1 - xc1 * yc0;
        const double ab = alpha * alpha + beta * beta;
        const double rad_ab = ab - gamma * gamma;
        const double sint = (alpha * gamma - beta * sqrt(fmax(rad_ab, 0.0))) / ab;
        const double rad_t = 1.0 - sint * sint;
        // written so that a NaN in any operand also fails
        if (!(rad_phi >= 0.0 && cosphi > 0.0 && rad_psi >= 0.0 && ab > 0.0 && rad_ab >= 0.0 &&
              rad_t >= 0.0)) {
            atomicOr(A.err, 1);
            return rr;
        }
        const double cost = sqrt(rad_t);
        const double p3[3][3] = {{-ya2 * sint, ya2 * cost, za1},
                                 {xb2 * cost - yb2 * sint, xb2 * sint + yb2 * cost, zb1},
                                 {-xb2 * cost - yc2 * sint, -xb2 * sint + yc2 * cost, zc1}};
        const double ms[3] = {mo, mh, mh};
        long long add[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            long long sum_h = 0;
#pragma unroll
            for (int a = 1; a < 3; ++a) {
                const double xnew = T[0][c] * p3[a][0] + T[1][c] * p3[a][1] + T[2][c] * p3[a][2] + com[c];
                const double f = ms[a] * (xnew - x1[a][c]) / A.dtsq;
                add[a][c] = to_fix(f);
                sum_h += add[a][c];
                vir[c] += (a == 1 ? b0[c] : c0[c]) * f;
            }
            add[0][c] = -sum_h;
        }
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                long long *p = &A.fix[(size_t)c * n + idx[a]];
                if (fused) *p = own[a][c] + add[a][c];
                else atomicAdd((unsigned long long *)p, (unsigned long long)add[a][c]);
            }
    }
    return rr;
}

// All engine constraints in one launch.  The first nb_it blocks run the iteratively solved
// clusters of kidx (kinds 1, 3, 4, -3 in that order, each kind padded with -1 to whole
// wavefronts; e1..e4 are the ends of the groups), so that a wavefront runs a single solver.
// Each wavefront of the other blocks owns WSPAN consecutive atoms in their current
// (cell-sorted) order: it queues the SETTLE waters whose oxygen lies there in LDS and solves
// them 64 at a time, so its waters come from a few neighbouring cells and share cache lines.
//
// Bound by the latency of one solve (dependent gathers, FP64 divisions and square roots), not
// by throughput, so the split aims at one solve per wavefront and many wavefronts: 160 atoms
// hold about 53 waters (rarely more than the 64 of one round), where 512 atoms took three
// rounds one after the other.  The energy and virial sums (ten 64-bit wave reductions and
// five atomics) run on energy launches only.
constexpr int WSPAN = 160;

// The end of an engine step, done by one extra workgroup of the constraint launch (the last of
// the step): rebuilt replicas counted, every flag down, the step counters on by one.
struct StepEnd {
    int32_t nrep;          // 0: nothing to end
    int32_t *rebuild, *nbuilds;
    uint64_t *step;
};
__device__ inline void end_step(const StepEnd &S) {
    for (int r = threadIdx.x; r <= S.nrep; r += blockDim.x) {
        if (r < S.nrep) {
            if (S.rebuild[r]) S.nbuilds[r] += 1;
            S.step[r] += 1;
        }
        S.rebuild[r] = 0;   // [nrep] is `any`
    }
}

template <bool ENERGY>
__global__ void __launch_bounds__(128)
k_constraints(const int32_t *__restrict__ kidx, int32_t e1, int32_t e2, int32_t e3, int32_t e4,
              int32_t nb_it, const int32_t *__restrict__ wclus, ShakeArgs A, StepEnd S,
              long long *__restrict__ eacc) {
    if (S.nrep && blockIdx.x == gridDim.x - 1) {
        end_step(S);
        return;
    }
    auto energies = [&](const double vir[3], long long eb, long long ea, bool live, int rr) {
        if (!ENERGY) return;
        wave_add(to_efix(vir[0]), live, rr, eacc, V_X);
        wave_add(to_efix(vir[1]), live, rr, eacc, V_Y);
        wave_add(to_efix(vir[2]), live, rr, eacc, V_Z);
        wave_add(eb, live, rr, eacc, E_BOND);
        wave_add(ea, live, rr, eacc, E_ANGLE);
    };
    if ((int)blockIdx.x < nb_it) {
        double vir[3] = {0.0, 0.0, 0.0};
        long long eb = 0, ea = 0;
        int rr = 0;
        const int t = blockIdx.x * blockDim.x + threadIdx.x;
        const int m = t < e4 ? kidx[t] : -1;
        if (m >= 0) {
            if (t >= e3) rr = shake_cluster<-3>(m, A, vir, eb, ea);
            else if (t >= e2) rr = shake_cluster<4>(m, A, vir, eb, ea);
            else if (t >= e1) rr = shake_cluster<3>(m, A, vir, eb, ea);
            else rr = shake_cluster<1>(m, A, vir, eb, ea);
        }
        energies(vir, eb, ea, m >= 0, rr);
        return;
    }
    __shared__ int32_t s_q[2][WSPAN];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int a0 = ((blockIdx.x - nb_it) * 2 + wave) * WSPAN;
    int cnt = 0;
    for (int k = 0; k < WSPAN; k += 64) {
        const int i = a0 + k + lane;
        const int m = (k + lane < WSPAN && i < A.n) ? wclus[i] : -1;
        const uint64_t b = __ballot(m >= 0);
        if (m >= 0) s_q[wave][cnt + __popcll(b & lt_mask)] = m;
        cnt += __popcll(b);
    }
    __builtin_amdgcn_wave_barrier();   // this wavefront's LDS writes precede its reads
    for (int base = 0; base < cnt; base += 64) {
        double vir[3] = {0.0, 0.0, 0.0};
        long long eb = 0, ea = 0;
        int rr = 0;
        const bool live = base + lane < cnt;
        if (live) rr = settle_water(s_q[wave][base + lane], A, vir, eb, ea);
        energies(vir, eb, ea, live, rr);
    }
}

// Plain streaming copy (16 B per thread per iteration): the HBM reference for traffic
// counters and for the achieved-bandwidth figure of the profiling helpers.
__global__ void k_copy16(size_t n16, const float4 *__restrict__ src, float4 *__restrict__ dst) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n16; k += stride) dst[k] = src[k];
}

// The force wrapper's merge: each term rounded to real*4 as its own routine returns it (the
// fixed-point sums as k_fix_to_aos rounds them), then pair + 1-4 + bonded summed in FP64 and
// stored real*4 into ff (which holds the pair term on entry).  Workgroups past the atoms'
// write the report, for which the merge need not wait.
__global__ void __launch_bounds__(256)
k_merge_report(int32_t n, float *__restrict__ ff, const long long *__restrict__ f14,
               const long long *__restrict__ fb, ReportArgs A) {
    const int merge = (n + 255) / 256;
    if ((int)blockIdx.x >= merge) {
        report_words(A, ((int)blockIdx.x - merge) * 256 + threadIdx.x);
        return;
    }
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float h = (float)((double)f14[(size_t)c * n + i] * FIX_INV);
        const float b = (float)((double)fb[(size_t)c * n + i] * FIX_INV);
        ff[3 * (size_t)i + c] = (float)(((double)ff[3 * (size_t)i + c] + (double)h) + (double)b);
    }
}

// An upload changes places with the state (positions, and v / q / gid where given), and a type
// (the int bits of pos.w) outside 1..ntypes is told to the host, which then runs the exchange
// once more and has the state as it was.  (A check of its own before the move was a launch in
// every call of the drop-in step: 3.4 us, and one in front of the other.)
__global__ void k_put_state(int32_t n, AtomArrays up, AtomArrays state, bool v, bool q, bool gid,
                            int32_t ntypes, HostWords *__restrict__ hw) {
    const int stride = gridDim.x * blockDim.x;
    bool out = false;
    auto exchange = [](auto &a, auto &b) {
        const auto x = a;
        a = b;
        b = x;
    };
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
        exchange(state.pos4[k], up.pos4[k]);
        const int t = __float_as_int(state.pos4[k].w);
        out |= (t < 1) | (t > ntypes);
        if (q) exchange(state.q[k], up.q[k]);
        if (gid) exchange(state.gid[k], up.gid[k]);
        if (v) {
#pragma unroll
            for (int d = 0; d < 3; ++d) exchange(state.v32[(size_t)d * n + k], up.v32[(size_t)d * n + k]);
        }
    }
    if (__ballot(out) && __lane_id() == 0) hw->type_err = 1;   // every lane writes the same
}

// The fused rigid-water bonded terms alone (steps that run no SHAKE: the minimiser).
__global__ void k_water_bonded(int32_t ns, const int32_t *__restrict__ num, ShakeArgs A) {
    water_terms(ns, num, A, blockIdx.x * blockDim.x + threadIdx.x);
}

// Capped steepest descent: every atom moves along its force by min(gamma |F|, max_disp); then,
// as in k_advance, the rebuild check, a cleared force sum and the pair kernel's record.
__global__ void k_minimize_step(int32_t n, double gamma, double max_disp, double *__restrict__ xd,
                                double *__restrict__ drd, const double *__restrict__ fnb,
                                float4 *__restrict__ pos4, const int32_t *__restrict__ rep,
                                const RepInfo *__restrict__ reps, StepOut O) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = rep[i];
    const RepInfo &R = reps[r];
    const double box = R.box;
    double f[3], x[3], dr[3], f2 = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        f[c] = fnb[o] + (double)O.fix[o] * FIX_INV;
        O.fix[o] = 0;
        f2 += f[c] * f[c];
    }
    const double fn = sqrt(f2);
    const double step = (fn > 0.0) ? fmin(gamma * fn, max_disp) / fn : 0.0;
    float4 p = pos4[i];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        const double d = isfinite(f[c]) ? step * f[c] : 0.0;
        dr[c] = drd[o] + d;
        drd[o] = dr[c];
        x[c] = wrap64(xd[o] + d, box);
        xd[o] = x[c];
    }
    p.x = (float)x[0]; p.y = (float)x[1]; p.z = (float)x[2];
    pos4[i] = p;
    flag_rebuild(O, r, dr, R.chk2);
    if (O.pf) write_record(O.pf, i, x[0], x[1], x[2], R.fscale, (uint32_t)__float_as_int(p.w), O.q);
}

__global__ void k_step_add(int32_t nrep, uint64_t *step, long long delta) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrep) step[r] += (uint64_t)delta;
}

}  // namespace

void launch_zero_forces(sofia_ctx *c, long long *f, bool energies) {
    if (energies) {
        launch_save_segment(c);
        c->eacc_zero = false;
    }
    const int n3 = 3 * c->N, ne = (int)eacc_len(c->nrep);
    hipLaunchKernelGGL(k_zero, dim3(nblocks(n3 > ne ? n3 : ne, 256)), dim3(256), 0, c->stream, n3, f,
                       ne, energies ? c->eacc : nullptr);
}

void launch_fix_to_coords(sofia_ctx *c, const long long *f, float *out) {
    hipLaunchKernelGGL(k_fix_to_aos, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, f, out);
}

void launch_nve_v32(sofia_ctx *c, float dt_partial, const float *ff) {
    hipLaunchKernelGGL(k_nve_v32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, dt_partial,
                       c->a.pos4, c->mass, c->a.v32, ff, c->rep, c->dp.amu2e, c->eacc);
}

void launch_nve_x32(sofia_ctx *c) {
    hipLaunchKernelGGL(k_nve_x32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->dp.dt,
                       c->a.v32, c->a.pos4, c->dr32);
}

void launch_berendsen32(sofia_ctx *c, const double *mu_dev) {
    hipLaunchKernelGGL(k_berendsen32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->dr32, c->rep, mu_dev);
}

void launch_pbc32(sofia_ctx *c) {
    hipLaunchKernelGGL(k_pbc32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->rep, c->reps_d);
}

void launch_shake32(sofia_ctx *c, int iflag, float *ff, double *) {
    if (!c->ns) return;
    const float dt = c->dp.dt, k2a = c->dp.kcal2amu;
    const double dtsq = (iflag == 0) ? (double)(((0.5f * dt) * dt) * k2a) : (double)((dt * dt) * k2a);
    hipLaunchKernelGGL(k_shake32, dim3(nblocks(c->ns, 64)), dim3(64), 0, c->stream, c->ns, c->shake_num,
                       (const int4 *)c->shake_atoms, c->shake_bond, c->a.pos4, c->a.v32, ff, c->mtab,
                       c->rep, c->reps_d, dt, dtsq, c->dp.shake_tol, c->dp.shake_maxiter,
                       c->shake_err, c->shake_iters, c->eacc);
}

void launch_langevin32(sofia_ctx *c, float fric, float gconst, uint64_t seed, uint64_t step, float *out) {
    hipLaunchKernelGGL(k_langevin32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->a.v32, c->a.gid, c->mass, fric, gconst, seed, step, out);
}

void launch_engine_from32(sofia_ctx *c) {
    hipLaunchKernelGGL(k_from32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->a.v32, c->a.xd, c->a.vd, c->drd);
}

void launch_engine_to32(sofia_ctx *c) {
    hipLaunchKernelGGL(k_to32, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.xd,
                       c->a.vd, c->a.pos4, c->a.v32);
}

void launch_nve_v64(sofia_ctx *c, bool ke) {
    const double dthalf = 0.5 * (double)c->dp.dt * (double)c->dp.kcal2amu;
    hipLaunchKernelGGL(k_nve_v64, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, dthalf,
                       c->a.pos4, c->mass, c->a.vd, c->fnb, c->fix, c->rep, c->dp.amu2e, ke ? 1 : 0,
                       c->eacc);
}

StepOut step_out(sofia_ctx *c) {
    const int rb = record_bytes(c);
    return StepOut{c->rebuild, c->rebuild + c->nrep, c->fix, rb ? c->pfix : nullptr,
                   rb == 16 ? c->a.q : nullptr};
}

void launch_advance(sofia_ctx *c, bool kick2) {
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N,
                           (double)c->dp.dt, c->mtab, c->a.xd, c->a.vd, c->drd, c->a.pos4, c->fnb,
                           c->a.gid, c->rep, c->reps_d, c->step_d, c->has_thermostat ? 1 : 0,
                           step_out(c));
    };
    if (kick2) go(k_advance<true>);
    else go(k_advance<false>);
}

// Energy sums start from zero; skipped where the last report left them so.
void launch_zero_energies(sofia_ctx *c) {
    launch_save_segment(c);
    const bool zero = c->eacc_zero;
    c->eacc_zero = false;
    if (zero) return;
    const int ne = (int)eacc_len(c->nrep);
    hipLaunchKernelGGL(k_zero, dim3(nblocks(ne, 256)), dim3(256), 0, c->stream, ne, c->eacc, 0,
                       (long long *)nullptr);
}

void launch_langevin64(sofia_ctx *c) {
    hipLaunchKernelGGL(k_langevin64, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->a.vd, c->a.gid, c->rep, c->reps_d, c->mass, c->step_d, c->fix);
}

ShakeArgs shake_args(sofia_ctx *c) {
    const double dt = c->dp.dt;
    const double dtsq = dt * dt * (double)c->dp.kcal2amu;
    ShakeArgs A;
    A.atoms = c->shake_atoms; A.bond = c->shake_bond; A.water = c->water;
    A.pos4 = c->a.pos4; A.xd = c->a.xd; A.vd = c->a.vd; A.fnb = c->fnb; A.fix = c->fix;
    A.mtab = c->mtab; A.rep = c->rep; A.reps = c->reps_d;
    A.bond_k = c->bond_k; A.bond_r0 = c->bond_r0; A.angle_k = c->angle_k; A.angle_th0 = c->angle_th0;
    A.n = c->N; A.dt = dt; A.dtsq = dtsq; A.tol = c->dp.shake_tol; A.maxiter = c->dp.shake_maxiter;
    A.err = c->shake_err;
    return A;
}

void launch_shake64(sofia_ctx *c, bool energies, bool step) {
    const int32_t *n = c->shake_kcount;   // group sizes in whole wavefronts
    const int e1 = n[0], e2 = e1 + n[1], e3 = e2 + n[2], e4 = e3 + n[3];
    const int nb_it = nblocks(e4, 128);
    const int nb_w = n[4] ? nblocks(c->N, 2 * WSPAN) : 0;
    const int grid = nb_it + nb_w + (step ? 1 : 0);
    if (grid == 0) return;
    StepEnd S{step ? c->nrep : 0, c->rebuild, c->nbuilds, c->step_d};
    if (energies)
        hipLaunchKernelGGL(k_constraints<true>, dim3(grid), dim3(128), 0, c->stream, c->shake_kidx,
                           e1, e2, e3, e4, nb_it, c->a.wclus, shake_args(c), S, c->eacc);
    else
        hipLaunchKernelGGL(k_constraints<false>, dim3(grid), dim3(128), 0, c->stream, c->shake_kidx,
                           e1, e2, e3, e4, nb_it, c->a.wclus, shake_args(c), S, c->eacc);
}

void launch_put_state(sofia_ctx *c, bool v, bool q, bool gid) {
    const int grid = std::min(nblocks(c->N, 256), 1024);
    hipLaunchKernelGGL(k_put_state, dim3(grid), dim3(256), 0, c->stream, c->N, c->b, c->a, v, q, gid,
                       c->p.ntypes, c->hw);
}

namespace {
ReportArgs report_args(sofia_ctx *c, bool clear_shake) {
    c->eacc_zero = true;
    return ReportArgs{c->nrep * NE, c->eacc, c->shake_err, c->shake_iters, c->maxcnt, c->hw, c->hw_e,
                      clear_shake};
}
inline int report_blocks(const sofia_ctx *c) { return nblocks((long long)c->nrep * NE * ESPREAD, 256); }
}  // namespace

void launch_report(sofia_ctx *c, bool clear_shake) {
    hipLaunchKernelGGL(k_report, dim3(report_blocks(c)), dim3(256), 0, c->stream,
                       report_args(c, clear_shake));
}

void launch_save_segment(sofia_ctx *c) {
    if (c->segment != sofia_ctx::SEG_EACC) return;
    ReportArgs A = report_args(c, false);
    A.hw_e = c->hw_seg;
    hipLaunchKernelGGL(k_report, dim3(report_blocks(c)), dim3(256), 0, c->stream, A);
    c->segment = sofia_ctx::SEG_SAVED;
}

void launch_merge_report(sofia_ctx *c, float *ff32, const long long *f14, const long long *fb) {
    hipLaunchKernelGGL(k_merge_report, dim3(nblocks(c->N, 256) + report_blocks(c)), dim3(256), 0,
                       c->stream, c->N, ff32, f14, fb, report_args(c, false));
}

void launch_start_forces(sofia_ctx *c, long long *a, long long *b, double *xd) {
    hipLaunchKernelGGL(k_start_forces, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, a, b,
                       c->a.pos4, xd);
}

void launch_soa_to_aos(sofia_ctx *c, const double *src, const long long *fix, const int32_t *gid, double *dst) {
    hipLaunchKernelGGL(k_soa_to_aos, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, src, fix,
                       gid, c->rep, c->reps_d, dst);
}

void launch_aos_to_soa(sofia_ctx *c, const double *src, double *dst) {
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, src, dst);
}

void launch_copy16(sofia_ctx *c, size_t n16, const void *src, void *dst) {
    hipLaunchKernelGGL(k_copy16, dim3(2048), dim3(256), 0, c->stream, n16, (const float4 *)src,
                       (float4 *)dst);
}

void launch_water_bonded(sofia_ctx *c) {
    if (!c->ns || !c->water_split) return;
    hipLaunchKernelGGL(k_water_bonded, dim3(nblocks(c->ns, 128)), dim3(128), 0, c->stream, c->ns,
                       c->shake_num, shake_args(c));
}

void launch_minimize_step(sofia_ctx *c, double gamma, double max_disp) {
    hipLaunchKernelGGL(k_minimize_step, dim3(nblocks(c->N, 256)), dim3(256), 0, c->stream, c->N, gamma,
                       max_disp, c->a.xd, c->drd, c->fnb, c->a.pos4, c->rep, c->reps_d, step_out(c));
}

void launch_step_add(sofia_ctx *c, long long delta) {
    hipLaunchKernelGGL(k_step_add, dim3(nblocks(c->nrep, 256)), dim3(256), 0, c->stream, c->nrep,
                       c->step_d, delta);
}

}  // namespace sofia
