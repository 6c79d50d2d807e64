// The cell sort's moves: every atom array into cell order, and back into its own place with the
// ids that name atoms re-indexed.
#pragma once

#include "sofia_device.h"

namespace sofia {

// What the step's sort carries beyond the per-atom arrays (SORT_STEP), else null.
struct StepArrays {
    long long *fix, *fixb;   // the step's fixed-point forces and their gather target
    int4 *pf;                // position records, rewritten from the moved positions
    const float *q;          // null: 12-byte records
};

// Atom o of src to place k of dst; specbond entries go along unmapped.
__device__ inline void move_atom(const AtomArrays &src, const AtomArrays &dst, int n, int o, int k,
                                 int mode, const StepArrays &T) {
    dst.pos4[k] = src.pos4[o];
    dst.q[k] = src.q[o];
    dst.gid[k] = src.gid[o];
    dst.num1[k] = src.num1[o];
    dst.num2[k] = src.num2[o];
    dst.num3[k] = src.num3[o];
    dst.mol[k] = src.mol[o];
    dst.wclus[k] = src.wclus[o];
    const int4 *s4 = (const int4 *)(src.spec + (size_t)o * SPEC);
    int4 *d4 = (int4 *)(dst.spec + (size_t)k * SPEC);
#pragma unroll
    for (int l = 0; l < SPEC / 4; ++l) d4[l] = s4[l];
#pragma unroll
    for (int d = 0; d < 3; ++d) dst.v32[3 * (size_t)k + d] = src.v32[3 * (size_t)o + d];
    if (mode != SORT_DROPIN) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            dst.xd[(size_t)d * n + k] = src.xd[(size_t)d * n + o];
            dst.vd[(size_t)d * n + k] = src.vd[(size_t)d * n + o];
        }
    }
    if (mode == SORT_STEP) {
#pragma unroll
        for (int d = 0; d < 3; ++d) T.fixb[(size_t)d * n + k] = T.fix[(size_t)d * n + o];
    }
}

// Every bonded list of the context: item t of the concatenation falls in list L of S, whose
// items are `width` ints with the first `nidx` atom ids (-1 = unused).  Items of replicas
// that rebuild nothing this step are skipped (their atoms keep their places).
struct RemapSet {
    int32_t *lst[8];
    int32_t end[8];           // cumulative item counts
    int32_t width[8], nidx[8];
    int32_t nlists;
};

// The sort's last phase: the moved data back to the state's own arrays (device pointers stay
// fixed, which keeps captured graphs valid), atom ids re-indexed, the binning counters cleared.
struct CopyArgs {
    int32_t n, ncell, mode;
    const int32_t *rep, *rebuild, *any, *tt, *cell_rep;
    const RepInfo *reps;
    AtomArrays src, dst;
    float *dr32;
    double *drd;
    StepArrays T;
    RemapSet S;
    int32_t *cbin, *nover;
};
__device__ inline void copy_back(const CopyArgs &A, int t0, int stride) {
    const int n = A.n, mode = A.mode;
    const AtomArrays &src = A.src, &dst = A.dst;
    const StepArrays &T = A.T;
    const RemapSet &S = A.S;
    const int32_t *__restrict__ rep = A.rep, *__restrict__ rebuild = A.rebuild;
    const int32_t *__restrict__ tt = A.tt, *__restrict__ cell_rep = A.cell_rep;
    const RepInfo *__restrict__ reps = A.reps;
    float *__restrict__ dr32 = A.dr32;
    double *__restrict__ drd = A.drd;
    int32_t *__restrict__ cbin = A.cbin;
    const int ncell = A.ncell;
    for (int k = t0; k < n; k += stride) {
        const int r = rep[k];
        if (!rebuild[r]) continue;
        move_atom(src, dst, n, k, k, mode == SORT_STEP ? (int)SORT_ENGINE : mode, T);
#pragma unroll
        for (int l = 0; l < SPEC; ++l) {
            const int s = src.spec[(size_t)k * SPEC + l];
            if (s >= 0) dst.spec[(size_t)k * SPEC + l] = tt[s];
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) dr32[(size_t)d * n + k] = 0.0f;
        if (mode != SORT_DROPIN) {
#pragma unroll
            for (int d = 0; d < 3; ++d) drd[(size_t)d * n + k] = 0.0;
        }
        if (mode == SORT_STEP) {
#pragma unroll
            for (int d = 0; d < 3; ++d) T.fix[(size_t)d * n + k] = T.fixb[(size_t)d * n + k];
            if (T.pf)
                write_record(T.pf, k, src.xd[k], src.xd[(size_t)n + k], src.xd[2 * (size_t)n + k],
                             reps[r].fscale, (uint32_t)__float_as_int(src.pos4[k].w), T.q ? src.q : nullptr);
        }
    }
    const int total = S.nlists ? S.end[S.nlists - 1] : 0;
    for (int t = t0; t < total; t += stride) {
        int L = 0;
        while (t >= S.end[L]) ++L;
        const int m = t - (L ? S.end[L - 1] : 0);
        int32_t *item = S.lst[L] + (size_t)m * S.width[L];
        const int a0 = item[0];
        if (a0 < 0 || !rebuild[rep[a0]]) continue;
        for (int k = 0; k < S.nidx[L]; ++k) {
            const int v = item[k];
            if (v >= 0) item[k] = tt[v];
        }
    }
    for (int c = t0; c < ncell; c += stride)
        if (rebuild[cell_rep[c]]) cbin[c] = 0;
    if (t0 == 0) *A.nover = 0;
}
// The arguments of the context's copy back; *items: how many threads find work.
CopyArgs copy_args(sofia_ctx *c, SortMode mode, int *items);

}  // namespace sofia
