// Cell binning, cell sort, permutation gather and Verlet-list build for gfx950.
//
// Semantics follow Source/mod_neighbor.f90 exactly (bit-exact list parity):
//   xyz2bin        1381-1424  cell = int(dble(x) * (1/dble(rn))), x >= box -> last cell
//   new_nlist +    923-1005   cells in id order; inside a cell, descending old index
//   sort_posit_charge          (the linked-list chain order)
//   build_neighbor_nonewton 90-303 / 622-809: stencil cells in cnum order, atoms of each
//                  cell in index order, real*4 minimum image with round-to-nearest,
//                  dr2 = (dx*dx + dy*dy) + dz*dz in real*4, kept if z != i,
//                  dble(dr2) < rv2 and z not in specbond(1:num3bond(i), i).
// This file is compiled with -ffp-contract=off so no FMA changes the real*4 distance.
//
// GPU design: one workgroup per cell stages the 27 stencil cells (x, y, z, index as a
// float4) in LDS in stencil order; each wavefront takes one i atom at a time and sweeps
// the staged candidates 64 at a time, compacting hits with a ballot + popcount prefix so
// the output keeps the reference's order.  Several replicas share one launch: every
// cell belongs to one replica and only replicas flagged for a rebuild do work.
#include <algorithm>

#include "sofia_device.h"

namespace sofia {
namespace {

constexpr int LIST_CAP = 4096;   // staged candidates per cell (64 KiB of LDS)

// real*4 minimum image: (s + sign(2^23,s)) - sign(2^23,dx) is round-to-nearest-even of
// s = dx*ibox for |s| < 2^22, i.e. rintf.
__device__ inline float mimg32(float dx, float box, float ibox) {
    const float s = __builtin_rintf(dx * ibox);
    return dx - s * box;
}

// The list-maintenance kernels below run every step and do work only for the replicas
// flagged in `rebuild`; `any` (the word after the nrep flags) is set whenever one is, so a
// step that rebuilds nothing ends each of them after one read.  They loop over their items
// with a fixed grid (at most GRID_CAP workgroups), which keeps such a step's launches short.
constexpr int GRID_CAP = 2048;

// The sort is three launches.  k_bin (in a step with bonded bundles k_bonded_bundles, which
// shares its launch) counts each cell's atoms and drops their ids into the cell's bucket;
// k_sort_gather orders a cell and moves its atoms' data to the gather target;
// k_copyback puts them back (device pointers stay fixed, which keeps captured graphs valid),
// re-indexes what names atoms and clears the binning counters for the next sort.
__global__ void k_bin(BinArgs A) {
    if (!*A.any) return;
    bin_atoms(A, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

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

// Atoms of a cell in descending old index (the chain order of the reference's linked cells),
// by ranking, which is deterministic.  A wavefront owns `per` consecutive cells; it finds
// their first atom by summing the replica's counts before its first cell (a scan kernel of one
// workgroup per replica in the launch sequence cost every step more than these sums cost the
// steps that rebuild).  A cell with more atoms than a bucket holds is read from acell.
__global__ void __launch_bounds__(256)
k_sort_gather(int32_t ncell, int32_t per, const int32_t *__restrict__ cell_rep,
              const RepInfo *__restrict__ reps, const int32_t *__restrict__ rebuild,
              const int32_t *__restrict__ any, const int32_t *__restrict__ cbin,
              const int32_t *__restrict__ acell, const int32_t *__restrict__ bucket, int32_t cap,
              int32_t *__restrict__ ccount, int32_t *__restrict__ cstart, int32_t *__restrict__ tt,
              int32_t *__restrict__ atombin, int32_t n, AtomArrays src, AtomArrays dst, int mode,
              StepArrays T) {
    if (!*any) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int c0 = wave * per, c1 = min(c0 + per, ncell);
    int rcur = -1, base = 0;
    for (int c = c0; c < c1; ++c) {
        const int r = cell_rep[c];
        if (!rebuild[r]) {
            rcur = -1;
            continue;
        }
        if (r != rcur) {   // first cell of this replica here: the atoms in the cells before it
            int s = 0;
            for (int k = reps[r].cell0 + lane; k < c; k += 64) s += cbin[k];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
            base = reps[r].atom0 + __builtin_amdgcn_readfirstlane(s);
            rcur = r;
        }
        const int cnt = cbin[c];
        if (lane == 0) {
            cstart[c] = base;
            ccount[c] = cnt;
        }
        auto place = [&](int me, int rank) {
            tt[me] = base + rank;
            atombin[base + rank] = c;
            move_atom(src, dst, n, me, base + rank, mode, T);
        };
        if (cnt <= cap) {
            const int32_t *ids = bucket + (size_t)c * cap;
            for (int e = lane; e < cnt; e += 64) {
                const int me = ids[e];
                int rank = 0;
                for (int f = 0; f < cnt; ++f) rank += ids[f] > me;
                place(me, rank);
            }
        } else {
            const int a0 = reps[r].atom0, a1 = a0 + reps[r].natom;
            const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
            int done = 0;
            for (int b = 0; b < a1 - a0; b += 64) {   // lanes in descending atom order
                const int i = a1 - 1 - b - lane;
                const bool in = i >= a0 && acell[i] == c;
                const uint64_t m = __ballot(in);
                if (in) place(i, done + __popcll(m & lt_mask));
                done += __popcll(m);
            }
        }
        base += cnt;
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

__global__ void k_copyback(int32_t n, const int32_t *__restrict__ rep,
                           const RepInfo *__restrict__ reps, const int32_t *__restrict__ rebuild,
                           const int32_t *__restrict__ any, const int32_t *__restrict__ tt,
                           AtomArrays src, AtomArrays dst, float *__restrict__ dr32,
                           double *__restrict__ drd, int mode, StepArrays T, RemapSet S,
                           int32_t ncell, const int32_t *__restrict__ cell_rep,
                           int32_t *__restrict__ cbin) {
    if (!*any) return;
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
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
}

// A device topology array in the host's layout: in the first nidx columns of each item a
// global 0-based atom id (-1 = empty) becomes the 1-based id within its replica (0 = empty);
// the other columns (types) are copied.
__global__ void k_host_ids(size_t count, int32_t width, int32_t nidx, const int32_t *__restrict__ src,
                           int32_t *__restrict__ dst, const int32_t *__restrict__ rep,
                           const RepInfo *__restrict__ reps) {
    for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < count;
         e += (size_t)gridDim.x * blockDim.x) {
        const int v = src[e];
        const bool is_id = (int)(e % (size_t)width) < nidx;
        dst[e] = !is_id ? v : (v < 0 ? 0 : v - reps[rep[v]].atom0 + 1);
    }
}

// RDF_calc (Source/mod_force_nonbond.f90:708-775): one wavefront per atom.  An atom of type
// itype walks its list row; each neighbour of type jtype with dr2 < rcut2 (FP64 distance, the
// real*8 minimum image, no contraction in this file) adds 1 to bin int(sqrt(dr2) / delta).
// The counts are integers, so the histogram does not depend on the order of the additions.
__global__ void k_rdf(int32_t n, const float4 *__restrict__ pos4, const int32_t *__restrict__ rep,
                      const RepInfo *__restrict__ reps, const int32_t *__restrict__ nlist,
                      const int32_t *__restrict__ numneigh, int32_t na, double rcut2,
                      double delta, int32_t itype, int32_t jtype, int32_t nbins,
                      uint32_t *__restrict__ hist) {
    const int i = blockIdx.x * (blockDim.x / 64) + (int)(threadIdx.x / 64);
    if (i >= n) return;
    const float4 xi = pos4[i];
    if (__float_as_int(xi.w) != itype) return;   // uniform across the wavefront
    const RepInfo R = reps[rep[i]];
    const double bx = R.box, ib = R.ibox;
    const double x1 = xi.x, y1 = xi.y, z1 = xi.z;
    const int nn = min(numneigh[i], na);
    const int32_t *row = nlist + (size_t)i * na;
    for (int k = (int)(threadIdx.x & 63); k < nn; k += 64) {
        const float4 pj = pos4[row[k]];
        if (__float_as_int(pj.w) != jtype) continue;
        double dx = x1 - (double)pj.x, dy = y1 - (double)pj.y, dz = z1 - (double)pj.z;
        dx = dx - bx * __builtin_rint(dx * ib);
        dy = dy - bx * __builtin_rint(dy * ib);
        dz = dz - bx * __builtin_rint(dz * ib);
        const double dr2 = dx * dx + dy * dy + dz * dz;
        if (dr2 < rcut2) {
            const int node = (int)(sqrt(dr2) / delta);
            if (node < nbins) atomicAdd(&hist[node], 1u);
        }
    }
}

template <int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
k_build_list(const float4 *__restrict__ pos4, const int32_t *__restrict__ num3,
             const int32_t *__restrict__ spec, const int32_t *__restrict__ cstart,
             const int32_t *__restrict__ ccount, const int32_t *__restrict__ cnum,
             const int32_t *__restrict__ cell_rep, const RepInfo *__restrict__ reps,
             const int32_t *__restrict__ rebuild, double rv2, int32_t na,
             int32_t *__restrict__ nlist, int32_t *__restrict__ numneigh,
             int32_t *__restrict__ maxcnt) {
    const int c = blockIdx.x;
    const int r = cell_rep[c];
    if (!rebuild[r] || reps[r].stencil5) return;
    const float box = reps[r].box, ibox = reps[r].ibox;

    __shared__ int32_t s_cell[27];
    __shared__ int32_t s_start[27];
    __shared__ int32_t s_off[28];
    __shared__ float4 s_j[LIST_CAP];

    const int tid = threadIdx.x;
    if (tid < 27) {
        const int nc = cnum[27 * c + tid];
        s_cell[tid] = nc;
        s_start[tid] = cstart[nc];
    }
    __syncthreads();
    if (tid == 0) {
        int acc = 0;
        for (int k = 0; k < 27; ++k) {
            s_off[k] = acc;
            acc += ccount[s_cell[k]];
        }
        s_off[27] = acc;
    }
    __syncthreads();
    const int total = s_off[27];
    const bool staged = total <= LIST_CAP;
    if (staged) {
        for (int k = 0; k < 27; ++k) {
            const int cnt = s_off[k + 1] - s_off[k], st = s_start[k];
            for (int t = tid; t < cnt; t += WAVES * 64) {
                float4 p = pos4[st + t];
                p.w = __int_as_float(st + t);
                s_j[s_off[k] + t] = p;
            }
        }
    }
    __syncthreads();

    const int wave = tid >> 6, lane = tid & 63;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int i0 = cstart[c], ni = ccount[c];
    for (int ii = blockIdx.y * WAVES + wave; ii < ni; ii += gridDim.y * WAVES) {
        const int i = i0 + ii;
        const float4 xi = pos4[i];
        const int n3 = num3[i];
        int ex[SPEC];
        int exmin = 0x7fffffff, exmax = -1;
#pragma unroll
        for (int l = 0; l < SPEC; ++l) {
            ex[l] = (l < n3) ? spec[(size_t)i * SPEC + l] : -1;
            if (l < n3) {
                exmin = min(exmin, ex[l]);
                exmax = max(exmax, ex[l]);
            }
        }
        int cnt = 0;
        int32_t *out = nlist + (size_t)i * na;
        for (int base = 0; base < total; base += 64) {
            const int t = base + lane;
            bool pred = false;
            int z = -1;
            if (t < total) {
                float4 pj;
                if (staged) {
                    pj = s_j[t];
                    z = __float_as_int(pj.w);
                } else {
                    int k = 0;
                    while (k < 26 && t >= s_off[k + 1]) ++k;
                    z = s_start[k] + (t - s_off[k]);
                    pj = pos4[z];
                }
                const float dx = mimg32(xi.x - pj.x, box, ibox);
                const float dy = mimg32(xi.y - pj.y, box, ibox);
                const float dz = mimg32(xi.z - pj.z, box, ibox);
                const float dr2 = (dx * dx + dy * dy) + dz * dz;
                pred = (z != i) && ((double)dr2 < rv2);
            }
            const bool maybe = pred && z >= exmin && z <= exmax;
            if (__any(maybe)) {
                if (maybe) {
#pragma unroll
                    for (int l = 0; l < SPEC; ++l)
                        if (ex[l] == z) pred = false;
                }
            }
            const uint64_t mask = __ballot(pred);
            const int pos = cnt + __popcll(mask & lt_mask);
            if (pred && pos < na) out[pos] = z;
            cnt += __popcll(mask);
        }
        if (lane == 0) {
            numneigh[i] = cnt;
            if (cnt > na) atomicMax(maxcnt, cnt);
        }
    }
}

// check_neighbor; the rebuild flags are cleared with it.
__global__ void k_check32(int32_t n, const float *__restrict__ dr, double rvrc2, int32_t nrep,
                          int32_t *__restrict__ rebuild, HostWords *__restrict__ hw) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool moved = false;
    if (i <= nrep) rebuild[i] = 0;   // [nrep] is `any`
    if (i < n) {
        const float x = dr[i], y = dr[(size_t)n + i], z = dr[2 * (size_t)n + i];
        moved = (double)((x * x + y * y) + z * z) >= rvrc2;
    }
    // any atom of any replica: every wavefront that writes, writes the same
    if (__ballot(moved) && (threadIdx.x & 63) == 0) hw->moved = 1;
}

// rebuild[0..nrep) and `any` = rebuild[nrep] to value
__global__ void k_set_flags(int32_t nrep, int32_t *__restrict__ rebuild, int32_t value) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= nrep) rebuild[r] = value;
}

__global__ void k_finish(int32_t nrep, int32_t *__restrict__ rebuild, int32_t *__restrict__ nbuilds) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= nrep) finish_rebuild(r, nrep, rebuild, nbuilds);
}

// The end of a rebuild: the largest count to the host; if the lists fit, k_finish's books.
__global__ void k_list_done(int32_t nrep, int32_t *__restrict__ rebuild, int32_t *__restrict__ nbuilds,
                            const int32_t *__restrict__ maxcnt, int32_t na, HostWords *__restrict__ hw,
                            int32_t n, const int32_t *__restrict__ tt, const int32_t *__restrict__ rep,
                            const RepInfo *__restrict__ reps, int32_t *__restrict__ local) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int mx = *maxcnt;
    if (t == 0) hw->maxcnt = mx;
    if (mx <= na && t <= nrep) {
        if (t < nrep && rebuild[t]) nbuilds[t] += 1;
        rebuild[t] = 0;   // [nrep] is `any`
    }
    if (local && t < n) local[t] = tt[t] - reps[rep[t]].atom0 + 1;
}

inline int nblk(int n, int b) { return (n + b - 1) / b; }

}  // namespace

// grid of the looping list-maintenance kernels
inline int capped(int n, int b) { return std::max(1, std::min(nblk(n, b), GRID_CAP)); }
inline const int32_t *any_flag(const sofia_ctx *c) { return c->rebuild + c->nrep; }

void launch_sort(sofia_ctx *c, SortMode mode, bool bonded, bool energies) {
    const BinArgs B{c->N, c->bucket_cap, c->a.pos4, c->rep, c->reps_d, c->rebuild, any_flag(c),
                    c->cbin, c->acell, c->bucket};
    const int bin_grid = capped(c->N, 256);
    if (bonded) launch_bundles_bin(c, B, bin_grid, energies);
    else hipLaunchKernelGGL(k_bin, dim3(bin_grid), dim3(256), 0, c->stream, B);
    StepArrays T{};
    if (mode == SORT_STEP) {
        const int rb = record_bytes(c);
        T = StepArrays{c->fix, c->fscratch, rb ? c->pfix : nullptr, rb == 16 ? c->a.q : nullptr};
    }
    const int per = nblk(c->ncell_total, 4 * GRID_CAP);   // cells per wavefront
    hipLaunchKernelGGL(k_sort_gather, dim3(nblk(nblk(c->ncell_total, per), 4)), dim3(256), 0, c->stream,
                       c->ncell_total, per, c->cell_rep, c->reps_d, c->rebuild, any_flag(c), c->cbin,
                       c->acell, c->bucket, c->bucket_cap, c->ccount, c->cstart, c->tt, c->atombin,
                       c->N, c->a, c->b, (int)mode, T);
    RemapSet S{};
    int total = 0;
    auto add = [&](int32_t *lst, int items, int width, int nidx) {
        if (!items) return;
        S.lst[S.nlists] = lst;
        total += items;
        S.end[S.nlists] = total;
        S.width[S.nlists] = width;
        S.nidx[S.nlists] = nidx;
        ++S.nlists;
    };
    add(c->bondlist, c->nb, 3, 2);
    add(c->anglelist, c->na, 4, 3);
    add(c->dihedlist, c->nd, 5, 4);
    add(c->torsions, c->ntor, 5, 4);
    add(c->improlist, c->nimp, 5, 4);
    add(c->shake_atoms, c->ns, 4, 4);
    add(c->ebond, c->nbe, 3, 2);
    add(c->eangle, c->nae, 4, 3);
    const int items = std::max({c->N, total, c->ncell_total});
    hipLaunchKernelGGL(k_copyback, dim3(capped(items, 256)), dim3(256), 0, c->stream, c->N, c->rep,
                       c->reps_d, c->rebuild, any_flag(c), c->tt, c->b, c->a, c->dr32, c->drd,
                       (int)mode, T, S, c->ncell_total, c->cell_rep, c->cbin);
}

void launch_rdf(sofia_ctx *c, int32_t itype, int32_t jtype, double delta, int32_t nbins,
                uint32_t *hist) {
    hipLaunchKernelGGL(k_rdf, dim3((c->N + 3) / 4), dim3(256), 0, c->stream, c->N, c->a.pos4,
                       c->rep, c->reps_d, c->nlist, c->numneigh, c->neigh_alloc, c->dp.rcut2,
                       delta, itype, jtype, nbins, hist);
}

void launch_host_ids(sofia_ctx *c, const int32_t *src, int32_t *dst, size_t items, int width,
                     int nidx) {
    const size_t count = items * (size_t)width;
    if (!count) return;
    const int grid = (int)std::min<size_t>((count + 255) / 256, GRID_CAP);
    hipLaunchKernelGGL(k_host_ids, dim3(grid), dim3(256), 0, c->stream, count, width, nidx, src,
                       dst, c->rep, c->reps_d);
}

void launch_build_list(sofia_ctx *c) {
    if (c->n_stencil5 > 0) launch_build_list_engine(c);
    if (c->n_stencil5 == c->nrep) return;
    // few cells (the reference's are a cutoff wide: 125 in a 13,500-atom box) leave most of the
    // chip idle: their atoms go to several workgroups, each staging the stencil for itself
    const int w = c->list_waves;
    const int parts = std::max(1, std::min(8, 1024 / c->ncell_total));
#define LB(W)                                                                                    \
    hipLaunchKernelGGL(k_build_list<W>, dim3(c->ncell_total, parts), dim3(W * 64), 0, c->stream, \
                       c->a.pos4, c->a.num3, c->a.spec, c->cstart, c->ccount, c->cnum,            \
                       c->cell_rep, c->reps_d, c->rebuild, c->dp.rv2, c->neigh_alloc, c->nlist,   \
                       c->numneigh, c->maxcnt)
    if (w <= 2) LB(2);
    else if (w <= 4) LB(4);
    else if (w <= 8) LB(8);
    else LB(16);
#undef LB
}

void launch_check_neighbor(sofia_ctx *c) {
    hipLaunchKernelGGL(k_check32, dim3(nblk(std::max(c->N, c->nrep + 1), 256)), dim3(256), 0, c->stream,
                       c->N, c->dr32, c->dp.rvrc2, c->nrep, c->rebuild, c->hw);
}

void launch_set_rebuild(sofia_ctx *c, int32_t value) {
    hipLaunchKernelGGL(k_set_flags, dim3(nblk(c->nrep + 1, 256)), dim3(256), 0, c->stream, c->nrep,
                       c->rebuild, value);
}

void launch_finish_rebuild(sofia_ctx *c) {
    hipLaunchKernelGGL(k_finish, dim3(nblk(c->nrep + 1, 256)), dim3(256), 0, c->stream, c->nrep,
                       c->rebuild, c->nbuilds);
}

void launch_list_done(sofia_ctx *c, int32_t *local) {
    const int threads = std::max(c->nrep + 1, local ? c->N : 1);
    hipLaunchKernelGGL(k_list_done, dim3(nblk(threads, 256)), dim3(256), 0, c->stream, c->nrep,
                       c->rebuild, c->nbuilds, c->maxcnt, c->neigh_alloc, c->hw, c->N, c->tt, c->rep,
                       c->reps_d, local);
}

}  // namespace sofia
