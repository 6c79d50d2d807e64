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
#include <cmath>

#include "sort_device.h"

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
// k_sort_gather orders a cell and moves its atoms' data to the gather target; k_copyback (in an
// engine step the first workgroups of the list build) puts them back.
__global__ void k_bin(BinArgs A) {
    if (!*A.any) return;
    bin_atoms(A, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// Atoms in each run of cells, a run a workgroup.
__global__ void __launch_bounds__(1 << CHUNK_SHIFT)
k_chunk_sums(int32_t ncell, const int32_t *__restrict__ any, const int32_t *__restrict__ cbin,
             int32_t *__restrict__ chunk) {
    if (!*any) return;
    __shared__ int32_t s_w[(1 << CHUNK_SHIFT) / 64];
    const int c = (blockIdx.x << CHUNK_SHIFT) + threadIdx.x;
    int s = c < ncell ? cbin[c] : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x) return;
    s = 0;
    for (int w = 0; w < (1 << CHUNK_SHIFT) / 64; ++w) s += s_w[w];
    chunk[blockIdx.x] = s;
}

// Atoms of a cell in descending old index (the chain order of the reference's linked cells), by
// ranking, which is deterministic.  A wavefront owns `per` consecutive cells; it finds their
// first atom by summing the replica's counts before its first cell (a scan kernel of one
// workgroup per replica in the launch sequence cost every step more than these sums cost the
// steps that rebuild), by runs of cells where k_chunk_sums counted those.  A cell with more atoms
// than a bucket holds first gathers them, from its bucket and the list of atoms past full
// buckets, where its places will be (in fat).
__global__ void __launch_bounds__(256)
k_sort_gather(int32_t ncell, int32_t per, int32_t split, const int32_t *__restrict__ cell_rep,
              const RepInfo *__restrict__ reps, const int32_t *__restrict__ rebuild,
              const int32_t *__restrict__ any, const int32_t *__restrict__ cbin,
              const int32_t *__restrict__ chunk, const int32_t *__restrict__ bucket, int32_t cap,
              const int32_t *__restrict__ nover, const int2 *__restrict__ over, int32_t *fat,
              int32_t *__restrict__ ccount, int32_t *__restrict__ cstart, int32_t *__restrict__ tt,
              int32_t *__restrict__ atombin, int32_t n, AtomArrays src, AtomArrays dst, int mode,
              StepArrays T) {
    if (!*any) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const int part = wave % split;   // split > 1: per = 1
    const int c0 = wave / split * per, c1 = min(c0 + per, ncell);
    int rcur = -1, base = 0;
    for (int c = c0; c < c1; ++c) {
        const int r = cell_rep[c];
        if (!rebuild[r]) {
            rcur = -1;
            continue;
        }
        if (r != rcur) {   // first cell of this replica here: the atoms in the cells before it
            int s = 0;
            const int first = reps[r].cell0;
            // whole runs of cells [h, t), the cells before and after them one by one
            const int h = chunk ? (first + (1 << CHUNK_SHIFT) - 1) >> CHUNK_SHIFT : 0;
            const int t = chunk ? c >> CHUNK_SHIFT : 0;
            const int a = h < t ? h << CHUNK_SHIFT : c, b = h < t ? t << CHUNK_SHIFT : c;
            for (int k = first + lane; k < a; k += 64) s += cbin[k];
            for (int k = h + lane; k < t; k += 64) s += chunk[k];
            for (int k = b + lane; k < c; k += 64) s += cbin[k];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
            base = reps[r].atom0 + __builtin_amdgcn_readfirstlane(s);
            rcur = r;
        }
        const int cnt = cbin[c];
        if (lane == 0 && part == 0) {
            cstart[c] = base;
            ccount[c] = cnt;
        }
        const int32_t *ids = bucket + (size_t)c * cap;
        if (cnt > cap) {   // every part of a split writes the same ids to the same places
            const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
            for (int e = lane; e < cap; e += 64) fat[base + e] = ids[e];
            const int no = *nover;
            int done = cap;
#pragma unroll 4
            for (int b = 0; b < no; b += 64) {
                const int2 o = over[min(b + lane, no - 1)];
                const bool in = b + lane < no && o.x == c;
                const uint64_t m = __ballot(in);
                if (in) fat[base + done + __popcll(m & lt_mask)] = o.y;
                done += __popcll(m);
            }
            __threadfence_block();   // other lanes read them
            ids = fat + base;
        }
        for (int e0 = 64 * part; e0 < cnt; e0 += 64 * split) {
            const bool in = e0 + lane < cnt;
            const int me = in ? ids[e0 + lane] : 0;
            int rank = 0;
            for (int f0 = 0; f0 < cnt; f0 += 64) {
                const int other = f0 + lane < cnt ? ids[f0 + lane] : -1;
                const int m = min(64, cnt - f0);
                for (int f = 0; f < m; ++f) rank += __builtin_amdgcn_readlane(other, f) > me;
            }
            if (in) {
                tt[me] = base + rank;
                atombin[base + rank] = c;
                move_atom(src, dst, n, me, base + rank, mode, T);
            }
        }
        base += cnt;
    }
}

__global__ void k_copyback(CopyArgs A) {
    if (!*A.any) return;
    copy_back(A, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
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

// The drop-in list of one cell (or of a share of its atoms, blockIdx.y).
//
// Where the box has at least 5 cells a side and every staged coordinate lies in [0, box], the
// image of a stencil cell is the same for all its atoms: separations inside the box are at
// most 0.4 box, across it at least 0.6 box, so the reference's rounded shift is 0 or +-1 as the
// cell lies, and the distance takes that shift directly -- the same two real*4 operations
// without the product and the rounding.  (4 cells a side: the two shifts can differ only at
// half a box, which is no neighbour by either where rv is less.)  A wavefront then sweeps two atoms at once over the
// cells that come within rv of either (CULL_MARGIN is far above the rounding of positions and
// cells).  Candidates are staged three loads at a time from all 27 cells, which one after the
// other were a chain of 27 loads.  97 -> 60 us at 13,500 atoms, 1010 -> 560 at 204,000; the
// second launch bound keeps two workgroups of 16 wavefronts on a CU.
constexpr float CULL_MARGIN = 0.01f;  // A

template <int WAVES>
__global__ void __launch_bounds__(WAVES * 64, WAVES >= 4 ? WAVES * 2 / 4 : 1)
k_build_list(const float4 *__restrict__ pos4, const int32_t *__restrict__ num3,
             const int32_t *__restrict__ spec, const int32_t *__restrict__ cstart,
             const int32_t *__restrict__ ccount, const int32_t *__restrict__ cnum,
             const int32_t *__restrict__ cell_rep, const RepInfo *__restrict__ reps,
             const int32_t *__restrict__ rebuild, float rv2, float rvm2, int32_t na,
             int32_t *__restrict__ nlist, int32_t *__restrict__ numneigh,
             int32_t *__restrict__ maxcnt) {
    const int c = blockIdx.x;
    const int r = cell_rep[c];
    if (!rebuild[r] || reps[r].stencil5) return;
    const float box = reps[r].box, ibox = reps[r].ibox, rn = reps[r].rn;
    const int nD = reps[r].ncellD, lc = c - reps[r].cell0;

    __shared__ int32_t s_start[27];
    __shared__ int32_t s_off[28];
    __shared__ float4 s_j[LIST_CAP];

    const int tid = threadIdx.x;
    if (tid < 64) {
        int start = 0, count = 0;
        if (tid < 27) {
            const int nc = cnum[27 * c + tid];
            start = cstart[nc];
            count = ccount[nc];
            s_start[tid] = start;
        }
        int v = count;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
            const int u = __shfl_up(v, o, 64);
            if (tid >= o) v += u;
        }
        if (tid < 28) s_off[tid] = v - count;
    }
    __syncthreads();
    const int total = s_off[27];
    const bool staged = total <= LIST_CAP;
    bool outside = false;
    if (staged) {
        constexpr int U = 3;   // loads in flight per thread
        for (int t0 = tid; t0 < total; t0 += U * WAVES * 64) {
            float4 p[U];
            int id[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = min(t0 + u * WAVES * 64, total - 1);
                int k = 0;   // the last cell that starts at or before t
#pragma unroll
                for (int s = 16; s > 0; s >>= 1)
                    if (k + s < 27 && s_off[k + s] <= t) k += s;
                id[u] = s_start[k] + t - s_off[k];
                p[u] = pos4[id[u]];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = t0 + u * WAVES * 64;
                if (t >= total) continue;
                outside |= !(p[u].x >= 0.0f && p[u].x <= box && p[u].y >= 0.0f && p[u].y <= box &&
                             p[u].z >= 0.0f && p[u].z <= box);
                p[u].w = __int_as_float(id[u]);
                s_j[t] = p[u];
            }
        }
    }
    const bool inside = !__syncthreads_or(outside);   // (and the staged candidates are there)
    const bool direct = staged && inside && (nD >= 5 || (nD == 4 && 0.49f * box > sqrtf(rvm2)));

    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int i0 = cstart[c], ni = ccount[c];
    const int first = blockIdx.y * WAVES + wave, step = gridDim.y * WAVES;

    if (direct) {
        // lane k < 27: stencil cell k's place (the centre first, then z, y, x ascending), the
        // shift of its image, and where its candidates lie
        const int j = lane == 0 ? 13 : (lane <= 13 ? lane - 1 : lane);
        const int at[3] = {lc % nD + j % 3 - 1, (lc / nD) % nD + j / 3 % 3 - 1, lc / (nD * nD) + j / 9 - 1};
        float sh[3], low[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            sh[d] = at[d] < 0 ? -box : (at[d] >= nD ? box : 0.0f);
            low[d] = (float)at[d] * rn;
        }
        const int o0 = s_off[min(lane, 27)], o1 = s_off[min(lane + 1, 27)];
        const int id0 = s_start[min(lane, 26)], id1 = id0 + o1 - o0;   // the cell's atom ids
        for (int ii = 2 * first; ii < ni; ii += 2 * step) {
            const int ia = i0 + ii;
            const bool two = ii + 1 < ni;
            const int ib = two ? ia + 1 : ia;
            const float4 xa = pos4[ia], xb = pos4[ib];
            const float lima = rv2, limb = two ? rv2 : -1.0f;
            // exclusions: lanes 0..11 those of a, 16..27 those of b
            const int who = lane < 16 ? ia : ib, e = lane & 15;
            const bool has = lane < 32 && e < SPEC && e < num3[who];
            const int ex = has ? spec[(size_t)who * SPEC + e] : -1;
            const uint64_t exs = __ballot(has);
            bool holds = false;   // an excluded atom of either
            for (uint64_t m = exs; m; m &= m - 1) {
                const int v = __builtin_amdgcn_readlane(ex, __builtin_ctzll(m));
                holds |= v >= id0 && v < id1;
            }
            const uint64_t excells = __ballot(lane < 27 && holds);
            auto gap = [&](const float4 &x) {
                const float g[3] = {x.x, x.y, x.z};
                float d2 = 0.0f;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const float w = fmaxf(0.0f, fmaxf(low[d] - g[d], g[d] - (low[d] + rn)) - CULL_MARGIN);
                    d2 += w * w;
                }
                return d2;
            };
            uint64_t cells = __ballot(lane < 27 && o1 > o0 && fminf(gap(xa), gap(xb)) < rvm2);
            int cnta = 0, cntb = 0;
            int32_t *outa = nlist + (size_t)ia * na, *outb = nlist + (size_t)ib * na;
            while (cells) {
                const int k = __builtin_ctzll(cells);
                cells &= cells - 1;
                const uint64_t exk = (excells >> k & 1) ? exs : 0ull;
                const int lo = __builtin_amdgcn_readlane(o0, k), hi = __builtin_amdgcn_readlane(o1, k);
                const float sx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sh[0]), k));
                const float sy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sh[1]), k));
                const float sz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sh[2]), k));
                for (int base = lo; base < hi; base += 64) {
                    const int t = base + lane;
                    const float4 pj = s_j[min(t, hi - 1)];
                    const int z = __float_as_int(pj.w);
                    const bool in = t < hi;
                    const float ax = (xa.x - pj.x) - sx, ay = (xa.y - pj.y) - sy, az = (xa.z - pj.z) - sz;
                    const float bx = (xb.x - pj.x) - sx, by = (xb.y - pj.y) - sy, bz = (xb.z - pj.z) - sz;
                    bool ha = in & ((ax * ax + ay * ay) + az * az <= lima) & (z != ia);
                    bool hb = in & ((bx * bx + by * by) + bz * bz <= limb) & (z != ib);
                    for (uint64_t m = exk; m; m &= m - 1) {   // exclusions of a and of b
                        const int l = __builtin_ctzll(m);
                        const int v = __builtin_amdgcn_readlane(ex, l);
                        if (l < 16) ha = ha & (z != v);
                        else hb = hb & (z != v);
                    }
                    const uint64_t ma = __ballot(ha), mb = __ballot(hb);
                    const int pa = cnta + (int)__builtin_amdgcn_mbcnt_hi(
                                              (uint32_t)(ma >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ma, 0u));
                    const int pb = cntb + (int)__builtin_amdgcn_mbcnt_hi(
                                              (uint32_t)(mb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mb, 0u));
                    if (ha & (pa < na)) outa[pa] = z;
                    if (hb & (pb < na)) outb[pb] = z;
                    cnta += __popcll(ma);
                    cntb += __popcll(mb);
                }
            }
            if (lane == 0) {
                numneigh[ia] = cnta;
                if (two) numneigh[ib] = cntb;
                const int mx = max(cnta, cntb);
                if (mx > na) atomicMax(maxcnt, mx);
            }
        }
        return;
    }

    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int ii = first; ii < ni; ii += step) {
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
                pred = (z != i) && (dr2 <= rv2);
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
    if (mx <= na && t <= nrep) finish_rebuild(t, nrep, rebuild, nbuilds);
    if (local && t < n) local[t] = tt[t] - reps[rep[t]].atom0 + 1;
}

inline int nblk(int n, int b) { return (n + b - 1) / b; }

}  // namespace

// grid of the looping list-maintenance kernels
inline int capped(int n, int b) { return std::max(1, std::min(nblk(n, b), GRID_CAP)); }
inline const int32_t *any_flag(const sofia_ctx *c) { return c->rebuild + c->nrep; }

StepArrays step_arrays(sofia_ctx *c, SortMode mode) {
    if (mode != SORT_STEP) return StepArrays{};
    const int rb = record_bytes(c);
    return StepArrays{c->fix, c->fscratch, rb ? c->pfix : nullptr, rb == 16 ? c->a.q : nullptr};
}

CopyArgs copy_args(sofia_ctx *c, SortMode mode, int *items) {
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
    *items = std::max({c->N, total, c->ncell_total});
    return CopyArgs{c->N, c->ncell_total, (int)mode, c->rep, c->rebuild, any_flag(c), c->tt, c->cell_rep,
                    c->reps_d, c->b, c->a, c->dr32, c->drd, step_arrays(c, mode), S, c->cbin, c->nover};
}

void launch_sort(sofia_ctx *c, SortMode mode, bool bonded, bool energies, bool leave_copy, bool water) {
    const BinArgs B{c->N, c->bucket_cap, c->a.pos4, c->rep, c->reps_d, c->rebuild, any_flag(c),
                    c->cbin, c->bucket, c->nover, c->over};
    const int bin_grid = capped(c->N, 256);
    if (bonded) launch_bundles_bin(c, B, bin_grid, energies, water);
    else hipLaunchKernelGGL(k_bin, dim3(bin_grid), dim3(256), 0, c->stream, B);
    const int32_t *chunk = c->chunked ? c->chunk : nullptr;
    if (chunk)
        hipLaunchKernelGGL(k_chunk_sums, dim3(nblk(c->ncell_total, 1 << CHUNK_SHIFT)), dim3(1 << CHUNK_SHIFT), 0,
                           c->stream, c->ncell_total, any_flag(c), c->cbin, c->chunk);
    const int per = nblk(c->ncell_total, 4 * GRID_CAP);   // cells per wavefront
    // or wavefronts per cell, where a cell holds more atoms than a wavefront has lanes (the
    // reference's cells: 30 -> 22 us at 13,500 atoms in 125 cells, 33 -> 15 at 31,000)
    const int split = per > 1 ? 1 : std::max(1, std::min(8, nblk(c->N, 64 * c->ncell_total)));
    hipLaunchKernelGGL(k_sort_gather, dim3(nblk(nblk(c->ncell_total, per) * split, 4)), dim3(256), 0, c->stream,
                       c->ncell_total, per, split, c->cell_rep, c->reps_d, c->rebuild, any_flag(c), c->cbin,
                       chunk, c->bucket, c->bucket_cap, c->nover, c->over, c->fat, c->ccount, c->cstart,
                       c->tt, c->atombin, c->N, c->a, c->b, (int)mode, step_arrays(c, mode));
    if (leave_copy) return;
    int items = 0;
    const CopyArgs A = copy_args(c, mode, &items);
    hipLaunchKernelGGL(k_copyback, dim3(capped(items, 256)), dim3(256), 0, c->stream, A);
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

// The sort's copy back rides with the engine's list build where that builds every list.
bool list_takes_copy(const sofia_ctx *c) { return c->n_stencil5 == c->nrep; }

void launch_build_list(sofia_ctx *c, bool copy) {
    if (c->n_stencil5 > 0) launch_build_list_engine(c, copy);
    if (c->n_stencil5 == c->nrep) return;
    // few cells (the reference's are a cutoff wide: 125 in a 13,500-atom box) leave most of the
    // chip idle: their atoms go to several workgroups, each staging the stencil for itself
    const int w = c->list_waves;
    const int parts = std::max(1, std::min(8, 1024 / c->ncell_total));
    // the largest real*4 value whose real*8 promotion is below rv2: the same comparison in real*4
    float rv2 = (float)c->dp.rv2;
    if ((double)rv2 >= c->dp.rv2) rv2 = std::nextafterf(rv2, 0.0f);
    const float rvm = (float)std::sqrt(c->dp.rv2) + CULL_MARGIN;
#define LB(W)                                                                                    \
    hipLaunchKernelGGL(k_build_list<W>, dim3(c->ncell_total, parts), dim3(W * 64), 0, c->stream, \
                       c->a.pos4, c->a.num3, c->a.spec, c->cstart, c->ccount, c->cnum,            \
                       c->cell_rep, c->reps_d, c->rebuild, rv2, rvm * rvm, c->neigh_alloc, c->nlist,  \
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
