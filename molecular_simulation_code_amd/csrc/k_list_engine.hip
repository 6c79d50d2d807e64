// Verlet-list build of the device-resident engine, on half-width cells.
//
// The engine's lists only have to hold every pair closer than rv (order and exact
// boundary rounding are free, unlike the drop-in build in k_neighbor.hip).  That allows a
// cheaper search:
//  * cells are at least rv/2 wide, so a pair closer than rv lies within +-2 cells on each
//    axis: 125 stencil cells, 15.6 rv^3 of candidate volume instead of 27 rv^3;
//  * one workgroup owns one cell and stages its stencil in LDS in (dz, dy, dx) order with
//    the periodic image shift already added, so a candidate costs 3 subtractions and a
//    squared norm (no minimum image) and the 5 cells of a (dy, dz) row are contiguous;
//  * for each atom, 25 lanes bound the 25 rows at once: a row whose y-z rectangle is
//    farther than rv is skipped, and of the others only the x-cells meeting the chord
//    [x - w, x + w], w = sqrt(rv^2 - d_yz^2), are swept -- about 45 % of the stencil;
//  * sweeps go 64 candidates at a time, hits compacted with a ballot + popcount prefix.
// Culling distances carry a 0.01 A margin, far above the float rounding of positions, cell
// indices and image shifts, so culling never drops a pair the distance test would keep.
// A stencil larger than the LDS capacity is staged in pieces; per-atom counts then carry
// over in numneigh (each atom stays with the same wavefront).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "sort_device.h"

namespace sofia {
namespace {

// staged candidates per pass, by cells a workgroup takes (64 and 74 KiB of LDS)
constexpr int ECAP[3] = {0, 4096, 4736};
constexpr float CULL_MARGIN = 0.01f;  // A

// Two workgroups fit a CU's LDS; the second bound (waves per SIMD) keeps the register
// budget that lets both run (64 VGPRs at 16 waves per workgroup).
//
// COPY: the step's copy back (copy_back) in the first ncopy workgroups, side by side with the
// builds, which read the moved atoms where the sort put them (pos4, num3, spec and, for the
// exclusions' new ids, tt): a launch less in every step, and a rebuild's copy overlapped.
// 49.7 -> 46.9 us a step at 5,000 atoms, 75 -> 72.5 at 20,000 (Ewald), 507 -> 500 at 264,000.
//
// NX: x-neighbouring cells a workgroup takes together.  Two share the staging (150 cells for
// two instead of 125 for each, and one chain of dependent loads) and their ~43 atoms leave
// fewer of 16 wavefronts idle at the end than ~21 do.  With the plain rows below, a full build
// (copy back beside it) took 761 -> 656 us at 264,000 atoms, 604 -> 517 at 204,000; 64 VGPRs.
template <int WAVES, bool COPY, int NX>
__global__ void __launch_bounds__(WAVES * 64, WAVES * 2 / 4)
k_build_engine(int32_t ncopy, CopyArgs C, int32_t ncell, const float4 *__restrict__ pos4, const int32_t *__restrict__ num3,
               const int32_t *__restrict__ spec, const int32_t *__restrict__ cstart,
               const int32_t *__restrict__ ccount, const int32_t *__restrict__ cell_rep,
               const RepInfo *__restrict__ reps, const int32_t *__restrict__ rebuild,
               const int32_t *__restrict__ any, float rv, float rv2, int32_t na,
               int32_t *__restrict__ nlist, int32_t *__restrict__ numneigh,
               int32_t *__restrict__ maxcnt) {
    if (!*any) return;   // no replica rebuilds this step
    if (COPY && (int)blockIdx.x < ncopy) {
        copy_back(C, blockIdx.x * (WAVES * 64) + threadIdx.x, ncopy * (WAVES * 64));
        return;
    }
    const int first = COPY ? (int)blockIdx.x - ncopy : (int)blockIdx.x;
    const int stride = COPY ? (int)gridDim.x - ncopy : (int)gridDim.x;
    const int32_t *__restrict__ tt = C.tt;
    constexpr int W = 4 + NX, CELLS = 25 * W;     // stencil cells: W a row, 25 rows
    constexpr int SC = (CELLS + 63) / 64, CAP = ECAP[NX];
    __shared__ int32_t s_src[64 * SC];
    __shared__ int32_t s_cnt[64 * SC];
    __shared__ int32_t s_off[64 * SC + 1];
    __shared__ int32_t s_rlo[32], s_rhi[32];   // least and greatest atom id of each stencil row
    __shared__ float4 s_j[CAP + 128];         // (a row's last chunks read past its end)

    // a fixed grid walks the cells; slot s and s + stride stay on one XCD, and
    // xcd_block gives each XCD runs of neighbouring cells
    const int nslot = (ncell + NX - 1) / NX;
    for (int slot = first; slot < nslot; slot += stride) {
      const int cb = NX * xcd_block(slot, nslot), ce = min(cb + NX, ncell);
      for (int c = cb, span; c < ce; c += span) {
        span = 1;
        const int r = cell_rep[c];
        if (!rebuild[r]) continue;
        const RepInfo R = reps[r];
        if (!R.stencil5) continue;
        const int n = R.ncellD, lc = c - R.cell0;
        const int cx = lc % n, cy = (lc / n) % n, cz = lc / (n * n);
        if (NX == 2 && c + 1 < ce && cx + 1 < n) span = 2;   // (else the next row's: by itself)
        const int i0 = cstart[c], n0 = ccount[c], ni = n0 + (span == 2 ? ccount[c + 1] : 0);
        if (ni == 0) continue;
        const float box = R.box, rn = R.rn;

        const int tid = threadIdx.x;
        if (tid < 64 * SC) {
            int cnt = 0, src = 0;
            if (tid < CELLS) {
                int x = cx + tid % W - 2, y = cy + (tid / W) % 5 - 2, z = cz + tid / (5 * W) - 2;
                x += (x < 0) ? n : ((x >= n) ? -n : 0);     // n >= 5: one wrap at most
                y += (y < 0) ? n : ((y >= n) ? -n : 0);
                z += (z < 0) ? n : ((z >= n) ? -n : 0);
                const int nc = R.cell0 + x + (y + z * n) * n;
                src = cstart[nc];
                cnt = ccount[nc];
            }
            s_src[tid] = src;
            s_cnt[tid] = cnt;
        }
        __syncthreads();
        if (tid < 64) {   // exclusive scan of the counts, SC per lane
            int v = 0;
#pragma unroll
            for (int q = 0; q < SC; ++q) v += s_cnt[SC * tid + q];
            int at = -v;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(v, o, 64);
                if (tid >= o) v += u;
            }
            at += v;
#pragma unroll
            for (int q = 0; q < SC; ++q) {
                s_off[SC * tid + q] = at;
                at += s_cnt[SC * tid + q];
            }
            if (tid == 63) s_off[64 * SC] = v;
        } else if (tid < 96) {
            const int row = tid - 64;
            int lo = 0x7fffffff, hi = -1;
            for (int q = W * row; q < W * row + W && row < 25; ++q) {
                if (s_cnt[q] == 0) continue;
                lo = min(lo, s_src[q]);
                hi = max(hi, s_src[q] + s_cnt[q] - 1);
            }
            s_rlo[row] = lo;
            s_rhi[row] = hi;
        }
        __syncthreads();
        const int total = s_off[CELLS];

        // the wave index is uniform: the atoms a wave takes, and their exclusions, stay scalar
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const float rvm = rv + CULL_MARGIN, rvm2 = rvm * rvm;
        const float irn = 1.0f / rn;

        for (int g0 = 0; g0 < total || g0 == 0; g0 += CAP) {
            const int g1 = min(total, g0 + CAP);
            if (g0 > 0) __syncthreads();   // the previous pass is done with s_j
            // a wave stages whole (dy, dz) rows: the row's cells are found with compares
            // against its (uniform) cell offsets, and the y / z image shifts are uniform
            for (int row = wave; row < 25; row += WAVES) {
                const int k0 = W * row;
                const int r0 = max(s_off[k0], g0), r1 = min(s_off[k0 + W], g1);
                if (r0 >= r1) continue;
                const int ay = cy + row % 5 - 2, az = cz + row / 5 - 2;
                const float sy = (ay < 0) ? -box : ((ay >= n) ? box : 0.0f);
                const float sz = (az < 0) ? -box : ((az >= n) ? box : 0.0f);
                int b[W - 1], d[W];
#pragma unroll
                for (int q = 0; q < W; ++q) {
                    if (q > 0) b[q - 1] = s_off[k0 + q];
                    d[q] = s_src[k0 + q] - s_off[k0 + q];   // staged index -> atom id
                }
                for (int f = r0 + lane; f < r1; f += 64) {
                    int dk = 0, dd = d[0];
#pragma unroll
                    for (int q = 1; q < W; ++q) {
                        dk += (int)(f >= b[q - 1]);
                        dd = (f >= b[q - 1]) ? d[q] : dd;
                    }
                    const int id = f + dd;
                    const int ax = cx + dk - 2;
                    float4 p = pos4[id];
                    p.x += (ax < 0) ? -box : ((ax >= n) ? box : 0.0f);
                    p.y += sy;
                    p.z += sz;
                    p.w = __int_as_float(id);
                    s_j[f - g0] = p;
                }
            }
            __syncthreads();

            for (int ii = wave; ii < ni; ii += WAVES) {
                const int i = i0 + ii;
                const float4 xi = pos4[i];
                const int n3 = num3[i];
                // the atom's exclusions (wave-uniform: scalar loads, held in scalar registers);
                // exmin..exmax holds them and the atom itself
                int ex[SPEC];
                int exmin = i, exmax = i;
#pragma unroll
                for (int l = 0; l < SPEC; ++l) {
                    int v = spec[(size_t)i * SPEC + l];
                    if (COPY) v = (l < n3) ? tt[v] : -1;
                    ex[l] = (l < n3) ? v : -1;
                    exmin = (l < n3) ? min(exmin, v) : exmin;
                    exmax = (l < n3) ? max(exmax, v) : exmax;
                }
                // row bounds: lane k < 25 takes row (dy, dz) = (k % 5 - 2, k / 5 - 2)
                int rlo = 0, rhi = 0;
                if (lane < 25) {
                    const float ylo = (float)(cy + lane % 5 - 2) * rn, zlo = (float)(cz + lane / 5 - 2) * rn;
                    const float ey = fmaxf(0.0f, fmaxf(ylo - xi.y, xi.y - (ylo + rn)) - CULL_MARGIN);
                    const float ez = fmaxf(0.0f, fmaxf(zlo - xi.z, xi.z - (zlo + rn)) - CULL_MARGIN);
                    const float dyz = ey * ey + ez * ez;
                    if (dyz < rvm2) {
                        const float w = sqrtf(rvm2 - dyz);
                        const int ox = (NX == 2 && ii >= n0) ? 1 : 0;   // the atom's own cell
                        const int a = min(ox + 2, max(ox - 2, (int)floorf((xi.x - w) * irn) - cx));
                        const int b = min(ox + 2, max(ox - 2, (int)floorf((xi.x + w) * irn) - cx));
                        rlo = max(s_off[lane * W + a + 2], g0);
                        rhi = min(s_off[lane * W + b + 3], g1);
                    }
                }
                uint64_t rows = __ballot(rhi > rlo);
                const uint64_t rows_ex =
                    __ballot(lane < 25 && s_rlo[lane & 31] <= exmax && s_rhi[lane & 31] >= exmin);
                int cnt = (g0 == 0) ? 0 : numneigh[i];
                int32_t *out = nlist + (size_t)i * na;
                // test one staged candidate per lane; hits appended in staged order.  PLAIN: a row
                // without the atom or an exclusion of it (all but one or two rows of a water), whose
                // hits the list has room for.  Else the tests combine without short-circuit (no
                // branch per condition) and the id compares run only for a chunk where some lane
                // falls in [exmin, exmax] (measured cheaper than compares bounded by the atom's
                // exclusion count).
                auto sweep = [&](auto plain, const float4 pj, const bool valid) {
                    constexpr bool PLAIN = decltype(plain)::value;
                    const int z = __float_as_int(pj.w);
                    const float dx = xi.x - pj.x, dy = xi.y - pj.y, dz = xi.z - pj.z;
                    bool pred = valid & (dx * dx + dy * dy + dz * dz < rv2);
                    if (!PLAIN && __ballot(pred & (z >= exmin) & (z <= exmax))) {
                        pred = pred & (z != i);
#pragma unroll
                        for (int l = 0; l < SPEC; ++l) pred = pred & (ex[l] != z);
                    }
                    const uint64_t mask = __ballot(pred);
                    const uint32_t pos = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)cnt));
                    if (PLAIN ? pred : pred & (pos < (uint32_t)na))
                        *(int32_t *)((char *)out + (pos << 2)) = z;   // na < 2^29: one row of a list
                    cnt += __popcll(mask);
                };
                // two chunks per iteration, both LDS reads issued before either is used; lanes
                // past the row are masked off
                auto sweep_row = [&](auto plain, const int lo, const int hi) {
                    for (int base = lo; base < hi; base += 128) {
                        const float4 p0 = s_j[base + lane];
                        const float4 p1 = s_j[base + 64 + lane];
                        sweep(plain, p0, lane < hi - base);
                        if (base + 64 < hi) sweep(plain, p1, lane < hi - base - 64);
                    }
                };
                while (rows) {
                    const int k = __builtin_ctzll(rows);
                    rows &= rows - 1;
                    const int lo = __builtin_amdgcn_readlane(rlo, k) - g0;
                    const int hi = __builtin_amdgcn_readlane(rhi, k) - g0;
                    if (!(rows_ex >> k & 1) && cnt + (hi - lo) <= na) sweep_row(std::true_type{}, lo, hi);
                    else sweep_row(std::false_type{}, lo, hi);
                }
                if (lane == 0) {
                    numneigh[i] = cnt;
                    if (g1 >= total && cnt > na) atomicMax(maxcnt, cnt);
                }
            }
            if (g1 >= total) break;
        }
        __syncthreads();   // the shared arrays are refilled for the next cell
      }
    }
}

inline int nblk(int n, int b) { return (n + b - 1) / b; }

}  // namespace

void launch_build_list_engine(sofia_ctx *c, bool copy) {
    const float rv2 = (float)c->dp.rv2;
    const float rv = std::sqrt(rv2);
    int items = 0;
    const CopyArgs C = copy ? copy_args(c, SORT_STEP, &items) : CopyArgs{};
    const AtomArrays &A = copy ? c->b : c->a;
    // two workgroups of 16 wavefronts fit a CU (64 KiB of staged candidates each): more would
    // only lengthen the launch of a step that rebuilds nothing
    // two cells a workgroup where the compute units have two rounds of them all the same, and
    // the stencil of two fits the staging in one pass: a full build by one / two cells 62 / 76 us
    // at 930 cells (20,000 atoms), 147 / 140 at 2,500, 709 / 656 at 12,000
    const double percell = (double)c->N / std::max(1, c->ncell_total);
    const int nx = (c->list_waves >= 16 && c->ncell_total >= 2048 && 150.0 * percell < 4300.0) ? 2 : 1;
    auto go = [&](auto kernel, int waves) {
        // (whole rounds of the XCDs, so that the builds' blocks keep theirs)
        const int ncopy = copy ? (std::min(nblk(items, waves * 64), 128) + 7) / 8 * 8 : 0;
        hipLaunchKernelGGL(kernel, dim3(ncopy + std::min((c->ncell_total + nx - 1) / nx, 8192 / waves)),
                           dim3(waves * 64), 0, c->stream, ncopy, C, c->ncell_total, A.pos4, A.num3, A.spec,
                           c->cstart, c->ccount, c->cell_rep, c->reps_d, c->rebuild, c->rebuild + c->nrep,
                           rv, rv2, c->neigh_alloc, c->nlist, c->numneigh, c->maxcnt);
    };
    if (c->list_waves >= 16 && nx == 2) copy ? go(k_build_engine<16, true, 2>, 16) : go(k_build_engine<16, false, 2>, 16);
    else if (c->list_waves >= 16) copy ? go(k_build_engine<16, true, 1>, 16) : go(k_build_engine<16, false, 1>, 16);
    else if (c->list_waves >= 8) copy ? go(k_build_engine<8, true, 1>, 8) : go(k_build_engine<8, false, 1>, 8);
    else copy ? go(k_build_engine<4, true, 1>, 4) : go(k_build_engine<4, false, 1>, 4);
}

}  // namespace sofia
