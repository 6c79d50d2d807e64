// Internal declarations shared by the HIP translation units of libsofia_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/sofia_hip.h"

namespace sofia {

constexpr int SPEC = 12;                     // specbond slots per atom
constexpr double FIX_SCALE = 4294967296.0;   // forces: 2^32 units per kcal/mol/A
constexpr double FIX_INV = 1.0 / FIX_SCALE;
constexpr double EFIX_SCALE = 16777216.0;    // energies and virial: 2^24 units per kcal/mol
constexpr double EFIX_INV = 1.0 / EFIX_SCALE;
constexpr float PAIR_QUANT = 16777216.0f;    // 2^24: per-pair quantum of the mixed kernel
constexpr int PAIR_SHIFT = 8;                // 2^32 / 2^24

// energy / virial accumulator slots (int64 fixed point, per replica)
enum {
    E_LJ = 0, E_COUL, E_POT14, E_COUL14, E_BOND, E_ANGLE, E_DIHED, E_KE,
    V_X, V_Y, V_Z, E_CORR, E_IMPRO, NE
};
// Each (replica, slot) accumulator exists in ESPREAD copies, one 128-byte line apart, and a
// workgroup adds to copy blockIdx % ESPREAD: tens of thousands of wavefronts adding to one
// address serialise at the L2, spreading them over lines does not.  The host sums the copies
// (integers: the total does not depend on which copy a wave used).
constexpr int ESPREAD = 16;
constexpr int ECOPY = 16;                       // int64 words between copies (128 B)
constexpr int EACC_PER_SLOT = ESPREAD * ECOPY;
inline size_t eacc_len(int nrep) { return (size_t)nrep * NE * EACC_PER_SLOT; }

// Per-replica geometry and thermostat (device table).
struct RepInfo {
    float box, ibox, rn;
    int32_t ncellD, ncellT;
    int32_t atom0, natom;
    int32_t cell0;
    int32_t stencil5; // engine grid of cells >= rv/2 with a +-2 stencil (k_build_engine)
    double fric;      // friction * amu2e (kcal/mol per amu*A/fs)
    double gconst;    // noise amplitude * amu2e
    uint64_t seed;
    double chk2;      // engine rebuild threshold on |displacement|^2 (complete-list criterion)
    double fscale;    // 2^32 / box: coordinate -> fixed-point record of the mixed pair kernel
};

// Scalars passed by value to every kernel.
struct DevParams {
    float coulpre, dt, kcal2amu;
    int32_t ntypes;
    double rcut2, cut_coulsq, rv2, rvrc2;
    double alpha, gewald, e_shift, f_shift, ewald_p, ewald_f;
    double a1, a2, a3, a4, a5, my_pis, my_pis_inv, amu2e;
    double fudge12, fudge13, fudge14;
    double shake_tol;
    int32_t shake_maxiter;
    int32_t nrep;
    int32_t natom;
    int32_t neigh_alloc;
    float tab_r0, tab_inv_h;     // DSF Coulomb table of the mixed kernel: r0 + k / inv_h
    int32_t tab_n;               // bins per table; each table has one more, all-zero bin
};

constexpr int DSF_TAB_BINS = 1024;

constexpr int CHUNK_SHIFT = 8;   // cells to a run of the sort's prefix: 256

// Engine bonded work in bundles of whole molecules: item kinds and the widths of their lists.
enum BondedKind { BK_PAIR14 = 0, BK_BOND = 1, BK_ANGLE = 2, BK_TORSION = 3, BK_IMPRO = 4, BK_COUNT = 5 };
constexpr int BUNDLE_SLOTS = 192;   // atoms per bundle (its forces sit in LDS)
constexpr int BUNDLE_TERMS = 256;   // items per bundle when molecules are packed together
constexpr int BUNDLE_THREADS = 256; // one workgroup per bundle
__host__ __device__ inline int bonded_width(int kind) {
    return kind == BK_BOND ? 3 : (kind == BK_ANGLE ? 4 : 5);
}

struct HostWords {
    int32_t maxcnt, shake_err, shake_iters, type_err, moved, pad[11];
};

// Per-atom arrays that the cell sort permutes (one set; the context keeps two).
struct AtomArrays {
    float4 *pos4 = nullptr;     // x, y, z, type (int bits)
    float *q = nullptr;
    int32_t *gid = nullptr;
    int32_t *num1 = nullptr, *num2 = nullptr, *num3 = nullptr;
    int32_t *spec = nullptr;    // [N][12] global 0-based, -1 = empty
    float *v32 = nullptr;       // AoS coords (3N)
    double *xd = nullptr;       // SoA x | y | z (3N)
    double *vd = nullptr;       // SoA (3N)
    int32_t *mol = nullptr;     // molecule id (cluster analysis), -1 = solvent
    int32_t *wclus = nullptr;   // engine: SETTLE water whose oxygen this atom is, -1 = none
};

}  // namespace sofia

struct sofia_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    sofia_params p{};
    sofia::DevParams dp{};
    int32_t nrep = 0, N = 0;
    std::vector<sofia::RepInfo> reps_h;
    sofia::RepInfo *reps_d = nullptr;
    int32_t ncell_total = 0, ncell_cap = 0;

    sofia::AtomArrays a, b;     // a = current, b = gather target
    int32_t *rep = nullptr;     // replica of each atom (invariant under the sort)

    // reference-format and engine state that is not permuted as a set
    float *dr32 = nullptr;      // drx | dry | drz (3N), real*4
    double *drd = nullptr;      // FP64 displacement since the last build (engine)
    double *fnb = nullptr;      // nonbond forces, SoA (3N)
    long long *fix = nullptr;   // fixed-point accumulator of every other force, SoA (3N)
    long long *fscratch = nullptr;   // fixed-point scratch for drop-in outputs (3N)
    float *stage32 = nullptr;        // AoS real*4 staging for drop-in inputs/outputs (3N)
    long long *fix14 = nullptr;      // force wrapper: the 1-4 term's fixed-point sums (3N, lazy)

    // cluster analysis: global solute-molecule index per atom lives in AtomArrays::mol
    int32_t nmol = 0;
    int32_t *mol_rep = nullptr, *uf_parent = nullptr, *uf_size = nullptr, *uf_largest = nullptr;
    // get_greatestCluster: first molecule of each replica (nrep + 1), per-molecule centres,
    // their construction, the density counts, and per-replica results
    int32_t *gc_first = nullptr, *gc_refgid = nullptr, *gc_cnt = nullptr, *gc_dens = nullptr;
    long long *gc_sum = nullptr;
    double *gc_refx = nullptr, *gc_com = nullptr;
    unsigned long long *gc_key = nullptr;
    int32_t *gc_surface = nullptr;

    // cells
    int32_t *ccount = nullptr, *cstart = nullptr, *cnum = nullptr, *cell_rep = nullptr;
    int32_t *cbin = nullptr;        // binning counters (zero between sorts)
    int32_t *bucket = nullptr;      // bucket_cap atom ids per cell, in binning order
    int32_t bucket_cap = 0;
    size_t bucket_len = 0;
    // atoms past a full bucket: how many (zero between sorts), their (cell, id), and the ids of
    // such cells' atoms gathered for the ranking
    int32_t *nover = nullptr, *fat = nullptr;
    int2 *over = nullptr;
    // where a replica has many cells: atoms in each run of 1 << CHUNK_SHIFT cells, which the
    // sort's prefix takes instead of their counts one by one
    int32_t *chunk = nullptr;
    bool chunked = false;
    int32_t *tt = nullptr, *atombin = nullptr;

    // Verlet list
    int32_t *nlist = nullptr, *numneigh = nullptr;
    int32_t neigh_alloc = 0;
    size_t nlist_cap = 0;
    int32_t *maxcnt = nullptr;  // device scalar
    bool have_list = false;

    // flags
    int32_t *rebuild = nullptr;     // per replica
    int32_t *nbuilds = nullptr;     // per replica
    int32_t *shake_err = nullptr;   // device scalar
    int32_t *shake_iters = nullptr; // device scalar

    // topology (global 0-based indices)
    int32_t *bondlist = nullptr, nb = 0;
    int32_t *anglelist = nullptr, na = 0;
    int32_t *dihedlist = nullptr, nd = 0;
    int32_t *torsions = nullptr, ntor = 0;
    int32_t *improlist = nullptr, nimp = 0;   // (i1, i2, i3 central, i4, type) per improper
    int32_t *shake_num = nullptr, *shake_atoms = nullptr, ns = 0;
    int32_t *topo_stage = nullptr;   // topology in the host's id layout, on its way out
    uint32_t *rdf_hist = nullptr;    // sofia_rdf_calc's counts (rdf_cap bins, lazy)
    int32_t rdf_cap = 0;
    size_t topo_stage_len = 0;
    // engine constraints: indices of the iteratively solved clusters grouped by kind 1, 3,
    // 4, -3 (each group padded with -1 to whole wavefronts, as the counts are), and the count
    // of symmetric rigid waters (SETTLE, found through AtomArrays::wclus);
    // built when the engine sets up its lists
    int32_t *shake_kidx = nullptr;
    int32_t shake_kcount[5] = {0, 0, 0, 0, 0};
    double *shake_bond = nullptr;
    int4 *water = nullptr;       // per SHAKE cluster: rigid-water bond/angle types + fused flag
    bool water_split = false;    // water bonds/angles moved into the SHAKE kernel
    int32_t *ebond = nullptr, nbe = 0;    // engine bond / angle lists without the fused waters
    int32_t *eangle = nullptr, nae = 0;
    // engine bonded bundles (k_bonded_bundles): per bundle the ranges of its term and atom-slot
    // records; nbundle = 0 runs the per-kind kernels instead
    int32_t nbundle = 0;
    // run the bundles (tuning choice) rather than one thread per item: 7 against 11 us at
    // 5,000 atoms, 8 / 17 at 55,000, 16 / 47 at 264,000, 12 / 39 at 204,000 (1,200 glycines)
    bool bonded_bundles = true;
    int4 *bund_heads = nullptr;   // first and last term, first slot, replica << 8 | slots
    int32_t *bund_slots = nullptr;
    int2 *bund_terms = nullptr;

    // force field
    float4 *ljtab = nullptr;    // (lj1, lj2, lj3, lj4) per type pair
    double4 *lj14 = nullptr;    // (lj14_1..4) per type pair
    double *mass = nullptr;     // per type
    double4 *mtab = nullptr;    // per type: m, dt/2 kcal2amu / m, sqrt(m), 1/m
    double *bond_k = nullptr, *bond_r0 = nullptr, *angle_k = nullptr, *angle_th0 = nullptr;
    double *tors_k = nullptr, *tors_n = nullptr, *tors_shift = nullptr;
    double *tors_cs = nullptr;  // per torsion type: cos(shift), sin(shift)
    double *impro_k = nullptr, *impro_chi0 = nullptr;   // per improper type
    int32_t *impro_dn = nullptr;   // cvff style: (d, n) per improper type
    int32_t impro_style = 0;       // 0 harmonic (lammps14), 1 cvff (amber wrapper)
    float4 *dsf_tab = nullptr;  // cubic pieces of the DSF Coulomb force / energy (mixed kernel)
    int4 *pfix = nullptr;       // mixed kernel positions: x 2^32 / box mod 2^32, type (per launch)
    // charges by atom type (every atom of a type carries the same charge): the pair kernels
    // then take C q_i q_j from ptab (lj1, lj2, C q_i q_j, q_j), the mixed one with 12-byte records
    bool q_by_type = false;
    float4 *ptab = nullptr;
    std::vector<float4> lj_host;   // lj1..lj4 per type pair, as uploaded
    int32_t nbt = 0, nat = 0, ntt = 0;
    bool have_ff = false;

    // energies (int64 fixed point, per replica x NE)
    long long *eacc = nullptr;
    bool eacc_zero = false;      // eacc is known to be all zero (launch_report cleared it)
    // page-locked words the device writes for the host (launch_report, launch_list_done,
    // k_check32): read after one synchronisation, with no copy of their own
    sofia::HostWords *hw = nullptr;
    long long *hw_e = nullptr;   // nrep x NE energy sums, behind hw
    // a launched segment whose energies the host has not taken yet: their sums stand in eacc,
    // or (another call needed eacc since) in hw_seg, which a report ahead of that call wrote
    enum { SEG_NONE, SEG_EACC, SEG_SAVED } segment = SEG_NONE;
    long long *hw_seg = nullptr; // nrep x NE, behind hw_e
    // blocks that hold the context's fixed-size arrays (one allocation instead of dozens)
    std::vector<void *> blocks;
    int gid_perm = -1;           // global ids of every replica a permutation: 1, 0, -1 unknown
    std::vector<double> last_e;

    // engine
    bool engine_ready = false;
    bool engine_grid = false;    // cells re-sized for complete lists (first md_init/md_resume)
    int32_t n_stencil5 = 0;      // replicas on the half-width engine grid
    double skin = -1.0;          // engine skin (A); < 0: the reference's pad
    uint64_t *step_d = nullptr;  // per-replica step counters (Langevin key)
    uint64_t step_h = 0;
    // lanes per atom of the pair kernels and threads per workgroup of the mixed one; < 0 and 0
    // until the caller tunes them: chosen by kernel and size (mixed_lanes and its neighbours)
    int lanes = -1, block = 0, list_waves = 16;
    hipGraphExec_t graph = nullptr;    // one MD step
    hipGraphExec_t graphk = nullptr;   // graph_steps MD steps
    int32_t graph_steps = 1;

    // Grow-and-redo of an MD segment whose Verlet list overflowed (the engine's form of the
    // reference's grow-and-rebuild, Source/mod_neighbor.f90:258-298): the state at the start
    // of each segment is kept on the device, and a segment that overflowed is run again
    // from it with a larger list stride.
    bool redo = true;
    sofia::AtomArrays snap{};
    int32_t *snap_topo = nullptr;
    size_t snap_topo_cap = 0;
    double *snap_fnb = nullptr, *snap_drd = nullptr;
    long long *snap_fix = nullptr;
    uint64_t *snap_step = nullptr;
    int32_t *snap_nbuilds = nullptr;
    bool snap_valid = false;
    int32_t snap_nsteps = 0, snap_graph = 0;
    int32_t redos = 0;
    int32_t stride_floor = 0;          // smallest stride the next engine list set-up uses
    double headroom = 1.5;             // engine list stride: headroom x the largest count
    bool has_thermostat = false;

    // host staging (pinned) for the asynchronous pair-kernel drop-in
    void *pinned = nullptr;
    size_t pinned_bytes = 0;
    int async_mode = -1;         // pair-kernel mode in flight, -1 = none
};

namespace sofia {

// ------------------------------------------------------------------ kernel launchers
// neighbor build (k_neighbor.hip)
// What the sort carries along with the atoms: the drop-in's real*4 state, the engine's FP64
// state too, or (inside an engine step) also the fixed-point forces already set for the step
// and the pair kernel's position records.
enum SortMode { SORT_DROPIN = 0, SORT_ENGINE = 1, SORT_STEP = 2 };
// bonded: with the step's bonded terms (where sort_takes_bonded)
// (leave_copy: its copy back is left to launch_build_list, where list_takes_copy; water: and
// with the rigid waters' own terms)
void launch_sort(sofia_ctx *c, SortMode mode, bool bonded = false, bool energies = false,
                 bool leave_copy = false, bool water = false);
bool list_takes_copy(const sofia_ctx *c);
bool sort_takes_bonded(const sofia_ctx *c);
struct BinArgs;
void launch_bundles_bin(sofia_ctx *c, const BinArgs &B, int bin_grid, bool energies, bool water);
void launch_host_ids(sofia_ctx *c, const int32_t *src, int32_t *dst, size_t items, int width,
                     int nidx);
void launch_rdf(sofia_ctx *c, int32_t itype, int32_t jtype, double delta, int32_t nbins,
                uint32_t *hist);
void launch_build_list(sofia_ctx *c, bool copy = false);   // copy: with a step's copy back
void launch_build_list_engine(sofia_ctx *c, bool copy);
void launch_check_neighbor(sofia_ctx *c);
void launch_set_rebuild(sofia_ctx *c, int32_t value);
void launch_finish_rebuild(sofia_ctx *c);
// Ends a rebuild whose lists fit (counts it, lowers the flags) and tells the host the largest
// count either way; local (optional): tt as 1-based ids within the replica.
void launch_list_done(sofia_ctx *c, int32_t *local);

// nonbond (k_nonbond.hip): mode 0 = DSF FP64, 1 = DSF mixed, 2 = Ewald real space (FP32)
// records: the mixed kernel's position records are already up to date
// close: the books of the rebuild before it
void launch_nonbond(sofia_ctx *c, int mode, bool energies, bool records = false, bool close = false);
void launch_count_pairs(sofia_ctx *c, unsigned long long *out);

// bonded (k_bonded.hip)
void launch_correct(sofia_ctx *c, int which, long long *fout);
void launch_pair14(sofia_ctx *c, long long *fout);
void launch_bonded_engine(sofia_ctx *c, bool energies);
void launch_bonded_dropin(sofia_ctx *c, long long *fout);
void launch_bonded_wrapper(sofia_ctx *c, const double *xd, long long *fout, long long *f14);
int build_bonded_bundles(sofia_ctx *c);   // host: molecules of the engine's bonded items
void drop_bonded_bundles(sofia_ctx *c);
void launch_dsf_mixed(sofia_ctx *c, bool energies, float *ff32, bool from_xd, bool records, bool close);
// bytes per position record the mixed pair kernel reads (12 or 16), 0 in the other modes
int record_bytes(const sofia_ctx *c);

// integration (k_integrate.hip)
void launch_zero_forces(sofia_ctx *c, long long *f, bool energies);
void launch_fix_to_coords(sofia_ctx *c, const long long *f, float *out_aos);
void launch_nve_v32(sofia_ctx *c, float dt_partial, const float *ff_aos);
void launch_nve_x32(sofia_ctx *c);
void launch_pbc32(sofia_ctx *c);
void launch_berendsen32(sofia_ctx *c, const double *mu_dev);
void launch_shake32(sofia_ctx *c, int iflag, float *ff_aos, double *vir_dev);
void launch_langevin32(sofia_ctx *c, float fric, float gconst, uint64_t seed, uint64_t step,
                       float *out_aos);
void launch_engine_from32(sofia_ctx *c);
void launch_engine_to32(sofia_ctx *c);
void launch_nve_v64(sofia_ctx *c, bool ke);
void launch_advance(sofia_ctx *c, bool kick2);
void launch_langevin64(sofia_ctx *c);
// step: the launch also ends the engine step (rebuild flags down, step counters on)
void launch_shake64(sofia_ctx *c, bool energies, bool step = false);
void launch_zero_energies(sofia_ctx *c);
void launch_water_bonded(sofia_ctx *c);
void launch_copy16(sofia_ctx *c, size_t n16, const void *src, void *dst);
void launch_put_state(sofia_ctx *c, bool v, bool q, bool gid);
// with the report of the call
void launch_merge_report(sofia_ctx *c, float *ff32, const long long *f14, const long long *fb);
// Energy sums (cleared on the device) and flags to the host words
void launch_report(sofia_ctx *c, bool clear_shake = false);
// ahead of whatever clears or reads the energy sums: those of a launched segment put aside
void launch_save_segment(sofia_ctx *c);
void launch_start_forces(sofia_ctx *c, long long *a, long long *b, double *xd);
// FP64 SoA (plus fixed point) <-> AoS; with gid, dst rows in global-id order of each replica
void launch_soa_to_aos(sofia_ctx *c, const double *src, const long long *fix, const int32_t *gid, double *dst);
void launch_aos_to_soa(sofia_ctx *c, const double *src, double *dst);
void launch_step_add(sofia_ctx *c, long long delta);
void launch_minimize_step(sofia_ctx *c, double gamma, double max_disp);

// cluster analysis (k_cluster.hip)
int cluster_largest(sofia_ctx *c, float rcontact, const std::vector<int> &o_types,
                    const std::vector<int> &n_types, int32_t *largest);
int cluster_greatest(sofia_ctx *c, double denscut, int32_t densmin, int32_t *total, int32_t *core,
                     int32_t *surface);
int cluster_greatest_noalloc(int32_t n, const double *x, const int32_t *gid, const int32_t *mol,
                             int32_t nmol, float box, double denscut, int32_t densmin,
                             int32_t *out, hipStream_t s);

// Lanes per atom of the mixed pair kernel while the caller has not tuned them: its exact force
// sums do not depend on them.  Small systems need more lanes to spread over the chip (one launch,
// 5,000 atoms: 12.7 us at 64 lanes, 13.6 at 32, 15.8 at 16), large ones fewer shuffles and
// idle row tails (55,000: 76 / 64 / 60; 264,000: 433 / 353 / 321).  An atom's energies and virial
// are summed in floating point, in an order set by the lanes: launches with energies take one
// value for every size, so that a replica's energies do not depend on what it is batched with.
inline int mixed_lanes(const sofia_ctx *c, bool energies = false) {
    if (c->lanes >= 0) return c->lanes;
    if (energies) return 16;
    return c->N < 12000 ? 64 : (c->N < 40000 ? 32 : 16);
}
// The FP64 and Ewald kernels sum in floating point, in an order set by the lanes: one value
// for every size, so that a replica's last bits do not depend on what it is batched with.
inline int ordered_lanes(const sofia_ctx *c) { return c->lanes >= 0 ? c->lanes : 16; }
// Threads per workgroup of the mixed pair kernel: each workgroup stages the DSF table (16 KB)
// and the type-pair tables in LDS, so large workgroups spend less of the load path on it
// (-4.8 % at 1,280,000 atoms), but a grid of few of them leaves compute units idle: by
// workgroups of 256 / 512 / 1024 threads and the lanes above, 12.6 / 13.1 / 14.8 us at 5,000
// atoms, 28.5 / 27.4 / 30.6 at 20,000, 63 / 61 / 66 at 55,000.
inline int mixed_block(const sofia_ctx *c, bool energies) {
    if (c->block > 0) return c->block;
    if (energies) return 512;   // two tables to stage
    if ((long long)c->N * mixed_lanes(c) / 1024 >= 1024) return 1024;
    return c->N < 6000 ? 256 : 512;
}

// error helpers (sofia_api.cpp)
int fail(int code, const std::string &msg);
int check_hip(hipError_t e, const char *what);

}  // namespace sofia

#define SOFIA_HIP(call)                                                   \
    do {                                                                  \
        hipError_t e_ = (call);                                           \
        if (e_ != hipSuccess) return sofia::check_hip(e_, #call);         \
    } while (0)
