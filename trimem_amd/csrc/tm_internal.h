// tm_internal.h -- launchers shared between the library's translation units.
#pragma once

#include "tm_common.h"

namespace tmh {

// Pair cache of the cell-list repulsion query (single meshes).  Between
// rebuilds of the cell list the candidates of a vertex are fixed (the stored
// stencil list of its cell, or the stencil rows of the cell it has moved
// to), and exclusion depends on the topology only.  A recording launch runs
// the full query with radius lc1 + skin and keeps, per vertex and lane, the
// non-excluded candidates it meets, in the lane's visit order; later
// launches replay a list with the exact lc1 test while neither the vertex nor
// one of its candidates has moved so far that another candidate can have come
// within lc1, and the vertex is in the cell it was recorded in (the full query
// would visit the same candidates in the same order).  Each lane then adds the
// same terms in the same order as the full query: the results are
// bit-identical.
constexpr int kPairLanes = 8;      // lanes per vertex of the query
// Recorded candidates per lane; a vertex with more takes the full query every
// time, and the launch waits for it.  With 4, and a thread for each vertex's
// replay, an evaluation of a disc of 40962 vertices whose sheets are 1.2 mean
// edges apart took 383 us at exclusion level 0, 179 at 1 and 63.8 at 2; with 8,
// and eight lanes for each replay, 61.2, 58.3 and 51.1.
constexpr int kPairCap = 8;
constexpr double kPairSkin = 0.2;  // skin = 0.2 lc1
// A vertex is slow while it has moved less than 0.25 skin from the snapshot of
// the last recording of all lists, else fast.  Lists are replayed for slow
// vertices with no fast one among their candidates.  A slow vertex that left the
// cell its list was recorded in records it again there (the snapshot stays, and
// again only while its candidates are slow), so two lists can be recorded at
// different times: a pair's distance then changed by at most 4 x 0.25 skin since
// either list was recorded.
constexpr double kPairLimit = 0.25;
// Recorded counts of a vertex without a non-excluded candidate within lc1 + skin
// in the stencil of any cell that a slow vertex can be in: no pairs, whichever of
// them it is in.
constexpr unsigned kEmptyAround = 0xf0000000u;    // no count reaches 15
// Looked for by recordings of meshes of at most this many vertices.  It costs the
// recording a chain of loads and spares the replays that of the vertices that
// change cells: at 2562 vertices a recording takes 15.3 us instead of 7.0, the
// queries of a trajectory 9.9 instead of 13.9 each.  At 163842, where a recording
// is bound by its loads, a step with its ten queries takes as long with it as
// without.
constexpr int kAroundVerts = 16384;
// Recording all lists again costs the query several times what the full queries
// round a few fast vertices do, but those are paid on every evaluation.  A
// trajectory that goes astray is rejected and takes its fast vertices back with it;
// vertices that drift stay fast.  So all lists are recorded again when the end of a
// trajectory with fast vertices is accepted, or after kPatience evaluations in a row
// (HMC without rebuilds: 1963 steps/s at 40962 vertices and 1471 at 163842 while fast
// vertices stayed until there were too many, 2470 and 1662 so).
constexpr int kPatience = 12;
// More fast vertices than this in one block, or in all, record at once.
constexpr int kFastSeg = 32, kFastMax = 256, kFastRow = kFastSeg + 1;
struct PairCache {
    double* x_snap;         // [3N] positions at the recording; null: no cache
    int* cell;              // [N] cell (query_cell) at the recording, -1: replay not allowed
    unsigned* cnt;          // [N] recorded candidates of each lane, 4 bits per lane
    int* ent;               // [8 kPairCap N] ids, lane-major per vertex
    double* disp_part;      // [disp_n] max |x - x_snap|^2 per pass-1 block (written by pass 1)
    int* fast;              // [kFastRow disp_n] per block with fast vertices: their number and build-time cells
    int disp_n;
    int* dforce;            // replica groups: device flag, nonzero records (the reduction clears it)
    // [0] evaluations in a row with fast vertices, [1] the same after this one: the
    // query stores it, the sums' last step takes it over
    int* streak;
    double skin;
    double limit2;          // fast: |x - x_snap|^2 >= limit2
    int force;              // single meshes: 1 records in this launch
};
constexpr int kCachedVerts = 256;    // vertices per block of the cached query
constexpr int kPass1Verts = 256;     // vertices (one lane each) per block of pass 1

// ------------------------------------------------------- block mapping ---
// Workgroups are dispatched round-robin over the 8 XCDs (block b on XCD
// b % 8), each with its own L2.  Launching a multiple of 8 blocks and giving
// XCD x the logical blocks [x * G/8, (x+1) * G/8) makes each XCD work on one
// contiguous range of (spatially ordered) vertices, so its L2 holds that
// region and its halo instead of a slice of the whole mesh.
constexpr int kXcds = 8;
__device__ __forceinline__ int logical_block()
{
    const int chunk = gridDim.x / kXcds;
    return (blockIdx.x % kXcds) * chunk + blockIdx.x / kXcds;
}

// energy passes (tm_energy.hip)
struct PassBuffers {
    double* q;          // [N] curvature / area per vertex
    double* gprops;     // [6N] properties of listed (boundary) vertices
    int* pair_cnt;      // [N] repulsion pairs per vertex (k_rep)
    double* rep_v;      // [N] repulsion property per vertex (k_rep)
    double* rep_g;      // [3N] repulsion gradient, rows of vertices with pairs (k_rep)
    double* partials;   // [6 * pass1 blocks]
    unsigned* count;    // [kLastCounters] zeros (tm_last.h)
    Globals* globals;
    Globals* host;      // pinned copy of globals the pass also writes; null: none
    const int* list;    // boundary / degenerate vertices
    int nlist;
    PairCache pc;       // x_snap null: the query runs in full every time
    // [kRingPad * N] dihedral angle of each ring slot of vertices of valence
    // <= kRingPad, column-major, in the precision of the pass (float or
    // double); written by pass 1, read by pass 2.  Null: pass 2 forms them
    void* theta;
};
int pass1_blocks(int nv);
// Up to this many rows of partials the pass's last workgroup sums them, above
// it a launch of its own does.  Counting the workgroups costs the pass about
// what the launch does where they are many: an evaluation (properties and
// gradient, mixed) takes 31.6 us with the tail and 33.3 with the launch at 642
// vertices (8 rows), 31.1 and 33.4 at 10242 (48), 36.5 and 36.7 at 23042 (96),
// 42.6 and 42.4 at 92162 (368), 51.9 and 51.8 at 163842 (648).  (Since then the
// query has become 4 to 6 us shorter at every size, on both sides alike.)
constexpr int kTailBlocks = 128;

// Everything the pass kernels read and write for one mesh.  A grouped launch
// takes a device array of these, one per replica, and a prefix table of
// pass-1 blocks: logical block b belongs to the replica r with
// block0[r] <= b < block0[r + 1] and is its local block b - block0[r], so
// every replica is partitioned and summed exactly as in a launch of its own.
struct PassArgs {
    MeshView m;
    NListView nl;
    EParams p;
    double* q;
    double* gprops;
    double* rep_v;       // null: repulsion off
    int* pair_cnt;
    double* rep_g;       // null: rows not stored (pass 1 only)
    double* partials;
    unsigned* count;
    int tail;            // the pass's last workgroup sums the partials (see kTailBlocks)
    Globals* globals;
    Globals* host;       // PassBuffers::host
    double* grad;
    double* vprops;      // optional per-vertex properties of pass 1
    void* theta;         // PassBuffers::theta
    const int* list;     // boundary / degenerate vertices
    int nlist;
    int nblocks;         // pass-1 blocks of kPass1Verts vertices (a multiple of 8)
    PairCache pc;
};
PassArgs pass_args(const MeshView& m, const NListView& nl, const EParams& p, const PassBuffers& b, double* vprops,
                   double* grad);
// Launch shapes that do not change any result bit: the repulsion query and
// pass 2 write per-vertex values only, and each lane visits its candidates in
// the same order whatever the batch.  (Pass 1's blocks fix the order of the
// global sums and stay at 256 threads.)
struct Tuning {
    int rep_threads = 256;    // 64, 128, 256 or 512
    int rep_batch = 2;        // candidates in flight per lane: 1, 2, 4 or 8
    int p2_threads = 256;     // 64, 128, 256 or 512
    int rep_fused = 0;        // taken and kept; the query has its own launch either way
    int pair_cache = 1;       // 1: replay recorded candidate lists (single meshes, cell list)
    int pflip_window = 256;   // proposals the pflip Metropolis scan tests at once (1..256)
    int serial_window = 256;  // proposals per window of the serial sweep (1..256), 0: one workgroup
};
bool tuning_valid(const Tuning& t);
int tuned_blocks(int nv, int threads);    // blocks of 8-lane groups (the query), a multiple of 8
int pass2_blocks(int nv, int threads);    // blocks of one lane per vertex (pass 2), a multiple of 8
// the repulsion query and the pass-2 kernel alone (for timing)
void launch_rep(const PassArgs& a, const Tuning& t, hipStream_t s);
// the repulsion query and the pass-1 kernel, the later of which finalizes;
// marks (optional): HIP events stamped at the pass-1 kernel's start and end
// (either may be null)
void launch_pass1_body(const PassArgs& a, int mixed, const Tuning& t, hipStream_t s,
                       const hipEvent_t* marks = nullptr);
void launch_pass2_kernel(const PassArgs& a, int mixed, const Tuning& t, hipStream_t s);
// R replicas: d_args in device memory, h_args its host copy (for the
// launches of the boundary kernels), one prefix table of blocks per kernel
// shape
struct GroupLaunch {
    const PassArgs* d_args;
    const PassArgs* h_args;
    int R;
    const int* d_block0_p1;
    int total_p1;
    const int* d_block0_rep;
    int total_rep;
    const int* d_block0_p2;
    int total_p2;
    Tuning tune;
    int mixed;
    // with the pair cache (h_args[r].pc.x_snap set): the cached query's
    // prefix table (pass-1 blocks of each replica)
    const int* d_block0_rc;
    int total_rc;
};
void launch_pass1_grouped(const GroupLaunch& g, hipStream_t s, const hipEvent_t* marks = nullptr);
void launch_pass2_grouped(const GroupLaunch& g, hipStream_t s);
void launch_rep_grouped(const GroupLaunch& g, hipStream_t s);
void launch_pass1(const MeshView& m, const NListView& nl, const EParams& p, int mixed, const PassBuffers& b,
                  double* vprops, hipStream_t s, const Tuning& t = Tuning(), const hipEvent_t* marks = nullptr);
void launch_pass2(const MeshView& m, const NListView& nl, const EParams& p, int mixed, const PassBuffers& b,
                  double* grad, hipStream_t s, const Tuning& t = Tuning());
void launch_halfedge_geometry(const MeshView& m, int h, double* out, hipStream_t s);
void launch_sum_geometry(const MeshView& m, int what, double* partials, unsigned* counter, double* result,
                         hipStream_t s);

// dst[i*w + c] = src[idx[i]*w + c] for i < n, c < w (tm_flips.hip)
void launch_gather_rows(const double* src, const int* idx, double* dst, int n, int w, hipStream_t s);

// topology helpers (tm_flips.hip)
// out[3 n]: the vertices of faces first .. first + n - 1 as user ids (perm:
// internal -> user)
void launch_faces(const MeshView& m, const int* perm, int* out, int first, int n, hipStream_t s);
// x[at[i]] = host[i] (n rows of 3) and host[i] = src[idx[first + i]] (n rows of
// w); host: pinned, 16-byte aligned
void launch_take_points(const double* host, const int* at, double* x, int n, hipStream_t s);
void launch_give_rows(const double* src, const int* idx, double* host, int first, int n, int w, hipStream_t s);
// Rebuild ring table and meta from the halfedge arrays; sets *overflow (pinned) to 1
// if a vertex has more than kMaxValence neighbours.
void launch_build_ring(const MeshView& m, int* ring, int* meta, int* overflow, hipStream_t s);

// neighbour lists (tm_nlist.hip)
int box_scratch_doubles();
void launch_fill_ints(int* a, int na, int va, int* b, int nb, int vb, int* c, int nc, int vc, hipStream_t s);
void launch_exclusive_scan(const int* in, int* out, int n, int* block_sums, hipStream_t s);
int scan_block_sums_size(int n);
// One list of a build.
struct NlistBuild {
    const double* x;
    const int* perm;
    int n, nc;                 // vertices, cells
    double* box;               // [box_scratch_doubles] pinned
    NListView nl;              // the grid, and the tables as they will be
    MeshView m;
    int *counts, *cell_start;  // [nc + 1]
    int *vert_cell, *place, *cell_verts;    // [n]
    int *cand_count, *cand_start;           // [n + 1]; a Verlet list: these and below null
    int* cand;                 // [27 n]
    int2* vcand;               // [n]
    unsigned long long* mask;  // [2 n]
    int* pc_cell;              // [n]
    int* pc_streak;            // [2]
    int* sums;                 // [scan_block_sums_size(max(n, nc) + 1)]
};
// Workgroups of a list in the launches of each shape.
enum {
    kShapeBox, kShapeVerts, kShapeCells, kShapeCand, kShapeStarts, kShapeFill, kShapeVertsSort, kShapeMask,
    kShapes
};
int nlist_blocks(const NlistBuild& b, int shape);
struct NlistGroup {
    const NlistBuild* h;       // [R]
    int R;
    const NlistBuild* d;       // R > 1: the same in device memory
    const int* block0;         // [kShapes][R + 1] prefix tables of nlist_blocks
    int total[kShapes];
};
void launch_nlist_box(const NlistGroup& g, hipStream_t s);
// everything after the host has set the grids
void launch_nlist_build(const NlistGroup& g, hipStream_t s);
void launch_nlist_masks(const NlistGroup& g, hipStream_t s);    // tm_energy.hip
// exclusion masks of the stored stencil lists (tm_energy.hip); nl needs
// vcand and cand, its excl_mask is ignored
void launch_excl_mask(const MeshView& m, const NListView& nl, unsigned long long* mask, hipStream_t s);
// distance_matrix (cell list or verlet) in two phases: counts then fill
void launch_dm_count(const MeshView& m, const NListView& nl, double dmax, int* counts, hipStream_t s);
void launch_dm_fill(const MeshView& m, const NListView& nl, double dmax, const int* offsets, double* d, int* i,
                    int* j, hipStream_t s);
// point_distances of one vertex in the reference's stencil order
void launch_point_distances(const MeshView& m, const NListView& nl, int pid, double dmax, int cap, int* count,
                            double* dist3, int* jdx, hipStream_t s);
// verlet adjacency from a cell list: counts, then fill (ascending ids)
void launch_verlet_count(const MeshView& m, const NListView& cl, double rlist, int* counts, hipStream_t s);
void launch_verlet_fill(const MeshView& m, const NListView& cl, double rlist, const int* offsets, int* adj,
                        hipStream_t s);

// flips (tm_flips.hip)
struct FlipMeshView {
    double* x;
    int* he_to;
    int* he_next;
    int* he_prev;
    int* he_face;
    int* v_he;
    int* f_he;
    int nv, nh, nf;
};
void launch_flip_serial(const FlipMeshView& fm, const NListView& nl, const EParams& p, int nflips,
                        const int* proposals, const double* uniforms, int n_uniforms, uint64_t seed, int injected,
                        const Globals* g0, int* result /* [accepted, used, error] */, hipStream_t s);

// Rows of the one-rings (tm_flips.hip), kMaxValence slots per vertex; er null
// where no sweep claims edges.
struct FlipRows {
    int* nb;     // [kMaxValence N] neighbours, ended by -1
    int2* er;    // [kMaxValence N] spoke and rim edge of each slot
};

// windowed serial sweep: the serial sweep's decisions and topology from
// windows of up to kSerialWindowMax proposals evaluated in parallel
constexpr int kSerialWindowMax = 256;
struct SerialState {
    int pos, done, used, acc, err, window;
    double props[6];
    double e0;
    unsigned count;    // workgroups of the window that have finished
};
constexpr int kFlipRecord = 32;      // ints per proposal record of the parallel sweep
constexpr int kSerialRecord = 40;    // ... and of the serial one
// rows, face stamps and the starting state
void launch_serial_begin(const FlipMeshView& fm, const FlipRows& rows, const Globals* g0, const EParams& p, int nflips,
                         SerialState* st, unsigned long long* fstamp, hipStream_t s);
// rec: [kSerialRecord W], fstamp: [faces]
void launch_serial_windows(const FlipMeshView& fm, const FlipRows& rows, const NListView& nl, const EParams& p,
                           int nflips, const int* proposals, const double* uniforms, int n_uniforms, uint64_t seed,
                           int injected, int W, SerialState* st, int* rec, unsigned long long* fstamp,
                           int n_windows, hipStream_t s);

// The claim-based parallel sweep of one mesh; state receives props[6], the
// final energy and the number of accepted flips.
struct PflipArgs {
    FlipMeshView fm;
    NListView nl;
    EParams p;
    FlipRows rows;
    uint64_t seed;
    int nflips, batch;
    const Globals* g0;
    unsigned long long* owner;    // [E] largest claim key
    int* rec;                     // [kFlipRecord batch] the proposals' records
    int* lost;                    // [batch] the last round + 1 in which a later claim beat one of its claims
    double* state;                // [8]
    unsigned* count;              // workgroups of the round that have finished
};
int pflip_round_blocks(int batch);    // workgroups of a round of `batch` proposals
void launch_flip_parallel(const PflipArgs& a, int window, hipStream_t s);

// The parallel sweep of many meshes at once: round r of every replica in one
// launch.  Each replica's workgroups run the single-mesh sweep's device
// functions on its own arguments, so its flips, decisions and state are those
// of launch_flip_parallel with the same arguments.
struct PflipGroup {
    const PflipArgs* d_args;
    int R;
    int rounds;            // the most rounds of any replica
    int window;
    const int* d_block0;   // prefix table of pflip_round_blocks per replica
    int total_blocks;
    int max_nv, max_nh, max_batch;
};
void launch_flip_parallel_grouped(const PflipGroup& g, hipStream_t s);

// replica of logical block lb in a grouped launch (block0 ascending,
// block0[0] = 0)
__device__ __forceinline__ int find_replica(const int* __restrict__ block0, int R, int lb)
{
    int lo = 0, hi = R - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (block0[mid] <= lb) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// device HMC step (tm_hmc.hip)
struct HmcState {
    double energy0, energy1, kinetic0, kinetic1, dh, uniform;
    int accepted, pad;
    unsigned long long n_accepted, n_steps;
    double props0[6];    // global properties at x0 (first force evaluation)
    double props[6];     // ... of the state after the step (x0 or xn)
};
enum { kHmcFirst = 1, kHmcKick = 2, kHmcDrift = 4, kHmcLast = 8 };
int hmc_blocks(int n3);
void launch_hmc_begin(int n3, const double* x, double* x0, double* p, const int* perm, int draw, uint64_t seed,
                      uint64_t step, double sigma, double* kpart, hipStream_t s);
void launch_hmc_leap(int n3, double* x, double* p, double* a, const double* g, double dt, double dt2, double mass,
                     int mode, const Globals* globals, HmcState* st, double* kpart, hipStream_t s);
void launch_hmc_accept(int n3, const double* kpart0, const double* kpart1, const double* x0, const double* x,
                       int harmonic, const Globals* globals, double mass, double temperature, double uniform,
                       uint64_t seed, uint64_t step, HmcState* st, int* streak, hipStream_t s);
void launch_hmc_restore(int n3, double* x, const double* x0, const HmcState* st, hipStream_t s);

// One replica of a grouped HMC step: device draws keyed by (seed, the
// replica's own step count), forces from grad, energies from globals.
struct HmcArgs {
    int n3;
    int nblocks;          // hmc_blocks(n3)
    double* x;
    double* x0;
    double* p;
    double* a;
    const double* grad;
    Globals* globals;
    const int* perm;
    HmcState* st;
    double* kpart0;
    double* kpart1;
    double mass, dt, dt2, temperature;
    uint64_t seed;
};
void launch_hmc_begin_grouped(const HmcArgs* d, const int* d_block0, int R, int total_blocks, hipStream_t s);
void launch_hmc_leap_grouped(const HmcArgs* d, const int* d_block0, int R, int total_blocks, int mode,
                             hipStream_t s);
void launch_hmc_accept_grouped(const HmcArgs* d, const PassArgs* a, int R, hipStream_t s);
void launch_hmc_restore_grouped(const HmcArgs* d, const int* d_block0, int R, int total_blocks, hipStream_t s);
// Parallel-tempering exchange over a kappa_b ladder: ladder slots s and s+1
// (s = parity, parity + 2, ...) swap their replicas with probability
// min(1, exp(-(k[s+1] - k[s]) (B_a - B_b) / T)), B the bending of the current
// states; pass parameters and the slot owners are updated in place.
void launch_pt_swap(PassArgs* d_args, const HmcArgs* d_hmc, int* owner, const double* ladder, int R,
                    uint64_t seed, unsigned long long* round, unsigned long long* swaps_accepted,
                    unsigned long long* swaps_tried, hipStream_t s);

}    // namespace tmh
