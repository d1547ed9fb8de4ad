// tm_flips.hip -- ring-table rebuild and the edge-flip sweeps: the serial
// sweep (one workgroup, k_flip_serial, or windows of proposals evaluated at
// once and committed in order, k_sf_window) and the parallel sweep
// (k_pflip_round).
//
// flip_serial (src/flips.cpp:22-80) is a Metropolis loop in which every
// proposal depends on the topology left by the previous one.  The
// one-workgroup kernel walks the proposal stream in order.  For each proposal:
//   * lane 0 tests OpenMesh is_flip_ok and the boundary condition;
//   * the workgroup evaluates vertex_properties of the four patch vertices
//     (flip_utils.cpp:19-41), 16 lanes per vertex (coop_patch), including
//     their repulsion queries;
//   * lane 0 flips (OpenMesh TriConnectivity::flip rewiring), the lanes
//     re-evaluate the patch, and lane 0 applies the FP64 Metropolis test
//     u <= (dE < 0 ? 1 : exp(-dE)) and flips back on rejection.
// A uniform is consumed only for proposals that pass the validity test
// (flips.cpp:45, 64).  Proposals and uniforms are either injected by the
// caller or drawn from a counter-based generator keyed by a seed.
#include "tm_internal.h"
#include "tm_om.h"
#include "tm_rng.h"
#include "tm_last.h"
#include "tm_wave.h"

#include <algorithm>

namespace tmh {

// ------------------------------------------------------- ring rebuild -----
__global__ void k_build_ring(MeshView m, int* __restrict__ ring, int* __restrict__ meta, int* __restrict__ overflow)
{
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m.nv) return;
    const int N = m.nv;
    int h0 = m.v_he[v];
    int n = 0, b = -1;
    if (h0 >= 0) {
        int h = h0;
        do {
            if (n < kMaxValence) ring[n * N + v] = m.he_to[h];
            if (m.he_face[h] < 0 && b < 0) b = n;
            n++;
            h = m.he_next[h ^ 1];
        } while (h != h0 && n <= kMaxValence);
    }
    if (n > kMaxValence) {
        *overflow = 1;    // pinned host memory
        n = kMaxValence;
        b = 0;    // route to the halfedge walker
    }
    for (int k = n; k < kRingPad; k++) ring[k * N + v] = -1;
    meta[v] = n | ((b + 1) << 16);
}

void launch_build_ring(const MeshView& m, int* ring, int* meta, int* overflow, hipStream_t s)
{
    if (m.nv == 0) return;
    hipLaunchKernelGGL(k_build_ring, dim3((m.nv + 255) / 256), dim3(256), 0, s, m, ring, meta, overflow);
}

// ------------------------------------------------------- permutations -----
__global__ void k_gather_rows(const double* __restrict__ src, const int* __restrict__ idx, double* __restrict__ dst,
                              int n, int w)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * w) return;
    int i = t / w, c = t - i * w;
    dst[t] = src[(size_t)idx[i] * w + c];
}

void launch_gather_rows(const double* src, const int* idx, double* dst, int n, int w, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_gather_rows, dim3((n * w + 255) / 256), dim3(256), 0, s, src, idx, dst, n, w);
}

// Rows between pinned host memory and the device, by kernels that reorder them
// on the way: no copy through a device buffer, and at small sizes one launch
// instead of a copy engine's start and a launch.  The link is what bounds them, so
// the host side is read and written in order, two doubles per thread, and the
// device side scattered or gathered: 3.0 us to take 642 points, 96 us (41 GB/s)
// 163842; 10.8 us (48 GB/s) to give 21845 rows.
// x[at[i]] = host[i], three doubles per row
__global__ void __launch_bounds__(256) k_take_points(const double* __restrict__ host, const int* __restrict__ at,
                                                     double* __restrict__ x, int n3)
{
    const int e = 2 * (blockIdx.x * 256 + threadIdx.x);
    if (e + 1 < n3) {
        const double2 v = *reinterpret_cast<const double2*>(host + e);
        x[3 * (size_t)at[e / 3] + e % 3] = v.x;
        x[3 * (size_t)at[(e + 1) / 3] + (e + 1) % 3] = v.y;
    } else if (e < n3) {
        x[3 * (size_t)at[e / 3] + e % 3] = host[e];
    }
}

// host[i] = src[idx[first + i]], i < n, w doubles per row
__global__ void __launch_bounds__(256) k_give_rows(const double* __restrict__ src, const int* __restrict__ idx,
                                                   double* __restrict__ host, int first, int n, int w)
{
    const int e = 2 * (blockIdx.x * 256 + threadIdx.x);
    if (e >= n * w) return;
    auto at = [&](int k) { return src[(size_t)idx[first + k / w] * w + k % w]; };
    if (e + 1 < n * w) *reinterpret_cast<double2*>(host + e) = make_double2(at(e), at(e + 1));
    else host[e] = at(e);
}

void launch_take_points(const double* host, const int* at, double* x, int n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_take_points, dim3((3 * n + 511) / 512), dim3(256), 0, s, host, at, x, 3 * n);
}

void launch_give_rows(const double* src, const int* idx, double* host, int first, int n, int w, hipStream_t s)
{
    if (n > 0)
        hipLaunchKernelGGL(k_give_rows, dim3((n * w + 511) / 512), dim3(256), 0, s, src, idx, host, first, n, w);
}

// The faces first .. first + n - 1 as user vertex ids (fv_indices): to(h),
// to(next h), to(next next h) of each face's halfedge, one thread per face.
__global__ void __launch_bounds__(256) k_faces(MeshView m, const int* __restrict__ perm, int* __restrict__ out,
                                               int first, int n)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= n) return;
    const int h0 = m.f_he[first + f], h1 = m.he_next[h0], h2 = m.he_next[h1];
    out[3 * f] = perm[m.he_to[h0]];
    out[3 * f + 1] = perm[m.he_to[h1]];
    out[3 * f + 2] = perm[m.he_to[h2]];
}

void launch_faces(const MeshView& m, const int* perm, int* out, int first, int n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_faces, dim3((n + 255) / 256), dim3(256), 0, s, m, perm, out, first, n);
}

// ---------------------------------------------------------------- RNG -----
__device__ __forceinline__ double rng_uniform(uint64_t seed, uint64_t i) { return rng_unit(rng_draw(seed, 1, i)); }
__device__ __forceinline__ int rng_edge(uint64_t seed, uint64_t i, int ne)
{
    return (int)(((rng_draw(seed, 0, i) >> 32) * (uint64_t)ne) >> 32);
}

// ------------------------------------------------------------ helpers -----
// OpenMesh TriConnectivity::is_flip_ok (not a boundary edge, the two
// opposite vertices distinct and not yet neighbours), plus one condition the
// reference does not have: a flip adds a neighbour to each opposite vertex,
// and it is refused when either would exceed the ring-table width
// kMaxValence.  Meshes are created with valences of at most kMaxValence, so
// every topology a sweep can reach stays within the table.  The two one-rings
// are walked in one loop so that their dependent loads overlap.
__device__ __forceinline__ bool flip_ok(const Topo& t, int e)
{
    if (t.edge_boundary(e)) return false;
    int ah = t.to(t.next(2 * e));
    int bh = t.to(t.next(2 * e + 1));
    if (ah == bh) return false;
    const int ha0 = t.vhe(ah), hb0 = t.vhe(bh);
    int ha = ha0, hb = hb0, na = 0, nb = 0;
    bool da = false, db = false, adjacent = false;
    do {
        if (!da) {
            adjacent = adjacent || t.to(ha) == bh;
            ha = t.cw(ha);
            da = ha == ha0 || ++na >= 4 * kMaxValence;
        }
        if (!db) {
            hb = t.cw(hb);
            db = hb == hb0 || ++nb >= 4 * kMaxValence;
        }
    } while (!(da && db));
    // na, nb count the steps before the walk closed: valence - 1
    return !adjacent && na + 1 < kMaxValence && nb + 1 < kMaxValence;
}

// An interior edge's two triangles: what a flip reads.  a0 = 2e, b0 = 2e + 1.
struct FlipEdge {
    int e;
    int pv[4];             // to(a0), to(a1), to(b0), to(b1)
    int a1, a2, b1, b2;    // the halfedges that follow a0 and b0
    int fa, fb;            // faces of a0 and b0 (-1 on a boundary, the rest then unset)
    int ha, hb;            // v_he of to(a0) and to(b0)
};
__device__ __forceinline__ FlipEdge load_flip_edge(const FlipMeshView& fm, int e)
{
    FlipEdge f{};
    f.e = e;
    const int2 nx = reinterpret_cast<const int2*>(fm.he_next)[e], to = reinterpret_cast<const int2*>(fm.he_to)[e];
    const int2 fc = reinterpret_cast<const int2*>(fm.he_face)[e];
    f.fa = fc.x;
    f.fb = fc.y;
    if (f.fa < 0 || f.fb < 0) return f;
    f.a1 = nx.x;
    f.b1 = nx.y;
    f.pv[0] = to.x;
    f.pv[2] = to.y;
    f.pv[1] = fm.he_to[f.a1];
    f.pv[3] = fm.he_to[f.b1];
    f.a2 = fm.he_next[f.a1];
    f.b2 = fm.he_next[f.b1];
    f.ha = fm.v_he[f.pv[0]];
    f.hb = fm.v_he[f.pv[2]];
    return f;
}

// OpenMesh TriConnectivity::flip of f.e
__device__ __forceinline__ void store_flip(const FlipMeshView& fm, const FlipEdge& f)
{
    const int a0 = 2 * f.e, b0 = a0 + 1;
    fm.he_to[a0] = f.pv[1];
    fm.he_to[b0] = f.pv[3];
    fm.he_next[a0] = f.a2; fm.he_prev[f.a2] = a0;
    fm.he_next[f.a2] = f.b1; fm.he_prev[f.b1] = f.a2;
    fm.he_next[f.b1] = a0; fm.he_prev[a0] = f.b1;
    fm.he_next[b0] = f.b2; fm.he_prev[f.b2] = b0;
    fm.he_next[f.b2] = f.a1; fm.he_prev[f.a1] = f.b2;
    fm.he_next[f.a1] = b0; fm.he_prev[b0] = f.a1;
    fm.he_face[f.a1] = f.fb;
    fm.he_face[f.b1] = f.fa;
    fm.f_he[f.fa] = a0;
    fm.f_he[f.fb] = b0;
    if (f.ha == b0) fm.v_he[f.pv[0]] = f.a1;
    if (f.hb == a0) fm.v_he[f.pv[2]] = f.b1;
}

// store_flip twice (a rejected proposal) in one pass.  The second flip
// undoes the connectivity but not the ids: the edge's two halfedges swap
// direction, the two faces swap triangles, and the v_he of the edge's
// endpoints move off the swapped halfedges exactly as the first flip moved
// them (the second flip's v_he tests cannot hold, since its endpoints'
// outgoing halfedges are not the edge's).
__device__ __forceinline__ void store_flip_twice(const FlipMeshView& fm, const FlipEdge& f)
{
    const int a0 = 2 * f.e, b0 = a0 + 1;
    fm.he_to[a0] = f.pv[2];
    fm.he_to[b0] = f.pv[0];
    fm.he_next[a0] = f.b1; fm.he_prev[f.b1] = a0;
    fm.he_next[f.b1] = f.b2; fm.he_prev[f.b2] = f.b1;
    fm.he_next[f.b2] = a0; fm.he_prev[a0] = f.b2;
    fm.he_next[b0] = f.a1; fm.he_prev[f.a1] = b0;
    fm.he_next[f.a1] = f.a2; fm.he_prev[f.a2] = f.a1;
    fm.he_next[f.a2] = b0; fm.he_prev[b0] = f.a2;
    fm.he_face[f.a1] = f.fb;
    fm.he_face[f.a2] = f.fb;
    fm.he_face[f.b1] = f.fa;
    fm.he_face[f.b2] = f.fa;
    fm.f_he[f.fa] = a0;
    fm.f_he[f.fb] = b0;
    if (f.ha == b0) fm.v_he[f.pv[0]] = f.a1;
    if (f.hb == a0) fm.v_he[f.pv[2]] = f.b1;
}

__device__ __forceinline__ void do_flip(const FlipMeshView& fm, int e) { store_flip(fm, load_flip_edge(fm, e)); }

__device__ __forceinline__ double energy_of(const double pr[6], const EParams& p)
{
    // trimem_energy (kernel.h:110-122)
    double e = 0.0, d;
    d = pr[0] / p.ref_area - 1.0;
    e += p.kappa_a * d * d;
    d = pr[1] / p.ref_volume - 1.0;
    e += p.kappa_v * d * d;
    d = pr[2] / p.ref_curvature - 1.0;
    e += p.kappa_c * d * d;
    e += p.kappa_t * pr[4];
    e += p.kappa_r * pr[5];
    e += p.kappa_b * pr[3];
    return e;
}

// ------------------------------------------ cooperative patch evaluation --
// vertex_properties (mesh_properties.cpp:12-49) of the four vertices of an
// edge's flip patch (flip_utils.cpp:19-41), to(2e), to(next(2e)), to(2e+1),
// to(next(2e+1)), by one 64-lane workgroup: lanes 16g .. 16g+15 evaluate
// patch vertex g.
//   phase 1  lane 0 of the group walks the one-ring (clockwise from v_he,
//            as the circulator does) and locates the candidate runs of the
//            repulsion query;
//   phase 2  the lanes compute the per-halfedge terms;
//   phase 3  the lanes test the candidates in chunks of 64, the exclusion
//            test reading the one-ring from LDS (coop_excluded);
//   phase 4  lane 0 adds the terms of each accumulator in the order the
//            single-thread walker (om_vertex_properties) adds them, so every
//            value is bit-identical to it; thread 0 adds the four vertices.
// A vertex whose valence exceeds kMaxValence is evaluated by its lane 0
// with om_vertex_properties.
constexpr int kCoopLanes = 16;
constexpr int kCoopChunk = 4 * kCoopLanes;

struct CoopShared {
    int h[4][kMaxValence];              // outgoing halfedges, circulator order
    int nb[4][kMaxValence];             // their target vertices (the one-ring)
    int bnd[4][kMaxValence];            // halfedge on the boundary
    int n[4];                           // valence; -1 above kMaxValence
    int total[4];                       // repulsion candidates
    double slot[4][kMaxValence][4];     // area, volume, edge curvature, tether
    int run_s[4][9], run_len[4][9];     // candidate runs (CandRuns) of the repulsion query
    double pos[4][3];                   // the patch vertex's position
    double rep[4][kCoopChunk];
    double vp[4][6];
    double sum[6];
};

template <class TP>
__device__ __forceinline__ int patch_vertex(const TP& t, int e, int g)
{
    int h = 2 * e + (g >> 1);
    return (g & 1) ? t.to(t.next(h)) : t.to(h);
}

// The candidate runs of a vertex's repulsion query, in the order
// nlist_visit walks them: the nine (dj, dk) rows of three consecutive cells
// of cell_verts, or the vertex's adj range of the Verlet list.  Rows that
// fall outside the grid are empty runs, so every index is a constant after
// unrolling and the runs stay in registers.
struct CandRuns {
    int s[9], len[9];
    int total;
};

__device__ __forceinline__ CandRuns cand_runs(const NListView& nl, int i, d3 pi)
{
    CandRuns r;
#pragma unroll
    for (int k = 0; k < 9; k++) r.s[k] = r.len[k] = 0;
    if (nl.kind == 0) {
        int c[3];
        cell_coords(nl, pi, c);
#pragma unroll
        for (int k = 0; k < 9; k++) {
            int kk = c[2] + k / 3 - 1, jj = c[1] + k % 3 - 1;
            int i0 = max(c[0] - 1, 0), i1 = min(c[0] + 1, nl.shape[0] - 1);
            if (kk >= 0 && kk < nl.shape[2] && jj >= 0 && jj < nl.shape[1] && i0 <= i1) {
                int base = jj * nl.strides[1] + kk * nl.strides[2];
                r.s[k] = nl.cell_start[base + i0];
                r.len[k] = nl.cell_start[base + i1 + 1] - r.s[k];
            }
        }
    } else if (nl.kind == 1) {
        r.s[0] = nl.adj_start[i];
        r.len[0] = nl.adj_start[i + 1] - r.s[0];
    }
    r.total = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) r.total += r.len[k];
    return r;
}

// Slot of the c-th candidate (0 <= c < total) in cell_verts / adj.
__device__ __forceinline__ int cand_slot(const CandRuns& r, int c)
{
    int q = -1;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        if (q < 0 && c < r.len[k]) q = r.s[k] + c;
        if (q < 0) c -= r.len[k];
    }
    return q;
}

__device__ __forceinline__ bool coop_in_ring(const CoopShared& S, int g, int n, int j)
{
    for (int k = 0; k < n; k++)
        if (S.nb[g][k] == j) return true;
    return false;
}

// om_excluded(ve, j) for patch vertex g (valence n <= kMaxValence, one-ring
// in S.nb).  Adjacency is symmetric, so j lies in the one-ring of a ring
// vertex of ve exactly when j's own one-ring meets ve's: the walk runs
// around j, and only for candidates within the cutoff that are not in ve's
// one-ring, instead of around every ring vertex of every patch vertex.  A
// candidate of valence above kMaxValence takes om_excluded.
template <class TP>
__device__ __forceinline__ bool coop_excluded(const TP& t, const CoopShared& S, int g, int n, int ve, int excl,
                                              int j)
{
    if (excl <= 0) return false;
    if (coop_in_ring(S, g, n, j)) return true;
    if (excl == 1) return false;
    const int h0 = t.vhe(j);
    if (h0 < 0) return false;
    int h = h0, m = 0;
    do {
        if (m == kMaxValence) return om_excluded(t, ve, j, excl);
        if (coop_in_ring(S, g, n, t.to(h))) return true;
        m++;
        h = t.cw(h);
    } while (h != h0);
    return false;
}

// Called by all 64 threads of the workgroup; S.vp and S.sum hold the result
// on return.
template <class TP>
__device__ void coop_patch(const TP& t, const NListView& nl, const EParams& p, int e, CoopShared& S)
{
    const int g = threadIdx.x / kCoopLanes, l = threadIdx.x % kCoopLanes;
    const int ve = patch_vertex(t, e, g);
    const bool rep_on = p.rep_lc1 > 0 && nl.kind >= 0;
    const int excl = nl.kind == 0 ? nl.exclusion : 0;

    // phase 1 (the candidate runs wait in LDS while phase 2 needs the registers)
    if (l == 0) {
        const d3 pv = t.P(ve);
        S.pos[g][0] = pv.x;
        S.pos[g][1] = pv.y;
        S.pos[g][2] = pv.z;
        const CandRuns runs = cand_runs(nl, ve, pv);
#pragma unroll
        for (int k = 0; k < 9; k++) {
            S.run_s[g][k] = runs.s[k];
            S.run_len[g][k] = runs.len[k];
        }
        S.total[g] = rep_on ? runs.total : 0;
        int n = 0;
        int h0 = t.vhe(ve);
        if (h0 >= 0) {
            int h = h0;
            do {
                if (n == kMaxValence) {
                    n = -1;
                    break;
                }
                S.h[g][n] = h;
                S.nb[g][n] = t.to(h);
                n++;
                h = t.cw(h);
            } while (h != h0);
        }
        S.n[g] = n;
        if (n < 0) S.total[g] = 0;
    }
    __syncthreads();
    const int n = S.n[g];

    // phase 2
    for (int s = l; s < n; s += kCoopLanes) {
        const int h = S.h[g][s];
        const int b = t.he_boundary(h);
        S.bnd[g][s] = b;
        if (!b) {
            double el = mu_edge_length(t, h);
            double da = om_dihedral_angle(t, h);
            S.slot[g][s][0] = mu_face_area(t, h);
            S.slot[g][s][1] = mu_face_volume(t, h);
            S.slot[g][s][2] = 0.5 * el * da;
            S.slot[g][s][3] = p.bond_type == 0 ? bond_edge_value(el, p) : bond_area_value(mu_face_area(t, h), p);
        }
    }
    __syncthreads();

    // phase 3
    const d3 pi{S.pos[g][0], S.pos[g][1], S.pos[g][2]};
    CandRuns runs;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        runs.s[k] = S.run_s[g][k];
        runs.len[k] = S.run_len[g][k];
    }
    const int total = S.total[g];
    const int tmax = max(max(S.total[0], S.total[1]), max(S.total[2], S.total[3]));
    const double dmax = p.rep_lc1;
    const double dmax2 = dmax * dmax * (1.0 + 1e-15);    // prefilter, as in nlist_visit
    double rep = 0.0;
    for (int base = 0; base < tmax; base += kCoopChunk) {
        double val[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = base + k * kCoopLanes + l;
            val[k] = 0.0;
            if (c < total) {
                const int q = cand_slot(runs, c);
                const int j = nl.kind == 0 ? nl.cell_verts[q] : nl.adj[q];
                const d3 d = pi - t.P(j);
                const double sq = sqnorm(d);
                bool in = sq <= dmax2 && sqrt(sq) < dmax;
                if (in && nl.kind == 0)
                    in = j != ve && !coop_excluded(t, S, g, n, ve, excl, j);
                if (in) val[k] = rep_value(norm(d), p.rep_lc1, p.rep_r);
            }
            S.rep[g][k * kCoopLanes + l] = val[k];
        }
        // a zero term leaves the (non-negative) sum unchanged: lane 0 adds
        // only the lanes whose term is non-zero, in candidate order
        unsigned long long mask[4];
#pragma unroll
        for (int k = 0; k < 4; k++) mask[k] = __ballot(val[k] != 0.0);
        __syncthreads();
        if (l == 0) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                unsigned bits = (unsigned)(mask[k] >> (kCoopLanes * g)) & 0xffffu;
                while (bits) {
                    const int b = __ffs(bits) - 1;
                    bits &= bits - 1;
                    rep += S.rep[g][k * kCoopLanes + b];
                }
            }
        }
        __syncthreads();
    }

    // phase 4
    if (l == 0) {
        VP r;
        if (n < 0) {
            r = om_vertex_properties(t, nl, p, ve);
        } else {
            double area = 0, vol = 0, curv = 0, teth = 0;
            for (int s = 0; s < n; s++) {
                if (S.bnd[g][s]) continue;
                area += S.slot[g][s][0];
                vol += S.slot[g][s][1];
                curv += S.slot[g][s][2];
                teth += S.slot[g][s][3];
            }
            area /= 3;
            vol /= 3;
            curv /= 2;
            teth /= (p.bond_type == 0 ? 2 : 3);
            r.v[0] = area;
            r.v[1] = vol;
            r.v[2] = curv;
            r.v[3] = 2 * curv * curv / area;
            r.v[4] = teth;
            r.v[5] = rep;
        }
        for (int k = 0; k < 6; k++) S.vp[g][k] = r.v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 0; k < 6; k++) S.sum[k] = 0.0;
        for (int i = 0; i < 4; i++)
            for (int k = 0; k < 6; k++) S.sum[k] += S.vp[i][k];
    }
    __syncthreads();
}

__global__ void __launch_bounds__(64) k_flip_serial(FlipMeshView fm, NListView nl, EParams p, int nflips,
                                                    const int* __restrict__ proposals,
                                                    const double* __restrict__ uniforms, int n_uniforms,
                                                    uint64_t seed, int injected, const Globals* __restrict__ g0,
                                                    int* __restrict__ result)
{
    __shared__ CoopShared S;
    __shared__ int s_go;
    __shared__ int s_stop;
    const int ne = fm.nh / 2;
    const Topo t{fm.x, fm.he_to, fm.he_next, fm.he_prev, fm.he_face, fm.v_he, fm.f_he};
    double props[6];
    for (int k = 0; k < 6; k++) props[k] = g0->props[k];
    double e0 = energy_of(props, p);
    int acc = 0, used = 0, err = 0;
    if (threadIdx.x == 0) s_stop = 0;
    __syncthreads();
    for (int i = 0; i < nflips; i++) {
        __syncthreads();
        if (threadIdx.x == 0) {
            int idx = injected ? proposals[i] : rng_edge(seed, (uint64_t)i, ne);
            if (idx < 0 || idx >= ne) {
                err = 1;
                s_stop = 1;
                s_go = -1;
            } else {
                s_go = (flip_ok(t, idx) && !t.edge_boundary(idx)) ? idx : -1;
            }
        }
        __syncthreads();
        if (s_stop) break;
        const int e = s_go;
        if (e < 0) continue;
        coop_patch(t, nl, p, e, S);
        double old_sum[6];
        if (threadIdx.x == 0) {
            for (int k = 0; k < 6; k++) {
                old_sum[k] = S.sum[k];
                props[k] -= old_sum[k];
            }
            do_flip(fm, e);
        }
        __threadfence_block();
        __syncthreads();
        coop_patch(t, nl, p, e, S);
        if (threadIdx.x == 0) {
            for (int k = 0; k < 6; k++) props[k] += S.sum[k];
            double en = energy_of(props, p);
            double de = en - e0;
            double alpha = de < 0.0 ? 1.0 : exp(-de);
            double u;
            if (injected) {
                if (used >= n_uniforms) {
                    err = 2;
                    s_stop = 1;
                    u = 2.0;
                } else {
                    u = uniforms[used];
                }
            } else {
                u = rng_uniform(seed, (uint64_t)used);
            }
            used++;
            if (u <= alpha) {
                e0 = en;
                acc += 1;
            } else {
                do_flip(fm, e);
                for (int k = 0; k < 6; k++) {
                    props[k] -= S.sum[k];
                    props[k] += old_sum[k];
                }
            }
        }
        __threadfence_block();
        __syncthreads();
        if (s_stop) break;
    }
    if (threadIdx.x == 0) {
        result[0] = acc;
        result[1] = used;
        result[2] = err;
    }
}

void launch_flip_serial(const FlipMeshView& fm, const NListView& nl, const EParams& p, int nflips,
                        const int* proposals, const double* uniforms, int n_uniforms, uint64_t seed, int injected,
                        const Globals* g0, int* result, hipStream_t s)
{
    hipLaunchKernelGGL(k_flip_serial, dim3(1), dim3(64), 0, s, fm, nl, p, nflips, proposals, uniforms, n_uniforms,
                       seed, injected, g0, result);
}

// ==================================================== rows of the one-rings ==
// The sweeps below read every vertex's one-ring from a row of its own instead
// of walking the halfedges: nb[kRowW v + k] is the k-th neighbour in the
// circulator's (clockwise) order, with kNoFace set when the halfedge to it has
// no face, and the row ends with -1 when it is shorter than kRowW.  er holds
// each slot's spoke edge and rim edge (the edge of the next halfedge in its
// face), the edges the parallel sweep claims.  A walk around a ring is a chain
// of about twelve dependent loads; a row is one, and a patch's four rows, the
// positions of their entries and the candidates of its repulsion query are
// five levels in all.  Rows are built at the start of a sweep and rewritten
// for the four vertices of every accepted flip; a rejected flip (do_flip
// twice) leaves every vertex's neighbours and their cyclic order.
constexpr int kRowW = kMaxValence;
constexpr int kRowPair = 8;    // slots read or written in one round of vector operations
constexpr int kNoFace = 1 << 30;

__device__ __forceinline__ void build_rows(const FlipMeshView& fm, const FlipRows& rows, int v)
{
    const int h0 = fm.v_he[v];
    int* nb = rows.nb + (size_t)kRowW * v;
    int2* er = rows.er ? rows.er + (size_t)kRowW * v : nullptr;
    // the leading kRowPair slots in registers, stored as vectors
    int id[kRowPair], sp[kRowPair], rm[kRowPair];
#pragma unroll
    for (int k = 0; k < kRowPair; k++) {
        id[k] = -1;
        sp[k] = rm[k] = 0;
    }
    int n = 0, h = h0;
    if (h0 >= 0) {
#pragma unroll
        for (int k = 0; k < kRowPair; k++) {
            if (k > 0 && h == h0) break;
            id[k] = fm.he_to[h] | (fm.he_face[h] < 0 ? kNoFace : 0);
            sp[k] = h >> 1;
            rm[k] = er ? fm.he_next[h] >> 1 : 0;
            n++;
            h = fm.he_next[h ^ 1];
        }
        if (h != h0)
            do {
                nb[n] = fm.he_to[h] | (fm.he_face[h] < 0 ? kNoFace : 0);
                if (er) er[n] = make_int2(h >> 1, fm.he_next[h] >> 1);
                n++;
                h = fm.he_next[h ^ 1];
            } while (h != h0 && n < kRowW);
    }
#pragma unroll
    for (int k = 0; k < kRowPair; k += 4) {
        reinterpret_cast<int4*>(nb)[k / 4] = make_int4(id[k], id[k + 1], id[k + 2], id[k + 3]);
        if (er) {
            reinterpret_cast<int4*>(er)[k / 2] = make_int4(sp[k], rm[k], sp[k + 1], rm[k + 1]);
            reinterpret_cast<int4*>(er)[k / 2 + 1] = make_int4(sp[k + 2], rm[k + 2], sp[k + 3], rm[k + 3]);
        }
    }
    if (n >= kRowPair && n < kRowW) nb[n] = -1;
}


// The row of patch vertex g after the flip of e.  With the edge's triangles
// (B, A, C) and (A, B, D), A = to(2e) (g 0) and B = to(2e + 1) (g 2) lose
// each other: the slot that follows takes the new edge, e again, as its rim.
// C = to(next(2e)) (g 1) and D (g 3) gain each other before their slot of B
// and of A, with rims ed[0] (of the new slot) and ed[1] (of the slot after).
// One thread per vertex; rows of at most kRowPair slots are read in one
// round of loads, longer ones are shifted in memory.
__device__ __forceinline__ void flip_row(const FlipRows& rows, int ve, int g, int partner, int opposite, int e,
                                         int2 ed)
{
    int* nb = rows.nb + (size_t)kRowW * ve;
    int2* er = rows.er ? rows.er + (size_t)kRowW * ve : nullptr;
    int id[kRowPair + 1];
    int2 ee[kRowPair + 1];
#pragma unroll
    for (int k = 0; k <= kRowPair; k++) {
        id[k] = nb[k];
        ee[k] = er ? er[k] : make_int2(0, 0);
    }
    int n = kRowPair + 1;
#pragma unroll
    for (int k = kRowPair; k >= 0; k--)
        if (id[k] < 0) n = k;
    if (n <= kRowPair) {
        int r = -1;
#pragma unroll
        for (int k = 0; k < kRowPair; k++)
            if (k < n && (id[k] & ~kNoFace) == partner) r = k;
        if (g & 1) {
            // slots r .. n-1 move up by one
#pragma unroll
            for (int k = kRowPair; k > 0; k--)
                if (k > r && k <= n) {
                    nb[k] = id[k - 1];
                    if (er) er[k] = make_int2(ee[k - 1].x, k == r + 1 ? ed.y : ee[k - 1].y);
                }
            nb[r] = opposite;
            if (er) er[r] = make_int2(e, ed.x);
            if (n + 1 < kRowW) nb[n + 1] = -1;
        } else {
#pragma unroll
            for (int k = 0; k < kRowPair; k++)
                if (k >= r && k + 1 < n) {
                    nb[k] = id[k + 1];
                    if (er) er[k] = make_int2(ee[k + 1].x, k == r ? e : ee[k + 1].y);
                }
            nb[n - 1] = -1;
            if (er && r == n - 1) er[0].y = e;    // the slot that follows the last is the first
        }
        return;
    }
    n = 0;
    int r = -1;
    while (n < kRowW && nb[n] >= 0) {
        if ((nb[n] & ~kNoFace) == partner) r = n;
        n++;
    }
    if (g & 1) {
        if (er) er[r].y = ed.y;
        for (int k = n; k > r; k--) {
            nb[k] = nb[k - 1];
            if (er) er[k] = er[k - 1];
        }
        nb[r] = opposite;
        if (er) er[r] = make_int2(e, ed.x);
        if (n + 1 < kRowW) nb[n + 1] = -1;
    } else {
        if (er) er[r + 1 < n ? r + 1 : 0].y = e;
        for (int k = r; k + 1 < n; k++) {
            nb[k] = nb[k + 1];
            if (er) er[k] = er[k + 1];
        }
        nb[n - 1] = -1;
    }
}

// ------------------------------------------------------- patch evaluation --
// Order between a wave's own LDS writes and reads (the LDS serves one wave's
// operations in order, so only the compiler must keep them).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

constexpr int kPatchWaves = 4;    // proposals per 256-thread workgroup, one wave each

constexpr int kCandBatch = 4;                 // candidates in flight per lane
constexpr int kListMax = 16 * kCandBatch;     // of one step of a vertex's 16 lanes
struct PatchShared {
    double pos[4][kRowW][3];    // positions of the one-rings
    double pv[4][3];            // positions of the patch vertices
    alignas(16) int nb[4][kRowW];    // the one-rings (kNoFace bits kept)
    int pre[4][9], st[4][9];    // candidate runs: inclusive prefix of their lengths, starts
    int list[4][kListMax];      // candidates inside the cutoff that a ring test has not excluded
    double term[4][2][8][4];    // eight slots' terms of a ring and side, on their way into a sum in order
};

struct PatchResult {
    bool ok;          // is_flip_ok and the valence cap (flip_ok)
    double val[6];    // lanes 0-7: sums before the flip, lanes 8-15: after it
    __device__ __forceinline__ void difference(double (&d)[6]) const
    {
#pragma unroll
        for (int c = 0; c < 6; c++) d[c] = __shfl(val[c], 8, 64) - __shfl(val[c], 0, 64);
    }
};

// A spoke a -> b with the two faces at it, (a, b, c) and (b, a, d), for the
// halfedge functions: halfedge 0 is the spoke, 1 its twin, 2 and 4 their next ones.
struct Hinge {
    d3 p[4];
    bool edge;    // the face of the twin is missing
    __device__ __forceinline__ d3 P(int v) const { return p[v]; }
    __device__ __forceinline__ int to(int h) const { return h == 0 ? 1 : (h == 1 ? 0 : (h == 2 ? 2 : 3)); }
    __device__ __forceinline__ int from(int h) const { return to(h ^ 1); }
    __device__ __forceinline__ int next(int h) const { return h == 0 ? 2 : 4; }
    __device__ __forceinline__ bool edge_boundary(int) const { return edge; }
};

// vertex_properties (mesh_properties.cpp:12-49) summed over the four vertices
// of interior edge e's flip patch (flip_utils.cpp:19-41), before and after the
// flip, by one wave.  Lanes 16 g .. 16 g + 15 serve patch vertex g (ve[g]: to(2e),
// to(next(2e)), to(2e+1), to(next(2e+1))): first its row, one slot per lane,
// and the ring positions, into LDS; then lanes 0-7 of the group take the
// slots of the ring before the flip and lanes 8-15 those after it, which is
// the same ring without the edge's other end (g 0, 2) or with the other
// opposite vertex (g 1, 3) in front of the slot of `partner`; then all 16
// test the repulsion candidates once, each against both rings.  What bounds
// it is the chain of dependent loads: rows, positions and cell ranges,
// candidate ids, candidate positions.  side_work is done meanwhile: PatchClaim
// claims every edge of the patch, and every sum is a fixed butterfly, whose bits
// depend on the rows alone; WalkOrder (kWalk) finds where each vertex's circulator
// starts, and every term and sum is computed as coop_patch computes it, in the
// order of its walks, so every value has its bits.
template <class SideWork>
__device__ __forceinline__ PatchResult patch_eval(const FlipMeshView& fm, const NListView& nl, const EParams& p,
                                                  const FlipRows& rows, const int (&pv)[4], PatchShared& S,
                                                  SideWork& side_work)
{
    constexpr bool kWalk = SideWork::kWalk;
    const int lane = threadIdx.x & 63, g = lane >> 4, q = lane & 15;
    const int side = (lane >> 3) & 1, k8 = lane & 7;
    const int ve = g == 0 ? pv[0] : (g == 1 ? pv[1] : (g == 2 ? pv[2] : pv[3]));
    const int partner = g < 2 ? pv[2] : pv[0];
    const int opp = g == 1 ? pv[3] : pv[1];    // of C: D, of D: C (g odd only)
    const bool rep_on = p.rep_lc1 > 0 && nl.kind >= 0;

    // rows (a second chunk of 16 slots only where the first is full), the
    // vertices' own positions
    const int* row = rows.nb + (size_t)kRowW * ve;
    int id = row[q];
    side_work.load(ve, q);
    const d3 xv{fm.x[3 * ve], fm.x[3 * ve + 1], fm.x[3 * ve + 2]};
    unsigned full = (unsigned)(__ballot(id >= 0) >> (16 * g)) & 0xffffu;
    int n0 = __ffs(~full) - 1;    // slots before the end mark
    int id2 = -1, n2 = 0;
    if (__ballot(n0 == 16)) {
        if (n0 == 16) id2 = row[16 + q];
        const unsigned f2 = (unsigned)(__ballot(id2 >= 0) >> (16 * g)) & 0xffffu;
        n2 = n0 == 16 ? __ffs(~f2) - 1 : 0;
    }
    const bool has = q < n0, has2 = q < n2;
    // cell ranges of the repulsion query: lane q < 9 takes row q of the stencil
    int rs = 0, rl = 0;
    if (rep_on && q < 9) {
        if (nl.kind == 0) {
            int c[3];
            cell_coords(nl, xv, c);
            const int kk = c[2] + q / 3 - 1, jj = c[1] + q % 3 - 1;
            const int i0 = max(c[0] - 1, 0), i1 = min(c[0] + 1, nl.shape[0] - 1);
            if (kk >= 0 && kk < nl.shape[2] && jj >= 0 && jj < nl.shape[1] && i0 <= i1) {
                const int base = jj * nl.strides[1] + kk * nl.strides[2];
                rs = nl.cell_start[base + i0];
                rl = nl.cell_start[base + i1 + 1] - rs;
            }
        } else if (q == 0) {
            rs = nl.adj_start[ve];
            rl = nl.adj_start[ve + 1] - rs;
        }
    }
    const int j0 = id & ~kNoFace, j2 = id2 & ~kNoFace;
    d3 xj{0, 0, 0};
    if (has) xj = d3{fm.x[3 * j0], fm.x[3 * j0 + 1], fm.x[3 * j0 + 2]};
    side_work.issue(has);
    if (__ballot(has2)) side_work.more(ve, 16 + q, has2);
    if (has) {
        S.nb[g][q] = id;
        S.pos[g][q][0] = xj.x;
        S.pos[g][q][1] = xj.y;
        S.pos[g][q][2] = xj.z;
    }
    if (has2) {
        S.nb[g][16 + q] = id2;
        for (int c = 0; c < 3; c++) S.pos[g][16 + q][c] = fm.x[3 * j2 + c];
    }
    if (q == 0) {
        S.pv[g][0] = xv.x;
        S.pv[g][1] = xv.y;
        S.pv[g][2] = xv.z;
    }
    n0 += n2;
    // the partner's slot, and flip_ok: opposite vertices distinct, not
    // adjacent, both below the valence cap
    const unsigned at = (unsigned)(__ballot(has && j0 == partner) >> (16 * g)) & 0xffffu;
    const unsigned at2 = (unsigned)(__ballot(has2 && j2 == partner) >> (16 * g)) & 0xffffu;
    const int r = at ? __ffs(at) - 1 : (at2 ? 16 + __ffs(at2) - 1 : -1);
    const bool bad = r < 0 || ((g & 1) && (n0 >= kMaxValence || ve == opp || (has && j0 == opp) || (has2 && j2 == opp)));
    PatchResult res;
    res.ok = __ballot(bad) == 0ull;
    if (!res.ok) return res;
    // inclusive prefix of the run lengths over lanes 0-8
    int pre = rl;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        const int y = __shfl_up(pre, o, 16);
        if (q >= o) pre += y;
    }
    const int total = __shfl(pre, 8, 16);
    if (q < 9) {
        S.pre[g][q] = pre;
        S.st[g][q] = rs - (pre - rl);
    }
    wave_sync();

    // the first candidates' ids, in flight during the ring terms
    int cand[kCandBatch];
    auto load_candidates = [&](int t0) {
        const int* ids = nl.kind == 0 ? nl.cell_verts : nl.adj;
#pragma unroll
        for (int u = 0; u < kCandBatch; u++) {
            const int t = t0 + 16 * u + q;
            cand[u] = -1;
            if (t < total) {
                int w = 0;
#pragma unroll
                for (int i = 0; i < 8; i++) w += t >= S.pre[g][i] ? 1 : 0;
                cand[u] = ids[S.st[g][w] + t];
            }
        }
    };
    load_candidates(0);

    // ring terms.  The walk starts at slot w0 of the stored ring and comes to the
    // partner as its step rw; where it starts with the partner, it goes on from the
    // slot after it once the two have lost each other, and still starts there when
    // a vertex is added in front
    const int nS = side ? ((g & 1) ? n0 + 1 : n0 - 1) : n0;
    int w0 = 0, rw = r;
    if constexpr (kWalk) {
        const unsigned a1 = (unsigned)(__ballot(has && j0 == side_work.from) >> (16 * g)) & 0xffffu;
        const unsigned a2 = (unsigned)(__ballot(has2 && j2 == side_work.from) >> (16 * g)) & 0xffffu;
        w0 = a1 ? __ffs(a1) - 1 : (a2 ? 16 + __ffs(a2) - 1 : 0);
        rw = r >= w0 ? r - w0 : r - w0 + n0;
    }
    auto stored = [&](int s) { return w0 + s < n0 ? w0 + s : w0 + s - n0; };
    auto slot_of = [&](int s) {    // slot of the stored ring, or -1 for the vertex the flip adds
        if (!side) return stored(s);
        if (g & 1) {
            const int at = kWalk && rw == 0 ? n0 : rw;
            return s < at ? stored(s) : (s == at ? -1 : stored(s - 1));
        }
        return stored(s < rw ? s : s + 1);
    };
    auto at_slot = [&](int i) {
        const double* a = i < 0 ? S.pv[4 - g] : S.pos[g][i];    // g odd: 4 - g is the other opposite vertex
        return d3{a[0], a[1], a[2]};
    };
    double area = 0, vol = 0, curv = 0, teth = 0;
    double walk = 0;    // kWalk: lane k8 < 4 of a side sums its k8-th quantity
    for (int c0 = 0; __ballot(c0 + k8 < nS); c0 += 8) {
        const int s = c0 + k8;
        const int i1 = s < nS ? slot_of(s) : 0, i2 = slot_of(s + 1 < nS ? s + 1 : 0);
        const bool nof = i1 >= 0 && (S.nb[g][i1] & kNoFace), nofn = i2 >= 0 && (S.nb[g][i2] & kNoFace);
        // a halfedge without a face contributes nothing
        const bool in = s < nS && !nof;
        if constexpr (kWalk) {
            double t[4] = {0, 0, 0, 0};
            if (in) {
                const Hinge hg{{xv, at_slot(i1), at_slot(slot_of(s > 0 ? s - 1 : nS - 1)), at_slot(i2)}, nofn};
                const double el = mu_edge_length(hg, 0), da = om_dihedral_angle(hg, 0);
                t[0] = mu_face_area(hg, 0);
                t[1] = mu_face_volume(hg, 0);
                t[2] = 0.5 * el * da;
                t[3] = p.bond_type == 0 ? bond_edge_value(el, p) : bond_area_value(t[0], p);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) S.term[g][side][k8][c] = t[c];
            wave_sync();
            // (a zero leaves a sum as it is: none of them is ever -0)
#pragma unroll
            for (int i = 0; i < 8; i++) walk += S.term[g][side][i][k8 & 3];
            wave_sync();
        } else if (in) {
            const d3 ec = at_slot(i1) - xv, ep = at_slot(slot_of(s > 0 ? s - 1 : nS - 1)) - xv, en = at_slot(i2) - xv;
            const d3 nc = cross(ec, ep), nn = cross(en, ec);
            const double nl0 = norm(nc), el = norm(ec);
            double da = 0.0;
            if (!nofn) {
                const double denom = nl0 * norm(nn);
                if (denom != 0) da = om_angle(dot(nc, nn) / denom, dot(cross(nc, nn), ec));
            }
            const double fa = nl0 / 2;
            curv += 0.5 * el * da;
            area += fa;
            vol += dot(xv, nc) / 6;
            teth += p.bond_type == 0 ? bond_edge_value(el, p) : bond_area_value(fa, p);
        }
    }
    if constexpr (kWalk) {
        area = __shfl(walk, lane & ~7, 64);
        vol = __shfl(walk, (lane & ~7) + 1, 64);
        curv = __shfl(walk, (lane & ~7) + 2, 64);
        teth = __shfl(walk, (lane & ~7) + 3, 64);
    } else {
        area = group_sum(area);
        vol = group_sum(vol);
        curv = group_sum(curv);
        teth = group_sum(teth);
    }
    area /= 3;
    vol /= 3;
    curv /= 2;
    teth /= (p.bond_type == 0 ? 2 : 3);

    // repulsion: each candidate inside the cutoff against the ring before the
    // flip and the one after it (mesh_repulsion.h:28-54; exclusion as in
    // ring_excluded of the energy passes: at level 2, when the candidate's own
    // ring, as it is on that side, meets the vertex's)
    double rep0 = 0.0, rep1 = 0.0;
    if (rep_on) {
        const double dmax = p.rep_lc1, dmax2 = dmax * dmax * (1.0 + 1e-15);
        const double dsure2 = dmax * dmax * (1.0 - 1e-15);    // surely inside: no root needed
        const int excl = nl.kind == 0 ? nl.exclusion : 0;
        const int lost = (g & 1) ? -1 : partner, gained = (g & 1) ? opp : -1;
        // the ring in registers, -2 past its end (rings above kRowPair: the
        // rest from LDS)
        int rg[kRowPair];
        const bool wide = __ballot(n0 > kRowPair) != 0ull;
#pragma unroll
        for (int i = 0; i < kRowPair; i++) rg[i] = S.nb[g][i];
#pragma unroll
        for (int i = 0; i < kRowPair; i++) rg[i] = i < n0 ? rg[i] & ~kNoFace : -2;
        auto in_ring = [&](int w) {
            bool hit = false;
#pragma unroll
            for (int i = 0; i < kRowPair; i++) hit |= rg[i] == w;
            if (wide)
                for (int i = kRowPair; i < n0; i++) hit |= (S.nb[g][i] & ~kNoFace) == w;
            return hit;
        };
        for (int t0 = 0;;) {
            d3 d[kCandBatch];
#pragma unroll
            for (int u = 0; u < kCandBatch; u++)
                if (cand[u] >= 0) d[u] = xv - d3{fm.x[3 * cand[u]], fm.x[3 * cand[u] + 1], fm.x[3 * cand[u] + 2]};
            // within the cutoff, excluded before (bit 30) and after (bit 31).
            // At level 2 the ring before the flip counts on both sides: the two
            // ends of the edge still share C and D after it, and C and D share
            // A and B before it.  Few candidates are left, if any: they are
            // collected, so that one step of the lanes deals with them
            int listed = 0;
#pragma unroll
            for (int u = 0; u < kCandBatch; u++) {
                const int c = cand[u];
                bool e0 = true, e1 = true;
                const double sq = c >= 0 ? sqnorm(d[u]) : 0.0;
                if (c >= 0 && sq <= dmax2 && (sq < dsure2 || sqrt(sq) < dmax)) {
                    e0 = e1 = nl.kind == 0 && c == ve;
                    if (excl >= 1 && !e0) {
                        e0 = in_ring(c);
                        e1 = (e0 && c != lost) || c == gained;
                        if (excl > 1) e0 = e1 = e0 || e1;
                    }
                }
                const bool left = !(e0 && e1);
                const unsigned b = (unsigned)(__ballot(left) >> (16 * g)) & 0xffffu;
                if (left) S.list[g][listed + __popc(b & ((1u << q) - 1u))] = c | (e0 ? 1 << 30 : 0) | (e1 ? 1 << 31 : 0);
                listed += __popc(b);
            }
            wave_sync();
            for (int i0 = 0; __ballot(i0 < listed); i0 += 16) {
                double v0 = 0.0, v1 = 0.0;
                if (i0 + q < listed) {
                    const int w = S.list[g][i0 + q], c = w & ~(3 << 30);
                    bool e0 = w & (1 << 30), e1 = w < 0;
                    const d3 dc = xv - d3{fm.x[3 * c], fm.x[3 * c + 1], fm.x[3 * c + 2]};
                    if (excl > 1) {
                        // the candidate's neighbours, as stored and on the flipped side
                        const int* cr = rows.nb + (size_t)kRowW * c;
                        const int4 w0 = reinterpret_cast<const int4*>(cr)[0], w1 = reinterpret_cast<const int4*>(cr)[1];
                        const int cw[kRowPair] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
                        const int cl = c == pv[0] ? pv[2] : (c == pv[2] ? pv[0] : -1);
                        const int cg = c == pv[1] ? pv[3] : (c == pv[3] ? pv[1] : -1);
                        auto meet = [&](int x) {
                            const bool in0 = in_ring(x);
                            e0 |= in0;
                            e1 |= x != cl && ((in0 && x != lost) || x == gained);
                        };
                        int n = 0;
                        for (; n < kRowPair; n++) {
                            int x = cw[0];
    #pragma unroll
                            for (int i = 1; i < kRowPair; i++) x = n == i ? cw[i] : x;
                            if (x < 0) break;
                            meet(x & ~kNoFace);
                        }
                        if (n == kRowPair)
                            for (; n < kRowW && cr[n] >= 0; n++) meet(cr[n] & ~kNoFace);
                        if (cg >= 0) e1 |= (in_ring(cg) && cg != lost) || cg == gained;
                    }
                    if (!(e0 && e1)) {
                        const double v = rep_value(norm(dc), p.rep_lc1, p.rep_r);
                        if (!e0) v0 = v;
                        if (!e1) v1 = v;
                    }
                }
                if constexpr (kWalk) {
                    // in the candidates' order, which the list keeps
                    for (int i = 0; i < 16 && __ballot(i0 + i < listed); i++) {
                        rep0 += __shfl(v0, i, 16);
                        rep1 += __shfl(v1, i, 16);
                    }
                } else {
                    rep0 += v0;
                    rep1 += v1;
                }
            }
            t0 += kListMax;
            if (!__ballot(t0 < total)) break;
            load_candidates(t0);
        }
        if constexpr (!kWalk) {
            rep0 = row_sum(rep0);
            rep1 = row_sum(rep1);
        }
    }
    res.val[0] = area;
    res.val[1] = vol;
    res.val[2] = curv;
    res.val[3] = 2 * curv * curv / area;
    res.val[4] = teth;
    res.val[5] = side ? rep1 : rep0;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        if constexpr (kWalk) {
            // vertex by vertex, as the edge's halfedges then name them: from
            // to(2e) on, which after the flip is the vertex that came second
            const int first = (side_work.swapped ? 32 : 0) + 16 * side;
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < 4; i++) sum += __shfl(res.val[k], ((first + 16 * i) & 48) + 8 * side, 64);
            res.val[k] = sum;
        } else {
            res.val[k] += __shfl_xor(res.val[k], 16, 64);
            res.val[k] += __shfl_xor(res.val[k], 32, 64);
        }
    }
    return res;
}

// A proposal's record, which its wave stores in one go: kD doubles (of the
// parallel sweep the patch differences, after minus before; of the serial sweep
// the sums before the flip, then after it) in words 0 .. 2 kD - 1, then its validity
// (1 flippable, 0 not, -1 index out of range) and the FlipEdge.  The readers take
// records with several lanes each: read by one thread each, a record would be
// a request for the same line per word pair.
template <int kD>
__device__ __forceinline__ void put_record(int* rec, int lane, int valid, const double (&d)[kD], const FlipEdge& f)
{
    int w = 0;
#pragma unroll
    for (int c = 0; c < kD; c++)
        if ((lane >> 1) == c) w = (lane & 1) ? __double2hiint(d[c]) : __double2loint(d[c]);
    const int rest[14] = {valid, f.e, f.pv[0], f.pv[1], f.pv[2], f.pv[3], f.a1, f.a2, f.b1, f.b2, f.fa, f.fb, f.ha,
                          f.hb};
#pragma unroll
    for (int c = 0; c < 14; c++)
        if (lane == 2 * kD + c) w = rest[c];
    if (lane < 2 * kD + 14) put(rec + lane, w);
}
__device__ __forceinline__ FlipEdge flip_edge_of(const int* m)    // the words after a record's validity
{
    return FlipEdge{m[0], {m[1], m[2], m[3], m[4]}, m[5], m[6], m[7], m[8], m[9], m[10], m[11], m[12]};
}

// The Metropolis test (flips.cpp:57-64) u <= min(1, exp(-de)) as de <= -log(u):
// the logarithm is taken once per proposal, not in every step of a walk.  The same
// test but for the rounding of its two sides: the serial sweep only looks ahead
// with it.  An injected u may lie outside [0, 1]: u <= 0 passes whatever the
// (ordered) de, as exp(-de) is never negative, u > 1 and NaN never pass.
__device__ __forceinline__ double minus_log(double u)
{
    if (u <= 0.0) return INFINITY;
    return u > 1.0 ? -INFINITY : -log(u);
}

// ================================================ windowed serial sweep ==
// The serial sweep's decisions, topology and running properties, bit for bit,
// from windows of W proposals evaluated at once.  One launch per window: a wave
// per proposal evaluates is_flip_ok and its patch before and after the flip on
// the topology at the window start, and the last workgroup commits the window in
// order up to the first proposal whose evaluation an earlier one has changed.
// What an earlier proposal j of the window changes for a later one k:
//   * accepted: the one-rings of j's four patch vertices V(j).  k read the
//     one-rings of its patch vertices P_k and, for exclusion level 2, the
//     neighbour sets of their one-ring vertices N(P_k); so V(j) meeting P_k (or
//     N(P_k)) makes k stale.
//   * rejected (do_flip twice): every vertex keeps its neighbours in the same
//     cyclic order, but the edge's halfedges swap direction, so a later
//     proposal of the same edge adds its patch vertices in another order, and
//     an endpoint whose circulator started on the edge starts at the next
//     spoke.  k is decided only while no accepted proposal has met P_k, so
//     every earlier one that could have done this to it was rejected, if it was
//     valid: WalkOrder works out the order from the window's proposals alone.
// The commit tests all proposals up to the first stale one against the current
// state at once and takes the first acceptance: a rejection leaves the state, so
// every decision is that of the sequential walk to rounding.  One wave then runs
// the one-workgroup sweep's rounding path (props -= old, += new; on rejection
// -= new, += old) through these decisions, a component per lane, and every thread
// takes its proposal's decision again, from the path's own states.  The window ends
// after the first one that this changes.
// The halfedge arrays are then rewritten (do_flip or do_flip twice) by one thread per
// committed proposal.  Proposals that share a face must follow each other (a
// stamp per face holds the window's first valid proposal on it): those
// connected through shared faces get ascending ranks, and the ranks are
// applied one after the other.
// A window commits at least its first proposal, which cannot be stale.
// At level 7 (491520 edges) a window of 256 takes 44 us, 6.2 of them for the
// rounding path and 1.3 for the decisions on it; evaluating by ring walks (30 us)
// and committing (51 us) were two launches.

// The proposals of its window before a wave's own, four per lane, and the spokes at
// which the circulators of its patch vertices start when it is decided.
struct WalkOrder {
    static constexpr bool kWalk = true;
    const FlipMeshView& fm;
    const FlipRows& rows;
    const int (&before)[kSerialWindowMax / 64];    // lane l: the edges of proposals l, l + 64, ..., -1: none
    bool swapped;    // the edge's halfedges have swapped direction
    int h = 0;       // lanes of a vertex: the halfedge at which its walk starts
    int from = 0;    // its target
    __device__ WalkOrder(const FlipMeshView& m, const FlipRows& r, const int (&b)[kSerialWindowMax / 64], int e)
        : fm(m), rows(r), before(b)
    {
        int n = 0;
#pragma unroll
        for (int u = 0; u < kSerialWindowMax / 64; u++) n += __popcll(__ballot(before[u] == e));
        swapped = n & 1;
    }
    __device__ __forceinline__ void load(int v, int) { h = fm.v_he[v]; }
    __device__ __forceinline__ void more(int, int, bool) {}
    __device__ __forceinline__ void issue(bool)
    {
        bool hit = false;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int e = __builtin_amdgcn_readlane(h, 16 * g) >> 1;
#pragma unroll
            for (int u = 0; u < kSerialWindowMax / 64; u++) hit |= before[u] == e;
        }
        if (__ballot(hit)) moved();
        from = fm.he_to[h];
    }
    // each valid earlier proposal of the edge a walk starts on moves it to the
    // next spoke, where a later one may move it again
    __device__ __forceinline__ void moved()
    {
        const int lane = threadIdx.x & 63;
        for (int g = 0; g < 4; g++) {
            int at = __builtin_amdgcn_readlane(h, 16 * g);
            for (int j = -1;;) {
                int next = kSerialWindowMax;
#pragma unroll
                for (int u = kSerialWindowMax / 64 - 1; u >= 0; u--) {
                    const unsigned long long b = __ballot(before[u] == at >> 1 && 64 * u + lane > j);
                    if (b) next = 64 * u + __ffsll((long long)b) - 1;
                }
                if (next == kSerialWindowMax || !flippable(at >> 1)) break;
                j = next;
                at = fm.he_next[at ^ 1];
            }
            if (lane >> 4 == g) h = at;
        }
    }
    // flip_ok of an edge, by the wave
    __device__ __forceinline__ bool flippable(int e)
    {
        static_assert(kRowW == 32, "a lane per slot of two rows");
        const FlipEdge f = load_flip_edge(fm, e);
        if (f.fa < 0 || f.fb < 0) return false;
        const int lane = threadIdx.x & 63;
        const int id = rows.nb[(size_t)kRowW * (lane < 32 ? f.pv[1] : f.pv[3]) + (lane & 31)];
        const unsigned long long b = __ballot(id >= 0);
        const unsigned c = (unsigned)b, d = (unsigned)(b >> 32);
        if (c == ~0u || d == ~0u || f.pv[1] == f.pv[3]) return false;
        const int n = __ffs(~c) - 1;    // slots of the first row before its end mark
        return !__ballot(lane < n && (id & ~kNoFace) == f.pv[3]);
    }
};

__global__ void __launch_bounds__(256) k_sf_begin(FlipMeshView fm, FlipRows rows, const Globals* __restrict__ g0,
                                                  EParams p, int nflips, SerialState* __restrict__ st,
                                                  unsigned long long* __restrict__ fstamp)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < fm.nv) build_rows(fm, rows, t);
    if (t < fm.nf) fstamp[t] = 0ull;
    if (t != 0) return;
    double props[6];
    for (int k = 0; k < 6; k++) props[k] = st->props[k] = g0->props[k];
    st->e0 = energy_of(props, p);
    st->pos = 0;
    st->done = nflips <= 0;
    st->used = st->acc = st->err = st->window = 0;
    st->count = 0u;
}

constexpr int kRecInts = 38;    // the used words of a record
constexpr int kRecValid = 24, kRecEdge = 25;
struct SerialShared {
    alignas(16) int rec[kSerialWindowMax * kRecInts];
    // the rounding path: properties after each proposal's flip, and their energies
    double after[kSerialWindowMax][6];
    double energy[kSerialWindowMax];
    unsigned long long acc[kPatchWaves];    // the accepted proposals
    // one-rings of every proposal's patch, kRowPair slots each and -1 past the
    // end, as int4 chunks rotated by the proposal's number (bank conflicts)
    int4 ring[kSerialWindowMax][kRowPair];
    alignas(16) int label[kSerialWindowMax];
    int slots[2][kPatchWaves];
    int wsum[kPatchWaves];
    unsigned long long wide[kPatchWaves];    // proposals with a ring longer than kRowPair
    int maxrank;
    int nflip, flip[kSerialWindowMax];
};

// a record's sums before the flip (0-5) and after it (6-11)
__device__ __forceinline__ const double* sums_of(const int* m) { return reinterpret_cast<const double*>(m); }

// One wave runs the serial sweep's rounding path from properties P through the
// proposals [0, end) and some after them, lane c < 6 the component c (an invalid
// proposal's sums are zeros); bit k of acc: proposal k is accepted.
__device__ __forceinline__ void serial_path(SerialShared& S, const double (&P)[6], int end)
{
    const int c = threadIdx.x & 63;
    if (c >= 6) return;
    double x = c == 0 ? P[0] : (c == 1 ? P[1] : (c == 2 ? P[2] : (c == 3 ? P[3] : (c == 4 ? P[4] : P[5]))));
    // kStep proposals in registers, the next ones' loads in flight, and nothing
    // but the chain of additions where none is accepted: one wave alone issues an
    // instruction at a time (256 proposals take 6.2 us; with bounds, register moves
    // and the choice between two states in the loop 12.3)
    constexpr int kStep = 16;
    static_assert(kSerialWindowMax % (2 * kStep) == 0, "two steps per round");
    struct Sums {
        double o[kStep], n[kStep];
    } a, b;
    auto load = [&](int i0, Sums& s) {
        const double* d = sums_of(S.rec + kRecInts * min(i0, kSerialWindowMax - kStep)) + c;
#pragma unroll
        for (int i = 0; i < kStep; i++) {
            s.o[i] = d[kRecInts / 2 * i];
            s.n[i] = d[kRecInts / 2 * i + 6];
        }
    };
    auto run = [&](int i0, const Sums& s) {
        double q[kStep];
        const unsigned acc =
            __builtin_amdgcn_readfirstlane((int)(unsigned)(S.acc[i0 >> 6] >> (i0 & 63))) & ((1u << kStep) - 1u);
        if (acc == 0u) {
#pragma unroll
            for (int i = 0; i < kStep; i++) {
                q[i] = x - s.o[i];
                q[i] += s.n[i];
                x = q[i] - s.n[i];
                x += s.o[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < kStep; i++) {
                q[i] = x - s.o[i];
                q[i] += s.n[i];
                double r = q[i] - s.n[i];
                r += s.o[i];
                x = (acc >> i) & 1u ? q[i] : r;
            }
        }
#pragma unroll
        for (int i = 0; i < kStep; i++) S.after[i0 + i][c] = q[i];
    };
    load(0, a);
    for (int i0 = 0; i0 < end; i0 += 2 * kStep) {
        load(i0 + kStep, b);
        run(i0, a);
        load(i0 + 2 * kStep, a);
        run(i0 + kStep, b);
    }
}

__device__ __forceinline__ void sf_commit(const FlipMeshView& fm, const FlipRows& rows, const EParams& p, int nflips,
                                          const double* __restrict__ uniforms, int n_uniforms, uint64_t seed,
                                          int injected, int W, int need_nb, SerialState* __restrict__ st,
                                          const int* rec, const unsigned long long* fstamp, SerialShared& S)
{
    const int tid = threadIdx.x, wave = tid >> 6;
    const int pos0 = st->pos, used0 = st->used, wid = st->window + 1;
    const int cnt = min(W, nflips - pos0);
    {
        // thirty-two lanes per record
        const unsigned long long* src = reinterpret_cast<const unsigned long long*>(rec);
        const int c = tid & 31, r0 = tid >> 5;
        unsigned long long w[32];
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const int r = r0 + 8 * i;
            w[i] = r < cnt && c < kRecInts / 2 ? get(src + (size_t)(kSerialRecord / 2) * r + c) : 0ull;
        }
#pragma unroll
        for (int i = 0; i < 32; i++)
            if (c < kRecInts / 2)
                *reinterpret_cast<unsigned long long*>(S.rec + kRecInts * (r0 + 8 * i) + 2 * c) = w[i];
    }
    double P[6], e0 = st->e0;
#pragma unroll
    for (int c = 0; c < 6; c++) P[c] = st->props[c];
    if (tid == 0) S.maxrank = S.nflip = 0;
    S.label[tid] = tid;
    __syncthreads();
    // thread k holds proposal k of the window
    const int k = tid;
    const int* m = S.rec + kRecInts * k;
    const int v = k < cnt ? m[kRecValid] : -2;
    const FlipEdge fe = flip_edge_of(m + kRecEdge);
    const int pv0 = fe.pv[0], pv1 = fe.pv[1], pv2 = fe.pv[2], pv3 = fe.pv[3];
    const bool inner = v >= 0 && fe.fa >= 0 && fe.fb >= 0;
    double dp[6];
#pragma unroll
    for (int c = 0; c < 6; c++) dp[c] = sums_of(m)[6 + c] - sums_of(m)[c];
    // window positions of the first valid proposals on its faces, and the
    // rings that acceptances are checked against
    int l0 = k, l1 = k;
    bool wide = false;
    if (v == 1) {
        const unsigned long long s0 = get(fstamp + fe.fa), s1 = get(fstamp + fe.fb);
        if (need_nb) {
            int4 w[8];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int4* row = reinterpret_cast<const int4*>(rows.nb + (size_t)kRowW * fe.pv[g]);
                w[2 * g] = row[0];
                w[2 * g + 1] = row[1];
            }
#pragma unroll
            for (int g = 0; g < 4; g++) {
                int x[kRowPair] = {w[2 * g].x, w[2 * g].y, w[2 * g].z, w[2 * g].w,
                                   w[2 * g + 1].x, w[2 * g + 1].y, w[2 * g + 1].z, w[2 * g + 1].w};
                bool more = true;
#pragma unroll
                for (int i = 0; i < kRowPair; i++) {
                    more = more && x[i] >= 0;
                    x[i] = more ? x[i] & ~kNoFace : -1;
                }
                wide = wide || more;
                S.ring[k][(2 * g + k) & 7] = make_int4(x[0], x[1], x[2], x[3]);
                S.ring[k][(2 * g + 1 + k) & 7] = make_int4(x[4], x[5], x[6], x[7]);
            }
        }
        l0 = W - (int)(unsigned)s0;
        l1 = W - (int)(unsigned)s1;
    }
    // rank among the valid proposals: the uniform's index
    const unsigned long long vb = __ballot(v == 1), wb = __ballot(wide);
    if ((tid & 63) == 0) {
        S.wsum[wave] = __popcll(vb);
        S.wide[wave] = wb;
    }
    __syncthreads();
    int mr = __popcll(vb & ((1ull << (tid & 63)) - 1ull)), nvalid = 0;
    for (int i = 0; i < kPatchWaves; i++) {
        if (i < wave) mr += S.wsum[i];
        nvalid += S.wsum[i];
    }
    // an injected stream too short: the proposal that finds it empty is
    // rejected and the sweep stops after it
    const int movf = injected ? max(n_uniforms - used0, 0) : INT_MAX;
    const bool ovf = v == 1 && mr == movf, can = v == 1 && mr < movf;
    const double u =
        !can ? __builtin_nan("") : (injected ? uniforms[used0 + mr] : rng_uniform(seed, (uint64_t)(used0 + mr)));
    const double nlu = minus_log(u);
    double P0[6], start0 = e0;
#pragma unroll
    for (int c = 0; c < 6; c++) P0[c] = P[c];

    // every thread carries the state; one barrier per step
    bool stale = false, accepted = false;
    int pos = 0, err = 0, it = 0;
    while (pos < cnt) {
        // the first proposal that is not to be decided now (1), finds the
        // uniform stream empty (2) or is likely to be accepted (3)
        int what = 0;
        if (k >= pos && k < cnt) {
            if (stale || v < 0) what = 1;
            else if (ovf) what = 2;
            else if (can) {
                double q[6];
#pragma unroll
                for (int c = 0; c < 6; c++) q[c] = P[c] + dp[c];
                what = energy_of(q, p) - e0 <= nlu ? 3 : 0;
            }
        }
        const unsigned long long b = __ballot(what != 0);
        const int lane1 = b ? __ffsll((long long)b) - 1 : 0;
        const int what1 = __builtin_amdgcn_readlane(what, lane1);
        int* slots = S.slots[it++ & 1];
        if ((tid & 63) == 0) slots[wave] = b ? (64 * wave + lane1) * 4 + what1 : INT_MAX;
        __syncthreads();
        int s = INT_MAX;
#pragma unroll
        for (int i = 0; i < kPatchWaves; i++) s = min(s, slots[i]);
        if (s == INT_MAX) {
            pos = cnt;
            break;
        }
        const int first = s >> 2;
        what = s & 3;
        pos = what == 1 ? first : first + 1;
        if (what == 2) err = 2;
        if (what != 3) break;
        const int* f = S.rec + kRecInts * first;
#pragma unroll
        for (int c = 0; c < 6; c++) P[c] += sums_of(f)[6 + c] - sums_of(f)[c];
        e0 = energy_of(P, p);
        if (k == first) accepted = true;
        // later proposals whose patch meets the accepted patch are stale; at
        // exclusion level 2 its one-rings count too (adjacency is symmetric:
        // they meet P_k exactly when V(j) meets N(P_k))
        bool hit = false;
        auto check = [&](int x) { hit |= (x == pv0) | (x == pv1) | (x == pv2) | (x == pv3); };
        if (need_nb) {
            int4 x[kRowPair];
#pragma unroll
            for (int i = 0; i < kRowPair; i++) x[i] = S.ring[first][i];
#pragma unroll
            for (int i = 0; i < kRowPair; i++) {
                check(x[i].x);
                check(x[i].y);
                check(x[i].z);
                check(x[i].w);
            }
            if ((S.wide[first >> 6] >> (first & 63)) & 1ull)
                for (int g = 0; g < 4; g++) {
                    const int* row = rows.nb + (size_t)kRowW * f[kRecEdge + 1 + g];
                    for (int i = 0; i < kRowW && row[i] >= 0; i++) check(row[i] & ~kNoFace);
                }
        }
#pragma unroll
        for (int g = 0; g < 4; g++) check(f[kRecEdge + 1 + g]);
        stale = stale || (hit && inner);
    }

    // the same decisions from the rounding path
    int nacc = 0;
    {
        const unsigned long long b = __ballot(accepted);
        if ((tid & 63) == 0) S.acc[wave] = b;
        __syncthreads();
        if (wave == 0) serial_path(S, P0, pos);
        __syncthreads();
        const double en = k < pos ? energy_of(S.after[k], p) : 0.0;
        S.energy[k] = en;
        __syncthreads();
        // the energy before this proposal: that of the acceptance before it
        int last = -1;
#pragma unroll
        for (int w = 0; w < kPatchWaves; w++) {
            unsigned long long a = S.acc[w];
            if (64 * w + 63 >= k) a &= 64 * w < k ? (1ull << (k - 64 * w)) - 1ull : 0ull;
            if (a) last = 64 * w + 63 - __clzll((long long)a);
        }
        const double de = en - (last < 0 ? start0 : S.energy[last]);
        const double alpha = de < 0.0 ? 1.0 : exp(-de);
        const bool take = k < pos && u <= alpha;
        const unsigned long long m = __ballot(take != accepted);
        int* slots = S.slots[it++ & 1];
        if ((tid & 63) == 0) slots[wave] = m ? 64 * wave + __ffsll((long long)m) - 1 : INT_MAX;
        __syncthreads();
        int changed = INT_MAX;
#pragma unroll
        for (int i = 0; i < kPatchWaves; i++) changed = min(changed, slots[i]);
        if (changed != INT_MAX) {
            pos = changed + 1;
            err = 0;
            accepted = k < changed ? accepted : k == changed && !accepted;
        }
        // the state after the last committed proposal
        if (pos > 0) {
            const bool now = (((S.acc[(pos - 1) >> 6] >> ((pos - 1) & 63)) & 1ull) != 0ull) != (pos - 1 == changed);
            const double* d = sums_of(S.rec + kRecInts * (pos - 1));
#pragma unroll
            for (int c = 0; c < 6; c++) {
                const double q = S.after[pos - 1][c];
                double r = q - d[6 + c];
                r += d[c];
                P[c] = now ? q : r;
            }
        }
        e0 = start0;
        int at = -1;
#pragma unroll
        for (int w = 0; w < kPatchWaves; w++) {
            unsigned long long a = S.acc[w];
            if (64 * w + 63 >= pos) a &= 64 * w < pos ? (1ull << (pos - 64 * w)) - 1ull : 0ull;
            if (changed != INT_MAX && changed >> 6 == w) a ^= 1ull << (changed & 63);
            nacc += __popcll(a);
            if (a) at = 64 * w + 63 - __clzll((long long)a);
        }
        if (at >= 0) e0 = S.energy[at];
    }

    // ranks of the committed flips along shared faces: the labels become the
    // least position of each connected set
    const bool commit = k < pos && v == 1;
    int rank = 0;
    if (!commit) l0 = l1 = k;
    if (__syncthreads_or(l0 != k || l1 != k)) {
        for (;;) {
            const int a = min(S.label[k], min(S.label[l0], S.label[l1]));
            const bool low = a < S.label[k] || a < S.label[l0] || a < S.label[l1];
            if (!__syncthreads_or(low)) break;
            if (low) {
                atomicMin(&S.label[k], a);
                atomicMin(&S.label[l0], a);
                atomicMin(&S.label[l1], a);
            }
            __syncthreads();
        }
        if (commit) {
            const int a = S.label[k];
            const int4* lab = reinterpret_cast<const int4*>(S.label);
#pragma unroll 8
            for (int i = 0; i < kSerialWindowMax / 4; i++) {
                const int4 x = lab[i];
                rank += (x.x == a && 4 * i < k) + (x.y == a && 4 * i + 1 < k) + (x.z == a && 4 * i + 2 < k) +
                        (x.w == a && 4 * i + 3 < k);
            }
            if (rank) atomicMax(&S.maxrank, rank);
        }
        __syncthreads();
    }
    if (accepted) S.flip[atomicAdd(&S.nflip, 1)] = k;
    // rank 0 from the records, later ranks from what the earlier ones left
    const int maxrank = S.maxrank;
    for (int i = 0; i <= maxrank; i++) {
        if (commit && rank == i) {
            const FlipEdge f = i == 0 ? fe : load_flip_edge(fm, fe.e);
            if (accepted) store_flip(fm, f);
            else store_flip_twice(fm, f);
        }
        __threadfence_block();
        __syncthreads();
    }
    // the rows of the accepted patches, one thread per vertex (accepted
    // proposals of a window have disjoint patches, which earlier flips left
    // as the records have them)
    for (int t = tid; t < 4 * S.nflip; t += 256) {
        const int g = t & 3;
        const int* f = S.rec + kRecInts * S.flip[t >> 2] + kRecEdge + 1;    // the patch vertices
        flip_row(rows, f[g], g, g < 2 ? f[2] : f[0], g == 1 ? f[3] : f[1], f[-1], make_int2(0, 0));
    }
    // state; the uniforms used are the valid proposals before pos
    if (pos < cnt ? k == pos : tid == 0) {
        st->used = used0 + (pos < cnt ? mr : nvalid);
        if (!err && pos < cnt && v == -1) err = 1;
        st->err = err;
        st->pos = pos0 + pos;
        st->done = (err || pos0 + pos >= nflips) ? 1 : 0;
    }
    if (tid == 0) {
#pragma unroll
        for (int c = 0; c < 6; c++) st->props[c] = P[c];
        st->e0 = e0;
        st->acc += nacc;
        st->window = wid;
    }
}

__global__ void __launch_bounds__(256) k_sf_window(FlipMeshView fm, FlipRows rows, NListView nl, EParams p,
                                                   int nflips, const int* __restrict__ proposals,
                                                   const double* __restrict__ uniforms, int n_uniforms, uint64_t seed,
                                                   int injected, int W, int need_nb, SerialState* __restrict__ st,
                                                   int* rec, unsigned long long* fstamp)
{
    __shared__ union Shared {
        PatchShared patch[kPatchWaves];
        SerialShared serial;
        __device__ Shared() {}
    } S;
    if (st->done) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int k = blockIdx.x * kPatchWaves + wave;
    const int cnt = min(W, nflips - st->pos);
    const int blocks = (cnt + kPatchWaves - 1) / kPatchWaves;
    if ((int)blockIdx.x >= blocks) return;
    if (k < cnt) {
        const int i = st->pos + k, ne = fm.nh / 2;
        const int e = injected ? proposals[i] : rng_edge(seed, (uint64_t)i, ne);
        int valid = -1;
        FlipEdge f{};
        double d[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (e >= 0 && e < ne) {
            f = load_flip_edge(fm, e);
            valid = 0;
            if (f.fa >= 0 && f.fb >= 0) {
                int before[kSerialWindowMax / 64];
#pragma unroll
                for (int u = 0; u < kSerialWindowMax / 64; u++) {
                    const int j = 64 * u + lane;
                    before[u] = -1;
                    if (j < k) before[u] = injected ? proposals[i - k + j] : rng_edge(seed, (uint64_t)(i - k + j), ne);
                }
                WalkOrder order(fm, rows, before, e);
                const PatchResult r = patch_eval(fm, nl, p, rows, f.pv, S.patch[wave], order);
                if (r.ok) {
                    valid = 1;
                    const unsigned long long key =
                        ((unsigned long long)(unsigned)(st->window + 1) << 32) | (unsigned)(W - k);
                    if (lane < 2) atomicMax(&fstamp[lane ? f.fb : f.fa], key);
#pragma unroll
                    for (int c = 0; c < 12; c++) d[c] = __shfl(r.val[c % 6], c < 6 ? 0 : 8, 64);
                }
            }
        }
        put_record(rec + (size_t)kSerialRecord * k, lane, valid, d, f);
    }
    if (!last_block(&st->count, (unsigned)blocks)) return;
    sf_commit(fm, rows, p, nflips, uniforms, n_uniforms, seed, injected, W, need_nb, st, rec, fstamp, S.serial);
}

void launch_serial_begin(const FlipMeshView& fm, const FlipRows& rows, const Globals* g0, const EParams& p, int nflips,
                         SerialState* st, unsigned long long* fstamp, hipStream_t s)
{
    const int n = std::max(std::max(fm.nv, fm.nf), 1);
    hipLaunchKernelGGL(k_sf_begin, dim3((n + 255) / 256), dim3(256), 0, s, fm, rows, g0, p, nflips, st, fstamp);
}

void launch_serial_windows(const FlipMeshView& fm, const FlipRows& rows, const NListView& nl, const EParams& p,
                           int nflips, const int* proposals, const double* uniforms, int n_uniforms, uint64_t seed,
                           int injected, int W, SerialState* st, int* rec, unsigned long long* fstamp,
                           int n_windows, hipStream_t s)
{
    const int need_nb = nl.kind == 0 && nl.exclusion > 1 && p.rep_lc1 > 0;
    for (int r = 0; r < n_windows; r++)
        hipLaunchKernelGGL(k_sf_window, dim3((W + kPatchWaves - 1) / kPatchWaves), dim3(256), 0, s, fm, rows, nl, p,
                           nflips, proposals, uniforms, n_uniforms, seed, injected, W, need_nb, st, rec, fstamp);
}

// ============================================ conflict-free parallel sweep ==
// pflip (flip_parallel_batches, flips.cpp:82-166) lets OpenMP threads lock
// the edge patch of their proposal (flip_patch, flip_utils.cpp:43-68), skip
// proposals whose patch is taken, flip and evaluate in parallel and apply the
// Metropolis test one flip at a time.  Here a round of B proposals is one
// launch:
//   claim   every proposal writes its priority key into all edges of its
//           patch with a 64-bit atomicMax (later rounds have larger keys, so
//           the owner array never needs clearing).  What the maximum replaced
//           tells the loser: a larger key of the same round is the winner's, a
//           smaller one belongs to a proposal that has just lost the edge.  Of
//           all proposals that claim an edge, every one but the largest is
//           told so by its own claim or by a later one;
//   eval    the same wave evaluates the patch before and after the flip
//           (patch_eval) without waiting for the outcome of its claims: the
//           evaluation after the flip sees the proposal's own flip only (the
//           reference's threads see whichever other flips have happened);
//   scan    the last workgroup of the mesh runs the FP64 Metropolis test in
//           proposal order on the running global properties, over the
//           proposals that lost no edge and pass is_flip_ok: their patches
//           are pairwise disjoint;
//   apply   the same workgroup flips the accepted ones.
// Proposals that lose a claim are skipped, like the reference's failed locks.
// No workgroup reads topology that another rewrites within a launch (the last
// one applies when all others have read); the result depends only on the seed.
// At level 7 (491520 edges, 480 proposals) a round takes 23 us, and 37 us for 8
// such meshes at once; claim, evaluation by ring walks, scan and application as
// launches of their own took 7.3 + 32.5 + 11.2 + 4.6 us and 9.8 + 64.8 + 14.0 +
// 4.7 us.

// The flip patch of edge e (flip_utils.cpp:43-68) is the set of edges of h
// and of next(h) over the outgoing halfedges h of its four vertices: the spoke
// and rim edges of their rows.

__device__ __forceinline__ int pflip_edge(uint64_t seed, int round, int B, int i, int ne)
{
    return rng_edge(seed ^ 0x5bd1e9955bd1e995ull, (uint64_t)round * (uint64_t)B + (uint64_t)i, ne);
}

__device__ __forceinline__ unsigned long long pflip_key(int round, int B, int i)
{
    return ((unsigned long long)(round + 1) << 32) | (unsigned)(B - i);
}

// proposals of replica a in round r (<= 0 once its sweep is done)
__device__ __forceinline__ int pflip_nprop(const PflipArgs& a, int round)
{
    return min(a.batch, a.nflips - round * a.batch);
}

// One wave's claims: lane 16 g + slot claims the spoke and the rim edge of that
// slot of patch vertex g's row.  The edges are loaded beside the row, the
// atomics go out behind the position loads, and what they replaced is looked
// at after the evaluation.
struct PatchClaim {
    static constexpr bool kWalk = false;
    const PflipArgs& a;
    const unsigned long long key;
    const int round;
    int2 er = make_int2(0, 0);
    unsigned long long o0 = 0ull, o1 = 0ull;
    bool lost = false;
    __device__ __forceinline__ void load(int v, int slot) { er = a.rows.er[(size_t)kRowW * v + slot]; }
    __device__ __forceinline__ void issue(bool has)
    {
        if (!has) return;
        o0 = atomicMax(&a.owner[er.x], key);
        o1 = atomicMax(&a.owner[er.y], key);
    }
    __device__ __forceinline__ void more(int v, int slot, bool has)
    {
        if (!has) return;
        const int2 e2 = a.rows.er[(size_t)kRowW * v + slot];
        told(atomicMax(&a.owner[e2.x], key));
        told(atomicMax(&a.owner[e2.y], key));
    }
    __device__ __forceinline__ void told(unsigned long long old)
    {
        if ((old >> 32) != (key >> 32) || old == key) return;
        if (old > key) lost = true;
        else put(a.lost + (a.batch - (int)(unsigned)old), round + 1);
    }
    __device__ __forceinline__ bool beaten()
    {
        told(o0);
        told(o1);
        return __ballot(lost) != 0ull;
    }
};

constexpr int kScanPer = 2;    // proposals per thread
struct ScanShared {
    double dp[256 * kScanPer][7];    // patch differences and (as an integer) the validity
    int slots[2][kPatchWaves];
    int acc[256 * kScanPer];
};

// state: props[6], e0, accepted count (as double).  The Metropolis test
// walks the winners in proposal order on the running properties
// (flips.cpp:146-163), with a rejected flip restoring the running properties
// exactly.  Most winners are rejected and a rejection leaves the state
// unchanged, so the workgroup tests the next `window` proposals of each half
// of a chunk of 512 (thread t holds proposals t and t + 256) against the
// current state at once, takes the first acceptance in proposal order, applies
// it and continues after it: every decision is the one the sequential walk
// makes, and the walk takes one parallel step, of one barrier, per acceptance
// instead of one dependent FP64 chain per winner.  Every thread carries the
// state and adds the accepted difference itself.
__device__ __forceinline__ void pflip_decide(const PflipArgs& a, int round, int nprop, int window, ScanShared& S)
{
    const int tid = threadIdx.x, wave = tid >> 6;
    const uint64_t useed = a.seed ^ 0x5bd1e9955bd1e995ull;
    double P[6], e0 = a.state[6], nacc = a.state[7];
#pragma unroll
    for (int c = 0; c < 6; c++) P[c] = a.state[c];
    constexpr int kChunk = 256 * kScanPer;
    int it = 0;
    for (int base = 0; base < nprop; base += kChunk) {
        const int cnt = min(kChunk, nprop - base);
        // eight lanes per record, its first seven pairs of words
        unsigned long long w[8 * kScanPer];
        int lost[kScanPer];
        const int c8 = tid & 7, r0 = tid >> 3;
#pragma unroll
        for (int i = 0; i < 8 * kScanPer; i++) {
            const int r = r0 + 32 * i;
            w[i] = r < cnt && c8 < 7 ? get(reinterpret_cast<const unsigned long long*>(a.rec) +
                                           (size_t)(kFlipRecord / 2) * (base + r) + c8)
                                     : 0ull;
        }
#pragma unroll
        for (int h = 0; h < kScanPer; h++) lost[h] = 256 * h + tid < cnt ? get(a.lost + base + 256 * h + tid) : 0;
        double nlu[kScanPer];
#pragma unroll
        for (int h = 0; h < kScanPer; h++)
            nlu[h] = minus_log(rng_uniform(
                useed, (uint64_t)round * (uint64_t)a.batch + (uint64_t)(base + 256 * h + tid)));
#pragma unroll
        for (int i = 0; i < 8 * kScanPer; i++)
            if (c8 < 7) S.dp[r0 + 32 * i][c8] = __longlong_as_double((long long)w[i]);
        __syncthreads();
        double dp[kScanPer][6];
        bool win[kScanPer];
#pragma unroll
        for (int h = 0; h < kScanPer; h++) {
            const double* d = S.dp[256 * h + tid];
#pragma unroll
            for (int c = 0; c < 6; c++) dp[h][c] = d[c];
            win[h] = 256 * h + tid < cnt && __double2loint(d[6]) == 1 && lost[h] != round + 1;
        }
        const int reach = window * kScanPer;
        int n = 0;
        for (int pos = 0; pos < cnt;) {
            bool take[kScanPer];
#pragma unroll
            for (int h = 0; h < kScanPer; h++) {
                const int i = 256 * h + tid;
                take[h] = false;
                if (win[h] && i >= pos && i < pos + reach) {
                    double q[6];
#pragma unroll
                    for (int c = 0; c < 6; c++) q[c] = P[c] + dp[h][c];
                    take[h] = energy_of(q, a.p) - e0 <= nlu[h];
                }
            }
            // the first acceptance: of the lower half, else of the upper
            static_assert(kScanPer == 2, "halves in order");
            const unsigned long long b0 = __ballot(take[0]), b1 = __ballot(take[1]);
            int* slots = S.slots[it++ & 1];
            if ((tid & 63) == 0)
                slots[wave] = b0 ? 64 * wave + __ffsll((long long)b0) - 1
                                 : (b1 ? 256 + 64 * wave + __ffsll((long long)b1) - 1 : INT_MAX);
            __syncthreads();
            int first = INT_MAX;
#pragma unroll
            for (int i = 0; i < kPatchWaves; i++) first = min(first, slots[i]);
            if (first == INT_MAX) {
                pos += reach;
                continue;
            }
#pragma unroll
            for (int c = 0; c < 6; c++) P[c] += S.dp[first][c];
            e0 = energy_of(P, a.p);
            nacc += 1.0;
            if (tid == 0) S.acc[n] = base + first;
            n++;
            pos = first + 1;
        }
        __syncthreads();
        // apply: four threads per accepted flip, one per patch vertex; their
        // patches are disjoint, and the records hold what do_flip reads
        for (int t = tid; t < 4 * n; t += 256) {
            const unsigned long long* r = reinterpret_cast<const unsigned long long*>(a.rec) +
                                          (size_t)(kFlipRecord / 2) * S.acc[t >> 2];
            int m[26];
#pragma unroll
            for (int c = 6; c < 13; c++) {
                const unsigned long long x = get(r + c);
                m[2 * c] = (int)(unsigned)x;
                m[2 * c + 1] = (int)(unsigned)(x >> 32);
            }
            const FlipEdge f = flip_edge_of(m + 13);
            const int g = t & 3;
            const int2 ed = g == 1 ? make_int2(f.b2 >> 1, f.b1 >> 1) : make_int2(f.a2 >> 1, f.a1 >> 1);
            const int me = g == 0 ? f.pv[0] : (g == 1 ? f.pv[1] : (g == 2 ? f.pv[2] : f.pv[3]));
            if (g == 0) store_flip(a.fm, f);
            flip_row(a.rows, me, g, g < 2 ? f.pv[2] : f.pv[0], g == 1 ? f.pv[3] : f.pv[1], f.e, ed);
        }
        __syncthreads();
    }
    if (tid == 0) {
#pragma unroll
        for (int c = 0; c < 6; c++) a.state[c] = P[c];
        a.state[6] = e0;
        a.state[7] = nacc;
    }
}

__device__ __forceinline__ void pflip_round_body(const PflipArgs& a, int round, int window, int lb)
{
    __shared__ union Shared {
        PatchShared patch[kPatchWaves];
        ScanShared scan;
        __device__ Shared() {}
    } S;
    const int nprop = pflip_nprop(a, round);
    const int blocks = nprop > 0 ? (nprop + kPatchWaves - 1) / kPatchWaves : 0;
    if (lb >= blocks) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = lb * kPatchWaves + wave;
    if (i < nprop) {
        const int e = pflip_edge(a.seed, round, a.batch, i, a.fm.nh / 2);
        const FlipEdge f = load_flip_edge(a.fm, e);
        int valid = 0;
        double d[6] = {0, 0, 0, 0, 0, 0};
        if (f.fa >= 0 && f.fb >= 0) {
            PatchClaim claim{a, pflip_key(round, a.batch, i), round};
            const PatchResult r = patch_eval(a.fm, a.nl, a.p, a.rows, f.pv, S.patch[wave], claim);
            valid = !claim.beaten() && r.ok ? 1 : 0;
            if (valid) r.difference(d);
        }
        put_record(a.rec + (size_t)kFlipRecord * i, lane, valid, d, f);
    }
    if (!last_block(a.count, (unsigned)blocks)) return;
    pflip_decide(a, round, nprop, window, S.scan);
}

__global__ void __launch_bounds__(256) k_pflip_round(PflipArgs a, int round, int window)
{
    pflip_round_body(a, round, window, blockIdx.x);
}

// rows, running state, claims and counters at the start of a sweep
__device__ __forceinline__ void pflip_begin_body(const PflipArgs& a, int t)
{
    if (t < a.fm.nv) build_rows(a.fm, a.rows, t);
    if (t < a.fm.nh / 2) a.owner[t] = 0ull;
    if (t < a.batch) a.lost[t] = 0;
    if (t == 0) {
        double props[6];
        for (int k = 0; k < 6; k++) props[k] = a.state[k] = a.g0->props[k];
        a.state[6] = energy_of(props, a.p);
        a.state[7] = 0.0;
        *a.count = 0u;
    }
}

__global__ void __launch_bounds__(256) k_pflip_begin(PflipArgs a)
{
    pflip_begin_body(a, blockIdx.x * blockDim.x + threadIdx.x);
}

// ---- many meshes: round r of every replica per launch ----
__global__ void __launch_bounds__(256) k_pflip_begin_grouped(const PflipArgs* __restrict__ A)
{
    pflip_begin_body(A[blockIdx.y], blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void __launch_bounds__(256) k_pflip_round_grouped(const PflipArgs* __restrict__ A,
                                                             const int* __restrict__ block0, int R, int round,
                                                             int window)
{
    const int r = find_replica(block0, R, blockIdx.x);
    pflip_round_body(A[r], round, window, blockIdx.x - block0[r]);
}

static inline int pflip_begin_blocks(int nv, int nh, int batch)
{
    return (std::max(std::max(nv, nh / 2), std::max(batch, 1)) + 255) / 256;
}

int pflip_round_blocks(int batch) { return (batch + kPatchWaves - 1) / kPatchWaves; }

void launch_flip_parallel(const PflipArgs& a, int window, hipStream_t s)
{
    hipLaunchKernelGGL(k_pflip_begin, dim3(pflip_begin_blocks(a.fm.nv, a.fm.nh, a.batch)), dim3(256), 0, s, a);
    const int rounds = (a.nflips + a.batch - 1) / a.batch;
    window = std::min(std::max(window, 1), 256);
    for (int r = 0; r < rounds; r++) {
        const int nprop = std::min(a.batch, a.nflips - r * a.batch);
        hipLaunchKernelGGL(k_pflip_round, dim3(pflip_round_blocks(nprop)), dim3(256), 0, s, a, r, window);
    }
}

void launch_flip_parallel_grouped(const PflipGroup& g, hipStream_t s)
{
    if (g.R <= 0) return;
    hipLaunchKernelGGL(k_pflip_begin_grouped, dim3(pflip_begin_blocks(g.max_nv, g.max_nh, g.max_batch), g.R),
                       dim3(256), 0, s, g.d_args);
    const int window = std::min(std::max(g.window, 1), 256);
    for (int r = 0; r < g.rounds; r++)
        hipLaunchKernelGGL(k_pflip_round_grouped, dim3(g.total_blocks), dim3(256), 0, s, g.d_args, g.d_block0, g.R,
                           r, window);
}

}    // namespace tmh
