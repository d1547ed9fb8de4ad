// tm_energy.hip -- the two energy passes and the global reduction.
//
// trimem evaluates the functional vertex by vertex (src/kernel.h:140-262,
// src/energy.cpp:63-124): a properties pass, a reduction of six globals, a
// gradient-gather pass and a combination.  The same two-pass structure is
// forced here (the gradient at v needs curvature/area of v's neighbours and
// the global A, V, C), but each pass is one kernel over vertices that reads
// the clockwise one-ring table:
//
//   pass 1  per vertex v: area, volume, curvature, tether, bending and
//           repulsion from the faces (v, j_m, j_{m-1}) and edges (v, j_m) of
//           its ring (mesh_properties.cpp:12-49); writes q_v = c_v / a_v and
//           block partial sums of the six globals in FP64; a one-block
//           kernel sums the partials in a fixed order and writes the energy
//           and the penalty factors (kernel.h:19-122), so the result is
//           deterministic and needs no float atomics.
//   pass 2  per vertex v: the gather of mesh_properties.cpp:51-148 (spoke
//           edges, faces and rim edges of the ring, tether, repulsion) fused
//           with the combination of kernel.h:124-137; writes grad_v.
//
// Precision: T = double gives the FP64 path.  T = float gives the mixed path:
// edge vectors, face normals and the arguments of every angle are formed in
// FP64 (they cancel), the square roots, reciprocals, cotangents and dihedral
// angles (atan2) built from them run in FP32, and accumulation, the global
// reduction and the penalty factors stay FP64.
//
// Boundary vertices (ring with a faceless slot) take the OpenMesh-semantics
// walker in FP64 in both paths, which reproduces the reference's boundary
// branches of calc_sector_angle / calc_dihedral_angle.
#include <hip/hip_ext.h>
#include "tm_internal.h"
#include "tm_last.h"
#include "tm_om.h"
#include "tm_wave.h"

#include <algorithm>

namespace tmh {

// Vector arithmetic of the ring passes' slot terms with explicit fused
// multiply-adds.  The library is built without FP contraction, so these are
// the only fusions: the bits depend on the source alone, not on the kernel a
// function is inlined into (a single-mesh launch and a replica group give the
// same bits).  The neighbour-list distance tests do not use these: their
// rounding decides which pairs exist and stays unfused, like the reference's.
__device__ __forceinline__ d3 cross_f(const d3& a, const d3& b)
{
    return d3{fma(a.y, b.z, -(a.z * b.y)), fma(a.z, b.x, -(a.x * b.z)), fma(a.x, b.y, -(a.y * b.x))};
}
__device__ __forceinline__ double dot_f(const d3& a, const d3& b)
{
    return fma(a.x, b.x, fma(a.y, b.y, a.z * b.z));
}
__device__ __forceinline__ d3 axpy_f(double s, const d3& a, const d3& y)    // s a + y
{
    return d3{fma(s, a.x, y.x), fma(s, a.y, y.y), fma(s, a.z, y.z)};
}

// Scalar kernels of the two precision modes.  Geometry vectors (edge vectors,
// face normals and the inputs of every angle) are always FP64; T is the type
// of the square roots, reciprocals, cotangents and angles built from them.
template <class T>
struct Prec;
template <>
struct Prec<double> {
    __device__ static __forceinline__ double sqrt_(double a) { return sqrt(a); }
    __device__ static __forceinline__ double rcp(double a) { return 1.0 / a; }
    __device__ static __forceinline__ double dihedral(const d3& n0, const d3& n1, const d3& e, double)
    {
        // OpenMesh calc_dihedral_angle: acos of the normalised dot, signed
        double denom = sqrt(dot_f(n0, n0)) * sqrt(dot_f(n1, n1));
        if (denom == 0) return 0;
        return om_angle(dot_f(n0, n1) / denom, dot_f(cross_f(n0, n1), e));
    }
};
template <>
struct Prec<float> {
    __device__ static __forceinline__ float sqrt_(double a) { return sqrtf((float)a); }
    // the hardware reciprocal (1 ulp) instead of the correctly rounded division
    __device__ static __forceinline__ float rcp(float a) { return __builtin_amdgcn_rcpf(a); }
    __device__ static __forceinline__ float dihedral(const d3& n0, const d3& n1, const d3& e, float l)
    {
        // the same angle as atan2(|n0 x n1|, n0.n1), signed by (n0 x n1).e;
        // n0 x n1 is parallel to e, so (n0 x n1).e = |e| x the signed sine
        // term, and atan2 of (sine |e|, cosine |e|) is the angle.  Both
        // products are formed in FP64 (they cancel for small angles) and
        // rounded once.
        double s = dot_f(cross_f(n0, n1), e);
        double c = dot_f(n0, n1) * (double)l;
        return atan2f((float)s, (float)c);
    }
};

// The edge tether (mesh_tether.h:40-82) amplifies a length error near its
// walls: exp(l / (l - lc1)) and (l - lc0)^r make dV/V ~ l lc1 / (l - lc1)^2
// x dl/l, hundreds of times the rounding of an FP32 length at the
// configurations' bond widths.  So both precisions evaluate it from the FP64
// length; the potential is zero between the walls, so the FP64 root is only
// taken for edges outside them (l2: the FP64 squared length).
__device__ __forceinline__ bool tether_active(double l2, const EParams& p)
{
    return l2 > p.bond_lc0 * p.bond_lc0 || l2 < p.bond_lc1 * p.bond_lc1;
}
template <class T>
__device__ __forceinline__ double tether_value(double l2, T l, const EParams& p)
{
    if constexpr (sizeof(T) == sizeof(double)) return bond_edge_value((double)l, p);
    else return tether_active(l2, p) ? bond_edge_value(sqrt(l2), p) : 0.0;
}
template <class T>
__device__ __forceinline__ double tether_dfac(double l2, T l, const EParams& p)
{
    if constexpr (sizeof(T) == sizeof(double)) return bond_edge_dfac((double)l, p);
    else return tether_active(l2, p) ? bond_edge_dfac(sqrt(l2), p) : 0.0;
}

__device__ __forceinline__ d3 load_p(const double* __restrict__ x, int v)
{
    return d3{x[3 * v], x[3 * v + 1], x[3 * v + 2]};
}

// ------------------------------------------------------------ reduction ---
// Column k of block_sum6 alone, by the same operations in the same order (a
// butterfly within each wave, then the waves in order), so its bits are those
// block_sum6 gives that column; the result is valid in thread 0.
__device__ __forceinline__ double block_sum1(double a, double* s_red /* [nwaves] */)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (lane == 0) s_red[wave] = a;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < nw; w++) r += s_red[w];
    return r;
}

// Sum six per-thread doubles over the block; result valid in s_out[0..5].
__device__ __forceinline__ void block_sum6(double v[6], double* s_red /* [nwaves*6] */, double* s_out)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        double a = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
        v[k] = a;
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 6; k++) s_red[wave * 6 + k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        double a = 0;
        for (int w = 0; w < nw; w++) a += s_red[w * 6 + threadIdx.x];
        s_out[threadIdx.x] = a;
    }
    __syncthreads();
}

// The energy (kernel.h:110-122) and the penalty factors 2 kappa / ref (X / ref -
// 1) (kernel.h:27-71) of the six global sums.
__device__ __forceinline__ Globals globals_of_sums(const double v[6], const EParams& p)
{
    Globals g;
    const double A = v[0], V = v[1], C = v[2], B = v[3], T = v[4], R = v[5];
    for (int k = 0; k < 6; k++) g.props[k] = v[k];
    double e = 0.0, d;
    d = A / p.ref_area - 1.0;
    e += p.kappa_a * d * d;
    g.fac_a = 2.0 * p.kappa_a / p.ref_area * d;
    d = V / p.ref_volume - 1.0;
    e += p.kappa_v * d * d;
    g.fac_v = 2.0 * p.kappa_v / p.ref_volume * d;
    g.fac_v6 = g.fac_v / 6.0;
    d = C / p.ref_curvature - 1.0;
    e += p.kappa_c * d * d;
    g.fac_c = 2.0 * p.kappa_c / p.ref_curvature * d;
    e += p.kappa_t * T;
    e += p.kappa_r * R;
    e += p.kappa_b * B;
    g.energy = e;
    return g;
}

// The end of a properties pass, by the workgroup of 256 threads that finishes
// last: the six globals from the block partials (stored column by column,
// partials[k * nblocks + b]) in a fixed order that depends on nothing but the
// number of rows -- lane i of a wave adds rows i, i + 64, ... of its column,
// then a butterfly joins the 64 lanes -- so every launch gets the same bits.
// Waves 0 and 1 take two columns each, waves 2 and 3 one.  A chain of two
// loads and a few barriers, run by the pass itself up to kTailBlocks rows.
__device__ __forceinline__ void finalize_tail(const PassArgs& A)
{
    __shared__ double s_sum[6];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int streak = A.pc.x_snap ? get(A.pc.streak + 1) : 0;
    const bool two = wave < 2;
    const double* c0 = A.partials + (size_t)wave * A.nblocks;
    const double* c1 = A.partials + (size_t)(wave + 4) * A.nblocks;
    double v0 = 0.0, v1 = 0.0;
    constexpr int kBatch = 12;    // rows in flight per lane
    for (int b0 = lane; b0 < A.nblocks; b0 += 64 * kBatch) {
        double r0[kBatch], r1[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int b = b0 + 64 * u;
            r0[u] = b < A.nblocks ? get(c0 + b) : 0.0;
            r1[u] = two && b < A.nblocks ? get(c1 + b) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (b0 + 64 * u < A.nblocks) {
                v0 += r0[u];
                v1 += r1[u];
            }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v0 += __shfl_xor(v0, off, 64);
        v1 += __shfl_xor(v1, off, 64);
    }
    if (lane == 0) {
        s_sum[wave] = v0;
        if (two) s_sum[wave + 4] = v1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const Globals g = globals_of_sums(s_sum, A.p);
        *A.globals = g;
        if (A.host) *A.host = g;
        if (A.pc.dforce) *A.pc.dforce = 0;    // replica groups: the query of this evaluation recorded
        if (A.pc.x_snap) A.pc.streak[0] = streak;
    }
}

// ------------------------------------------------------- lane groups -----
// Each vertex is handled by a group of kGroup lanes: lane k of the group owns
// ring slot k (and k + kGroup, ... for valence above kGroup).  All loads of a
// vertex's ring are issued at once instead of as a chain of dependent
// round trips, and the group sums its per-slot terms with lane shuffles.
constexpr int kGroup = 8;
static_assert(kGroup == kRingPad, "exclusion tests read kGroup ring columns without the valence");
static_assert(kGroup == kPairLanes && kPairCap <= 15, "pair-cache counts are 4 bits per lane");

// Exclusion test of the cell list (cell_list.h:170-202) on the ring table:
// j is excluded at level 1 if it is in ring(v), and at level 2 also if ring(j)
// and ring(v) intersect (j is then a neighbour of a neighbour of v).
__device__ __forceinline__ bool ring_excluded(const MeshView& m, int v, int n, int j, int excl)
{
    if (j == v) return true;
    if (excl <= 0) return false;
    const int N = m.nv;
    for (int k = 0; k < n; k++)
        if (m.ring[k * N + v] == j) return true;
    if (excl == 1) return false;
    const int nj = meta_valence(m.meta[j]);
    for (int a = 0; a < nj; a++) {
        int w = m.ring[a * N + j];
        for (int k = 0; k < n; k++)
            if (m.ring[k * N + v] == w) return true;
    }
    return false;
}

// One vertex's ring held in registers for exclusion tests: slots beyond the
// valence hold -1.  Rings longer than kGroup fall back to ring_excluded.
struct RingRegs {
    int r[kGroup];
    int n;
};
__device__ __forceinline__ RingRegs load_ring(const MeshView& m, int v, int n)
{
    RingRegs R;
    R.n = n;
#pragma unroll
    for (int k = 0; k < kGroup; k++) R.r[k] = k < n ? m.ring[k * m.nv + v] : -1;
    return R;
}
__device__ __forceinline__ bool in_ring(const RingRegs& R, int j)
{
    bool hit = false;
#pragma unroll
    for (int k = 0; k < kGroup; k++) hit |= R.r[k] == j;
    return hit;
}
// Same answer as ring_excluded(m, v, n, j, excl) for n <= kGroup, with the
// ring of v in registers.  The first kGroup columns of the ring of j are
// read without its valence (unused columns hold -1); meta[j] and the
// columns beyond are read only when j has kGroup or more neighbours.
__device__ __forceinline__ bool excluded_fast(const MeshView& m, const RingRegs& R, int v, int j, int excl)
{
    if (j == v) return true;
    if (excl <= 0) return false;
    if (R.n > kGroup) return ring_excluded(m, v, R.n, j, excl);
    if (in_ring(R, j)) return true;
    if (excl == 1) return false;
    int w[kGroup];
#pragma unroll
    for (int a = 0; a < kGroup; a++) w[a] = m.ring[a * m.nv + j];
    bool hit = false;
#pragma unroll
    for (int a = 0; a < kGroup; a++) hit |= w[a] >= 0 && in_ring(R, w[a]);
    if (hit) return true;
    if (w[kGroup - 1] >= 0) {
        const int nj = meta_valence(m.meta[j]);
        for (int a = kGroup; a < nj; a++)
            if (in_ring(R, m.ring[a * m.nv + j])) return true;
    }
    return false;
}

// The neighbour query of point_distances (cell_list.h:133-219,
// verlet_list.h:76-101) shared by the lanes of a group: the candidates (the
// stored stencil list of the vertex's cell, the stencil rows of its current
// cell if it has moved to another cell, or its Verlet adjacency) are strided
// over the lanes.  f(j, d) sees the pairs of this lane; together the lanes
// see the reference's set exactly once.
template <int kBatch = 1, class F>
__device__ __forceinline__ void group_neighbours(const MeshView& m, const NListView& nl, int v, int n, d3 pi,
                                                 double dmax, int lane, F&& f)
{
    // list range and build-time cell of v: independent of the ring loads
    int2 vr = make_int2(0, 0);
    int vc = -1;
    if (nl.kind == 0 && nl.vcand) {
        vr = nl.vcand[v];
        vc = nl.vert_cell[v];
    }
    const double dmax2 = dmax * dmax * (1.0 + 1e-15);
    const RingRegs R = load_ring(m, v, n);
    auto test = [&](int j, d3 pj) {
        const d3 d = pi - pj;
        const double sq = sqnorm(d);
        if (sq <= dmax2 && sqrt(sq) < dmax) {
            if (nl.kind == 1 || !excluded_fast(m, R, v, j, nl.exclusion)) f(j, d);
        }
    };
    // kBatch candidates per lane and step: their ids, then their positions,
    // are all in flight before the first test
    auto scan = [&](const int* ids, int s, int e) {
        for (int q0 = s + lane; q0 < e; q0 += kBatch * kGroup) {
            int j[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int q = q0 + u * kGroup;
                j[u] = q < e ? ids[q] : -1;
            }
            d3 pj[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) pj[u] = load_p(m.x, j[u] >= 0 ? j[u] : v);
#pragma unroll
            for (int u = 0; u < kBatch; u++)
                if (j[u] >= 0) test(j[u], pj[u]);
        }
    };
    if (nl.kind == 0) {
        int c[3];
        cell_coords(nl, pi, c);
        // a vertex still in its build-time cell scans that cell's stored
        // stencil list: the same candidates as the 27-cell walk below
        const bool inside = c[0] >= 0 && c[0] < nl.shape[0] && c[1] >= 0 && c[1] < nl.shape[1] && c[2] >= 0 &&
                            c[2] < nl.shape[2];
        const int flat = c[0] * nl.strides[0] + c[1] * nl.strides[1] + c[2] * nl.strides[2];
        if (inside && flat == vc) {
            if (!nl.excl_mask) {
                scan(nl.cand, vr.x, vr.y);
                return;
            }
            // excluded candidates are skipped without a position load; the
            // rest need only the distance test (the first 128 of the list)
            const unsigned long long m0 = nl.excl_mask[2 * v], m1 = nl.excl_mask[2 * v + 1];
            for (int q0 = vr.x + lane; q0 < vr.y; q0 += kBatch * kGroup) {
                int j[kBatch];
                int ex[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; u++) {
                    const int q = q0 + u * kGroup;
                    const int i = q - vr.x;
                    ex[u] = i < 64 ? (int)((m0 >> i) & 1ull) : (i < 128 ? (int)((m1 >> (i - 64)) & 1ull) : -1);
                    j[u] = (q < vr.y && ex[u] != 1) ? nl.cand[q] : -1;
                }
                d3 pj[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; u++)
                    if (j[u] >= 0) pj[u] = load_p(m.x, j[u]);
#pragma unroll
                for (int u = 0; u < kBatch; u++) {
                    if (j[u] < 0) continue;
                    if (ex[u] < 0) {
                        test(j[u], pj[u]);
                        continue;
                    }
                    const d3 d = pi - pj[u];
                    const double sq = sqnorm(d);
                    if (sq <= dmax2 && sqrt(sq) < dmax) f(j[u], d);
                }
            }
            return;
        }
        // moved vertex: the stored list of its current cell when that cell was
        // occupied at the build (the same candidates as its 9 stencil rows,
        // in the same order), else the 9 rows of x-consecutive cells of its
        // stencil, each strided over the lanes
        if (inside && nl.cand_start) {
            const int s0 = nl.cell_start[flat];
            if (nl.cell_start[flat + 1] > s0) {
                scan(nl.cand, nl.cand_start[s0], nl.cand_start[s0 + 1]);
                return;
            }
        }
        const int i0 = max(c[0] - 1, 0), i1 = min(c[0] + 1, nl.shape[0] - 1);
        if (i0 > i1) return;
        for (int r = 0; r < 9; r++) {
            const int kk = c[2] + r / 3 - 1, jj = c[1] + r % 3 - 1;
            if (kk < 0 || kk >= nl.shape[2] || jj < 0 || jj >= nl.shape[1]) continue;
            const int base = jj * nl.strides[1] + kk * nl.strides[2];
            scan(nl.cell_verts, nl.cell_start[base + i0], nl.cell_start[base + i1 + 1]);
        }
    } else if (nl.kind == 1) {
        scan(nl.adj, nl.adj_start[v], nl.adj_start[v + 1]);
    }
}

// ---------------------------------------------------- repulsion terms ---
// One lane's running repulsion terms over the pairs it visits: the property
// sum(rep(l)) (mesh_repulsion.h:28-54), the pair count and the gradient at
// v, 2 kappa_r sum(dfac(l) d) (mesh_repulsion.h:56-79, doubled as in
// mesh_properties.cpp:138-146).  The query kernels sum them over the lanes
// with group_sum; pass 2 adds the gradient of the vertices with pairs.
struct RepTerms {
    double rep = 0.0;
    d3 g{0.0, 0.0, 0.0};
    int cnt = 0;
    __device__ __forceinline__ void add(d3 d, const EParams& p)
    {
        const double l = norm(d);
        rep += rep_value(l, p.rep_lc1, p.rep_r);
        g += (p.kappa_r * 2.0 * rep_dfac(l, p.rep_lc1, p.rep_r)) * d;
        cnt++;
    }
    __device__ __forceinline__ void group_reduce()
    {
        rep = group_sum(rep);
        g.x = group_sum(g.x);
        g.y = group_sum(g.y);
        g.z = group_sum(g.z);
        cnt = group_sum(cnt);
    }
};
// the gradient row of a vertex with pairs (pass 2 reads it only then)
__device__ __forceinline__ void store_rep_g(const PassArgs& A, int v, const RepTerms& t)
{
    if (A.rep_g && t.cnt > 0) {
        A.rep_g[3 * v] = t.g.x;
        A.rep_g[3 * v + 1] = t.g.y;
        A.rep_g[3 * v + 2] = t.g.z;
    }
}

// ------------------------------------------------------------ pair cache ---
// (PairCache in tm_internal.h.)  The cell of position pi, as an id that no other
// cell has: the flat id inside the grid, -2 and below outside it, where a
// sphere's outermost vertices move and their stencils still reach into the
// grid.  (-1, no replay, only where the ids would not fit.)  While those
// vertices had no cell and took the full query on every evaluation, the launch
// waited for them: the same positions, 0.5% of an edge from those of the list,
// evaluated again and again took 31.8 us at 642 vertices, now 27.6; 36.5 and 32.7
// at 40962, 51.2 and 45.6 at 163842.
__device__ __forceinline__ int query_cell(const NListView& nl, d3 pi)
{
    int c[3];
    cell_coords(nl, pi, c);
    const bool inside = c[0] >= 0 && c[0] < nl.shape[0] && c[1] >= 0 && c[1] < nl.shape[1] && c[2] >= 0 &&
                        c[2] < nl.shape[2];
    if (inside) return c[0] * nl.strides[0] + c[1] * nl.strides[1] + c[2] * nl.strides[2];
    const long long w0 = nl.shape[0] + 4, w1 = nl.shape[1] + 4;    // cell_coords: -2 .. shape + 1
    const long long id = c[0] + 2 + w0 * (c[1] + 2 + w1 * (c[2] + 2));
    return id < 0x7fffff00ll ? -2 - (int)id : -1;
}

// Build-time cells of the fast vertices, in LDS.
struct FastCells {
    int n;
    int4 c[kFastMax];
};

// Block-uniform: 2 to record (forced, or too many vertices are fast or for too
// long), 1 to replay; F (F.n 0 on entry) then holds the fast vertices' cells.
// Contains a barrier.
__device__ __forceinline__ int pair_cache_mode(const PairCache& pc, const NListView& nl, FastCells& F)
{
    __shared__ int s_mode;
    if (pc.force || (pc.dforce && *pc.dforce)) {
        __syncthreads();
        return 2;
    }
    if (threadIdx.x < 64) {
        // one partial per pass-1 block: each lane has a batch of loads in
        // flight before it compares them, instead of one round trip per partial
        constexpr int kBatchLoads = 16;
        bool some = false, over = false;
        for (int i0 = threadIdx.x; i0 < pc.disp_n; i0 += 64 * kBatchLoads) {
            double d[kBatchLoads];
#pragma unroll
            for (int u = 0; u < kBatchLoads; u++) {
                const int i = i0 + 64 * u;
                d[u] = i < pc.disp_n ? pc.disp_part[i] : 0.0;
            }
            bool any = false;
#pragma unroll
            for (int u = 0; u < kBatchLoads; u++) any |= !(d[u] < pc.limit2);
            if (__builtin_expect(!__any(any), 1)) continue;
            some = true;
            unsigned hit = 0;
#pragma unroll
            for (int u = 0; u < kBatchLoads; u++) hit |= (d[u] < pc.limit2 ? 0u : 1u) << u;
            while (hit) {
                const int i = i0 + 64 * (__ffs(hit) - 1);
                hit &= hit - 1u;
                const int* f = pc.fast + (size_t)kFastRow * i;
                const int n = f[0];
                const int at = n > kFastSeg ? kFastMax : atomicAdd(&F.n, n);
                if (at + n > kFastMax) {
                    over = true;
                    break;
                }
                for (int k = 0; k < n; k++) {
                    const int id = f[1 + k], r = id % nl.strides[2];
                    F.c[at + k] = make_int4(r % nl.strides[1], r / nl.strides[1], id / nl.strides[2], 0);
                }
            }
        }
        int mode = 1;
        if (__builtin_expect(some, 0)) mode = __any(over) || pc.streak[0] >= kPatience ? 2 : 1;
        if (threadIdx.x == 0) s_mode = mode;
    }
    __syncthreads();
    return s_mode;
}

// Whether vertex v, recorded at pi in cell c, has a non-excluded candidate within
// `radius` in the stencil of another cell that it reaches while it is slow (the
// cells of pi -+ kPairLimit skin), by its lane group.
__device__ __forceinline__ bool candidate_around(const MeshView& m, const NListView& nl, const PairCache& pc, int v,
                                                 int n, d3 pi, double radius, int lane)
{
    const double reach = kPairLimit * pc.skin * (1.0 + 1e-12);
    int c[3], lo[3], hi[3];
    cell_coords(nl, pi, c);
    cell_coords(nl, d3{pi.x - reach, pi.y - reach, pi.z - reach}, lo);
    cell_coords(nl, d3{pi.x + reach, pi.y + reach, pi.z + reach}, hi);
    if (lo[0] == hi[0] && lo[1] == hi[1] && lo[2] == hi[2]) return false;
    const RingRegs R = load_ring(m, v, n);
    const double r2 = radius * radius * (1.0 + 1e-15);
    const int ny = hi[1] - lo[1] + 3, nz = hi[2] - lo[2] + 3;
    int found = 0;
    for (int i = lane; i < ny * nz && !found; i += kGroup) {
        const int y = lo[1] - 1 + i % ny, z = lo[2] - 1 + i / ny;
        if (y < 0 || y >= nl.shape[1] || z < 0 || z >= nl.shape[2]) continue;
        const int base = y * nl.strides[1] + z * nl.strides[2];
        const bool own = abs(y - c[1]) <= 1 && abs(z - c[2]) <= 1;    // its middle cells were searched
        for (int side = 0; side < (own ? 2 : 1); side++) {
            const int x0 = max(own && side == 1 ? c[0] + 2 : lo[0] - 1, 0);
            const int x1 = min(own && side == 0 ? c[0] - 2 : hi[0] + 1, nl.shape[0] - 1);
            if (x0 > x1) continue;
            const int end = nl.cell_start[base + x1 + 1];
            for (int q = nl.cell_start[base + x0]; q < end; q++) {
                const int j = nl.cell_verts[q];
                const d3 d = pi - load_p(m.x, j);
                const double sq = sqnorm(d);
                if (!(sq > r2) && !excluded_fast(m, R, v, j, nl.exclusion)) found = 1;
            }
        }
    }
    return group_sum(found) > 0;
}

// The full query with radius dmax + skin, keeping each lane's non-excluded
// candidates in its visit order; f sees the pairs within dmax, in the order
// and with the test of the plain query.  Lane 0 stores the counts and the
// cell the lists are valid in (-1 when a lane overflows).  kAround: look for
// candidates that the vertex may reach too (pi is the snapshot's position).
template <int kBatch, bool kAround = false, class F>
__device__ __forceinline__ void record_neighbours(const MeshView& m, const NListView& nl, const PairCache& pc, int v,
                                                  int n, d3 pi, double dmax, int lane, F&& f)
{
    int* e = pc.ent + ((size_t)v * kGroup + lane) * kPairCap;
    const double dmax2 = dmax * dmax * (1.0 + 1e-15);
    int rec = 0;
    group_neighbours<kBatch>(m, nl, v, n, pi, dmax + pc.skin, lane, [&](int j, d3 d) {
        if (rec < kPairCap) e[rec] = j;
        rec++;
        const double sq = sqnorm(d);
        if (sq <= dmax2 && sqrt(sq) < dmax) f(j, d);
    });
    const int over = group_sum(rec > kPairCap ? 1 : 0);
    unsigned word = (unsigned)group_sum(min(rec, kPairCap) << (4 * lane));
    const int cell = query_cell(nl, pi);
    if (kAround && word == 0u && !candidate_around(m, nl, pc, v, n, pi, dmax + pc.skin, lane)) word = kEmptyAround;
    if (lane == 0) {
        pc.cnt[v] = word;
        pc.cell[v] = over == 0 ? cell : -1;
    }
}

// Exclusion masks of the stored stencil lists: bit i of vertex v is set if
// the i-th candidate of the list of v's build-time cell is excluded from v
// (excluded_fast, which depends on the ring tables only).  8-lane groups,
// lane l takes candidates l, l + 8, ...; the group ORs its words.
// The group first gathers v's excluded set, v, its ring and (exclusion 2)
// the rings of its ring vertices, into an LDS hash set (open addressing,
// linear probing, -1 empty), one ring vertex per lane; each candidate then
// costs a probe or two instead of reading its own ring.  Membership is exact
// (adjacency is symmetric, so this is the set excluded_fast tests).  A ring
// above kGroup, or a set above kMaskSetMax entries, takes excluded_fast.
constexpr int kMaskTab = 128;
constexpr int kMaskSetMax = 96;

__device__ __forceinline__ unsigned mask_hash(int j)
{
    return ((unsigned)j * 2654435761u) >> 25;    // 7 bits: kMaskTab == 128
}

__device__ __forceinline__ bool mask_insert(int* tab, int* cnt, int j)
{
    const unsigned h = mask_hash(j);
    for (int q = 0; q < kMaskTab; q++) {
        const int at = (h + q) & (kMaskTab - 1);
        const int old = atomicCAS(&tab[at], -1, j);
        if (old == -1) return atomicAdd(cnt, 1) < kMaskSetMax;
        if (old == j) return true;
    }
    return false;
}

// a set of at most kMaskSetMax entries: the probe ends at j or at an empty slot
__device__ __forceinline__ bool mask_member(const int* tab, int j)
{
    const unsigned h = mask_hash(j);
    for (int q = 0; q < kMaskTab; q++) {
        const int x = tab[(h + q) & (kMaskTab - 1)];
        if (x == j) return true;
        if (x < 0) return false;
    }
    return false;
}

__device__ __forceinline__ void excl_mask_body(const MeshView& m, const NListView& nl,
                                               unsigned long long* __restrict__ mask, int lb)
{
    constexpr int kGroups = 256 / kGroup;
    __shared__ int s_tab[kGroups][kMaskTab];
    __shared__ int s_cnt[kGroups];
    __shared__ int s_ovf[kGroups];
    const int t = lb * 256 + threadIdx.x;
    const int gi = threadIdx.x / kGroup;
    const int v = t / kGroup, lane = t % kGroup;
    const bool active = v < m.nv;
    const int excl = nl.exclusion;
    for (int i = lane; i < kMaskTab; i += kGroup) s_tab[gi][i] = -1;
    if (lane == 0) {
        s_cnt[gi] = 0;
        s_ovf[gi] = 0;
    }
    int n = 0;
    RingRegs R;
    R.n = 0;
    if (active) {
        n = meta_valence(m.meta[v]);
        R = load_ring(m, v, n);
    }
    const bool use_set = active && excl >= 1 && n <= kGroup;
    __syncthreads();
    if (use_set) {
        bool ok = lane != 0 || mask_insert(s_tab[gi], &s_cnt[gi], v);
        int w = -1;
#pragma unroll
        for (int k = 0; k < kGroup; k++)
            if (k == lane) w = R.r[k];
        if (w >= 0) {
            ok = mask_insert(s_tab[gi], &s_cnt[gi], w) && ok;
            if (excl > 1) {
                const int N = m.nv;
                int c[kGroup];
#pragma unroll
                for (int a = 0; a < kGroup; a++) c[a] = m.ring[a * N + w];
#pragma unroll
                for (int a = 0; a < kGroup; a++)
                    if (c[a] >= 0) ok = mask_insert(s_tab[gi], &s_cnt[gi], c[a]) && ok;
                if (c[kGroup - 1] >= 0) {
                    const int nw = meta_valence(m.meta[w]);
                    for (int a = kGroup; a < nw; a++) ok = mask_insert(s_tab[gi], &s_cnt[gi], m.ring[a * N + w]) && ok;
                }
            }
        }
        if (!ok) s_ovf[gi] = 1;
    }
    __syncthreads();
    unsigned long long w0 = 0ull, w1 = 0ull;
    if (active) {
        const bool set = use_set && !s_ovf[gi];
        const int2 vr = nl.vcand[v];
        const int cnt = min(vr.y - vr.x, 128);
        for (int i = lane; i < cnt; i += kGroup) {
            const int j = nl.cand[vr.x + i];
            if (set ? mask_member(s_tab[gi], j) : excluded_fast(m, R, v, j, excl)) {
                if (i < 64) w0 |= 1ull << i;
                else w1 |= 1ull << (i - 64);
            }
        }
    }
#pragma unroll
    for (int o = 1; o < kGroup; o <<= 1) {
        w0 |= __shfl_xor(w0, o, 64);
        w1 |= __shfl_xor(w1, o, 64);
    }
    if (active && lane == 0) {
        mask[2 * v] = w0;
        mask[2 * v + 1] = w1;
    }
}

__global__ void __launch_bounds__(256) k_excl_mask(MeshView m, NListView nl, unsigned long long* __restrict__ mask)
{
    excl_mask_body(m, nl, mask, logical_block());
}
__global__ void __launch_bounds__(256) k_excl_mask_grouped(const NlistBuild* __restrict__ b,
                                                           const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    if (lb >= block0[R]) return;
    const int r = find_replica(block0, R, lb);
    excl_mask_body(b[r].m, b[r].nl, b[r].mask, lb - block0[r]);
}

void launch_excl_mask(const MeshView& m, const NListView& nl, unsigned long long* mask, hipStream_t s)
{
    if (m.nv <= 0) return;
    hipLaunchKernelGGL(k_excl_mask, dim3(tuned_blocks(m.nv, 256)), dim3(256), 0, s, m, nl, mask);
}

void launch_nlist_masks(const NlistGroup& g, hipStream_t s)
{
    if (g.total[kShapeMask] <= 0) return;
    if (g.R == 1) launch_excl_mask(g.h[0].m, g.h[0].nl, g.h[0].mask, s);
    else
        hipLaunchKernelGGL(k_excl_mask_grouped, dim3((g.total[kShapeMask] + kXcds - 1) / kXcds * kXcds), dim3(256), 0, s, g.d,
                           g.block0 + kShapeMask * (g.R + 1), g.R);
}

// --------------------------------------------------------------- pass 1 ---
// Ring slot k of an interior vertex v: halfedge v -> j_k, its face
// F_k = (v, j_k, j_{k-1}) and the twin face (j_k, v, j_{k+1}) = F_{k+1}.
// With e_k = x_{j_k} - x_v, the OpenMesh sector normal of v -> j_k is
// n_k = e_k x e_{k-1} (|n_k| = 2 area(F_k)) and that of j_k -> v is n_{k+1}.
// One slot contributes area(F_k), vol(F_k) = x_v . n_k / 6, l_k theta_k / 2
// and the tether term of halfedge v -> j_k (mesh_properties.cpp:19-33).
// Slot k's terms from its spoke e_k = x_{j_k} - x_v and the sector normals
// n_k = e_k x e_{k-1} and n_{k+1}.
template <class T>
__device__ __forceinline__ T slot_properties_at(const EParams& p, d3 xv, d3 e_cur, d3 n_cur, d3 n_next,
                                                double& area, double& vol, double& curv, double& teth)
{
    T af = Prec<T>::sqrt_(dot_f(n_cur, n_cur)) * (T)0.5;
    const double l2 = dot_f(e_cur, e_cur);
    T l = Prec<T>::sqrt_(l2);
    T th = Prec<T>::dihedral(n_cur, n_next, e_cur, l);
    curv += (double)((T)0.5 * l * th);
    area += (double)af;
    vol += dot_f(xv, n_cur);    // 6 x the signed volume x_v . (x_j x x_k) / 6 (mesh_util.h:94-101)
    if (p.bond_type == 0) teth += tether_value<T>(l2, l, p);
    else teth += bond_area_value((double)af, p);
    return th;
}

// One lane per vertex.  Lane v walks the clockwise ring of v once, carrying
// the spoke e_k and the sector normal n_k from one slot to the next, so every
// normal of the ring is formed once, and the per-vertex work (the sums, the
// bending ratio, the stores) runs once per vertex instead of once per lane of
// a lane group.  Column k of the ring table holds the k-th neighbours of all
// vertices, so each slot's load is coalesced across the wave; columns below
// kRingPad hold -1 past the valence, so a ring of at most kRingPad slots is
// loaded in full before its valence is known, and its position loads issue
// together.  Longer rings walk the table slot by slot.
// use: v is an interior vertex (its sums are wanted).  The leading kRingPad
// columns and their positions are loaded whether or not they are used, so
// they need not wait for the meta word that decides it.  theta (optional):
// the dihedral angle of each slot of a ring of at most kRingPad slots is
// stored at theta[k * N + v] for pass 2, which then need not form it again.
template <class T>
__device__ __forceinline__ void ring_properties(const MeshView& m, const EParams& p, int v, bool use, int n, d3 xv,
                                                double& area, double& vol, double& curv, double& teth,
                                                T* __restrict__ theta)
{
    const int N = m.nv;
    d3 e[kRingPad];
#pragma unroll
    for (int k = 0; k < kRingPad; k++) {
        const int j = m.ring[k * N + v];
        e[k] = load_p(m.x, j >= 0 ? j : v) - xv;    // past the valence: x_v, never used
    }
    if (!use) return;
    if (n <= kRingPad) {
        d3 e_last = e[kRingPad - 1];
#pragma unroll
        for (int k = kRingPad - 2; k >= 2; k--)
            if (k == n - 1) e_last = e[k];
        d3 n_cur = cross_f(e[0], e_last);
#pragma unroll
        for (int k = 0; k < kRingPad; k++) {
            if (k < n) {
                const d3 e_next = k + 1 < n ? e[(k + 1) % kRingPad] : e[0];
                const d3 n_next = cross_f(e_next, e[k]);
                const T th = slot_properties_at<T>(p, xv, e[k], n_cur, n_next, area, vol, curv, teth);
                if (theta) theta[k * N + v] = th;
                n_cur = n_next;
            }
        }
        return;
    }
    const d3 e_first = load_p(m.x, m.ring[v]) - xv;
    d3 e_cur = e_first;
    d3 n_cur = cross_f(e_first, load_p(m.x, m.ring[(n - 1) * N + v]) - xv);
    for (int k = 0; k < n; k++) {
        const d3 e_next = k + 1 < n ? load_p(m.x, m.ring[(k + 1) * N + v]) - xv : e_first;
        const d3 n_next = cross_f(e_next, e_cur);
        slot_properties_at<T>(p, xv, e_cur, n_cur, n_next, area, vol, curv, teth);
        e_cur = e_next;
        n_cur = n_next;
    }
}

__device__ __forceinline__ bool is_generic(int meta)
{
    return meta_bslot(meta) >= 0 || meta_valence(meta) < 3;
}


// Pass 1 over the kPass1Verts vertices of block lb; vertices on the boundary
// (or with fewer than three neighbours) read the properties that
// k_generic_props wrote.  Writes q_v, optionally the per-vertex properties,
// and the block's partial sums of the six globals (FP64, block_sum6's fixed
// butterfly order, so the result does not depend on timing).
//
// The repulsion property (column 5) comes from the query kernel.  Without
// the pair cache that kernel runs first and this one reads rep_v.  With it
// (kApart) the cached query runs after this kernel and sums column 5 of
// the same 256-vertex blocks itself, in the same order; this kernel then
// measures how far every vertex has moved since the cache's recording (the
// largest squared displacement of the block, NaN counting as infinite) and
// lists the cells of the fast ones, the query's replay condition.  kFinal: nothing of the pass follows, and the last
// workgroup sums the partials (finalize_tail).
template <class T, bool kApart = false, bool kFinal = !kApart>
__device__ __forceinline__ void pass1_body(const PassArgs& A, int lb)
{
    const MeshView& m = A.m;
    const EParams& p = A.p;
    __shared__ double s_red[(kPass1Verts / 64) * 6];
    const int v = lb * kPass1Verts + threadIdx.x;
    const bool active = v < m.nv;
    const int vc = active ? v : m.nv - 1;    // lanes past the last vertex load a valid one
    const int meta = m.meta[vc];
    const double rv = (!kApart && A.rep_v && active) ? A.rep_v[v] : 0.0;
    double disp = 0.0, own = 0.0;
    if (kApart && A.pc.x_snap && active) {
        const double* xs = A.pc.x_snap;
        const double dx = m.x[3 * v] - xs[3 * v], dy = m.x[3 * v + 1] - xs[3 * v + 1];
        const double dz = m.x[3 * v + 2] - xs[3 * v + 2];
        disp = dx * dx + dy * dy + dz * dz;
        if (!(disp == disp)) disp = INFINITY;
        own = disp;
    }
    const int n = meta_valence(meta);
    const bool ring = active && !is_generic(meta);
    double pr[6] = {0, 0, 0, 0, 0, 0};
    double area = 0, vol = 0, curv = 0, teth = 0;
    ring_properties<T>(m, p, vc, ring, n, load_p(m.x, vc), area, vol, curv, teth, (T*)A.theta);
    if (ring) {
        // a third of the face areas and volumes, half the edge terms (by
        // the rounded reciprocals: at most the last bit differs from a
        // division, far inside the parity tolerance)
        const double a = area * (1.0 / 3.0), c = curv * 0.5;
        const double q = c / a;    // curvature / area
        pr[0] = a;
        pr[1] = vol * (1.0 / 18.0);
        pr[2] = c;
        pr[3] = 2 * c * q;
        pr[4] = p.bond_type == 0 ? teth * 0.5 : teth * (1.0 / 3.0);
        pr[5] = rv;
        A.q[v] = q;
    } else if (active) {
        for (int k = 0; k < 6; k++) pr[k] = A.gprops[6 * v + k];
        A.q[v] = pr[2] / pr[0];
    }
    if (A.vprops && active)
        for (int k = 0; k < (kApart ? 5 : 6); k++) A.vprops[6 * v + k] = pr[k];
    // the block's partial sums by block_sum6's tree (the cached query sums
    // column 5 of the same vertices by that tree) and, with the cache, its
    // largest displacement, in one round through LDS
    constexpr int kWaves = kPass1Verts / 64;
    static_assert(kWaves == 4, "the displacement maximum below reads four waves");
    __shared__ double s_disp[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        double a = pr[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
        if (lane == 0) s_red[wave * 6 + k] = a;
    }
    if (kApart && A.pc.x_snap) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) disp = fmax(disp, __shfl_xor(disp, off, 64));
        if (lane == 0) s_disp[wave] = disp;
    }
    __syncthreads();
    if (threadIdx.x < (kApart ? 5 : 6)) {
        double a = 0;
        for (int w = 0; w < kWaves; w++) a += s_red[w * 6 + threadIdx.x];
        put(A.partials + (size_t)threadIdx.x * A.nblocks + lb, a);
    }
    if (kApart && A.pc.x_snap) {
        const double mx = fmax(fmax(s_disp[0], s_disp[1]), fmax(s_disp[2], s_disp[3]));
        if (threadIdx.x == 63) A.pc.disp_part[lb] = mx;
        if (!(mx < A.pc.limit2)) {
            __shared__ int s_fast;
            if (threadIdx.x == 0) s_fast = 0;
            __syncthreads();
            int* row = A.pc.fast + (size_t)kFastRow * lb;
            if (active && !(own < A.pc.limit2)) {
                const int i = atomicAdd(&s_fast, 1);
                if (i < kFastSeg) row[1 + i] = A.nl.vert_cell[v];
            }
            __syncthreads();
            if (threadIdx.x == 0) row[0] = s_fast;
        }
    }
    if constexpr (kFinal)
        if (A.tail && last_block_of_many(A.count, lb, A.nblocks)) finalize_tail(A);
}

template <class T>
__global__ void __launch_bounds__(kPass1Verts) k_pass1(PassArgs A)
{
    pass1_body<T>(A, logical_block());
}

// pass 1 before the cached repulsion query (column 5 left to it)
template <class T>
__global__ void __launch_bounds__(kPass1Verts) k_pass1_apart(PassArgs A)
{
    pass1_body<T, true>(A, logical_block());
}

template <class T>
__global__ void __launch_bounds__(kPass1Verts) k_pass1_grouped(const PassArgs* __restrict__ A,
                                                               const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    const int r = find_replica(block0, R, lb);
    pass1_body<T>(A[r], lb - block0[r]);
}

// replica groups with the cached query: every replica with repulsion leaves
// column 5 to it, and every replica its globals
template <class T>
__global__ void __launch_bounds__(kPass1Verts) k_pass1_apart_grouped(const PassArgs* __restrict__ A,
                                                                     const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    const int r = find_replica(block0, R, lb);
    if (A[r].rep_v) pass1_body<T, true>(A[r], lb - block0[r]);
    else pass1_body<T, false, false>(A[r], lb - block0[r]);
}

// Repulsion property of every ring vertex (mesh_repulsion.h:28-54):
// rep_v[v] = sum of rep(|x_v - x_j|) over the neighbours j of v within lc1,
// pair_cnt[v] = their number (0 for listed boundary vertices, whose
// properties k_generic_props computes).  A kernel of its own: the query is a
// chain of dependent loads (cell, candidate id, position, ring of the
// candidate) and needs few registers, so it runs apart from the
// register-heavy ring work of pass 1.
template <int kThreads, int kBatch>
__device__ __forceinline__ void rep_body(const PassArgs& A, int lb)
{
    if (!A.rep_v) return;
    const MeshView& m = A.m;
    const EParams& p = A.p;
    __shared__ double s_rep[kThreads / kGroup];
    __shared__ int s_cnt[kThreads / kGroup];
    const int t = lb * kThreads + threadIdx.x;
    const int v = t / kGroup, lane = t % kGroup;
    const bool active = v < m.nv;
    const int meta = active ? m.meta[v] : 0;
    const bool ring = active && !is_generic(meta);
    RepTerms tr;
    if (ring) {
        const d3 xv = load_p(m.x, v);
        group_neighbours<kBatch>(m, A.nl, v, meta_valence(meta), xv, p.rep_lc1, lane,
                                 [&](int, d3 d) { tr.add(d, p); });
    }
    tr.group_reduce();
    const double rep = tr.rep;
    if (lane == 0) {
        s_rep[threadIdx.x / kGroup] = rep;
        s_cnt[threadIdx.x / kGroup] = tr.cnt;
        if (ring) store_rep_g(A, v, tr);
    }
    __syncthreads();
    const int v0 = (lb * kThreads) / kGroup;
    const int i = threadIdx.x;
    if (i < kThreads / kGroup && v0 + i < m.nv) {
        A.rep_v[v0 + i] = s_rep[i];
        A.pair_cnt[v0 + i] = s_cnt[i];
    }
}

template <int kThreads, int kBatch>
__global__ void __launch_bounds__(kThreads) k_rep(PassArgs A)
{
    rep_body<kThreads, kBatch>(A, logical_block());
}

// The repulsion query with the pair cache (PairCache), kVertsPerBlock
// vertices per block of 256 threads.  Phase 1, one thread per vertex: a vertex
// whose lists may be replayed is done if nothing was recorded, else goes to a
// block-local list; the other ring vertices (all of them in a recording launch)
// go to a second one.  Phase 2: the block's 32 lane groups replay the first list,
// lane l the pairs that lane l of the query recorded, in their order, and
// group_sum over the lanes, which gives the bits of the 8-lane query.  A chain of
// two loads per vertex, its entries as one vector, two vertices of a group in
// flight.
// Phase 3: the lane groups run the full query (recording when the mode says so)
// over the second list.  Replays are the common case and want few,
// full blocks; a recording launch the device decides on (some vertex moved
// too far) is slower than k_rep, as each group takes 8 vertices in turn.
// Without cache buffers (a replica with a Verlet list in a cached group
// launch) every ring vertex takes phase 2 without recording (mode 0).
constexpr int kVertsPerBlock = kCachedVerts;
constexpr int kWaveVerts = 16;

// record_neighbours by one 64-lane wave instead of an 8-lane group, with
// the same result bits.  The candidates are laid out as group_neighbours
// walks them: runs (one range of the vertex's stored stencil list, with the
// exclusion masks when it is in its build-time cell; the stored list of the
// occupied cell it moved to; or the nine stencil rows of cell_verts), lane l
// of the group visiting indices l, l + 8, ... of each run in turn.  Lane L of
// the wave tests candidate L, L + 64, ... of the concatenated runs and
// computes its terms; then, in candidate order, the lanes whose candidate is
// within lc1 + skin pass it (lane shuffles) to lane (index in its run) % 8,
// which records and adds it as RepTerms::add would.  Lanes 0-7 end with the
// group's lane state; the caller reduces them with group_sum.
__device__ __forceinline__ void wide_record(const MeshView& m, const NListView& nl, const PairCache& pc,
                                            const EParams& p, int u, int n, d3 pu, bool keep, RepTerms& tr)
{
    const int L = threadIdx.x & 63;
    int rs[9], rl[9];
#pragma unroll
    for (int k = 0; k < 9; k++) rs[k] = rl[k] = 0;
    const int* ids = nl.cand;
    bool masked = false;
    unsigned long long m0 = 0ull, m1 = 0ull;
    {
        int2 vr = make_int2(0, 0);
        int vc = -1;
        if (nl.vcand) {
            vr = nl.vcand[u];
            vc = nl.vert_cell[u];
        }
        int c[3];
        cell_coords(nl, pu, c);
        const bool inside = c[0] >= 0 && c[0] < nl.shape[0] && c[1] >= 0 && c[1] < nl.shape[1] && c[2] >= 0 &&
                            c[2] < nl.shape[2];
        const int flat = c[0] * nl.strides[0] + c[1] * nl.strides[1] + c[2] * nl.strides[2];
        bool done = false;
        if (inside && flat == vc) {
            rs[0] = vr.x;
            rl[0] = vr.y - vr.x;
            if (nl.excl_mask) {
                masked = true;
                m0 = nl.excl_mask[2 * u];
                m1 = nl.excl_mask[2 * u + 1];
            }
            done = true;
        } else if (inside && nl.cand_start) {
            const int s0 = nl.cell_start[flat];
            if (nl.cell_start[flat + 1] > s0) {
                rs[0] = nl.cand_start[s0];
                rl[0] = nl.cand_start[s0 + 1] - rs[0];
                done = true;
            }
        }
        if (!done) {
            ids = nl.cell_verts;
            const int i0 = max(c[0] - 1, 0), i1 = min(c[0] + 1, nl.shape[0] - 1);
#pragma unroll
            for (int r = 0; r < 9; r++) {
                const int kk = c[2] + r / 3 - 1, jj = c[1] + r % 3 - 1;
                if (i0 <= i1 && kk >= 0 && kk < nl.shape[2] && jj >= 0 && jj < nl.shape[1]) {
                    const int base = jj * nl.strides[1] + kk * nl.strides[2];
                    rs[r] = nl.cell_start[base + i0];
                    rl[r] = nl.cell_start[base + i1 + 1] - rs[r];
                }
            }
        }
    }
    int total = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) total += rl[k];
    const RingRegs R = load_ring(m, u, n);
    const double dsk = keep ? p.rep_lc1 + pc.skin : p.rep_lc1, dsk2 = dsk * dsk * (1.0 + 1e-15);
    const double dmax = p.rep_lc1, dmax2 = dmax * dmax * (1.0 + 1e-15);
    int* ent = pc.ent + ((size_t)u * kGroup + (L & 7)) * kPairCap;
    int rec = 0;
    for (int t0 = 0; t0 < total; t0 += 64) {
        const int t = t0 + L;
        int j = -1, flag = 0, owner = 0;
        double val = 0.0;
        d3 gv{0.0, 0.0, 0.0};
        if (t < total) {
            // run and index of candidate t
            int i = t, q = -1;
#pragma unroll
            for (int k = 0; k < 9; k++) {
                if (q < 0 && i < rl[k]) q = rs[k] + i;
                if (q < 0) i -= rl[k];
            }
            owner = i & 7;
            // the masks cover the first 128 of the stored list: 1 excluded,
            // 0 not (no ring test needed), -1 beyond (ring test)
            const int ex = masked ? (i < 64 ? (int)((m0 >> i) & 1ull) : (i < 128 ? (int)((m1 >> (i - 64)) & 1ull) : -1))
                                  : -1;
            if (ex != 1) {
                j = ids[q];
                const d3 d = pu - load_p(m.x, j);
                const double sq = sqnorm(d);
                if (sq <= dsk2 && sqrt(sq) < dsk && (ex == 0 || !excluded_fast(m, R, u, j, nl.exclusion))) {
                    flag = 1;
                    if (sq <= dmax2 && sqrt(sq) < dmax) {
                        const double len = norm(d);
                        val = rep_value(len, p.rep_lc1, p.rep_r);
                        gv = (p.kappa_r * 2.0 * rep_dfac(len, p.rep_lc1, p.rep_r)) * d;
                        flag = 3;
                    }
                }
            }
        }
        unsigned long long bits = __ballot(flag != 0);
        while (bits) {
            const int src = __ffsll((long long)bits) - 1;
            bits &= bits - 1ull;
            const int fo = __shfl(owner, src), ff = __shfl(flag, src), fj = __shfl(j, src);
            const double fv = __shfl(val, src);
            const double gx = __shfl(gv.x, src), gy = __shfl(gv.y, src), gz = __shfl(gv.z, src);
            if (L == fo) {
                if (keep && rec < kPairCap) ent[rec] = fj;
                rec++;
                if (ff & 2) {
                    tr.rep += fv;
                    tr.g += d3{gx, gy, gz};
                    tr.cnt++;
                }
            }
        }
    }
    if (!keep) return;
    const int over = group_sum(rec > kPairCap ? 1 : 0);
    const int word = group_sum(min(rec, kPairCap) << (4 * (L & 7)));
    const int cell = query_cell(nl, pu);
    if (L == 0) {
        pc.cnt[u] = (unsigned)word;
        pc.cell[u] = over == 0 ? cell : -1;
    }
}

template <int kBatch>
__device__ __forceinline__ void rep_cached_body(const PassArgs& A, int lb)
{
    if (lb >= A.nblocks) return;    // padding of a grouped launch
    if (!A.rep_v) {
        if (A.tail && lb == 0) finalize_tail(A);    // no query: pass 1's partials are complete
        return;
    }
    const MeshView& m = A.m;
    const EParams& p = A.p;
    const PairCache& pc = A.pc;
    const int base = lb * kVertsPerBlock;
    const int v = base + threadIdx.x;
    const bool mine = threadIdx.x < kVertsPerBlock && v < m.nv;
    // this thread's vertex data, in flight while the mode is decided
    const int meta = mine ? m.meta[v] : 0;
    const d3 xv = mine ? load_p(m.x, v) : d3{0.0, 0.0, 0.0};
    const int rec_cell = mine && pc.x_snap ? pc.cell[v] : -1;    // -1: none
    const unsigned rec_word = mine && pc.x_snap ? pc.cnt[v] : 0u;
    __shared__ FastCells s_fast;
    __shared__ int s_list[kVertsPerBlock];
    __shared__ double s_val[kVertsPerBlock];    // repulsion property per vertex (column 5 of pass 1)
    __shared__ int s_n;
    __shared__ int s_rep[kVertsPerBlock];
    __shared__ unsigned s_word[kVertsPerBlock];
    __shared__ int s_nrep;
    if (threadIdx.x == 0) s_n = s_nrep = s_fast.n = 0;
    s_val[threadIdx.x] = 0.0;
    if (!pc.x_snap) __syncthreads();
    const int mode = pc.x_snap ? pair_cache_mode(pc, A.nl, s_fast) : 0;    // block-uniform: 1 replay, 2 record, 0 full
    if (pc.x_snap && lb == 0 && threadIdx.x == 0)
        put(pc.streak + 1, mode == 1 && s_fast.n > 0 ? pc.streak[0] + 1 : 0);
    const int nfast = s_fast.n;
    if (mine) {
        const bool ring = !is_generic(meta);
        bool done = !ring;
        bool keep = true;    // its list may be replayed, or recorded
        bool listed = false;
        if (mode == 2) {
            pc.x_snap[3 * v] = xv.x;
            pc.x_snap[3 * v + 1] = xv.y;
            pc.x_snap[3 * v + 2] = xv.z;
            if (!ring) pc.cell[v] = -1;
        } else if (ring && mode == 1) {
            if (nfast > 0) {
                const double dx = xv.x - pc.x_snap[3 * v], dy = xv.y - pc.x_snap[3 * v + 1];
                const double dz = xv.z - pc.x_snap[3 * v + 2];
                keep = dx * dx + dy * dy + dz * dz < pc.limit2;
                int c[3];
                cell_coords(A.nl, xv, c);
                // (as vectors, several in flight: 16 us of a block's time with
                // a hundred of them read one component after the other)
                bool near = false;
#pragma unroll 8
                for (int i = 0; i < nfast; i++) {
                    const int4 q = s_fast.c[i];
                    near |= ((unsigned)(c[0] - q.x + 1) <= 2u) & ((unsigned)(c[1] - q.y + 1) <= 2u) &
                            ((unsigned)(c[2] - q.z + 1) <= 2u);
                }
                keep = keep && !near;
            }
            const int cell = rec_cell;
            const unsigned word = rec_word;
            const bool around = keep && cell != -1 && word == kEmptyAround;
            const bool replay = around || (keep && cell != -1 && query_cell(A.nl, xv) == cell);
            if (around || (replay && word == 0u)) {
                done = true;    // nothing recorded: no pairs (the sums over none are +0)
            } else if (replay) {
                const int at = atomicAdd(&s_nrep, 1);
                s_rep[at] = v;
                s_word[at] = word;
                listed = true;
            }
        }
        if (done) {
            A.rep_v[v] = 0.0;
            A.pair_cnt[v] = 0;
            if (!ring) s_val[threadIdx.x] = A.gprops[6 * v + 5];
        } else if (!listed) {
            s_list[atomicAdd(&s_n, 1)] = keep ? v : ~v;
        }
    }
    __syncthreads();
    const int g = threadIdx.x / kGroup, lane = threadIdx.x % kGroup;
    constexpr int kGroups = 256 / kGroup, kAhead = 2;
    // (the phases that most launches on a sphere skip lie behind the rest: their
    // code in the way cost 0.3 us)
    for (int i0 = g; __builtin_expect(i0 < s_nrep, 0); i0 += kAhead * kGroups) {
        static_assert(kPairCap == 8, "a lane's entries are two vectors, the second rarely used");
        const double dmax = p.rep_lc1, dmax2 = dmax * dmax * (1.0 + 1e-15);
        int u[kAhead], k[kAhead];
        const int4* ent[kAhead];
        int4 e[kAhead];
        d3 xu[kAhead], pj[kAhead][4];
        auto positions = [&](int4 id, int n, d3 (&out)[4]) {
            if (n > 0) out[0] = load_p(m.x, id.x);
            if (n > 1) out[1] = load_p(m.x, id.y);
            if (n > 2) out[2] = load_p(m.x, id.z);
            if (n > 3) out[3] = load_p(m.x, id.w);
        };
#pragma unroll
        for (int a = 0; a < kAhead; a++) {
            const int i = i0 + a * kGroups, ic = i < s_nrep ? i : i0;
            u[a] = s_rep[ic];
            k[a] = i < s_nrep ? (int)((s_word[ic] >> (4 * lane)) & 15u) : 0;
            xu[a] = load_p(m.x, u[a]);
            ent[a] = reinterpret_cast<const int4*>(pc.ent + ((size_t)u[a] * kGroup + lane) * kPairCap);
            e[a] = k[a] > 0 ? *ent[a] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int a = 0; a < kAhead; a++) positions(e[a], k[a], pj[a]);
#pragma unroll
        for (int a = 0; a < kAhead; a++) {
            RepTerms t;
            auto add = [&](int n) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (q >= n) continue;
                    const d3 d = xu[a] - pj[a][q];
                    const double sq = sqnorm(d);
                    if (sq <= dmax2 && sqrt(sq) < dmax) t.add(d, p);
                }
            };
            add(k[a]);
            if (k[a] > 4) {
                positions(ent[a][1], k[a] - 4, pj[a]);
                add(k[a] - 4);
            }
            t.group_reduce();
            if (lane == 0 && i0 + a * kGroups < s_nrep) {
                A.rep_v[u[a]] = t.rep;
                A.pair_cnt[u[a]] = t.cnt;
                s_val[u[a] - base] = t.rep;
                store_rep_g(A, u[a], t);
            }
        }
    }
    const int n_full = s_n;
    // a replay launch leaves few vertices per block to the full query, so its
    // latency counts: up to kWaveVerts take a whole wave each (wide_record)
    const bool waves = mode == 1 && n_full <= kWaveVerts;
    for (int i = threadIdx.x / 64; waves && i < n_full; i += 256 / 64) {
        const int e = s_list[i], u = e < 0 ? ~e : e;
        RepTerms tr;
        wide_record(m, A.nl, pc, p, u, meta_valence(m.meta[u]), load_p(m.x, u), e >= 0, tr);
        tr.group_reduce();
        if ((threadIdx.x & 63) == 0) {
            A.rep_v[u] = tr.rep;
            A.pair_cnt[u] = tr.cnt;
            s_val[u - base] = tr.rep;
            store_rep_g(A, u, tr);
        }
    }
    for (int i = g; __builtin_expect(!waves && i < n_full, 0); i += kGroups) {
        const int e = s_list[i], u = e < 0 ? ~e : e;
        const d3 xu = load_p(m.x, u);
        const int n = meta_valence(m.meta[u]);
        RepTerms tr;
        auto add = [&](int, d3 d) { tr.add(d, p); };
        // a replay launch records the lists of the vertices that left
        // their recorded cell (in the cell they are in now), so each pays
        // the full query once per cell it enters; a vertex that is fast or has
        // a fast candidate records nothing
        if (mode != 0 && e >= 0) record_neighbours<kBatch>(m, A.nl, pc, u, n, xu, p.rep_lc1, lane, add);
        else group_neighbours<kBatch>(m, A.nl, u, n, xu, p.rep_lc1, lane, add);
        tr.group_reduce();
        if (lane == 0) {
            A.rep_v[u] = tr.rep;
            A.pair_cnt[u] = tr.cnt;
            s_val[u - base] = tr.rep;
            store_rep_g(A, u, tr);
        }
    }
    __syncthreads();
    // column 5 of pass-1 block lb (the same 256 vertices), summed by the
    // function and in the order pass 1 sums its columns
    static_assert(kVertsPerBlock == kPass1Verts, "the cached query covers one pass-1 block");
    const int vi = base + threadIdx.x;
    if (A.vprops && vi < m.nv) A.vprops[6 * vi + 5] = s_val[threadIdx.x];
    __shared__ double s_red[kPass1Verts / 64];
    const double col5 = block_sum1(s_val[threadIdx.x], s_red);
    if (threadIdx.x == 0) put(A.partials + 5 * (size_t)A.nblocks + lb, col5);
    if (A.tail && last_block_of_many(A.count, lb, A.nblocks)) finalize_tail(A);
}

template <int kBatch>
__global__ void __launch_bounds__(256) k_rep_cached(PassArgs A)
{
    rep_cached_body<kBatch>(A, logical_block());
}

// replica groups: block0 gives each replica its pass1_blocks, a workgroup for each
// pass-1 block of 256 vertices
template <int kBatch>
__global__ void __launch_bounds__(256) k_rep_cached_grouped(const PassArgs* __restrict__ A,
                                                            const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    const int r = find_replica(block0, R, lb);
    rep_cached_body<kBatch>(A[r], lb - block0[r]);
}

// A recording launch the host asks for (new list or topology): the layout
// of k_rep (32 vertices per block, one lane group each), recording every
// ring vertex's lists and every vertex's position.
template <int kBatch, bool kAround>
__global__ void __launch_bounds__(256) k_rep_record(PassArgs A)
{
    const MeshView& m = A.m;
    const EParams& p = A.p;
    const PairCache& pc = A.pc;
    __shared__ double s_rep[256 / kGroup];
    __shared__ int s_cnt[256 / kGroup];
    const int lb = logical_block();
    const int t = lb * 256 + threadIdx.x;
    const int v = t / kGroup, lane = t % kGroup;
    const bool active = v < m.nv;
    const int meta = active ? m.meta[v] : 0;
    const bool ring = active && !is_generic(meta);
    if (t == 0) pc.streak[1] = 0;
    RepTerms tr;
    if (active) {
        const d3 xv = load_p(m.x, v);
        if (lane == 0) {
            pc.x_snap[3 * v] = xv.x;
            pc.x_snap[3 * v + 1] = xv.y;
            pc.x_snap[3 * v + 2] = xv.z;
            if (!ring) pc.cell[v] = -1;
        }
        if (ring)
            record_neighbours<kBatch, kAround>(m, A.nl, pc, v, meta_valence(meta), xv, p.rep_lc1, lane,
                                               [&](int, d3 d) { tr.add(d, p); });
    }
    tr.group_reduce();
    const double rep = tr.rep;
    if (lane == 0) {
        s_rep[threadIdx.x / kGroup] = rep;
        s_cnt[threadIdx.x / kGroup] = tr.cnt;
        if (ring) store_rep_g(A, v, tr);
    }
    __syncthreads();
    const int v0 = lb * (256 / kGroup);
    const int i = threadIdx.x;
    if (i < 256 / kGroup && v0 + i < m.nv) {
        A.rep_v[v0 + i] = s_rep[i];
        A.pair_cnt[v0 + i] = s_cnt[i];
    }
}

template <int kThreads, int kBatch>
__global__ void __launch_bounds__(kThreads) k_rep_grouped(const PassArgs* __restrict__ A,
                                                          const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    const int r = find_replica(block0, R, lb);
    rep_body<kThreads, kBatch>(A[r], lb - block0[r]);
}

// the sums of the meshes of more than kTailBlocks rows, whose pass leaves them
// to a launch of its own
__global__ void __launch_bounds__(256) k_finalize(PassArgs A) { finalize_tail(A); }
__global__ void __launch_bounds__(256) k_finalize_grouped(const PassArgs* __restrict__ A)
{
    if (!A[blockIdx.x].tail) finalize_tail(A[blockIdx.x]);
}

// OpenMesh-semantics properties of the listed vertices (boundary and
// degenerate rings), FP64.
__global__ void __launch_bounds__(128) k_generic_props(MeshView m, NListView nl, EParams p,
                                                       const int* __restrict__ list, int nlist,
                                                       double* __restrict__ gprops)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlist) return;
    int v = list[i];
    VP r = om_vertex_properties(topo_of(m), nl, p, v);
    for (int k = 0; k < 6; k++) gprops[6 * v + k] = r.v[k];
}

__global__ void __launch_bounds__(128) k_generic_grad(MeshView m, NListView nl, EParams p,
                                                      const double* __restrict__ q, const Globals* __restrict__ gp,
                                                      const int* __restrict__ list, int nlist,
                                                      double* __restrict__ grad)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlist) return;
    int v = list[i];
    d3 out = om_vertex_gradient(topo_of(m), nl, p, *gp, q, v);
    grad[3 * v] = out.x;
    grad[3 * v + 1] = out.y;
    grad[3 * v + 2] = out.z;
}

// the same for replica r of a grouped launch, with its parameters read from
// the device table (parallel tempering changes them there)
__global__ void __launch_bounds__(128) k_generic_props_at(const PassArgs* __restrict__ A, int r)
{
    const PassArgs& a = A[r];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.nlist) return;
    int v = a.list[i];
    VP res = om_vertex_properties(topo_of(a.m), a.nl, a.p, v);
    for (int k = 0; k < 6; k++) a.gprops[6 * v + k] = res.v[k];
}

__global__ void __launch_bounds__(128) k_generic_grad_at(const PassArgs* __restrict__ A, int r)
{
    const PassArgs& a = A[r];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.nlist) return;
    int v = a.list[i];
    d3 out = om_vertex_gradient(topo_of(a.m), a.nl, a.p, *a.globals, a.q, v);
    a.grad[3 * v] = out.x;
    a.grad[3 * v + 1] = out.y;
    a.grad[3 * v + 2] = out.z;
}

// --------------------------------------------------------------- pass 2 ---
// Gradient at an interior vertex v.  Mathematically this is the gather of
// mesh_properties.cpp:51-148 combined as in kernel.h:124-137, regrouped so
// that no term relies on cancellation of large contributions:
//
//  * The l * dtheta parts of the spoke edges (v, j_k) and rim edges
//    (j_k, j_{k-1}) meet face by face.  For F_k with interior angles
//    alpha_j at j_k and alpha_i at j_{k-1} and unit normal u_k, the spoke
//    terms give w_{v j_k} cot(alpha_j) u_k + w_{v j_{k-1}} cot(alpha_i) u_k and
//    the rim term -w_{j_k j_{k-1}} (cot(alpha_j) + cot(alpha_i)) u_k, so with
//    edge weights w_{ab} = q_a + q_b (bending, mesh_properties.cpp:88-98,
//    121-129) the face contributes
//        [cot(alpha_j) (q_v - q_{k-1}) + cot(alpha_i) (q_v - q_k)] u_k
//    and with the constant weight of the curvature penalty it contributes 0
//    (Schlaefli's identity).  Only curvature/area differences remain.
//  * The theta * dl parts of the spokes stay as they are: -(q_v + q_k) theta e_hat.
//  * The face-volume gradients cross(x_j, x_k)/6 sum to sum_k n_k / 6 around a
//    closed ring (the x_v x rim terms telescope to zero).
// The penalty factors are known when pass 2 runs, so every contribution goes
// straight into one accumulator.
template <class T>
__device__ __forceinline__ d3 slot_gradient_at(const EParams& p, const Globals& g, double qv, d3 e_prev, d3 e_cur,
                                               double q_prev, double q_cur, d3 n_cur, d3 n_next, const T* th_given)
{
    const double kb = p.kappa_b, kt = p.kappa_t;
    // face F_k = (v, j_k, j_{k-1})
    T n0l = Prec<T>::sqrt_(dot_f(n_cur, n_cur));
    T inv0 = Prec<T>::rcp(n0l);
    d3 rim = e_prev - e_cur;                               // x_{k-1} - x_k
    T cot_j = (T)(-dot_f(rim, e_cur)) * inv0;              // angle at j_k
    T cot_i = (T)dot_f(e_prev, rim) * inv0;                // angle at j_{k-1}
    d3 u = (double)inv0 * n_cur;
    d3 dA = 0.5 * cross_f(u, rim);                         // d area(F_k) / d x_v
    double wq = fma((double)cot_j, qv - q_prev, (double)cot_i * (qv - q_cur));
    double q2 = fma(qv, qv, fma(q_cur, q_cur, q_prev * q_prev));
    double fdA = fma(-kb * (2.0 / 3.0), q2, g.fac_a);
    if (p.bond_type == 1) fdA = fma(kt, bond_area_dfac((double)(n0l * (T)0.5), p), fdA);
    d3 acc = fdA * dA;
    acc = axpy_f(g.fac_v6, n_cur, acc);
    acc = axpy_f(kb * wq, u, acc);
    // spoke (v, j_k) with faces F_k and F_{k+1}
    const double l2 = dot_f(e_cur, e_cur);
    T l = Prec<T>::sqrt_(l2);
    // the angle pass 1 stored (the same operations on the same values), or
    // formed here
    const T th = th_given ? *th_given : Prec<T>::dihedral(n_cur, n_next, e_cur, l);
    double fe = -fma(kb, qv + q_cur, 0.5 * g.fac_c) * (double)th;
    if (p.bond_type == 0) fe = fma(-kt, tether_dfac<T>(l2, l, p), fe);
    return axpy_f(fe * (double)Prec<T>::rcp(l), e_cur, acc);
}

// The gradient at interior vertex v, one lane per vertex, walking the ring
// as pass 1 does (ring_properties): slot k needs the spokes e_{k-1}, e_k,
// e_{k+1}, the curvature ratios q of j_{k-1} and j_k, and the normals n_k and
// n_{k+1}, each carried over from the slot before.  A ring of at most
// kRingPad slots is loaded in full first.
// The gradient of a ring of at most kRingPad neighbours.  Every lane loads
// the leading kRingPad ring columns of vc (they hold -1 past the valence,
// which loads vc itself) and their positions and q before it knows whether
// it needs them (use: an interior vertex with such a ring), so the loads do
// not wait for the vertex's meta word.  kStored: the slots' dihedral angles
// are read from theta (pass 1 stored them), coalesced like the ring columns.
template <class T, bool kStored>
__device__ __forceinline__ d3 ring_gradient_short(const MeshView& m, const EParams& p, const Globals* __restrict__ gp,
                                                  const double* __restrict__ q, int vc, bool use, int n, d3 xv,
                                                  double qv, const T* __restrict__ theta)
{
    const int N = m.nv;
    d3 e[kRingPad];
    double qj[kRingPad];
    T th[kRingPad];
#pragma unroll
    for (int k = 0; k < kRingPad; k++) {
        const int j = m.ring[k * N + vc];
        const int jj = j >= 0 ? j : vc;
        e[k] = load_p(m.x, jj) - xv;
        qj[k] = q[jj];
        if constexpr (kStored) th[k] = theta[k * N + vc];
    }
    d3 acc{0, 0, 0};
    if (!use) return acc;
    const Globals g = *gp;
    d3 e_last = e[kRingPad - 1];
    double q_last = qj[kRingPad - 1];
#pragma unroll
    for (int k = kRingPad - 2; k >= 2; k--)
        if (k == n - 1) {
            e_last = e[k];
            q_last = qj[k];
        }
    d3 n_cur = cross_f(e[0], e_last);
#pragma unroll
    for (int k = 0; k < kRingPad; k++) {
        if (k < n) {
            const d3 e_next = k + 1 < n ? e[(k + 1) % kRingPad] : e[0];
            const d3 e_prev = k == 0 ? e_last : e[(k + kRingPad - 1) % kRingPad];
            const double q_prev = k == 0 ? q_last : qj[(k + kRingPad - 1) % kRingPad];
            const d3 n_next = cross_f(e_next, e[k]);
            acc += slot_gradient_at<T>(p, g, qv, e_prev, e[k], q_prev, qj[k], n_cur, n_next,
                                       kStored ? &th[k] : nullptr);
            n_cur = n_next;
        }
    }
    return acc;
}

// rings longer than kRingPad, slot by slot
template <class T>
__device__ __forceinline__ d3 ring_gradient_walk(const MeshView& m, const EParams& p, const Globals& g,
                                                 const double* __restrict__ q, int v, int n, d3 xv, double qv)
{
    const int N = m.nv;
    d3 acc{0, 0, 0};
    const int j0 = m.ring[v], jl = m.ring[(n - 1) * N + v];
    const d3 e_first = load_p(m.x, j0) - xv;
    const double q_first = q[j0];
    d3 e_prev = load_p(m.x, jl) - xv;
    double q_prev = q[jl];
    d3 e_cur = e_first;
    double q_cur = q_first;
    d3 n_cur = cross_f(e_cur, e_prev);
    for (int k = 0; k < n; k++) {
        d3 e_next = e_first;
        double q_next = q_first;
        if (k + 1 < n) {
            const int j = m.ring[(k + 1) * N + v];
            e_next = load_p(m.x, j) - xv;
            q_next = q[j];
        }
        const d3 n_next = cross_f(e_next, e_cur);
        acc += slot_gradient_at<T>(p, g, qv, e_prev, e_cur, q_prev, q_cur, n_cur, n_next, nullptr);
        e_prev = e_cur;
        q_prev = q_cur;
        e_cur = e_next;
        q_cur = q_next;
        n_cur = n_next;
    }
    return acc;
}

// Pass 2 over the kThreads vertices of block lb, one lane per vertex.
template <class T, int kThreads>
__device__ __forceinline__ void pass2_body(const PassArgs& A, int lb)
{
    const MeshView& m = A.m;
    const EParams& p = A.p;
    const int v = lb * kThreads + threadIdx.x;
    const bool active = v < m.nv;
    // every lane loads (lanes past the last vertex a valid one, discarded)
    const int vc = active ? v : m.nv - 1;
    const int meta = m.meta[vc];
    const d3 xv = load_p(m.x, vc);
    const double qv = A.q[vc];
    const int n = meta_valence(meta);
    const bool ring = active && !is_generic(meta);    // listed vertices: k_generic_grad
    const bool use = ring && n <= kRingPad;
    d3 acc = A.theta ? ring_gradient_short<T, true>(m, p, A.globals, A.q, vc, use, n, xv, qv, (const T*)A.theta)
                     : ring_gradient_short<T, false>(m, p, A.globals, A.q, vc, use, n, xv, qv, nullptr);
    if (ring && n > kRingPad) acc = ring_gradient_walk<T>(m, p, *A.globals, A.q, v, n, xv, qv);
    // repulsion gradient of the vertices the query found pairs for (written
    // by the query kernel of this evaluation)
    if (ring && A.rep_v && p.kappa_r != 0 && A.pair_cnt[v] > 0)
        acc += d3{A.rep_g[3 * v], A.rep_g[3 * v + 1], A.rep_g[3 * v + 2]};
    // stage the block's gradient rows and store them as contiguous doubles;
    // rows of listed (boundary) vertices are left to k_generic_grad
    __shared__ double s_gr[3 * kThreads];
    __shared__ int s_ring[kThreads];
    s_gr[3 * threadIdx.x] = acc.x;
    s_gr[3 * threadIdx.x + 1] = acc.y;
    s_gr[3 * threadIdx.x + 2] = acc.z;
    s_ring[threadIdx.x] = ring;
    __syncthreads();
    const int v0 = lb * kThreads;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const int i = c * kThreads + threadIdx.x;
        const int r = i / 3;
        if (v0 + r < m.nv && s_ring[r]) A.grad[3 * v0 + i] = s_gr[i];
    }
}

template <class T, int kThreads>
__global__ void __launch_bounds__(kThreads) k_pass2(PassArgs A)
{
    pass2_body<T, kThreads>(A, logical_block());
}

template <class T, int kThreads>
__global__ void __launch_bounds__(kThreads) k_pass2_grouped(const PassArgs* __restrict__ A,
                                                            const int* __restrict__ block0, int R)
{
    const int lb = logical_block();
    const int r = find_replica(block0, R, lb);
    pass2_body<T, kThreads>(A[r], lb - block0[r]);
}

// ------------------------------------------------------------ launchers ---
static inline int nblocks(int n, int b) { return (n + b - 1) / b; }

int pass1_blocks(int nv) { return nblocks(nblocks(nv, kPass1Verts), kXcds) * kXcds; }

PassArgs pass_args(const MeshView& m, const NListView& nl, const EParams& p, const PassBuffers& b, double* vprops,
                   double* grad)
{
    PassArgs a{};
    a.m = m;
    a.nl = nl;
    a.p = p;
    a.q = b.q;
    a.gprops = b.gprops;
    a.rep_v = (p.rep_lc1 > 0 && nl.kind >= 0) ? b.rep_v : nullptr;
    a.pair_cnt = b.pair_cnt;
    a.rep_g = b.rep_g;
    a.partials = b.partials;
    a.globals = b.globals;
    a.host = b.host;
    a.grad = grad;
    a.vprops = vprops;
    a.list = b.list;
    a.nlist = b.nlist;
    a.nblocks = pass1_blocks(m.nv);
    a.count = b.count;
    a.tail = a.nblocks > 0 && a.nblocks <= kTailBlocks;    // no vertices, no last workgroup
    a.pc = a.rep_v ? b.pc : PairCache{};
    a.theta = b.theta;
    return a;
}

bool tuning_valid(const Tuning& t)
{
    auto th = [](int x) { return x == 64 || x == 128 || x == 256 || x == 512; };
    return th(t.rep_threads) && th(t.p2_threads) &&
           (t.rep_batch == 1 || t.rep_batch == 2 || t.rep_batch == 4 || t.rep_batch == 8) &&
           (t.rep_fused == 0 || t.rep_fused == 1) && (t.pair_cache == 0 || t.pair_cache == 1) &&
           t.pflip_window >= 1 && t.pflip_window <= 256 && t.serial_window >= 0 && t.serial_window <= 256;
}

int tuned_blocks(int nv, int threads) { return nblocks(nblocks(nv * kGroup, threads), kXcds) * kXcds; }
int pass2_blocks(int nv, int threads) { return nblocks(nblocks(nv, threads), kXcds) * kXcds; }

template <int TH, int B>
static void rep_go(bool grouped, const PassArgs& a, const GroupLaunch* g, hipStream_t s)
{
    if (grouped)
        hipLaunchKernelGGL((k_rep_grouped<TH, B>), dim3(g->total_rep), dim3(TH), 0, s, g->d_args, g->d_block0_rep,
                           g->R);
    else hipLaunchKernelGGL((k_rep<TH, B>), dim3(tuned_blocks(a.m.nv, TH)), dim3(TH), 0, s, a);
}
template <int TH>
static void rep_batch(int batch, bool grouped, const PassArgs& a, const GroupLaunch* g, hipStream_t s)
{
    switch (batch) {
    case 1: rep_go<TH, 1>(grouped, a, g, s); break;
    case 2: rep_go<TH, 2>(grouped, a, g, s); break;
    case 8: rep_go<TH, 8>(grouped, a, g, s); break;
    default: rep_go<TH, 4>(grouped, a, g, s); break;
    }
}
static void rep_dispatch(const Tuning& t, bool grouped, const PassArgs& a, const GroupLaunch* g, hipStream_t s)
{
    switch (t.rep_threads) {
    case 64: rep_batch<64>(t.rep_batch, grouped, a, g, s); break;
    case 128: rep_batch<128>(t.rep_batch, grouped, a, g, s); break;
    case 512: rep_batch<512>(t.rep_batch, grouped, a, g, s); break;
    default: rep_batch<256>(t.rep_batch, grouped, a, g, s); break;
    }
}

template <class T, int TH>
static void p2_go(bool grouped, const PassArgs& a, const GroupLaunch* g, hipStream_t s)
{
    if (grouped)
        hipLaunchKernelGGL((k_pass2_grouped<T, TH>), dim3(g->total_p2), dim3(TH), 0, s, g->d_args, g->d_block0_p2,
                           g->R);
    else hipLaunchKernelGGL((k_pass2<T, TH>), dim3(pass2_blocks(a.m.nv, TH)), dim3(TH), 0, s, a);
}
template <class T>
static void p2_threads(int th, bool grouped, const PassArgs& a, const GroupLaunch* g, hipStream_t s)
{
    switch (th) {
    case 64: p2_go<T, 64>(grouped, a, g, s); break;
    case 128: p2_go<T, 128>(grouped, a, g, s); break;
    case 512: p2_go<T, 512>(grouped, a, g, s); break;
    default: p2_go<T, 256>(grouped, a, g, s); break;
    }
}
static void p2_dispatch(int mixed, const Tuning& t, bool grouped, const PassArgs& a, const GroupLaunch* g,
                        hipStream_t s)
{
    if (mixed) p2_threads<float>(t.p2_threads, grouped, a, g, s);
    else p2_threads<double>(t.p2_threads, grouped, a, g, s);
}

// Pass 1 and the repulsion query (its own launch: a chain of dependent loads
// with few registers).  The full query, and a recording the host asks for,
// run first and pass 1 reads their rep_v; the cached query runs after pass
// 1, which measures the displacements its replay decision needs, and adds
// column 5 of the partials itself.
// A launch that, given marks, stamps marks[0] and marks[1] (either may be
// null) at the kernel's own start and end (hipExtLaunchKernel), so a caller
// can time one kernel of a launch sequence without an event packet between
// launches.
template <class F, class... Args>
void launch_marked(F kernel, dim3 grid, dim3 block, hipStream_t s, const hipEvent_t* marks, Args... args)
{
    if (marks && (marks[0] || marks[1]))
        hipExtLaunchKernelGGL(kernel, grid, block, 0, s, marks[0], marks[1], 0, args...);
    else
        hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
}

void launch_pass1_body(const PassArgs& a, int mixed, const Tuning& t, hipStream_t s, const hipEvent_t* marks)
{
    if (a.m.nv == 0) return;
    const dim3 grid(a.nblocks), block(kPass1Verts);
    if (a.rep_v && a.pc.x_snap && !a.pc.force) {
        if (mixed) launch_marked(k_pass1_apart<float>, grid, block, s, marks, a);
        else launch_marked(k_pass1_apart<double>, grid, block, s, marks, a);
        launch_rep(a, t, s);
        return;
    }
    launch_rep(a, t, s);
    if (mixed) launch_marked(k_pass1<float>, grid, block, s, marks, a);
    else launch_marked(k_pass1<double>, grid, block, s, marks, a);
}

template <bool kAround>
static void record_dispatch(const Tuning& t, dim3 grid, dim3 block, const PassArgs& a, hipStream_t s)
{
    switch (t.rep_batch) {
    case 1: hipLaunchKernelGGL((k_rep_record<1, kAround>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_rep_record<2, kAround>), grid, block, 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_rep_record<8, kAround>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((k_rep_record<4, kAround>), grid, block, 0, s, a); break;
    }
}

void launch_rep(const PassArgs& a, const Tuning& t, hipStream_t s)
{
    if (!a.rep_v || a.m.nv == 0) return;
    if (!a.pc.x_snap) {
        rep_dispatch(t, false, a, nullptr, s);
        return;
    }
    const dim3 block(256);
    if (a.pc.force) {
        const dim3 grid(tuned_blocks(a.m.nv, 256));
        if (a.m.nv <= kAroundVerts) record_dispatch<true>(t, grid, block, a, s);
        else record_dispatch<false>(t, grid, block, a, s);
        return;
    }
    const dim3 grid(nblocks(nblocks(a.m.nv, kVertsPerBlock), kXcds) * kXcds);
    switch (t.rep_batch) {
    case 1: hipLaunchKernelGGL(k_rep_cached<1>, grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL(k_rep_cached<2>, grid, block, 0, s, a); break;
    case 8: hipLaunchKernelGGL(k_rep_cached<8>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(k_rep_cached<4>, grid, block, 0, s, a); break;
    }
}

void launch_pass2_kernel(const PassArgs& a, int mixed, const Tuning& t, hipStream_t s)
{
    if (a.m.nv > 0) p2_dispatch(mixed, t, false, a, nullptr, s);
}

void launch_pass1(const MeshView& m, const NListView& nl, const EParams& p, int mixed, const PassBuffers& b,
                  double* vprops, hipStream_t s, const Tuning& t, const hipEvent_t* marks)
{
    const PassArgs a = pass_args(m, nl, p, b, vprops, nullptr);
    if (b.nlist > 0)
        hipLaunchKernelGGL(k_generic_props, dim3(nblocks(b.nlist, 128)), dim3(128), 0, s, m, nl, p, b.list, b.nlist,
                           b.gprops);
    launch_pass1_body(a, mixed, t, s, marks);
    if (!a.tail) hipLaunchKernelGGL(k_finalize, dim3(1), dim3(256), 0, s, a);
}

void launch_pass2(const MeshView& m, const NListView& nl, const EParams& p, int mixed, const PassBuffers& b,
                  double* grad, hipStream_t s, const Tuning& t)
{
    const PassArgs a = pass_args(m, nl, p, b, nullptr, grad);
    launch_pass2_kernel(a, mixed, t, s);
    if (b.nlist > 0)
        hipLaunchKernelGGL(k_generic_grad, dim3(nblocks(b.nlist, 128)), dim3(128), 0, s, m, nl, p, b.q, b.globals,
                           b.list, b.nlist, grad);
}

static bool group_repels(const GroupLaunch& g)
{
    for (int r = 0; r < g.R; r++)
        if (g.h_args[r].rep_v) return true;
    return false;
}

void launch_rep_grouped(const GroupLaunch& g, hipStream_t s)
{
    if (!group_repels(g)) return;
    if (g.total_rc > 0) {
        const dim3 grid(g.total_rc), block(256);
        switch (g.tune.rep_batch) {
        case 1: hipLaunchKernelGGL(k_rep_cached_grouped<1>, grid, block, 0, s, g.d_args, g.d_block0_rc, g.R); break;
        case 2: hipLaunchKernelGGL(k_rep_cached_grouped<2>, grid, block, 0, s, g.d_args, g.d_block0_rc, g.R); break;
        case 8: hipLaunchKernelGGL(k_rep_cached_grouped<8>, grid, block, 0, s, g.d_args, g.d_block0_rc, g.R); break;
        default: hipLaunchKernelGGL(k_rep_cached_grouped<4>, grid, block, 0, s, g.d_args, g.d_block0_rc, g.R); break;
        }
        return;
    }
    rep_dispatch(g.tune, true, g.h_args[0], &g, s);
}

void launch_pass1_grouped(const GroupLaunch& g, hipStream_t s, const hipEvent_t* marks)
{
    for (int r = 0; r < g.R; r++)
        if (g.h_args[r].nlist > 0)
            hipLaunchKernelGGL(k_generic_props_at, dim3(nblocks(g.h_args[r].nlist, 128)), dim3(128), 0, s, g.d_args,
                               r);
    const dim3 grid(g.total_p1), block(kPass1Verts);
    if (g.total_rc > 0 && group_repels(g)) {
        // the cached query after pass 1, as for single meshes
        if (g.mixed) launch_marked(k_pass1_apart_grouped<float>, grid, block, s, marks, g.d_args, g.d_block0_p1, g.R);
        else launch_marked(k_pass1_apart_grouped<double>, grid, block, s, marks, g.d_args, g.d_block0_p1, g.R);
        launch_rep_grouped(g, s);
    } else {
        launch_rep_grouped(g, s);
        if (g.mixed) launch_marked(k_pass1_grouped<float>, grid, block, s, marks, g.d_args, g.d_block0_p1, g.R);
        else launch_marked(k_pass1_grouped<double>, grid, block, s, marks, g.d_args, g.d_block0_p1, g.R);
    }
    bool tail = true;
    for (int r = 0; r < g.R; r++) tail = tail && g.h_args[r].tail;
    if (!tail) hipLaunchKernelGGL(k_finalize_grouped, dim3(g.R), dim3(256), 0, s, g.d_args);
}

void launch_pass2_grouped(const GroupLaunch& g, hipStream_t s)
{
    p2_dispatch(g.mixed, g.tune, true, g.h_args[0], &g, s);
    for (int r = 0; r < g.R; r++)
        if (g.h_args[r].nlist > 0)
            hipLaunchKernelGGL(k_generic_grad_at, dim3(nblocks(g.h_args[r].nlist, 128)), dim3(128), 0, s, g.d_args,
                               r);
}

// --------------------------------------------- single-halfedge geometry ---
// out: [l, dl(2x3), A, dA(3x3), V, dV(3x3), theta, dtheta(4x3)]  (47 doubles)
__global__ void k_halfedge_geometry(MeshView m, int h, double* out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const Topo t = topo_of(m);
    int k = 0;
    out[k++] = mu_edge_length(t, h);
    d3 g0 = mu_edge_length_grad_from(t, h);
    d3 gs[4];
    gs[0] = g0;
    gs[1] = -g0;
    for (int i = 0; i < 2; i++) { out[k++] = gs[i].x; out[k++] = gs[i].y; out[k++] = gs[i].z; }
    out[k++] = mu_face_area(t, h);
    for (int i = 0; i < 3; i++) { d3 a = mu_face_area_grad(t, h, i); out[k++] = a.x; out[k++] = a.y; out[k++] = a.z; }
    out[k++] = mu_face_volume(t, h);
    for (int i = 0; i < 3; i++) { d3 a = mu_face_volume_grad(t, h, i); out[k++] = a.x; out[k++] = a.y; out[k++] = a.z; }
    out[k++] = om_dihedral_angle(t, h);
    for (int i = 0; i < 4; i++) { d3 a = mu_dihedral_angle_grad(t, h, i); out[k++] = a.x; out[k++] = a.y; out[k++] = a.z; }
}

void launch_halfedge_geometry(const MeshView& m, int h, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(k_halfedge_geometry, dim3(1), dim3(64), 0, s, m, h, out);
}

// -------------------------------------------------- mesh-wide utilities ---
// sum of face areas (util.cpp:9-21) or edge lengths (util.cpp:23-35)
__global__ void k_sum_geometry(MeshView m, int what, double* partials, unsigned* counter, double* result)
{
    __shared__ double s_red[4 * 6];
    __shared__ double s_out[6];
    __shared__ int s_last;
    const Topo t = topo_of(m);
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (what == 0 && i < m.nf) v[0] = mu_face_area(t, m.f_he[i]);
    if (what == 1 && i < m.nh / 2) v[0] = mu_edge_length(t, 2 * i);
    block_sum6(v, s_red, s_out);
    if (threadIdx.x == 0) partials[blockIdx.x] = s_out[0];
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) s_last = (atomicAdd(counter, 1u) == gridDim.x - 1);
    __syncthreads();
    if (s_last) {
        __threadfence();
        double a[6] = {0, 0, 0, 0, 0, 0};
        for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x) a[0] += partials[b];
        block_sum6(a, s_red, s_out);
        if (threadIdx.x == 0) {
            *result = s_out[0];
            *counter = 0u;
        }
    }
}

void launch_sum_geometry(const MeshView& m, int what, double* partials, unsigned* counter, double* result,
                         hipStream_t s)
{
    int n = what == 0 ? m.nf : m.nh / 2;
    hipLaunchKernelGGL(k_sum_geometry, dim3(nblocks(n > 0 ? n : 1, 256)), dim3(256), 0, s, m, what, partials,
                       counter, result);
}

}    // namespace tmh
