// tm_nlist.hip -- cell-list binning and neighbour queries on the GPU.
//
// Reference: src/nlists/cell_list.h:28-313 and verlet_list.h:14-103.
//
// Build (cell list): a box reduction reproducing the reference's partial
// initialisation (cell_list.h:46-47: only component 0 of each bound starts at
// +max / -1, components 1 and 2 start at 0), the per-dimension cell size
// r_list = dim / int(dim / rlist) (cell_list.h:59-66, computed on the host in
// FP64 from the reduced box), flat cell ids sum_k int((p_k - min_k) / r_k)
// * stride_k (cell_list.h:70-79), then a counting sort: histogram, exclusive
// scan, scatter, and a per-cell sort by vertex id so that the order inside a
// cell is ascending like the reference's push_back order.  Every kernel of the
// build takes one list (its arguments by value) or many (a table of them and a
// prefix table of workgroups): the lists of a replica group are built together,
// with the launches and the one host round trip of a single list.  The reference keys
// its cells in a map (cell_list.h:31), so only occupied cells cost memory;
// here the table is dense over the occupied sub-grid, the global cells lo ..
// hi that hold a vertex at build time, which is the mesh's own bounding box
// in cells whatever the reference's box (anchored at 0 in y and z) spans.
// Stencils clipped to the sub-grid visit the same vertices as stencils
// clipped to the global grid: every cell outside the sub-grid is empty.
//
// Queries use the current positions with the cells frozen at build time,
// exactly as the reference does between two update_repulsion calls.  All
// distance tests are IEEE FP64 sqrt(dx*dx + dy*dy + dz*dz) (the library is
// built with -ffp-contract=off), compared with < dmax (point_distances,
// cell_list.h:208) or <= rlist (distance_matrix, cell_list.h:294).
#include "tm_internal.h"
#include "tm_om.h"

#include <cfloat>

namespace tmh {

// ----------------------------------------------------------------- box ----
// Bounding box of the vertices, as kBoxBlocks per-block partial minima and
// maxima (part[6 b + k], min in k < 3, max in k >= 3; +DBL_MAX and -DBL_MAX
// for a block without vertices).  They go to pinned host memory: the host needs
// the box anyway, to size the grid, so it combines them (min and max are exact in
// any order) and applies the reference's initial values (cell_list.h:46-47).
constexpr int kBoxBlocks = 64;
__device__ __forceinline__ void box_body(const NlistBuild& b, int lb)
{
    const double* __restrict__ x = b.x;
    const int n = b.n;
    __shared__ double s[6][4];
    double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX};
    double mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    // kBoxBatch points per thread and step, all their loads in flight before
    // the first comparison
    constexpr int kBoxBatch = 8;
    const int stride = kBoxBlocks * blockDim.x;
    for (int i0 = lb * blockDim.x + threadIdx.x; i0 < n; i0 += kBoxBatch * stride) {
        double v[kBoxBatch][3];
#pragma unroll
        for (int u = 0; u < kBoxBatch; u++) {
            const int i = i0 + u * stride;
#pragma unroll
            for (int k = 0; k < 3; k++) v[u][k] = i < n ? x[3 * i + k] : __builtin_nan("");    // neither test takes NaN
        }
#pragma unroll
        for (int u = 0; u < kBoxBatch; u++)
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if (v[u][k] < mn[k]) mn[k] = v[u][k];
                if (v[u][k] > mx[k]) mx[k] = v[u][k];
            }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < 3; k++) {
        for (int off = 32; off > 0; off >>= 1) {
            mn[k] = fmin(mn[k], __shfl_xor(mn[k], off, 64));
            mx[k] = fmax(mx[k], __shfl_xor(mx[k], off, 64));
        }
    }
    if (lane == 0) {
        for (int k = 0; k < 3; k++) {
            s[k][wave] = mn[k];
            s[3 + k][wave] = mx[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        int k = threadIdx.x;
        double r = s[k][0];
        for (int w = 1; w < 4; w++) r = k < 3 ? fmin(r, s[k][w]) : fmax(r, s[k][w]);
        b.box[lb * 6 + k] = r;
    }
}

int box_scratch_doubles() { return kBoxBlocks * 6; }

// Up to three int ranges set to a value each, in one launch (the list build
// issues these fills back to back after its one host round trip).
__global__ void k_fill_ints(int* a, int na, int va, int* b, int nb, int vb, int* c, int nc, int vc)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < na) a[i] = va;
    if (i < nb) b[i] = vb;
    if (i < nc) c[i] = vc;
}

void launch_fill_ints(int* a, int na, int va, int* b, int nb, int vb, int* c, int nc, int vc, hipStream_t s)
{
    const int n = std::max(na, std::max(nb, nc));
    if (n <= 0) return;
    hipLaunchKernelGGL(k_fill_ints, dim3((n + 255) / 256), dim3(256), 0, s, a, na, va, b, nb, vb, c, nc, vc);
}


// ------------------------------------------------------------- binning ----
// Build-time cell of vertex v in the occupied sub-grid.  The coordinate is
// clamped into the sub-grid: the reference's box epsilon (1e-6) vanishes in
// rounding for coordinates beyond ~1e9, where int((max - min) / r) can reach
// the grid size.
__device__ __forceinline__ int flat_cell(const NListView& nl, const double* x, int v)
{
    int id = 0;
    for (int k = 0; k < 3; k++) {
        int c = cell_coord(nl, x[3 * v + k], k);
        c = min(max(c, 0), nl.shape[k] - 1);
        id += c * nl.strides[k];
    }
    return id;
}

// all cells empty
constexpr int kClearTile = 4096;
__device__ __forceinline__ void clear_body(const NlistBuild& b, int lb)
{
    const int end = min((lb + 1) * kClearTile, b.nc + 1);
    for (int i = lb * kClearTile + threadIdx.x; i < end; i += 256) b.counts[i] = 0;
}

// each vertex's cell and its place among the cell's vertices as they come (the
// count that it found), which makes the scatter a plain store; the pair cache
// starts with nothing to replay
__device__ __forceinline__ void cells_body(const NlistBuild& b, int lb)
{
    const int v = lb * 256 + threadIdx.x;
    if (v >= b.n) return;
    const int c = flat_cell(b.nl, b.x, v);
    b.vert_cell[v] = c;
    b.place[v] = atomicAdd(&b.counts[c], 1);
    if (!b.cand) return;
    b.pc_cell[v] = -1;    // no replay
    if (v == 0) b.cand_count[b.n] = b.pc_streak[0] = b.pc_streak[1] = 0;
}

// ------------------------------------------------ stencil candidate lists
// The 27-cell stencil of cell c as 9 rows of x-consecutive cells, clipped to the
// grid like the query of cell_list.h:133-219: each row's range in cell_verts,
// all loads in flight at once.
struct StencilRows {
    int start[9], len[9];
};
__device__ __forceinline__ StencilRows stencil_rows(const NListView& nl, int cell)
{
    const int c2 = cell / nl.strides[2], c1 = (cell - c2 * nl.strides[2]) / nl.strides[1];
    const int c0 = cell - c2 * nl.strides[2] - c1 * nl.strides[1];
    const int i0 = max(c0 - 1, 0), i1 = min(c0 + 1, nl.shape[0] - 1);
    StencilRows r;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const int kk = c2 + k / 3 - 1, jj = c1 + k % 3 - 1;
        const bool in = kk >= 0 && kk < nl.shape[2] && jj >= 0 && jj < nl.shape[1];
        const int base = in ? jj * nl.strides[1] + kk * nl.strides[2] : 0;
        r.start[k] = in ? nl.cell_start[base + i0] : 0;
        r.len[k] = in ? nl.cell_start[base + i1 + 1] : 0;
    }
#pragma unroll
    for (int k = 0; k < 9; k++) r.len[k] -= r.start[k];
    return r;
}

// the counting sort's scatter; with it the stencil size of each occupied cell at
// its first slot, 0 at the others
__device__ __forceinline__ void scatter_body(const NlistBuild& b, int lb)
{
    const int v = lb * 256 + threadIdx.x;
    if (v >= b.n) return;
    const int c = b.vert_cell[v], place = b.place[v], slot = b.nl.cell_start[c] + place;
    b.cell_verts[slot] = v;
    if (!b.cand) return;
    int total = 0;
    if (place == 0) {
        const StencilRows r = stencil_rows(b.nl, c);
#pragma unroll
        for (int k = 0; k < 9; k++) total += r.len[k];
    }
    b.cand_count[slot] = total;
}

// The thread at the start of a cell's segment sorts it by user vertex id (cells
// hold a handful of vertices), the order in which the reference fills its cells.
__device__ __forceinline__ void sort_segment(const NlistBuild& b, int i)
{
    int* cell_verts = b.cell_verts;
    const int c = b.vert_cell[cell_verts[i]];
    if (b.nl.cell_start[c] != i) return;
    const int e = b.nl.cell_start[c + 1];
    for (int a = i + 1; a < e; a++) {
        const int key = cell_verts[a], kp = b.perm[key];
        int q = a - 1;
        while (q >= i && b.perm[cell_verts[q]] > kp) {
            cell_verts[q + 1] = cell_verts[q];
            q--;
        }
        cell_verts[q + 1] = key;
    }
}
__device__ __forceinline__ void sort_body(const NlistBuild& b, int lb)
{
    const int i = lb * 256 + threadIdx.x;
    if (i < b.n) sort_segment(b, i);
}

// The stencil lists, eight lanes per slot: the slots of a cell take its candidates
// in turns of eight, each lane its own from its row, and the first lane stores the
// range of the slot's vertex.  A chain of five loads, whatever the list's length
// (16.9 us at 163842 vertices, 5.5 at 2562; with one thread per slot copying whole
// rows 22.5 and 15.1).
__device__ __forceinline__ void fill_body(const NlistBuild& b, int lb)
{
    const int t = lb * 256 + threadIdx.x, i = t / 8, lane = t % 8;
    if (i >= b.n) return;
    const int v = b.cell_verts[i], c = b.vert_cell[v];
    const int s0 = b.nl.cell_start[c], verts = b.nl.cell_start[c + 1] - s0;
    const StencilRows r = stencil_rows(b.nl, c);
    const int first = b.cand_start[s0], total = b.cand_start[s0 + 1] - first;
    if (lane == 0) b.vcand[v] = make_int2(first, first + total);
    for (int k = 8 * (i - s0) + lane; k < total; k += 8 * verts) {
        int q = k, at = 0;
        bool found = false;
#pragma unroll
        for (int w = 0; w < 9; w++) {
            if (!found && q < r.len[w]) {
                at = r.start[w] + q;
                found = true;
            }
            if (!found) q -= r.len[w];
        }
        b.cand[first + k] = b.cell_verts[at];
    }
}

// ---------------------------------------------------- exclusive scan ------
// Block-local scans of 4096 elements with block totals, and the add-back of the
// totals before each block.
constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

int scan_block_sums_size(int n) { return (n + kScanTile - 1) / kScanTile + 1; }

__device__ __forceinline__ int block_exclusive_scan(int v, int* s_warp, int* total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
    for (int off = 1; off < 64; off <<= 1) {
        int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_warp[wave] = x;
    __syncthreads();
    if (wave == 0) {
        int nw = blockDim.x >> 6;
        int w = lane < nw ? s_warp[lane] : 0;
        for (int off = 1; off < 64; off <<= 1) {
            int y = __shfl_up(w, off, 64);
            if (lane >= off) w += y;
        }
        if (lane < nw) s_warp[lane] = w;
    }
    __syncthreads();
    int base = wave > 0 ? s_warp[wave - 1] : 0;
    *total = s_warp[(blockDim.x >> 6) - 1];
    __syncthreads();
    return base + x - v;
}

__device__ __forceinline__ void scan_tile(const int* __restrict__ in, int* __restrict__ out, int n,
                                          int* __restrict__ sums, int lb)
{
    __shared__ int s_warp[16];
    static_assert(kScanItems == 4, "a thread's elements are one vector");
    const int base = lb * kScanTile + threadIdx.x * kScanItems;
    int4 v = make_int4(0, 0, 0, 0);
    if (base + 3 < n) {
        v = *reinterpret_cast<const int4*>(in + base);
    } else {
        if (base < n) v.x = in[base];
        if (base + 1 < n) v.y = in[base + 1];
        if (base + 2 < n) v.z = in[base + 2];
    }
    int total;
    const int off = block_exclusive_scan(v.x + v.y + v.z + v.w, s_warp, &total);
    const int4 o = make_int4(off, off + v.x, off + v.x + v.y, off + v.x + v.y + v.z);
    if (base + 3 < n) {
        *reinterpret_cast<int4*>(out + base) = o;
    } else {
        if (base < n) out[base] = o.x;
        if (base + 1 < n) out[base + 1] = o.y;
        if (base + 2 < n) out[base + 2] = o.z;
    }
    if (threadIdx.x == 0) sums[lb] = total;
}
__global__ void __launch_bounds__(kScanThreads) k_scan_tiles(const int* __restrict__ in, int* __restrict__ out,
                                                             int n, int* __restrict__ sums)
{
    scan_tile(in, out, n, sums, blockIdx.x);
}

__global__ void __launch_bounds__(kScanThreads) k_scan_sums(int* __restrict__ sums, int nb)
{
    __shared__ int s_warp[16];
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += kScanThreads) {
        int i = b0 + threadIdx.x;
        int v = i < nb ? sums[i] : 0;
        int total;
        int ex = block_exclusive_scan(v, s_warp, &total);
        if (i < nb) sums[i] = carry + ex;
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[nb] = carry;
}

// The add-back of tile lb.  Every workgroup adds up the totals before it for
// itself (few, and read once each), which saves the launch that scans them;
// kScanned: that launch has run (more than kSumTiles tiles).
constexpr int kSumTiles = 2048;
template <bool kScanned>
__device__ __forceinline__ void scan_add(int* __restrict__ out, int n, const int* __restrict__ sums, int lb)
{
    __shared__ int s_part[kScanThreads / 64];
    int before = 0;
    if constexpr (kScanned) {
        before = sums[lb];
    } else {
        for (int i = threadIdx.x; i < lb; i += kScanThreads) before += sums[i];
        for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
        if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = before;
        __syncthreads();
        before = 0;
        for (int w = 0; w < kScanThreads / 64; w++) before += s_part[w];
    }
    for (int k = 0; k < kScanItems; k++) {
        const int i = lb * kScanTile + k * kScanThreads + threadIdx.x;
        if (i < n) out[i] += before;
    }
}
template <bool kScanned>
__global__ void __launch_bounds__(kScanThreads) k_scan_add(int* __restrict__ out, int n, const int* __restrict__ sums)
{
    scan_add<kScanned>(out, n, sums, blockIdx.x);
}

void launch_exclusive_scan(const int* in, int* out, int n, int* block_sums, hipStream_t s)
{
    const int nb = (n + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_tiles, dim3(nb), dim3(kScanThreads), 0, s, in, out, n, block_sums);
    if (nb > kSumTiles) {
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanThreads), 0, s, block_sums, nb);
        hipLaunchKernelGGL(k_scan_add<true>, dim3(nb), dim3(kScanThreads), 0, s, out, n, block_sums);
    } else {
        hipLaunchKernelGGL(k_scan_add<false>, dim3(nb), dim3(kScanThreads), 0, s, out, n, block_sums);
    }
}

// the build's two scans: the cells' counts, and the stencil sizes, whose add-back
// launch also sorts the cells' segments
__device__ __forceinline__ void cell_tiles_body(const NlistBuild& b, int lb)
{
    scan_tile(b.counts, b.cell_start, b.nc + 1, b.sums, lb);
}
__device__ __forceinline__ void cell_starts_body(const NlistBuild& b, int lb)
{
    scan_add<false>(b.cell_start, b.nc + 1, b.sums, lb);
}
__device__ __forceinline__ void cand_tiles_body(const NlistBuild& b, int lb)
{
    scan_tile(b.cand_count, b.cand_start, b.n + 1, b.sums, lb);
}
__device__ __forceinline__ void cand_starts_body(const NlistBuild& b, int lb)
{
    // a thread per slot, for the sort's sake (at 163842 vertices 28.8 us with
    // the scan's tiles, 11.3 with these); few totals, so every
    // workgroup adds up those before its tile
    __shared__ int s_part[4];
    const int i = lb * 256 + threadIdx.x;
    int before = 0;
    for (int k = threadIdx.x; k < lb * 256 / kScanTile; k += 256) before += b.sums[k];
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = before;
    __syncthreads();
    before = s_part[0] + s_part[1] + s_part[2] + s_part[3];
    if (i <= b.n) b.cand_start[i] += before;
    if (i < b.n) sort_segment(b, i);
}

// ---------------------------------------------------------- the build ----
// kNear: the kernels of vertices and slots, whose neighbours read the same lines
// (logical_block); their grids are rounded up to it.
template <bool kNear>
__device__ __forceinline__ int build_block()
{
    return kNear ? logical_block() : (int)blockIdx.x;
}
#define TM_BUILD_KERNEL(name, threads, near)                                                                    \
    __global__ void __launch_bounds__(threads) k_nl_##name(NlistBuild b) { name##_body(b, build_block<near>()); } \
    __global__ void __launch_bounds__(threads) k_nl_##name##_grouped(const NlistBuild* __restrict__ b,          \
                                                                    const int* __restrict__ block0, int R)      \
    {                                                                                                           \
        const int lb = build_block<near>();                                                                     \
        if (lb >= block0[R]) return;                                                                            \
        const int r = find_replica(block0, R, lb);                                                              \
        name##_body(b[r], lb - block0[r]);                                                                      \
    }
TM_BUILD_KERNEL(box, 256, false)
TM_BUILD_KERNEL(clear, 256, false)
TM_BUILD_KERNEL(cells, 256, true)
TM_BUILD_KERNEL(cell_tiles, kScanThreads, false)
TM_BUILD_KERNEL(cell_starts, kScanThreads, false)
TM_BUILD_KERNEL(scatter, 256, true)
TM_BUILD_KERNEL(sort, 256, true)
TM_BUILD_KERNEL(cand_tiles, kScanThreads, false)
TM_BUILD_KERNEL(cand_starts, 256, true)
TM_BUILD_KERNEL(fill, 256, true)
#undef TM_BUILD_KERNEL

static int ceil_div(int a, int b) { return (a + b - 1) / b; }
int nlist_blocks(const NlistBuild& b, int shape)
{
    switch (shape) {
    case kShapeBox: return kBoxBlocks;
    case kShapeVerts: return ceil_div(b.n, 256);
    case kShapeCells: return ceil_div(b.nc + 1, kScanTile);
    case kShapeCand: return b.cand ? ceil_div(b.n + 1, kScanTile) : 0;
    case kShapeStarts: return b.cand ? ceil_div(b.n + 1, 256) : 0;
    case kShapeFill: return b.cand ? ceil_div(b.n, 32) : 0;
    case kShapeVertsSort: return b.cand ? 0 : ceil_div(b.n, 256);
    default: return b.cand ? ceil_div(b.n * kPairLanes, 256) : 0;    // kShapeMask
    }
}
static_assert(kClearTile == kScanTile, "kShapeCells");

#define TM_BUILD_LAUNCH(name, shape, threads, near)                                                             \
    if (g.total[shape] > 0) {                                                                                   \
        const dim3 grid(near ? ceil_div(g.total[shape], kXcds) * kXcds : g.total[shape]);                       \
        if (g.R == 1)                                                                                           \
            hipLaunchKernelGGL(k_nl_##name, grid, dim3(threads), 0, s, g.h[0]);                                 \
        else                                                                                                    \
            hipLaunchKernelGGL(k_nl_##name##_grouped, grid, dim3(threads), 0, s, g.d,                           \
                               g.block0 + shape * (g.R + 1), g.R);                                              \
    }
void launch_nlist_box(const NlistGroup& g, hipStream_t s) { TM_BUILD_LAUNCH(box, kShapeBox, 256, false) }
void launch_nlist_build(const NlistGroup& g, hipStream_t s)
{
    TM_BUILD_LAUNCH(clear, kShapeCells, 256, false)
    TM_BUILD_LAUNCH(cells, kShapeVerts, 256, true)
    int tiles = 0;
    for (int r = 0; r < g.R; r++) tiles = std::max(tiles, nlist_blocks(g.h[r], kShapeCells));
    if (tiles > kSumTiles) {
        for (int r = 0; r < g.R; r++)
            launch_exclusive_scan(g.h[r].counts, g.h[r].cell_start, g.h[r].nc + 1, g.h[r].sums, s);
    } else {
        TM_BUILD_LAUNCH(cell_tiles, kShapeCells, kScanThreads, false)
        TM_BUILD_LAUNCH(cell_starts, kShapeCells, kScanThreads, false)
    }
    TM_BUILD_LAUNCH(scatter, kShapeVerts, 256, true)
    TM_BUILD_LAUNCH(sort, kShapeVertsSort, 256, true)
    // (at most 2^31 / 27 vertices: 19419 tiles)
    tiles = 0;
    for (int r = 0; r < g.R; r++) tiles = std::max(tiles, nlist_blocks(g.h[r], kShapeCand));
    if (tiles > kSumTiles) {
        for (int r = 0; r < g.R; r++)
            if (g.h[r].cand) {
                launch_exclusive_scan(g.h[r].cand_count, g.h[r].cand_start, g.h[r].n + 1, g.h[r].sums, s);
                hipLaunchKernelGGL(k_nl_sort, dim3(ceil_div(nlist_blocks(g.h[r], kShapeVerts), kXcds) * kXcds), dim3(256),
                                   0, s, g.h[r]);
            }
    } else {
        TM_BUILD_LAUNCH(cand_tiles, kShapeCand, kScanThreads, false)
        TM_BUILD_LAUNCH(cand_starts, kShapeStarts, 256, true)
    }
    TM_BUILD_LAUNCH(fill, kShapeFill, 256, true)
    launch_nlist_masks(g, s);
}
#undef TM_BUILD_LAUNCH

// ------------------------------------------------------ distance matrix ---
__device__ __forceinline__ double dist_ab(const double* x, int a, int b)
{
    // cell_list.h:11-25 squ_distance / distance
    double d0 = x[3 * a] - x[3 * b], d1 = x[3 * a + 1] - x[3 * b + 1], d2 = x[3 * a + 2] - x[3 * b + 2];
    double s = 0.0;
    s += d0 * d0;
    s += d1 * d1;
    s += d2 * d2;
    return sqrt(s);
}

// Visit the pairs a emits: for the cell list, b in the 27 cells around a's
// build-time cell with (cell(b) > cell(a)) or (same cell and b > a), not
// excluded, distance <= dmax -- each unordered pair of the reference's
// cell-pair enumeration exactly once (cell_list.h:221-312); for the Verlet
// list, b in adj(a) with distance < dmax (verlet_list.h:39-72).
template <class F>
__device__ __forceinline__ void dm_visit(const MeshView& m, const NListView& nl, double dmax, int a, F&& f)
{
    if (nl.kind == 0) {
        const Topo t = topo_of(m);
        int ca = nl.vert_cell[a];
        int kc = ca / nl.strides[2];
        int rem = ca % nl.strides[2];
        int jc = rem / nl.strides[1];
        int ic = rem % nl.strides[1];
        for (int di = -1; di < 2; di++) {
            int ii = ic + di;
            if (ii < 0 || ii >= nl.shape[0]) continue;
            for (int dj = -1; dj < 2; dj++) {
                int jj = jc + dj;
                if (jj < 0 || jj >= nl.shape[1]) continue;
                for (int dk = -1; dk < 2; dk++) {
                    int kk = kc + dk;
                    if (kk < 0 || kk >= nl.shape[2]) continue;
                    int oc = ii * nl.strides[0] + jj * nl.strides[1] + kk * nl.strides[2];
                    if (oc < ca) continue;
                    for (int q = nl.cell_start[oc]; q < nl.cell_start[oc + 1]; q++) {
                        int b = nl.cell_verts[q];
                        if (oc == ca && b <= a) continue;
                        double d = dist_ab(m.x, a, b);
                        if (d <= dmax && !om_excluded(t, a, b, nl.exclusion)) f(b, d);
                    }
                }
            }
        }
    } else if (nl.kind == 1) {
        for (int q = nl.adj_start[a]; q < nl.adj_start[a + 1]; q++) {
            int b = nl.adj[q];
            double d = dist_ab(m.x, a, b);
            if (d < dmax) f(b, d);
        }
    }
}

__global__ void k_dm_count(MeshView m, NListView nl, double dmax, int* __restrict__ counts)
{
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= m.nv) return;
    int c = 0;
    dm_visit(m, nl, dmax, a, [&](int, double) { c++; });
    counts[a] = c;
}

__global__ void k_dm_fill(MeshView m, NListView nl, double dmax, const int* __restrict__ offsets, double* d,
                          int* ii, int* jj)
{
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= m.nv) return;
    int o = offsets[a];
    const bool ordered = nl.kind == 0;
    const int ua = nl.perm[a];
    dm_visit(m, nl, dmax, a, [&](int b, double dd) {
        const int ub = nl.perm[b];
        d[o] = dd;
        if (ordered) {
            ii[o] = ua < ub ? ua : ub;
            jj[o] = ua < ub ? ub : ua;
        } else {
            ii[o] = ua;
            jj[o] = ub;
        }
        o++;
    });
}

void launch_dm_count(const MeshView& m, const NListView& nl, double dmax, int* counts, hipStream_t s)
{
    hipLaunchKernelGGL(k_dm_count, dim3((m.nv + 127) / 128), dim3(128), 0, s, m, nl, dmax, counts);
}

void launch_dm_fill(const MeshView& m, const NListView& nl, double dmax, const int* offsets, double* d, int* i,
                    int* j, hipStream_t s)
{
    hipLaunchKernelGGL(k_dm_fill, dim3((m.nv + 127) / 128), dim3(128), 0, s, m, nl, dmax, offsets, d, i, j);
}

// ------------------------------------------------------ point distances ---
// One vertex, in the reference's output order: stencil loops i (x), j (y),
// k (z) around the cell of the current position (cell_list.h:147-213), then
// ascending ids inside a cell; Verlet: adjacency order.
__global__ void k_point_distances(MeshView m, NListView nl, int pid, double dmax, int cap, int* count,
                                  double* dist3, int* jdx)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const Topo t = topo_of(m);
    const d3 p = t.P(pid);
    int c = 0;
    auto emit = [&](int j) {
        d3 d = p - t.P(j);
        if (norm(d) < dmax) {
            if (c < cap) {
                dist3[3 * c] = d.x;
                dist3[3 * c + 1] = d.y;
                dist3[3 * c + 2] = d.z;
                jdx[c] = nl.perm[j];
            }
            c++;
        }
    };
    if (nl.kind == 0) {
        int co[3];
        cell_coords(nl, p, co);
        for (int i = -1; i < 2; i++) {
            int ii = co[0] + i;
            if (ii < 0 || ii >= nl.shape[0]) continue;
            for (int j = -1; j < 2; j++) {
                int jj = co[1] + j;
                if (jj < 0 || jj >= nl.shape[1]) continue;
                for (int k = -1; k < 2; k++) {
                    int kk = co[2] + k;
                    if (kk < 0 || kk >= nl.shape[2]) continue;
                    int oc = ii * nl.strides[0] + jj * nl.strides[1] + kk * nl.strides[2];
                    for (int q = nl.cell_start[oc]; q < nl.cell_start[oc + 1]; q++) {
                        int jid = nl.cell_verts[q];
                        if (om_excluded(t, pid, jid, nl.exclusion)) continue;
                        emit(jid);
                    }
                }
            }
        }
    } else if (nl.kind == 1) {
        for (int q = nl.adj_start[pid]; q < nl.adj_start[pid + 1]; q++) emit(nl.adj[q]);
    }
    *count = c;
}

void launch_point_distances(const MeshView& m, const NListView& nl, int pid, double dmax, int cap, int* count,
                            double* dist3, int* jdx, hipStream_t s)
{
    hipLaunchKernelGGL(k_point_distances, dim3(1), dim3(64), 0, s, m, nl, pid, dmax, cap, count, dist3, jdx);
}

// --------------------------------------------------------- verlet build ---
// VerletList ctor (verlet_list.h:18-35): the symmetric adjacency of the cell
// list's distance_matrix(rlist) pairs.  Per vertex a: every b in the stencil
// of a's cell (either side of the cell ordering), not excluded, distance <=
// rlist; stored ascending.
template <class F>
__device__ __forceinline__ void verlet_visit(const MeshView& m, const NListView& nl, double rlist, int a, F&& f)
{
    const Topo t = topo_of(m);
    int ca = nl.vert_cell[a];
    int kc = ca / nl.strides[2];
    int rem = ca % nl.strides[2];
    int jc = rem / nl.strides[1];
    int ic = rem % nl.strides[1];
    for (int dk = -1; dk < 2; dk++) {
        int kk = kc + dk;
        if (kk < 0 || kk >= nl.shape[2]) continue;
        for (int dj = -1; dj < 2; dj++) {
            int jj = jc + dj;
            if (jj < 0 || jj >= nl.shape[1]) continue;
            int i0 = max(ic - 1, 0), i1 = min(ic + 1, nl.shape[0] - 1);
            int base = jj * nl.strides[1] + kk * nl.strides[2];
            for (int q = nl.cell_start[base + i0]; q < nl.cell_start[base + i1 + 1]; q++) {
                int b = nl.cell_verts[q];
                if (b == a) continue;
                if (dist_ab(m.x, a, b) <= rlist && !om_excluded(t, a, b, nl.exclusion)) f(b);
            }
        }
    }
}

__global__ void k_verlet_count(MeshView m, NListView nl, double rlist, int* __restrict__ counts)
{
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= m.nv) return;
    int c = 0;
    verlet_visit(m, nl, rlist, a, [&](int) { c++; });
    counts[a] = c;
}

__global__ void k_verlet_fill(MeshView m, NListView nl, double rlist, const int* __restrict__ offsets,
                              int* __restrict__ adj)
{
    int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= m.nv) return;
    int s = offsets[a];
    int o = s;
    verlet_visit(m, nl, rlist, a, [&](int b) { adj[o++] = b; });
    for (int p = s + 1; p < o; p++) {
        int key = adj[p];
        int q = p - 1;
        while (q >= s && adj[q] > key) {
            adj[q + 1] = adj[q];
            q--;
        }
        adj[q + 1] = key;
    }
}

void launch_verlet_count(const MeshView& m, const NListView& cl, double rlist, int* counts, hipStream_t s)
{
    hipLaunchKernelGGL(k_verlet_count, dim3((m.nv + 127) / 128), dim3(128), 0, s, m, cl, rlist, counts);
}

void launch_verlet_fill(const MeshView& m, const NListView& cl, double rlist, const int* offsets, int* adj,
                        hipStream_t s)
{
    hipLaunchKernelGGL(k_verlet_fill, dim3((m.nv + 127) / 128), dim3(128), 0, s, m, cl, rlist, offsets, adj);
}

}    // namespace tmh
