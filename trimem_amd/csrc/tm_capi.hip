// tm_capi.hip -- host side of libtrimem_hip: mesh construction, device
// buffers and the C ABI declared in include/trimem_hip.h.
//
// Every compute entry point enqueues gfx950 kernels on one library stream;
// there is no CPU compute path.  Host work is limited to building the
// half-edge arrays from a face list (OpenMesh add_face numbering), scalar
// parameter arithmetic, and copying inputs and results.
#include "../../include/trimem_hip.h"
#include "tm_internal.h"
#include "tm_last.h"
#include "tm_surrogate.h"

#include <cfloat>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <numeric>
#include <random>
#include <stdexcept>
#include <unordered_set>
#include <string>
#include <unordered_map>
#include <vector>

using namespace tmh;

// ------------------------------------------------------------- errors -----
namespace {

thread_local std::string g_err;

struct TmError : std::runtime_error {
    int code;
    TmError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define HIPCHECK(expr)                                                                             \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            throw TmError(TM_E_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));        \
    } while (0)

#define API_BEGIN try {
#define API_END                                          \
    }                                                    \
    catch (const TmError& ex) {                          \
        g_err = ex.what();                               \
        return ex.code;                                  \
    }                                                    \
    catch (const std::exception& ex) {                   \
        g_err = ex.what();                               \
        return TM_E_INVALID;                             \
    }                                                    \
    return TM_OK;

// ------------------------------------------------------------ runtime -----
// Scratch of tm_mesh_sum_noalloc: the arrival counter of its reduction (the
// first kNoAllocCounterBytes) and one partial sum per block of 256 faces or
// edges, in memory the library owns for the life of the process (one copy on
// every GPU it runs on), so that entry point allocates nothing.  Host code
// never passes this name to a kernel: it stands for a host-side shadow, and
// the device address comes from hipGetSymbolAddress (g_rt.scratch).
constexpr int kNoAllocMaxBlocks = 32768;                     // at most 32768 * 256 faces or edges
constexpr size_t kNoAllocCounterBytes = 256;
constexpr int kNoAllocScratchDoubles = kNoAllocCounterBytes / sizeof(double) + kNoAllocMaxBlocks;
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];
constexpr int kMaxDevices = 64;

constexpr size_t kRingPiece = 512 << 10;    // HostRing
constexpr int kRingPieces = 8;

struct Runtime {
    bool init = false;
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t arrived[kRingPieces] = {};    // HostRing's: events of the stream's device, whichever thread is first
    void* scratch[kMaxDevices] = {};    // device address of `scratch` on each device
    hipEvent_t pass1_marks[2] = {};     // tm_mark_pass1: taken by the next properties pass
};
Runtime g_rt;

void ensure_runtime()
{
    if (g_rt.init) return;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) throw TmError(TM_E_DEVICE, "no HIP device available");
    if (g_rt.device < 0 || g_rt.device >= n || g_rt.device >= kMaxDevices)
        throw TmError(TM_E_DEVICE, "device index out of range");
    HIPCHECK(hipSetDevice(g_rt.device));
    HIPCHECK(hipStreamCreateWithFlags(&g_rt.stream, hipStreamNonBlocking));
    for (hipEvent_t& e : g_rt.arrived) HIPCHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // the scratch array's address on this device, with the device current
    void* sp = nullptr;
    HIPCHECK(hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)));
    if (!sp) throw TmError(TM_E_DEVICE, "no device address for the library scratch");
    g_rt.scratch[g_rt.device] = sp;
    g_rt.init = true;
}

template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    void alloc(size_t count)
    {
        if (count <= n && p) return;
        release();
        size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
        HIPCHECK(hipMalloc((void**)&p, bytes));
        n = count;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    ~DevBuf() { release(); }
};

void h2d(void* d, const void* h, size_t bytes)
{
    if (bytes) HIPCHECK(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, g_rt.stream));
}
void d2h(void* h, const void* d, size_t bytes)
{
    if (bytes) HIPCHECK(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, g_rt.stream));
}
void sync() { HIPCHECK(hipStreamSynchronize(g_rt.stream)); }
void check_launch() { HIPCHECK(hipGetLastError()); }

// Pinned memory that kernels read and write (coherent: neither side caches it).
template <class T>
struct HostBuf {
    T* p = nullptr;
    void alloc(size_t count)
    {
        if (!p) HIPCHECK(hipHostMalloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T), hipHostMallocCoherent));
    }
    ~HostBuf()
    {
        if (p) (void)hipHostFree(p);
    }
};

// Rows of a device result into the caller's memory.  Kernels write pieces into
// a small pinned ring, and the host copies a piece on while the next ones
// arrive: the link and the host's copy overlap, and no result needs a device
// buffer in its own order or a pinned one of its size.  One ring for the
// process, its pieces written in stream order; the lock is held until the last
// piece has been copied.  A gradient of 163842 vertices takes 250 us with 8 pieces
// of 512 KB, 266 with 4, 283 and 304 with 8 and 4 of 256 KB (a wait per piece),
// 299 with 2 of 2 MB (no overlap); one copy into pageable memory took 404.
struct HostRing {
    std::mutex lock;
    HostBuf<char> buf;
};
HostRing& host_ring()
{
    static HostRing* ring = new HostRing;    // for the life of the process
    return *ring;
}
// piece(p, first, n): enqueue the kernel that writes rows first .. first + n - 1 to p
template <class F>
void to_host(void* dst, size_t rows, size_t row_bytes, F&& piece)
{
    if (rows == 0) return;
    HostRing& R = host_ring();
    std::lock_guard<std::mutex> guard(R.lock);
    R.buf.alloc(kRingPiece * kRingPieces);
    const size_t per = kRingPiece / row_bytes, pieces = (rows + per - 1) / per;
    auto slot = [&](size_t k) { return R.buf.p + (k % kRingPieces) * kRingPiece; };
    auto start = [&](size_t k) {
        piece(slot(k), (int)(k * per), (int)std::min(per, rows - k * per));
        check_launch();
        if (pieces > 1) HIPCHECK(hipEventRecord(g_rt.arrived[k % kRingPieces], g_rt.stream));
    };
    for (size_t k = 0; k < std::min<size_t>(pieces, kRingPieces); k++) start(k);
    for (size_t k = 0; k < pieces; k++) {
        if (pieces > 1) HIPCHECK(hipEventSynchronize(g_rt.arrived[k % kRingPieces]));
        else sync();
        std::memcpy((char*)dst + k * per * row_bytes, slot(k), std::min(per, rows - k * per) * row_bytes);
        if (k + kRingPieces < pieces) start(k + kRingPieces);
    }
}

}    // namespace

// --------------------------------------------------------------- mesh -----
struct tm_mesh {
    int nv = 0, nh = 0, nf = 0;
    double* points = nullptr;    // host (N,3), pinned when a device exists
    bool pinned = false;
    // host mirror of the topology
    std::vector<int> he_to, he_next, he_prev, he_face, v_he, f_he;
    bool host_stale = false;     // device topology changed (flips)
    bool faces_read = false;     // ... and its faces have been read since
    void flipped()
    {
        host_stale = true;
        faces_read = false;
    }
    bool device_ahead = false;   // device positions moved by a device-resident step
    unsigned topo_version = 0;   // bumped by every topology change (flips)
    bool has_boundary = false;
    // device state
    bool dev = false;
    DevBuf<double> x;
    DevBuf<int> d_to, d_next, d_prev, d_face, d_vhe, d_fhe, ring, meta;
    // what the host waits for after a sweep
    struct Report {
        int overflow;         // a vertex has more neighbours than the ring table has columns
        SerialState serial;
        double parallel[8];
    };
    HostBuf<Report> report;
    // vertices evaluated by the half-edge walker: boundary, isolated or with
    // fewer than three neighbours (flips preserve this set on valid meshes)
    DevBuf<int> generic;
    int n_generic = 0;
    // the sweeps' rows (FlipRows), allocated by the first sweep and rebuilt by each
    DevBuf<int> flip_nb;
    DevBuf<int2> flip_er;
    // Internal vertex order (Morton order of the creation-time positions):
    // perm[i] = user id of internal vertex i, iperm[u] = internal id of user
    // vertex u.  Topology and device arrays use internal ids; every id or
    // per-vertex row that crosses the API is mapped back to user ids.
    std::vector<int> perm, iperm;
    DevBuf<int> d_perm, d_iperm;
    DevBuf<double> stage;    // user-order rows on their way into internal order

    MeshView view() const
    {
        return MeshView{x.p, d_to.p, d_next.p, d_prev.p, d_face.p, d_vhe.p, d_fhe.p, ring.p, meta.p, nv, nh, nf};
    }
    FlipMeshView flip_view()
    {
        return FlipMeshView{x.p, d_to.p, d_next.p, d_prev.p, d_face.p, d_vhe.p, d_fhe.p, nv, nh, nf};
    }
    FlipRows flip_rows(bool edges)
    {
        const size_t n = (size_t)kMaxValence * nv;
        flip_nb.alloc(n);
        if (edges) flip_er.alloc(n);
        return FlipRows{flip_nb.p, edges ? flip_er.p : nullptr};
    }
    ~tm_mesh()
    {
        if (points) {
            if (pinned) (void)hipHostFree(points);
            else std::free(points);
        }
    }
};

namespace {

// Face list -> half-edge arrays with OpenMesh's numbering
// (PolyConnectivity::add_face as used by from_points_cells, mesh_py.cpp:53-67):
// face ids outside [0, n) are dropped, faces with fewer than three valid ids
// are skipped, a new edge e gets halfedge 2e = v_i -> v_{i+1}, the face's
// halfedge is v_2 -> v_0, and faces that would create a complex vertex (one
// whose fan is already closed) or a complex edge (a halfedge that already has
// a face) are rejected.  Remaining boundary halfedges are linked into loops
// and boundary vertices point at their boundary outgoing halfedge.
void build_topology(tm_mesh& M, const int* faces, int m)
{
    const int n = M.nv;
    M.v_he.assign(n, -1);
    M.he_to.clear(); M.he_next.clear(); M.he_prev.clear(); M.he_face.clear(); M.f_he.clear();
    if (n < 3 || m == 0) return;
    std::unordered_map<uint64_t, int> he_of;
    he_of.reserve((size_t)m * 4);
    auto key = [](int a, int b) { return ((uint64_t)(uint32_t)a << 32) | (uint32_t)b; };
    std::vector<int> n_out(n, 0), n_bout(n, 0);
    for (int f = 0; f < m; f++) {
        int vh[3], nvh = 0;
        for (int j = 0; j < 3; j++) {
            int c = faces[3 * f + j];
            if (c >= 0 && c < n) vh[nvh++] = c;
        }
        if (nvh < 3) continue;
        int hh[3];
        bool ok = true;
        for (int i = 0; i < 3 && ok; i++) {
            int a = vh[i], b = vh[(i + 1) % 3];
            if (n_out[a] > 0 && n_bout[a] == 0) ok = false;
            auto it = he_of.find(key(a, b));
            hh[i] = it == he_of.end() ? -1 : it->second;
            if (hh[i] >= 0 && M.he_face[hh[i]] >= 0) ok = false;
        }
        if (!ok) continue;
        int fid = (int)M.f_he.size();
        for (int i = 0; i < 3; i++) {
            if (hh[i] >= 0) continue;
            int a = vh[i], b = vh[(i + 1) % 3];
            int e = (int)M.he_to.size() / 2;
            M.he_to.push_back(b); M.he_to.push_back(a);
            M.he_next.push_back(-1); M.he_next.push_back(-1);
            M.he_prev.push_back(-1); M.he_prev.push_back(-1);
            M.he_face.push_back(-1); M.he_face.push_back(-1);
            he_of[key(a, b)] = 2 * e;
            he_of[key(b, a)] = 2 * e + 1;
            hh[i] = 2 * e;
            n_out[a]++; n_bout[a]++;
            n_out[b]++; n_bout[b]++;
            if (M.v_he[a] < 0) M.v_he[a] = 2 * e;
            if (M.v_he[b] < 0) M.v_he[b] = 2 * e + 1;
        }
        for (int i = 0; i < 3; i++) {
            M.he_face[hh[i]] = fid;
            M.he_next[hh[i]] = hh[(i + 1) % 3];
            M.he_prev[hh[(i + 1) % 3]] = hh[i];
            n_bout[vh[i]]--;
        }
        M.f_he.push_back(hh[2]);
    }
    const int nh = (int)M.he_to.size();
    std::vector<int> bout(n, -1);
    for (int h = 0; h < nh; h++)
        if (M.he_face[h] < 0) bout[M.he_to[h ^ 1]] = h;
    for (int h = 0; h < nh; h++) {
        if (M.he_face[h] < 0) {
            int nx = bout[M.he_to[h]];
            M.he_next[h] = nx;
            if (nx >= 0) M.he_prev[nx] = h;
        }
    }
    M.has_boundary = false;
    for (int v = 0; v < n; v++) {
        if (bout[v] >= 0) {
            M.v_he[v] = bout[v];
            M.has_boundary = true;
        }
    }
    M.nh = nh;
    M.nf = (int)M.f_he.size();
}

// Morton (Z-order) key of each vertex on a 1024^3 grid over the bounding box,
// ties broken by id; vertices close in space get close internal ids, which
// keeps the gathers of one wavefront in few cache lines.
void reorder_vertices(tm_mesh& M)
{
    const int n = M.nv;
    M.perm.resize(n);
    M.iperm.resize(n);
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int v = 0; v < n; v++)
        for (int k = 0; k < 3; k++) {
            double c = M.points[3 * v + k];
            if (c < lo[k]) lo[k] = c;
            if (c > hi[k]) hi[k] = c;
        }
    auto spread = [](uint64_t x) {
        x &= 0x3ff;
        x = (x | (x << 16)) & 0x030000ffull;
        x = (x | (x << 8)) & 0x0300f00full;
        x = (x | (x << 4)) & 0x030c30c3ull;
        x = (x | (x << 2)) & 0x09249249ull;
        return x;
    };
    std::vector<uint64_t> key(n);
    for (int v = 0; v < n; v++) {
        uint64_t code = 0;
        for (int k = 0; k < 3; k++) {
            double span = hi[k] - lo[k];
            double t = span > 0 ? (M.points[3 * v + k] - lo[k]) / span : 0.0;
            if (!(t >= 0)) t = 0;    // also catches NaN
            if (t > 1) t = 1;
            code |= spread((uint64_t)(t * 1023.0)) << k;
        }
        key[v] = (code << 32) | (uint32_t)v;
    }
    std::sort(key.begin(), key.end());
    for (int i = 0; i < n; i++) {
        M.perm[i] = (int)(key[i] & 0xffffffffu);
        M.iperm[M.perm[i]] = i;
    }
    for (int h = 0; h < M.nh; h++) M.he_to[h] = M.iperm[M.he_to[h]];
    std::vector<int> vhe(n);
    for (int i = 0; i < n; i++) vhe[i] = M.v_he[M.perm[i]];
    M.v_he.swap(vhe);
}

// the ring table of the current half-edge arrays; report->overflow is set when
// this has run
void queue_ring(tm_mesh& M)
{
    M.report.p->overflow = 0;
    launch_build_ring(M.view(), M.ring.p, M.meta.p, &M.report.p->overflow, g_rt.stream);
    check_launch();
}

void ensure_device(tm_mesh& M)
{
    ensure_runtime();
    if (M.dev) return;
    M.x.alloc((size_t)M.nv * 3);
    M.d_to.alloc(M.nh);
    M.d_next.alloc(M.nh);
    M.d_prev.alloc(M.nh);
    M.d_face.alloc(M.nh);
    M.d_vhe.alloc(M.nv);
    M.d_fhe.alloc(M.nf);
    M.ring.alloc((size_t)kMaxValence * M.nv);
    M.meta.alloc(M.nv);
    M.d_perm.alloc(M.nv);
    M.d_iperm.alloc(M.nv);
    M.stage.alloc((size_t)M.nv * 3);
    h2d(M.d_perm.p, M.perm.data(), sizeof(int) * M.nv);
    h2d(M.d_iperm.p, M.iperm.data(), sizeof(int) * M.nv);
    M.report.alloc(1);
    h2d(M.d_to.p, M.he_to.data(), sizeof(int) * M.nh);
    h2d(M.d_next.p, M.he_next.data(), sizeof(int) * M.nh);
    h2d(M.d_prev.p, M.he_prev.data(), sizeof(int) * M.nh);
    h2d(M.d_face.p, M.he_face.data(), sizeof(int) * M.nh);
    h2d(M.d_vhe.p, M.v_he.data(), sizeof(int) * M.nv);
    h2d(M.d_fhe.p, M.f_he.data(), sizeof(int) * M.nf);
    std::vector<int> gl;
    for (int v = 0; v < M.nv; v++) {
        int h0 = M.v_he[v];
        if (h0 < 0 || M.he_face[h0] < 0) {
            gl.push_back(v);
            continue;
        }
        int n = 0, h = h0;
        do {
            n++;
            h = M.he_next[h ^ 1];
        } while (h != h0 && n < 4);
        if (n < 3) gl.push_back(v);
    }
    M.n_generic = (int)gl.size();
    M.generic.alloc(std::max<size_t>(gl.size(), 1));
    h2d(M.generic.p, gl.data(), sizeof(int) * gl.size());
    queue_ring(M);
    sync();
    if (M.report.p->overflow) throw TmError(TM_E_UNSUPPORTED, "vertex valence exceeds the ring-table width (32)");
    M.dev = true;
}

// Below this many vertices a kernel reads the pinned positions itself, above it
// the copy engine, which starts later and needs a kernel to reorder after it, is
// ahead (49 GB/s over the link, the kernel 41): an upload takes 12.7 us by the
// kernel and 14.7 by the engine at 642 vertices, 34.9 and 37.5 at 40962, 58.1 and
// 54.8 at 81002, 105 and 91 at 163842.
constexpr int kTakeVerts = 65536;

// three doubles per vertex from host memory, in internal order
void upload_rows(tm_mesh& M, const double* host, double* dst)
{
    h2d(M.stage.p, host, sizeof(double) * 3 * M.nv);
    launch_gather_rows(M.stage.p, M.d_perm.p, dst, M.nv, 3, g_rt.stream);
}

void push_points(tm_mesh& M)
{
    ensure_device(M);
    M.device_ahead = false;
    if (M.nv == 0) return;
    if (M.pinned && M.nv < kTakeVerts) launch_take_points(M.points, M.d_iperm.p, M.x.p, M.nv, g_rt.stream);
    else upload_rows(M, M.points, M.x.p);
    check_launch();
}

// Host-facing calls take positions from the host array (the reference's
// points() view, mesh_py.cpp:96-105).  When a device-resident step has moved
// the device copy since, the device holds the newer state and is used as it
// is; the host array is refreshed only when it is read (tm_mesh_sync_host).
void upload_points(tm_mesh& M)
{
    ensure_device(M);
    if (!M.device_ahead) push_points(M);
}

// rows of an internal-order device array -> user order on the host, there when
// this returns
void download_rows(tm_mesh& M, const double* d_src, int width, double* host)
{
    to_host(host, M.nv, sizeof(double) * width, [&](void* p, int first, int n) {
        launch_give_rows(d_src, M.d_iperm.p, (double*)p, first, n, width, g_rt.stream);
    });
}

void pull_points(tm_mesh& M)
{
    if (M.pinned) {
        launch_give_rows(M.x.p, M.d_iperm.p, M.points, 0, M.nv, 3, g_rt.stream);
        check_launch();
        sync();
    } else {
        download_rows(M, M.x.p, 3, M.points);
    }
    M.device_ahead = false;
}

void refresh_host_topology(tm_mesh& M)
{
    if (!M.host_stale) return;
    struct {
        std::vector<int>& host;
        const int* dev;
    } a[] = {{M.he_to, M.d_to.p},     {M.he_next, M.d_next.p}, {M.he_prev, M.d_prev.p},
             {M.he_face, M.d_face.p}, {M.v_he, M.d_vhe.p},     {M.f_he, M.d_fhe.p}};
    size_t bytes = 0;
    for (auto& x : a) bytes += sizeof(int) * x.host.size();
    HostRing& R = host_ring();
    if (bytes <= kRingPiece * kRingPieces) {
        // through pinned memory with one wait (each copy to pageable memory waits)
        std::lock_guard<std::mutex> guard(R.lock);
        R.buf.alloc(kRingPiece * kRingPieces);
        char* at = R.buf.p;
        for (auto& x : a) {
            d2h(at, x.dev, sizeof(int) * x.host.size());
            at += sizeof(int) * x.host.size();
        }
        sync();
        at = R.buf.p;
        for (auto& x : a) {
            std::memcpy(x.host.data(), at, sizeof(int) * x.host.size());
            at += sizeof(int) * x.host.size();
        }
    } else {
        for (auto& x : a) d2h(x.host.data(), x.dev, sizeof(int) * x.host.size());
        sync();
    }
    M.host_stale = false;
}

}    // namespace

// ---------------------------------------------------------- nlist ---------
struct tm_nlist {
    int kind = 0;    // 0 cell, 1 verlet
    int exclusion = 0;
    double rlist = 0.1;
    NListView v{};
    DevBuf<int> cell_start, cell_verts, vert_cell, counts, place, scan_tmp, adj_start, adj, adj_counts;
    DevBuf<int> cand_count, cand_start, cand;
    DevBuf<int2> vcand;
    DevBuf<unsigned long long> excl_mask;
    unsigned mask_topo = ~0u;    // topology version the masks were built for
    // pair cache of the query (PairCache): recorded lists, valid for this
    // list and topology once a recording launch has been queued
    DevBuf<double> pc_x, pc_disp;
    DevBuf<int> pc_fast, pc_streak;
    DevBuf<int> pc_cell, pc_ent;
    DevBuf<unsigned> pc_cnt;
    bool pc_ok = false;
    // distance-matrix scratch
    DevBuf<int> dm_counts, dm_off;
    DevBuf<double> dm_d;
    DevBuf<int> dm_i, dm_j;
    DevBuf<double> pd_dist;
    DevBuf<int> pd_j, pd_count;
    int nv = 0;
    NListView view() const { return v; }
};

namespace {

// (Re)build the exclusion masks of a cell list when the mesh topology has
// changed since they were built; the view carries them only while valid.
void ensure_masks(tm_nlist& L, tm_mesh& M)
{
    if (L.kind != 0 || !L.excl_mask.p || M.nv == 0) return;
    if (L.mask_topo != M.topo_version) {
        NListView nv = L.v;
        nv.excl_mask = nullptr;
        launch_excl_mask(M.view(), nv, L.excl_mask.p, g_rt.stream);
        check_launch();
        L.mask_topo = M.topo_version;
        L.pc_ok = false;    // exclusion may have changed
    }
    L.v.excl_mask = L.excl_mask.p;
}

void scan(const int* in, int* out, int n, DevBuf<int>& tmp)
{
    tmp.alloc(scan_block_sums_size(n) + 1);
    launch_exclusive_scan(in, out, n, tmp.p, g_rt.stream);
    check_launch();
}

// the Verlet adjacency from the cells of its list
void build_verlet(tm_nlist& L, tm_mesh& M)
{
    const int n = M.nv;
    NListView& v = L.v;
    L.adj_counts.alloc(n + 1);
    L.adj_start.alloc(n + 1);
    HIPCHECK(hipMemsetAsync(L.adj_counts.p, 0, sizeof(int) * (n + 1), g_rt.stream));
    launch_verlet_count(M.view(), v, L.rlist, L.adj_counts.p, g_rt.stream);
    check_launch();
    scan(L.adj_counts.p, L.adj_start.p, n + 1, L.scan_tmp);
    int total = 0;
    d2h(&total, L.adj_start.p + n, sizeof(int));
    sync();
    L.adj.alloc(total);
    launch_verlet_fill(M.view(), v, L.rlist, L.adj_start.p, L.adj.p, g_rt.stream);
    check_launch();
    v.kind = 1;
    v.adj_start = L.adj_start.p;
    v.adj = L.adj.p;
}

// The grid of a list from the box partials of its vertices; returns the number of
// cells.
long long nlist_grid(tm_nlist& L, int n, const double* part)
{
    const int nbox = box_scratch_doubles();
    double tight[6] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX};    // the vertices' own box
    for (int b = 0; b < nbox / 6; b++)
        for (int k = 0; k < 3; k++) {
            tight[k] = std::fmin(tight[k], part[6 * b + k]);
            tight[3 + k] = std::fmax(tight[3 + k], part[6 * b + 3 + k]);
        }
    // the reference's box (cell_list.h:46-56): its bounds start at min =
    // (+max, 0, 0) and max = (-1, 0, 0), so it spans 0 in y and z
    double box[6];
    for (int k = 0; k < 3; k++) {
        box[k] = k == 0 ? tight[0] : std::min(0.0, tight[k]);
        box[3 + k] = std::max(k == 0 ? -1.0 : 0.0, tight[3 + k]);
    }
    const double box_eps = 1.0e-6;
    NListView v{};
    v.kind = 0;
    v.exclusion = L.exclusion;
    long long ncells = 1;
    for (int k = 0; k < 3; k++) {
        if (n == 0) {
            v.box_min[k] = 0.0;
            v.r_list[k] = 1.0;
            v.lo[k] = 0;
            v.shape[k] = 1;
            continue;
        }
        const double dim = box[3 + k] - box[k] + box_eps;
        const double q = dim / L.rlist;
        if (!(q < 1073741824.0))
            throw TmError(TM_E_UNSUPPORTED, "cell grid too fine along axis " + std::to_string(k) + " (" +
                                                std::to_string(q) + " cells); coordinates must be finite");
        const int nk = int(q);
        const int gk = (nk > 0) ? nk : 1;
        v.box_min[k] = box[k];
        v.r_list[k] = (nk > 0) ? dim / nk : dim;
        // global cells of the lowest and highest vertex; the cell index is
        // monotone in the coordinate, so they bound every vertex's cell
        auto cell = [&](double p) { return std::min(std::max(int((p - box[k]) / v.r_list[k]), 0), gk - 1); };
        v.lo[k] = cell(tight[k]);
        v.shape[k] = cell(tight[3 + k]) - v.lo[k] + 1;
        ncells *= v.shape[k];
    }
    if (ncells > (1ll << 28))
        throw TmError(TM_E_UNSUPPORTED, "occupied cell sub-grid too large (" + std::to_string(ncells) +
                                            " cells): the mesh spans more than 2^28 cells of size rlist");
    v.strides[0] = 1;
    v.strides[1] = v.shape[0];
    v.strides[2] = v.shape[0] * v.shape[1];
    L.v = v;
    return ncells;
}

// CellList ctor (cell_list.h:43-87) and, for kind 1, VerletList ctor
// (verlet_list.h:18-35), on the meshes' current device positions, of up to
// kBuildLists distinct lists together: one round trip for all boxes (in the ring),
// then one launch of each kind for all.
constexpr size_t kBuildLists = 1024;
struct NlistJob {
    tm_nlist* L;
    tm_mesh* M;
};
struct NlistTables {    // a build's arguments, and on the device those of several lists
    std::vector<NlistBuild> h;
    std::vector<int> h_block0;
    DevBuf<NlistBuild> builds;
    DevBuf<int> block0;
};
void build_nlists(const std::vector<NlistJob>& jobs, NlistTables& T)
{
    const int R = (int)jobs.size();
    if (R == 0) return;
    std::vector<NlistBuild>& h = T.h;
    std::vector<int>& block0 = T.h_block0;
    h.assign(R, NlistBuild{});
    block0.resize((size_t)kShapes * (R + 1));
    NlistGroup g{h.data(), R, nullptr, nullptr, {}};
    for (int r = 0; r < R; r++) {
        tm_nlist& L = *jobs[r].L;
        if (!(L.rlist > 0) || !std::isfinite(L.rlist)) throw TmError(TM_E_INVALID, "rlist must be positive");
        L.nv = jobs[r].M->nv;
        h[r].x = jobs[r].M->x.p;
        h[r].n = L.nv;
    }
    auto tabulate = [&]() {
        for (int k = 0; k < kShapes; k++) {
            int* b0 = block0.data() + (size_t)k * (R + 1);
            b0[0] = 0;
            for (int r = 0; r < R; r++) b0[r + 1] = b0[r] + nlist_blocks(h[r], k);
            g.total[k] = b0[R];
        }
        if (R == 1) return;
        T.builds.alloc(R);
        T.block0.alloc(block0.size());
        h2d(T.builds.p, h.data(), sizeof(NlistBuild) * R);
        h2d(T.block0.p, block0.data(), sizeof(int) * block0.size());
        g.d = T.builds.p;
        g.block0 = T.block0.p;
    };
    {
        const size_t nbox = box_scratch_doubles();
        HostRing& ring = host_ring();
        std::lock_guard<std::mutex> guard(ring.lock);
        ring.buf.alloc(kRingPiece * kRingPieces);
        if (nbox * sizeof(double) * R > kRingPiece * kRingPieces) throw TmError(TM_E_INVALID, "too many lists");
        double* box = reinterpret_cast<double*>(ring.buf.p);
        for (int r = 0; r < R; r++) h[r].box = box + nbox * r;
        tabulate();
        launch_nlist_box(g, g_rt.stream);
        check_launch();
        sync();
        for (int r = 0; r < R; r++) {
            const long long ncells = nlist_grid(*jobs[r].L, jobs[r].M->nv, h[r].box);
            h[r].nc = (int)ncells;
        }
    }
    for (int r = 0; r < R; r++) {
        tm_nlist& L = *jobs[r].L;
        tm_mesh& M = *jobs[r].M;
        const int n = M.nv, nc = h[r].nc;
        NlistBuild& b = h[r];
        L.counts.alloc(nc + 1);
        L.cell_start.alloc(nc + 1);
        L.place.alloc(n);
        L.vert_cell.alloc(n);
        L.cell_verts.alloc(n);
        L.scan_tmp.alloc(scan_block_sums_size(std::max(n, nc) + 1) + 1);
        b.perm = M.d_perm.p;
        b.m = M.view();
        b.counts = L.counts.p;
        b.cell_start = L.cell_start.p;
        b.vert_cell = L.vert_cell.p;
        b.place = L.place.p;
        b.cell_verts = L.cell_verts.p;
        b.sums = L.scan_tmp.p;
        L.v.cell_start = L.cell_start.p;
        L.v.cell_verts = L.cell_verts.p;
        L.v.vert_cell = L.vert_cell.p;
        L.v.perm = M.d_perm.p;
        if (L.kind == 0 && n > 0) {
            if ((long long)27 * n > INT_MAX) throw TmError(TM_E_UNSUPPORTED, "mesh too large for the candidate table");
            L.cand_count.alloc(n + 1);
            L.cand_start.alloc(n + 1);
            // a vertex is in the stencil lists of at most 27 cells: 27 N bounds
            // the total without reading it back
            L.cand.alloc((size_t)27 * n);
            L.vcand.alloc(n);
            L.excl_mask.alloc((size_t)2 * n);
            L.pc_x.alloc((size_t)3 * n);
            L.pc_cell.alloc(n);
            L.pc_streak.alloc(2);
            L.pc_cnt.alloc(n);
            L.pc_ent.alloc((size_t)kPairLanes * kPairCap * n);
            L.pc_disp.alloc(pass1_blocks(n));    // one displacement partial per pass-1 block
            L.pc_fast.alloc((size_t)kFastRow * pass1_blocks(n));
            b.cand_count = L.cand_count.p;
            b.cand_start = L.cand_start.p;
            b.cand = L.cand.p;
            b.vcand = L.vcand.p;
            b.mask = L.excl_mask.p;
            b.pc_cell = L.pc_cell.p;
            b.pc_streak = L.pc_streak.p;
            L.v.vcand = L.vcand.p;
            L.v.cand = L.cand.p;
            L.v.cand_start = L.cand_start.p;
        }
        b.nl = L.v;    // masks not set: they are what the build makes
    }
    tabulate();
    launch_nlist_build(g, g_rt.stream);
    check_launch();
    for (int r = 0; r < R; r++) {
        tm_nlist& L = *jobs[r].L;
        tm_mesh& M = *jobs[r].M;
        if (L.kind == 1) build_verlet(L, M);
        if (L.kind == 0 && M.nv > 0) {
            L.mask_topo = M.topo_version;
            L.v.excl_mask = L.excl_mask.p;
            L.pc_ok = false;
        }
    }
    // no wait here: everything that reads the lists is queued behind them on the
    // library stream (the host already waited once, for the bounding boxes)
}

void build_nlist(tm_nlist& L, tm_mesh& M)
{
    NlistTables one;
    build_nlists({NlistJob{&L, &M}}, one);
}

void check_params(const tm_params& p)
{
    if (p.bond_type != 0 && p.bond_type != 1) throw TmError(TM_E_INVALID, "Unknown bond potential");
    if (p.rep_nlist != 0 && p.rep_nlist != 1) throw TmError(TM_E_INVALID, "Unknown neighbour search algorithm.");
    if (p.rep_exclusion < 0 || p.rep_exclusion > 2) throw TmError(TM_E_INVALID, "Unsupported exclusion level");
}

tm_nlist* make_nlist(tm_mesh& M, const tm_params& p)
{
    check_params(p);
    auto L = std::make_unique<tm_nlist>();
    L->kind = p.rep_nlist;
    L->exclusion = p.rep_exclusion;
    L->rlist = p.rep_rlist;
    build_nlist(*L, M);
    return L.release();
}

}    // namespace

// --------------------------------------------------------- energy ---------
struct tm_energy {
    tm_params params{};
    tm_props initial{};
    int precision = TM_PREC_FP64;
    tm_nlist* nlist = nullptr;
    int nv = 0;
    DevBuf<double> q, partials, grad, vprops, gprops;
    DevBuf<int> pair_cnt;
    DevBuf<double> rep_v, rep_g;
    DevBuf<unsigned> pass_count;
    DevBuf<double> theta;    // pass 1's dihedral angles for pass 2 (kRingPad per vertex, float or double)
    DevBuf<Globals> globals;
    HostBuf<Globals> host_globals;    // written by the passes whose sums the host waits for
    DevBuf<int> flip_result, proposals, pf_rec, pf_lost;
    DevBuf<double> uniforms, pf_state;
    DevBuf<unsigned> pf_count;
    double pf_last[8] = {};    // pf_state at the end of the last parallel sweep (tm_energy_pflip_state)
    DevBuf<unsigned long long> pf_owner;
    DevBuf<SerialState> sf_state;
    DevBuf<int> sf_rec;
    DevBuf<unsigned long long> sf_fstamp;
    Tuning tune;
    tm_nlist* spare = nullptr;    // the previous list, rebuilt in place by update_repulsion
    // bumped whenever something a replica group copies into its device
    // table changes: the neighbour list, the reference values, the precision
    unsigned gen = 0;
    ~tm_energy()
    {
        delete nlist;
        delete spare;
    }
};

namespace {

EParams eparams_of(const tm_energy& E)
{
    const tm_params& P = E.params;
    EParams p{};
    p.kappa_b = P.kappa_b; p.kappa_a = P.kappa_a; p.kappa_v = P.kappa_v;
    p.kappa_c = P.kappa_c; p.kappa_t = P.kappa_t; p.kappa_r = P.kappa_r;
    p.bond_lc0 = P.bond_lc0; p.bond_lc1 = P.bond_lc1; p.bond_a0 = P.bond_a0;
    p.bond_r = P.bond_r; p.bond_type = P.bond_type;
    p.rep_lc1 = P.rep_lc1; p.rep_r = P.rep_r; p.rep_exclusion = P.rep_exclusion;
    // interpolate_reference_properties (energy.cpp:30-45)
    double lam = P.cont_lambda;
    p.ref_area = (1.0 - lam * (1.0 - P.area_frac)) * E.initial.area;
    p.ref_volume = (1.0 - lam * (1.0 - P.volume_frac)) * E.initial.volume;
    p.ref_curvature = (1.0 - lam * (1.0 - P.curvature_frac)) * E.initial.curvature;
    return p;
}

// the counters of `passes` properties passes, zero between launches
void alloc_pass_count(DevBuf<unsigned>& c, int passes = 1)
{
    c.alloc((size_t)kLastCounters * passes);
    launch_fill_ints(reinterpret_cast<int*>(c.p), kLastCounters * passes, 0, nullptr, 0, 0, nullptr, 0, 0,
                     g_rt.stream);
    check_launch();
}

void ensure_energy_buffers(tm_energy& E, const tm_mesh& M)
{
    if (E.nv == M.nv && E.q.p) return;
    E.nv = M.nv;
    E.q.alloc(M.nv);
    E.gprops.alloc((size_t)M.nv * 6);
    E.pair_cnt.alloc(M.nv);
    HIPCHECK(hipMemsetAsync(E.pair_cnt.p, 0, sizeof(int) * M.nv, g_rt.stream));
    E.rep_v.alloc(M.nv);
    E.rep_g.alloc((size_t)M.nv * 3);
    E.partials.alloc((size_t)pass1_blocks(M.nv) * 6);
    E.grad.alloc((size_t)M.nv * 3);
    E.theta.alloc((size_t)kRingPad * M.nv);
    E.globals.alloc(1);
    E.host_globals.alloc(1);
    alloc_pass_count(E.pass_count);
    E.flip_result.alloc(4);
}

// update_repulsion (energy.cpp:57-61) without new device allocations: the
// list is built into the energy manager's spare, whose buffers remain from
// the rebuild before, and swapped in only when complete, so a failed build
// leaves the current list in place.
tm_nlist& spare_nlist(tm_energy& E)
{
    check_params(E.params);
    if (!E.spare) E.spare = new tm_nlist();
    tm_nlist& L = *E.spare;
    L.kind = E.params.rep_nlist;
    L.exclusion = E.params.rep_exclusion;
    L.rlist = E.params.rep_rlist;
    return L;
}
void take_spare(tm_energy& E)
{
    std::swap(E.nlist, E.spare);
    E.gen++;
}
void rebuild_nlist(tm_energy& E, tm_mesh& M)
{
    build_nlist(spare_nlist(E), M);
    take_spare(E);
}

// the list's count of evaluations in a row with fast vertices (null: none kept)
int* streak_of(tm_energy* E)
{
    return E && E->tune.pair_cache && E->nlist && E->nlist->kind == 0 ? E->nlist->pc_streak.p : nullptr;
}

// The pair-cache buffers of the energy manager's cell list (x_snap null when
// it has none: a Verlet list, or no repulsion); the caller adds the
// displacement partials and the recording flag.
PairCache pair_cache_of(tm_energy& E, tm_mesh& M)
{
    PairCache pc{};
    tm_nlist& L = *E.nlist;
    if (L.kind == 0 && L.pc_x.p && L.nv == M.nv && E.params.rep_lc1 > 0) {
        const double skin = kPairSkin * E.params.rep_lc1;
        pc.x_snap = L.pc_x.p;
        pc.cell = L.pc_cell.p;
        pc.cnt = L.pc_cnt.p;
        pc.ent = L.pc_ent.p;
        pc.streak = L.pc_streak.p;
        pc.skin = skin;
        pc.limit2 = (kPairLimit * skin) * (kPairLimit * skin);
    }
    return pc;
}

PassBuffers buffers(tm_energy& E, tm_mesh& M)
{
    PassBuffers b{};
    b.q = E.q.p;
    b.gprops = E.gprops.p;
    b.pair_cnt = E.pair_cnt.p;
    b.rep_v = E.rep_v.p;
    b.rep_g = E.rep_g.p;
    b.partials = E.partials.p;
    b.count = E.pass_count.p;
    b.globals = E.globals.p;
    b.theta = E.theta.p;
    b.list = M.generic.p;
    b.nlist = M.n_generic;
    tm_nlist& L = *E.nlist;
    if (E.tune.pair_cache) {
        b.pc = pair_cache_of(E, M);
        if (b.pc.x_snap) {
            b.pc.disp_part = L.pc_disp.p;
            b.pc.fast = L.pc_fast.p;
            b.pc.disp_n = pass1_blocks(M.nv);
            b.pc.force = L.pc_ok ? 0 : 1;
        }
    }
    return b;
}

// to_host: the sums also go to E.host_globals (read_globals)
void run_pass1(tm_energy& E, tm_mesh& M, int mixed, double* vprops, bool to_host = false)
{
    ensure_energy_buffers(E, M);
    if (E.nlist->nv != M.nv) throw TmError(TM_E_INVALID, "mesh does not match the energy manager");
    if (M.nv == 0) {
        HIPCHECK(hipMemsetAsync(E.globals.p, 0, sizeof(Globals), g_rt.stream));
        if (to_host) *E.host_globals.p = Globals{};
        return;
    }
    ensure_masks(*E.nlist, M);
    PassBuffers b = buffers(E, M);
    if (to_host) b.host = E.host_globals.p;
    hipEvent_t marks[2] = {g_rt.pass1_marks[0], g_rt.pass1_marks[1]};
    g_rt.pass1_marks[0] = g_rt.pass1_marks[1] = nullptr;
    launch_pass1(M.view(), E.nlist->view(), eparams_of(E), mixed, b, vprops, g_rt.stream, E.tune, marks);
    check_launch();
    if (b.pc.x_snap) E.nlist->pc_ok = true;    // recorded by this launch, or still valid
}

void run_pass2(tm_energy& E, tm_mesh& M, int mixed)
{
    if (M.nv == 0) return;
    ensure_masks(*E.nlist, M);
    launch_pass2(M.view(), E.nlist->view(), eparams_of(E), mixed, buffers(E, M), E.grad.p, g_rt.stream, E.tune);
    check_launch();
}

// the sums of a pass that was told to hand them over
Globals read_globals(tm_energy& E)
{
    sync();
    return *E.host_globals.p;
}

tm_props props_of(const Globals& g)
{
    return tm_props{g.props[0], g.props[1], g.props[2], g.props[3], g.props[4], g.props[5]};
}

// trimem_energy (kernel.h:110-122) on host-supplied properties
double energy_from(const tm_energy& E, const tm_props& pr)
{
    EParams p = eparams_of(E);
    double e = 0.0, d;
    d = pr.area / p.ref_area - 1.0;
    e += p.kappa_a * d * d;
    d = pr.volume / p.ref_volume - 1.0;
    e += p.kappa_v * d * d;
    d = pr.curvature / p.ref_curvature - 1.0;
    e += p.kappa_c * d * d;
    e += p.kappa_t * pr.tethering;
    e += p.kappa_r * pr.repulsion;
    e += p.kappa_b * pr.bending;
    return e;
}

void require(bool c, const char* msg)
{
    if (!c) throw TmError(TM_E_INVALID, msg);
}

}    // namespace

// ================================================================ C ABI ====
extern "C" {

const char* tm_last_error(void) { return g_err.c_str(); }

int tm_device_count(int* count)
{
    API_BEGIN
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    *count = n;
    API_END
}

int tm_set_device(int device)
{
    API_BEGIN
    require(!g_rt.init || g_rt.device == device, "device already selected");
    g_rt.device = device;
    API_END
}

int tm_mesh_create(const double* points, int n_points, const int* faces, int n_faces, tm_mesh** out)
{
    API_BEGIN
    require(out != nullptr, "null output");
    require(n_points >= 0 && n_faces >= 0, "negative size");
    auto M = std::make_unique<tm_mesh>();
    M->nv = n_points;
    size_t bytes = sizeof(double) * 3 * std::max(n_points, 1);
    // pinned host memory when a device is present (fast uploads); plain
    // memory otherwise so that meshes can be built on a host without a GPU
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0 &&
        hipHostMalloc((void**)&M->points, bytes, hipHostMallocCoherent) == hipSuccess) {
        M->pinned = true;
    } else {
        (void)hipGetLastError();
        M->points = (double*)std::malloc(bytes);
        if (!M->points) throw TmError(TM_E_INVALID, "out of host memory");
    }
    if (n_points) std::memcpy(M->points, points, sizeof(double) * 3 * n_points);
    build_topology(*M, faces, n_faces);
    reorder_vertices(*M);
    *out = M.release();
    API_END
}

int tm_mesh_destroy(tm_mesh* mesh)
{
    delete mesh;
    return TM_OK;
}

int tm_mesh_counts(const tm_mesh* mesh, int* nv, int* ne, int* nf)
{
    API_BEGIN
    if (nv) *nv = mesh->nv;
    if (ne) *ne = mesh->nh / 2;
    if (nf) *nf = mesh->nf;
    API_END
}

double* tm_mesh_points(tm_mesh* mesh) { return mesh->points; }

int tm_mesh_fv_indices(tm_mesh* mesh, int* out)
{
    API_BEGIN
    // flips have changed the device topology: the faces from there, instead of all
    // six halfedge arrays and a walk over them here.  Faces that are read again
    // are walked here where that is faster than a launch and a wait: 0.7 against
    // 12.8 us at 320 faces, 5.5 and 15 at 5120, but 85 and 46 at 81920
    constexpr int kWalkFaces = 20480;
    if (mesh->faces_read && mesh->nf < kWalkFaces) refresh_host_topology(*mesh);
    if (mesh->host_stale) {
        mesh->faces_read = true;
        to_host(out, mesh->nf, 3 * sizeof(int), [&](void* p, int first, int n) {
            launch_faces(mesh->view(), mesh->d_perm.p, (int*)p, first, n, g_rt.stream);
        });
        return TM_OK;
    }
    for (int f = 0; f < mesh->nf; f++) {
        int h = mesh->f_he[f];
        out[3 * f] = mesh->perm[mesh->he_to[h]];
        h = mesh->he_next[h];
        out[3 * f + 1] = mesh->perm[mesh->he_to[h]];
        h = mesh->he_next[h];
        out[3 * f + 2] = mesh->perm[mesh->he_to[h]];
    }
    API_END
}

int tm_mesh_next_halfedge(tm_mesh* mesh, int he, int* out)
{
    API_BEGIN
    refresh_host_topology(*mesh);
    *out = (he >= 0 && he < mesh->nh) ? mesh->he_next[he] : -1;
    API_END
}

int tm_mesh_topology(tm_mesh* mesh, int* he_to, int* he_next, int* he_face, int* v_he, int* f_he)
{
    API_BEGIN
    refresh_host_topology(*mesh);
    if (he_to)
        for (int h = 0; h < mesh->nh; h++) he_to[h] = mesh->perm[mesh->he_to[h]];
    if (he_next) std::memcpy(he_next, mesh->he_next.data(), sizeof(int) * mesh->nh);
    if (he_face) std::memcpy(he_face, mesh->he_face.data(), sizeof(int) * mesh->nh);
    if (v_he)
        for (int u = 0; u < mesh->nv; u++) v_he[u] = mesh->v_he[mesh->iperm[u]];
    if (f_he) std::memcpy(f_he, mesh->f_he.data(), sizeof(int) * mesh->nf);
    API_END
}

double* tm_mesh_device_points(tm_mesh* mesh)
{
    try {
        ensure_device(*mesh);
    } catch (const std::exception& ex) {
        g_err = ex.what();
        return nullptr;
    }
    return mesh->x.p;
}

int tm_mesh_upload_points(tm_mesh* mesh)
{
    API_BEGIN
    push_points(*mesh);
    sync();
    API_END
}

int tm_mesh_download_points(tm_mesh* mesh)
{
    API_BEGIN
    ensure_device(*mesh);
    pull_points(*mesh);
    API_END
}

int tm_mesh_sync_host(tm_mesh* mesh)
{
    API_BEGIN
    if (mesh->device_ahead) pull_points(*mesh);
    API_END
}

int tm_halfedge_geometry(tm_mesh* mesh, int he, double* out47)
{
    API_BEGIN
    require(he >= 0 && he < mesh->nh, "halfedge out of range");
    upload_points(*mesh);
    DevBuf<double> d;
    d.alloc(47);
    launch_halfedge_geometry(mesh->view(), he, d.p, g_rt.stream);
    check_launch();
    d2h(out47, d.p, sizeof(double) * 47);
    sync();
    API_END
}

static int sum_geometry(tm_mesh* mesh, int what, double* out)
{
    API_BEGIN
    upload_points(*mesh);
    int n = what == 0 ? mesh->nf : mesh->nh / 2;
    DevBuf<double> part, res;
    DevBuf<unsigned> cnt;
    part.alloc((n + 255) / 256 + 1);
    res.alloc(1);
    cnt.alloc(1);
    HIPCHECK(hipMemsetAsync(cnt.p, 0, sizeof(unsigned), g_rt.stream));
    HIPCHECK(hipMemsetAsync(res.p, 0, sizeof(double), g_rt.stream));
    if (n > 0) {
        launch_sum_geometry(mesh->view(), what, part.p, cnt.p, res.p, g_rt.stream);
        check_launch();
    }
    d2h(out, res.p, sizeof(double));
    sync();
    API_END
}

int tm_area(tm_mesh* mesh, double* out) { return sum_geometry(mesh, 0, out); }
int tm_edges_length(tm_mesh* mesh, double* out) { return sum_geometry(mesh, 1, out); }

// tm_area / tm_edges_length without allocating: the device-resident
// positions, the partials and counter in the library's scratch, the sum
// written to the caller's device double, nothing synchronised.
int tm_mesh_sum_noalloc(tm_mesh* mesh, int what, double* out)
{
    API_BEGIN
    require(mesh != nullptr && out != nullptr, "null argument");
    require(what == 0 || what == 1, "what must be 0 (face areas) or 1 (edge lengths)");
    ensure_runtime();
    require(mesh->dev, "the mesh is not on the device yet (upload its points first)");
    const int n = what == 0 ? mesh->nf : mesh->nh / 2;
    require((n + 255) / 256 <= kNoAllocMaxBlocks, "too many faces or edges for the allocation-free sum (at most 8388608)");
    char* base = (char*)g_rt.scratch[g_rt.device];
    unsigned* counter = (unsigned*)base;
    double* partials = (double*)(base + kNoAllocCounterBytes);
    if (n > 0) {
        // the last-block counter starts at zero (a fill kernel, not a memset:
        // the call may be captured into a graph)
        launch_fill_ints((int*)counter, 1, 0, nullptr, 0, 0, nullptr, 0, 0, g_rt.stream);
        launch_sum_geometry(mesh->view(), what, partials, counter, out, g_rt.stream);
    } else {
        launch_fill_ints((int*)out, 2, 0, nullptr, 0, 0, nullptr, 0, 0, g_rt.stream);    // +0.0
    }
    check_launch();
    API_END
}

// ---- energy ----
int tm_energy_create(tm_mesh* mesh, const tm_params* params, tm_energy** out)
{
    API_BEGIN
    check_params(*params);
    auto E = std::make_unique<tm_energy>();
    E->params = *params;
    upload_points(*mesh);
    E->nlist = make_nlist(*mesh, E->params);
    // initial_props = properties(mesh) (energy.cpp:27); reference values
    // are not needed for the sums, unit placeholders keep the factors finite
    E->initial = tm_props{1, 1, 1, 0, 0, 0};
    run_pass1(*E, *mesh, 0, nullptr, true);
    E->initial = props_of(read_globals(*E));
    *out = E.release();
    API_END
}

int tm_energy_destroy(tm_energy* em)
{
    delete em;
    return TM_OK;
}

int tm_energy_get_params(const tm_energy* em, tm_params* out)
{
    *out = em->params;
    return TM_OK;
}

int tm_energy_initial_props(const tm_energy* em, tm_props* out)
{
    *out = em->initial;
    return TM_OK;
}

int tm_energy_set_precision(tm_energy* em, int precision)
{
    API_BEGIN
    require(precision == TM_PREC_FP64 || precision == TM_PREC_MIXED, "unknown precision");
    if (em->precision != precision) em->gen++;
    em->precision = precision;
    API_END
}

int tm_energy_get_precision(const tm_energy* em, int* precision)
{
    *precision = em->precision;
    return TM_OK;
}

int tm_energy_properties(tm_energy* em, tm_mesh* mesh, tm_props* out)
{
    API_BEGIN
    upload_points(*mesh);
    run_pass1(*em, *mesh, em->precision, nullptr, true);
    *out = props_of(read_globals(*em));
    API_END
}

int tm_energy_vertex_properties(tm_energy* em, tm_mesh* mesh, double* out)
{
    API_BEGIN
    upload_points(*mesh);
    em->vprops.alloc((size_t)mesh->nv * 6);
    run_pass1(*em, *mesh, em->precision, em->vprops.p);
    download_rows(*mesh, em->vprops.p, 6, out);
    API_END
}

int tm_energy_energy(tm_energy* em, tm_mesh* mesh, double* out)
{
    API_BEGIN
    upload_points(*mesh);
    run_pass1(*em, *mesh, em->precision, nullptr, true);
    *out = read_globals(*em).energy;
    API_END
}

int tm_energy_energy_props(tm_energy* em, const tm_props* props, double* out)
{
    *out = energy_from(*em, *props);
    return TM_OK;
}

int tm_energy_gradient(tm_energy* em, tm_mesh* mesh, double* out)
{
    API_BEGIN
    upload_points(*mesh);
    run_pass1(*em, *mesh, em->precision, nullptr);
    run_pass2(*em, *mesh, em->precision);
    download_rows(*mesh, em->grad.p, 3, out);
    API_END
}

int tm_energy_energy_gradient(tm_energy* em, tm_mesh* mesh, double* energy, double* grad)
{
    API_BEGIN
    upload_points(*mesh);
    run_pass1(*em, *mesh, em->precision, nullptr, true);
    run_pass2(*em, *mesh, em->precision);
    download_rows(*mesh, em->grad.p, 3, grad);
    *energy = read_globals(*em).energy;
    API_END
}

int tm_energy_update_reference_properties(tm_energy* em)
{
    // energy.cpp:47-55
    if (em->params.cont_lambda < 1.0) {
        em->params.cont_lambda += em->params.cont_delta;
        em->gen++;
    }
    return TM_OK;
}

int tm_energy_update_repulsion(tm_energy* em, tm_mesh* mesh)
{
    API_BEGIN
    upload_points(*mesh);
    rebuild_nlist(*em, *mesh);
    API_END
}

int tm_energy_eval_device(tm_energy* em, tm_mesh* mesh, int flags)
{
    API_BEGIN
    ensure_device(*mesh);
    if (flags & TM_EVAL_PROPS) run_pass1(*em, *mesh, em->precision, nullptr);
    if (flags & TM_EVAL_GRAD) run_pass2(*em, *mesh, em->precision);
    API_END
}

const double* tm_energy_device_gradient(tm_energy* em) { return em->grad.p; }
const double* tm_energy_device_globals(tm_energy* em) { return (const double*)em->globals.p; }

int tm_stream(void** out)
{
    API_BEGIN
    ensure_runtime();
    *out = (void*)g_rt.stream;
    API_END
}

int tm_mark_pass1(void* before, void* after)
{
    API_BEGIN
    ensure_runtime();
    g_rt.pass1_marks[0] = (hipEvent_t)before;
    g_rt.pass1_marks[1] = (hipEvent_t)after;
    API_END
}

int tm_sync(void)
{
    API_BEGIN
    ensure_runtime();
    sync();
    API_END
}

// ---- neighbour lists ----
int tm_nlist_create(tm_mesh* mesh, const tm_params* params, tm_nlist** out)
{
    API_BEGIN
    upload_points(*mesh);
    *out = make_nlist(*mesh, *params);
    API_END
}

int tm_nlist_destroy(tm_nlist* nl)
{
    delete nl;
    return TM_OK;
}

int tm_energy_nlist(tm_energy* em, tm_nlist** out)
{
    *out = em->nlist;
    return TM_OK;
}

int tm_nlist_distance_matrix(tm_nlist* nl, tm_mesh* mesh, double dmax, double* d, int* i, int* j, long cap,
                             long* count)
{
    API_BEGIN
    require(nl->nv == mesh->nv, "mesh does not match the neighbour list");
    upload_points(*mesh);
    const int n = mesh->nv;
    nl->dm_counts.alloc(n + 1);
    nl->dm_off.alloc(n + 1);
    HIPCHECK(hipMemsetAsync(nl->dm_counts.p, 0, sizeof(int) * (n + 1), g_rt.stream));
    launch_dm_count(mesh->view(), nl->view(), dmax, nl->dm_counts.p, g_rt.stream);
    check_launch();
    scan(nl->dm_counts.p, nl->dm_off.p, n + 1, nl->scan_tmp);
    int total = 0;
    d2h(&total, nl->dm_off.p + n, sizeof(int));
    sync();
    *count = total;
    if (d && i && j && total > 0) {
        nl->dm_d.alloc(total);
        nl->dm_i.alloc(total);
        nl->dm_j.alloc(total);
        launch_dm_fill(mesh->view(), nl->view(), dmax, nl->dm_off.p, nl->dm_d.p, nl->dm_i.p, nl->dm_j.p,
                       g_rt.stream);
        check_launch();
        long k = std::min<long>(cap, total);
        d2h(d, nl->dm_d.p, sizeof(double) * k);
        d2h(i, nl->dm_i.p, sizeof(int) * k);
        d2h(j, nl->dm_j.p, sizeof(int) * k);
        sync();
    }
    API_END
}

int tm_nlist_point_distances(tm_nlist* nl, tm_mesh* mesh, int pid, double dmax, double* dist3, int* jdx, long cap,
                             long* count)
{
    API_BEGIN
    require(pid >= 0 && pid < mesh->nv, "pid out of range");
    require(nl->nv == mesh->nv, "mesh does not match the neighbour list");
    upload_points(*mesh);
    pid = mesh->iperm[pid];
    // first pass counts, second pass fills a buffer of that size
    nl->pd_count.alloc(1);
    launch_point_distances(mesh->view(), nl->view(), pid, dmax, 0, nl->pd_count.p, nullptr, nullptr, g_rt.stream);
    check_launch();
    int c = 0;
    d2h(&c, nl->pd_count.p, sizeof(int));
    sync();
    *count = c;
    if (dist3 && jdx && c > 0) {
        nl->pd_dist.alloc((size_t)c * 3);
        nl->pd_j.alloc(c);
        launch_point_distances(mesh->view(), nl->view(), pid, dmax, c, nl->pd_count.p, nl->pd_dist.p, nl->pd_j.p,
                               g_rt.stream);
        check_launch();
        long k = std::min<long>(cap, c);
        d2h(dist3, nl->pd_dist.p, sizeof(double) * 3 * k);
        d2h(jdx, nl->pd_j.p, sizeof(int) * k);
        sync();
    }
    API_END
}

// ---- flips ----
// Arguments of one parallel sweep, its buffers allocated.
static PflipArgs pflip_args(tm_energy& E, tm_mesh& M, const EParams& ep, uint64_t seed, int nflips, int batch)
{
    E.pf_owner.alloc(M.nh / 2);
    E.pf_rec.alloc((size_t)kFlipRecord * batch);
    E.pf_lost.alloc(batch);
    E.pf_state.alloc(8);
    E.pf_count.alloc(1);
    return PflipArgs{M.flip_view(), E.nlist->view(), ep, M.flip_rows(true), seed, nflips, batch, E.globals.p,
                     E.pf_owner.p, E.pf_rec.p, E.pf_lost.p, E.pf_state.p, E.pf_count.p};
}

// The serial sweep in windows of W proposals (launch_serial_windows).  The
// number of windows a sweep needs depends on how many proposals each
// commits, so they are launched in batches sized from the rate so far, with
// the state read back between batches; surplus windows return at once.  The ring
// table is rebuilt behind each batch (the sweep does not read it), so that after
// the last one the host has waited for everything.
static SerialState serial_windows(tm_energy& E, tm_mesh& M, int nflips, const int* proposals, const double* uniforms,
                           int n_uniforms, uint64_t seed, int injected, int W)
{
    const size_t w = (size_t)W;
    E.sf_state.alloc(1);
    E.sf_rec.alloc(w * kSerialRecord);
    E.sf_fstamp.alloc(M.nf);
    const FlipRows rows = M.flip_rows(false);
    const EParams p = eparams_of(E);
    const NListView nl = E.nlist->view();
    launch_serial_begin(M.flip_view(), rows, E.globals.p, p, nflips, E.sf_state.p, E.sf_fstamp.p, g_rt.stream);
    int batch = std::max(1, std::min(1024, nflips / W + 1));
    for (;;) {
        launch_serial_windows(M.flip_view(), rows, nl, p, nflips, proposals, uniforms, n_uniforms, seed, injected, W,
                              E.sf_state.p, E.sf_rec.p, E.sf_fstamp.p, batch, g_rt.stream);
        check_launch();
        queue_ring(M);
        d2h(&M.report.p->serial, E.sf_state.p, sizeof(SerialState));
        sync();
        const SerialState h = M.report.p->serial;
        if (h.done) return h;
        const double per_window = std::max(1.0, (double)h.pos / std::max(h.window, 1));
        batch = std::min(4096, (int)std::ceil((nflips - h.pos) / per_window * 1.1) + 1);
    }
}

static int flip_impl(tm_energy* em, tm_mesh* mesh, int nflips, const int* proposals, const double* uniforms,
                     int n_uniforms, uint64_t seed, int injected, int* accepted, int* n_used)
{
    API_BEGIN
    upload_points(*mesh);
    // initial properties and energy (flips.cpp:30-31), FP64
    run_pass1(*em, *mesh, 0, nullptr);
    if (injected && nflips > 0) {
        em->proposals.alloc(nflips);
        h2d(em->proposals.p, proposals, sizeof(int) * nflips);
        em->uniforms.alloc(std::max(n_uniforms, 1));
        if (n_uniforms > 0) h2d(em->uniforms.p, uniforms, sizeof(double) * n_uniforms);
    }
    const int W = em->tune.serial_window;
    int res[3] = {0, 0, 0};
    if (W == 0) {
        launch_flip_serial(mesh->flip_view(), em->nlist->view(), eparams_of(*em), nflips,
                           injected ? em->proposals.p : nullptr, injected ? em->uniforms.p : nullptr, n_uniforms,
                           seed, injected, em->globals.p, em->flip_result.p, g_rt.stream);
        check_launch();
        queue_ring(*mesh);
        d2h(res, em->flip_result.p, sizeof(res));
        sync();
    } else {
        const SerialState st =
            serial_windows(*em, *mesh, nflips, injected ? em->proposals.p : nullptr,
                           injected ? em->uniforms.p : nullptr, n_uniforms, seed, injected, W);
        res[0] = st.acc;
        res[1] = st.used;
        res[2] = st.err;
    }
    const int ovf = mesh->report.p->overflow;
    mesh->flipped();
    if (res[0] > 0 || res[2] != 0 || ovf) mesh->topo_version++;   // only accepted flips change topology
    if (res[2] == 1) throw TmError(TM_E_INVALID, "flip proposal out of range");
    if (res[2] == 2) throw TmError(TM_E_INVALID, "uniform stream exhausted");
    if (ovf) throw TmError(TM_E_UNSUPPORTED, "vertex valence exceeds the ring-table width (32)");
    if (accepted) *accepted = res[0];
    if (n_used) *n_used = res[1];
    API_END
}

int tm_flip_parallel(tm_energy* em, tm_mesh* mesh, double flip_ratio, uint64_t seed, int batch, int* accepted)
{
    API_BEGIN
    // flips.cpp:84-85
    if (flip_ratio > 1.0) throw TmError(TM_E_RANGE, "flip_ratio must be <= 1.0");
    const int ne = mesh->nh / 2;
    const int nflips = (int)(ne * flip_ratio);
    // a patch conflicts with proposals on ~100 nearby edges: B = E / 1024
    // keeps the expected fraction of skipped proposals near 10%
    if (batch <= 0) batch = std::max(1, ne / 1024);
    upload_points(*mesh);
    run_pass1(*em, *mesh, 0, nullptr);
    if (nflips > 0)
        launch_flip_parallel(pflip_args(*em, *mesh, eparams_of(*em), seed, nflips, batch), em->tune.pflip_window,
                             g_rt.stream);
    check_launch();
    queue_ring(*mesh);
    double* st = mesh->report.p->parallel;
    std::fill(st, st + 8, 0.0);
    if (nflips > 0) d2h(st, em->pf_state.p, 8 * sizeof(double));
    sync();
    const int ovf = mesh->report.p->overflow;
    mesh->flipped();
    if (st[7] > 0 || ovf) mesh->topo_version++;
    if (nflips > 0) std::copy(st, st + 8, em->pf_last);
    if (ovf) throw TmError(TM_E_UNSUPPORTED, "vertex valence exceeds the ring-table width (32)");
    if (accepted) *accepted = (int)st[7];
    API_END
}

int tm_energy_pflip_state(tm_energy* em, double* out)
{
    API_BEGIN
    require(em != nullptr && out != nullptr, "null argument");
    std::copy(em->pf_last, em->pf_last + 8, out);
    API_END
}

int tm_flip_serial(tm_energy* em, tm_mesh* mesh, double flip_ratio, uint64_t seed, int* accepted)
{
    // flip_ratio > 1 is not rejected here, like flips.cpp:24-25
    int nflips = (int)((mesh->nh / 2) * flip_ratio);
    return flip_impl(em, mesh, nflips, nullptr, nullptr, 0, seed, 0, accepted, nullptr);
}

int tm_flip_serial_injected(tm_energy* em, tm_mesh* mesh, int n_proposals, const int* proposals,
                            const double* uniforms, int n_uniforms, int* accepted, int* n_used)
{
    return flip_impl(em, mesh, n_proposals, proposals, uniforms, n_uniforms, 0, 1, accepted, n_used);
}

}    // extern "C"

// ---- device-resident HMC step ----

struct tm_hmc {
    tm_mesh* mesh = nullptr;
    tm_energy* em = nullptr;
    int model = TM_HMC_ENERGY;
    int n3 = 0;
    DevBuf<double> x0, p, a, kpart0, kpart1;
    DevBuf<HmcState> state;
};

extern "C" {

int tm_hmc_create(tm_mesh* mesh, tm_energy* em, int model, tm_hmc** out)
{
    API_BEGIN
    require(mesh != nullptr && out != nullptr, "null argument");
    require(model == TM_HMC_ENERGY || model == TM_HMC_HARMONIC, "unknown HMC energy model");
    require(model != TM_HMC_ENERGY || em != nullptr, "the energy model needs an energy manager");
    ensure_device(*mesh);
    if (em) require(em->nlist && em->nlist->nv == mesh->nv, "mesh does not match the energy manager");
    auto H = std::make_unique<tm_hmc>();
    H->mesh = mesh;
    H->em = model == TM_HMC_ENERGY ? em : nullptr;
    H->model = model;
    H->n3 = 3 * mesh->nv;
    const size_t n3 = std::max(H->n3, 1);
    H->x0.alloc(n3);
    H->p.alloc(n3);
    H->a.alloc(n3);
    H->kpart0.alloc(hmc_blocks(H->n3));
    H->kpart1.alloc(hmc_blocks(H->n3));
    H->state.alloc(1);
    HIPCHECK(hipMemsetAsync(H->state.p, 0, sizeof(HmcState), g_rt.stream));
    sync();
    *out = H.release();
    API_END
}

int tm_hmc_destroy(tm_hmc* hmc)
{
    delete hmc;
    return TM_OK;
}

int tm_hmc_step(tm_hmc* hmc, const tm_hmc_params* prm, double temperature, const double* momenta, double uniform,
                uint64_t seed, uint64_t step)
{
    API_BEGIN
    require(hmc != nullptr && prm != nullptr, "null argument");
    require(prm->num_integration_steps >= 0, "num_integration_steps must be >= 0");
    tm_mesh& M = *hmc->mesh;
    require(3 * M.nv == hmc->n3, "mesh size changed since the HMC handle was created");
    // the device positions are the state; the host array is taken only when
    // it is the newer copy
    if (!M.device_ahead) push_points(M);
    const int n3 = hmc->n3;
    const double mass = prm->mass, dt = prm->time_step;
    const double dt2 = prm->time_step_sq != 0.0 ? prm->time_step_sq : dt * dt;
    const int L = prm->num_integration_steps;
    const int harmonic = hmc->model == TM_HMC_HARMONIC;
    if (momenta && M.nv > 0) {
        upload_rows(M, momenta, hmc->p.p);
        check_launch();
        sync();    // the caller's array may be reused on return
    }
    // p_var = m T (hmc.py:137); sigma = sqrt(p_var) (hmc.py:140)
    launch_hmc_begin(n3, M.x.p, hmc->x0.p, hmc->p.p, M.d_perm.p, momenta ? 0 : 1, seed, step,
                     std::sqrt(mass * temperature), hmc->kpart0.p, g_rt.stream);
    check_launch();
    HmcState* st = hmc->state.p;
    const Globals* globals = nullptr;
    const double* g = M.x.p;    // harmonic: dE/dx = x
    if (!harmonic) {
        tm_energy& E = *hmc->em;
        ensure_energy_buffers(E, M);
        globals = E.globals.p;
        g = E.grad.p;
    }
    // force at x0 (hmc.py:19), then L drift / force / kick steps (hmc.py:20-24)
    for (int i = 0; i <= L; i++) {
        if (!harmonic) {
            run_pass1(*hmc->em, M, hmc->em->precision, nullptr);
            run_pass2(*hmc->em, M, hmc->em->precision);
        }
        int mode = i == 0 ? kHmcFirst : kHmcKick;
        mode |= i < L ? kHmcDrift : kHmcLast;
        launch_hmc_leap(n3, M.x.p, hmc->p.p, hmc->a.p, g, dt, dt2, mass, mode, globals, st, hmc->kpart1.p,
                        g_rt.stream);
        check_launch();
    }
    launch_hmc_accept(n3, hmc->kpart0.p, hmc->kpart1.p, hmc->x0.p, M.x.p, harmonic, globals, mass, temperature,
                      uniform, seed, step, st, streak_of(harmonic ? nullptr : hmc->em), g_rt.stream);
    check_launch();
    launch_hmc_restore(n3, M.x.p, hmc->x0.p, st, g_rt.stream);
    check_launch();
    M.device_ahead = true;
    API_END
}

int tm_hmc_result(tm_hmc* hmc, tm_hmc_outcome* out)
{
    API_BEGIN
    require(hmc != nullptr && out != nullptr, "null argument");
    HmcState st;
    d2h(&st, hmc->state.p, sizeof(HmcState));
    sync();
    out->dh = st.dh;
    out->energy0 = st.energy0;
    out->energy1 = st.energy1;
    out->kinetic0 = st.kinetic0;
    out->kinetic1 = st.kinetic1;
    out->uniform = st.uniform;
    out->accepted = st.accepted;
    out->n_accepted = (long long)st.n_accepted;
    out->n_steps = (long long)st.n_steps;
    API_END
}

}    // extern "C"


// ---- replica groups ----
struct tm_replicas {
    int R = 0;
    int mixed = 0;
    std::vector<tm_mesh*> meshes;
    std::vector<tm_energy*> ems;
    // energy passes
    std::vector<PassArgs> h_args;
    DevBuf<PassArgs> d_args;
    std::vector<int> h_block0;
    DevBuf<int> d_block0;
    int total_blocks = 0;
    Tuning tune;
    DevBuf<int> d_block0_rep, d_block0_p2;
    int total_rep = 0, total_p2 = 0;
    // pair cache: per-replica recording flags (device; the reduction clears
    // them), displacement partials, and the prefix tables of the
    // displacement check and of the cached query
    NlistTables nl_tables;    // of the group's list builds
    DevBuf<int> force_flags, d_block0_rc;
    DevBuf<double> disp_parts;
    DevBuf<int> fast_parts;
    // parallel flip sweeps of the group: per-replica arguments and block
    // prefix tables (rebuilt by every sweep)
    DevBuf<PflipArgs> pf_args;
    DevBuf<int> pf_block0;
    HostBuf<double> pf_report;    // [8 R] the sweeps' final states
    std::vector<int> h_ones;
    int total_disp = 0, total_rc = 0;    // displacement partials, cached-query blocks
    std::vector<unsigned> gens;    // each member's tm_energy::gen when the table was built
    // zeros, the properties pass's counters of each member: a manager may be a
    // member more than once
    DevBuf<unsigned> pass_counts;
    GroupLaunch group() const
    {
        return GroupLaunch{d_args.p,  h_args.data(), R, d_block0.p, total_blocks, d_block0_rep.p, total_rep,
                           d_block0_p2.p, total_p2, tune, mixed, d_block0_rc.p,
                           tune.pair_cache ? total_rc : 0};
    }
    // every replica records at its next evaluation
    void force_all() { h2d(force_flags.p, h_ones.data(), sizeof(int) * R); }
    void force(int r) { h2d(force_flags.p + r, h_ones.data() + r, sizeof(int)); }
    // HMC
    bool hmc_ready = false;
    long long steps_run = 0;    // HMC steps run since the setup
    int L = 0;
    std::vector<HmcArgs> h_hmc;
    DevBuf<HmcArgs> d_hmc;
    std::vector<int> h_hblock0;
    DevBuf<int> d_hblock0;
    int hmc_total = 0;
    std::vector<DevBuf<double>> x0, p, a, kp0, kp1;
    DevBuf<HmcState> states;
    // tempering
    bool has_ladder = false;
    uint64_t pt_seed = 0;
    std::vector<double> h_ladder;
    DevBuf<double> ladder;
    DevBuf<int> owner;
    DevBuf<unsigned long long> pt_round, swaps_acc, swaps_tried;
    // graph of one HMC step
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    void drop_graph()
    {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        if (graph) (void)hipGraphDestroy(graph);
        graph_exec = nullptr;
        graph = nullptr;
    }
    ~tm_replicas() { drop_graph(); }
};

namespace {

void set_group_shape(tm_replicas& S, const Tuning& t, bool force);

// whether each member is the first, or the last, with its energy manager
std::vector<char> first_members(const tm_replicas& S)
{
    std::vector<char> first(S.R);
    std::unordered_set<const tm_energy*> seen;
    for (int r = 0; r < S.R; r++) first[r] = seen.insert(S.ems[r]).second;
    return first;
}
std::vector<char> last_members(const tm_replicas& S)
{
    std::vector<char> last(S.R);
    std::unordered_set<const tm_energy*> seen;
    for (int r = S.R; r-- > 0;) last[r] = seen.insert(S.ems[r]).second;
    return last;
}

// Rebuild the device table of pass arguments from the replicas' current
// buffers and neighbour lists.  With a ladder, each replica's kappa_b is that
// of the slot it holds on the device.
void refresh_replica_args(tm_replicas& S)
{
    std::vector<int> slot_of(S.R);
    if (S.has_ladder) {
        std::vector<int> owner(S.R);
        d2h(owner.data(), S.owner.p, sizeof(int) * S.R);
        sync();
        for (int s = 0; s < S.R; s++) slot_of[owner[s]] = s;
    }
    S.h_args.resize(S.R);
    S.h_block0.assign(S.R + 1, 0);
    // displacement partials and blocks of the cached query: one per pass-1
    // block (256 vertices) of each replica
    std::vector<int> b0d(S.R + 1, 0), b0c(S.R + 1, 0);
    for (int r = 0; r < S.R; r++) {
        b0d[r + 1] = b0d[r] + pass1_blocks(S.meshes[r]->nv);
        b0c[r + 1] = b0c[r] + pass1_blocks(S.meshes[r]->nv);
    }
    S.total_disp = b0d[S.R];
    S.total_rc = (b0c[S.R] + 7) / 8 * 8;    // a multiple of the 8 XCDs; padding blocks fall past the last replica's vertices
    S.d_block0_rc.alloc(S.R + 1);
    S.disp_parts.alloc(S.total_disp);
    S.fast_parts.alloc((size_t)kFastRow * S.total_disp);
    S.force_flags.alloc(S.R);
    S.h_ones.assign(S.R, 1);
    if (!S.pass_counts.p) alloc_pass_count(S.pass_counts, S.R);
    const std::vector<char> first = first_members(S);
    for (int r = 0; r < S.R; r++) {
        tm_mesh& M = *S.meshes[r];
        tm_energy& E = *S.ems[r];
        ensure_device(M);
        ensure_energy_buffers(E, M);
        ensure_masks(*E.nlist, M);
        EParams ep = eparams_of(E);
        if (S.has_ladder) ep.kappa_b = S.h_ladder[slot_of[r]];
        PassBuffers b = buffers(E, M);
        b.count = S.pass_counts.p + (size_t)kLastCounters * r;
        // one member keeps a list's recordings
        b.pc = first[r] ? pair_cache_of(E, M) : PairCache{};
        if (b.pc.x_snap) {
            b.pc.disp_part = S.disp_parts.p + b0d[r];
            b.pc.fast = S.fast_parts.p + (size_t)kFastRow * b0d[r];
            b.pc.disp_n = b0d[r + 1] - b0d[r];
            b.pc.dforce = S.force_flags.p + r;
        }
        S.h_args[r] = pass_args(M.view(), E.nlist->view(), ep, b, nullptr, E.grad.p);
        S.h_block0[r + 1] = S.h_block0[r] + S.h_args[r].nblocks;
    }
    S.total_blocks = S.h_block0[S.R];
    S.gens.resize(S.R);
    for (int r = 0; r < S.R; r++) S.gens[r] = S.ems[r]->gen;
    S.d_args.alloc(S.R);
    S.d_block0.alloc(S.R + 1);
    h2d(S.d_args.p, S.h_args.data(), sizeof(PassArgs) * S.R);
    h2d(S.d_block0.p, S.h_block0.data(), sizeof(int) * (S.R + 1));
    h2d(S.d_block0_rc.p, b0c.data(), sizeof(int) * (S.R + 1));
    set_group_shape(S, S.tune, true);
}

// block prefix tables of the repulsion query and pass 2 for tuning t; force:
// every replica records at its next evaluation (new tables, or a pair cache
// switched back on, which must not replay lists it did not keep).  The
// recorded lists do not depend on the launch shape.
void set_group_shape(tm_replicas& S, const Tuning& t, bool force)
{
    std::vector<int> rep(S.R + 1, 0), p2(S.R + 1, 0);
    for (int r = 0; r < S.R; r++) {
        rep[r + 1] = rep[r] + tuned_blocks(S.meshes[r]->nv, t.rep_threads);
        p2[r + 1] = p2[r] + pass2_blocks(S.meshes[r]->nv, t.p2_threads);
    }
    S.tune = t;
    S.tune.rep_fused = 0;     // grouped launches keep the query apart
    if (force) S.force_all();
    S.total_rep = rep[S.R];
    S.total_p2 = p2[S.R];
    S.d_block0_rep.alloc(S.R + 1);
    S.d_block0_p2.alloc(S.R + 1);
    h2d(S.d_block0_rep.p, rep.data(), sizeof(int) * (S.R + 1));
    h2d(S.d_block0_p2.p, p2.data(), sizeof(int) * (S.R + 1));
    sync();
}

// every replica's positions on the device (host arrays win where newer)
void replicas_device_points(tm_replicas& S)
{
    for (tm_mesh* M : S.meshes)
        if (!M->device_ahead) push_points(*M);
}

// The device table current for every member: a member whose manager
// rebuilt its neighbour list (update_repulsion swaps in the spare list),
// advanced its continuation or changed precision since the table was built
// makes the group rebuild the table and drop its captured graph, whose
// launches read the old list.  A precision different from the group's is
// refused.
void replicas_current(tm_replicas& S)
{
    bool stale = false;
    for (int r = 0; r < S.R; r++) {
        if (S.ems[r]->precision != S.mixed)
            throw TmError(TM_E_INVALID, "a replica's precision differs from the group's");
        stale = stale || S.ems[r]->gen != S.gens[r];
    }
    if (!stale) return;
    S.drop_graph();
    refresh_replica_args(S);
}

// exclusion masks current for every replica's topology (the table holds
// the mask buffers, whose addresses do not change)
void replicas_masks(tm_replicas& S)
{
    replicas_current(S);
    for (int r = 0; r < S.R; r++) {
        tm_nlist& L = *S.ems[r]->nlist;
        const unsigned before = L.mask_topo;
        ensure_masks(L, *S.meshes[r]);
        if (L.mask_topo != before) S.force(r);    // new topology: exclusion may have changed
    }
}

void replicas_hmc_step(tm_replicas& S)
{
    launch_hmc_begin_grouped(S.d_hmc.p, S.d_hblock0.p, S.R, S.hmc_total, g_rt.stream);
    for (int i = 0; i <= S.L; i++) {
        launch_pass1_grouped(S.group(), g_rt.stream);
        launch_pass2_grouped(S.group(), g_rt.stream);
        int mode = i == 0 ? kHmcFirst : kHmcKick;
        mode |= i < S.L ? kHmcDrift : kHmcLast;
        launch_hmc_leap_grouped(S.d_hmc.p, S.d_hblock0.p, S.R, S.hmc_total, mode, g_rt.stream);
    }
    launch_hmc_accept_grouped(S.d_hmc.p, S.d_args.p, S.R, g_rt.stream);
    launch_hmc_restore_grouped(S.d_hmc.p, S.d_hblock0.p, S.R, S.hmc_total, g_rt.stream);
}

}    // namespace

extern "C" {

int tm_replicas_create(tm_mesh* const* meshes, tm_energy* const* ems, int n_replicas, tm_replicas** out)
{
    API_BEGIN
    require(meshes && ems && out && n_replicas > 0, "null argument or no replicas");
    auto S = std::make_unique<tm_replicas>();
    S->R = n_replicas;
    for (int r = 0; r < n_replicas; r++) {
        require(meshes[r] && ems[r], "null replica");
        require(ems[r]->nlist && ems[r]->nlist->nv == meshes[r]->nv, "mesh does not match the energy manager");
        require(ems[r]->precision == ems[0]->precision, "replicas must share one precision");
        S->meshes.push_back(meshes[r]);
        S->ems.push_back(ems[r]);
    }
    S->mixed = ems[0]->precision;
    refresh_replica_args(*S);
    replicas_device_points(*S);
    *out = S.release();
    API_END
}

int tm_replicas_destroy(tm_replicas* rs)
{
    delete rs;
    return TM_OK;
}

// One sweep of each of these members, whose meshes and managers are distinct, their
// final states into pf_report; whether a valence became too large.
static bool pflip_members(tm_replicas& S, const std::vector<int>& members, const std::vector<int>& slot_of,
                          double flip_ratio, const uint64_t* seeds)
{
    const int R = (int)members.size();
    std::vector<PflipArgs> h(R);
    std::vector<int> b0(R + 1, 0);
    int rounds = 0, max_nv = 0, max_nh = 0, max_batch = 0;
    for (int i = 0; i < R; i++) {
        const int r = members[i];
        tm_mesh& M = *S.meshes[r];
        tm_energy& E = *S.ems[r];
        // as tm_flip_parallel: the FP64 properties at the current positions
        // start each replica's Metropolis walk
        upload_points(M);
        run_pass1(E, M, 0, nullptr);
        const int ne = M.nh / 2, nflips = (int)(ne * flip_ratio), batch = std::max(1, ne / 1024);
        EParams ep = eparams_of(E);
        if (S.has_ladder) ep.kappa_b = S.h_ladder[slot_of[r]];
        h[i] = pflip_args(E, M, ep, seeds[r], nflips, batch);
        if (nflips > 0) rounds = std::max(rounds, (nflips + batch - 1) / batch);
        b0[i + 1] = b0[i] + pflip_round_blocks(batch);
        max_nv = std::max(max_nv, M.nv);
        max_nh = std::max(max_nh, M.nh);
        max_batch = std::max(max_batch, batch);
    }
    S.pf_args.alloc(R);
    S.pf_block0.alloc(R + 1);
    h2d(S.pf_args.p, h.data(), sizeof(PflipArgs) * R);
    h2d(S.pf_block0.p, b0.data(), sizeof(int) * (R + 1));
    const PflipGroup g{S.pf_args.p, R, rounds, S.ems[0]->tune.pflip_window, S.pf_block0.p, b0[R],
                       max_nv, max_nh, max_batch};
    launch_flip_parallel_grouped(g, g_rt.stream);
    check_launch();
    for (int i = 0; i < R; i++) {
        const int r = members[i];
        queue_ring(*S.meshes[r]);
        if (h[i].nflips > 0) d2h(S.pf_report.p + 8 * (size_t)r, S.ems[r]->pf_state.p, 8 * sizeof(double));
    }
    sync();
    bool overflow = false;
    for (int i = 0; i < R; i++) {
        const int r = members[i];
        tm_mesh& M = *S.meshes[r];
        const double* st = S.pf_report.p + 8 * (size_t)r;
        const int ovf = M.report.p->overflow;
        M.flipped();
        if (st[7] > 0 || ovf) M.topo_version++;
        if (h[i].nflips > 0) std::copy(st, st + 8, S.ems[r]->pf_last);
        overflow = overflow || ovf;
    }
    return overflow;
}

int tm_replicas_pflip(tm_replicas* rs, double flip_ratio, const uint64_t* seeds, int* accepted)
{
    API_BEGIN
    require(seeds != nullptr, "null seeds");
    // flips.cpp:84-85
    if (flip_ratio > 1.0) throw TmError(TM_E_RANGE, "flip_ratio must be <= 1.0");
    tm_replicas& S = *rs;
    // each replica's kappa_b is that of the ladder slot it holds now
    std::vector<int> slot_of(S.R);
    if (S.has_ladder) {
        std::vector<int> owner(S.R);
        d2h(owner.data(), S.owner.p, sizeof(int) * S.R);
        sync();
        for (int s = 0; s < S.R; s++) slot_of[owner[s]] = s;
    }
    S.pf_report.alloc(8 * (size_t)S.R);
    std::fill(S.pf_report.p, S.pf_report.p + 8 * (size_t)S.R, 0.0);
    bool overflow = false;
    // members with a mesh or a manager in common sweep one after another
    std::vector<int> todo(S.R), now, later;
    std::iota(todo.begin(), todo.end(), 0);
    for (; !todo.empty(); todo.swap(later)) {
        now.clear();
        later.clear();
        std::unordered_set<const void*> taken;
        for (int r : todo) {
            const bool mesh = taken.insert(S.meshes[r]).second, em = taken.insert(S.ems[r]).second;
            (mesh && em ? now : later).push_back(r);
        }
        overflow = pflip_members(S, now, slot_of, flip_ratio, seeds) || overflow;
    }
    for (int r = 0; accepted && r < S.R; r++) accepted[r] = (int)S.pf_report.p[8 * (size_t)r + 7];
    if (overflow) throw TmError(TM_E_UNSUPPORTED, "vertex valence exceeds the ring-table width (32)");
    API_END
}

int tm_replicas_eval(tm_replicas* rs, int flags)
{
    API_BEGIN
    replicas_masks(*rs);
    if (flags & TM_EVAL_PROPS) {
        hipEvent_t marks[2] = {g_rt.pass1_marks[0], g_rt.pass1_marks[1]};
        g_rt.pass1_marks[0] = g_rt.pass1_marks[1] = nullptr;
        launch_pass1_grouped(rs->group(), g_rt.stream, marks);
    }
    if (flags & TM_EVAL_GRAD) launch_pass2_grouped(rs->group(), g_rt.stream);
    check_launch();
    API_END
}

int tm_replicas_globals(tm_replicas* rs, double* out)
{
    API_BEGIN
    std::vector<Globals> g(rs->R);
    for (int r = 0; r < rs->R; r++) d2h(&g[r], rs->ems[r]->globals.p, sizeof(Globals));
    sync();
    for (int r = 0; r < rs->R; r++) {
        for (int k = 0; k < 6; k++) out[7 * r + k] = g[r].props[k];
        out[7 * r + 6] = g[r].energy;
    }
    API_END
}

int tm_replicas_gradient(tm_replicas* rs, int r, double* out)
{
    API_BEGIN
    require(r >= 0 && r < rs->R, "replica index out of range");
    download_rows(*rs->meshes[r], rs->ems[r]->grad.p, 3, out);
    API_END
}

int tm_replicas_hmc_setup(tm_replicas* rs, const double* mass, const double* time_step, const double* temperature,
                          const uint64_t* seeds, int num_integration_steps)
{
    API_BEGIN
    require(mass && time_step && temperature && seeds, "null argument");
    require(num_integration_steps >= 0, "num_integration_steps must be >= 0");
    tm_replicas& S = *rs;
    S.drop_graph();
    S.L = num_integration_steps;
    const int R = S.R;
    if (!S.hmc_ready) {
        S.x0.resize(R);
        S.p.resize(R);
        S.a.resize(R);
        S.kp0.resize(R);
        S.kp1.resize(R);
        S.states.alloc(R);
        HIPCHECK(hipMemsetAsync(S.states.p, 0, sizeof(HmcState) * R, g_rt.stream));
    }
    S.h_hmc.resize(R);
    S.h_hblock0.assign(R + 1, 0);
    for (int r = 0; r < R; r++) {
        tm_mesh& M = *S.meshes[r];
        tm_energy& E = *S.ems[r];
        const int n3 = 3 * M.nv;
        const size_t n3a = std::max(n3, 1);
        S.x0[r].alloc(n3a);
        S.p[r].alloc(n3a);
        S.a[r].alloc(n3a);
        S.kp0[r].alloc(hmc_blocks(n3));
        S.kp1[r].alloc(hmc_blocks(n3));
        HmcArgs h{};
        h.n3 = n3;
        h.nblocks = hmc_blocks(n3);
        h.x = M.x.p;
        h.x0 = S.x0[r].p;
        h.p = S.p[r].p;
        h.a = S.a[r].p;
        h.grad = E.grad.p;
        h.globals = E.globals.p;
        h.perm = M.d_perm.p;
        h.st = S.states.p + r;
        h.kpart0 = S.kp0[r].p;
        h.kpart1 = S.kp1[r].p;
        h.mass = mass[r];
        h.dt = time_step[r];
        h.dt2 = time_step[r] * time_step[r];
        h.temperature = temperature[r];
        require(!S.has_ladder || temperature[r] == temperature[0],
                "replica exchange over a kappa_b ladder needs one temperature for all replicas");
        h.seed = seeds[r];
        S.h_hmc[r] = h;
        S.h_hblock0[r + 1] = S.h_hblock0[r] + h.nblocks;
    }
    S.hmc_total = S.h_hblock0[R];
    S.d_hmc.alloc(R);
    S.d_hblock0.alloc(R + 1);
    h2d(S.d_hmc.p, S.h_hmc.data(), sizeof(HmcArgs) * R);
    h2d(S.d_hblock0.p, S.h_hblock0.data(), sizeof(int) * (R + 1));
    sync();
    S.hmc_ready = true;
    API_END
}

int tm_replicas_set_ladder(tm_replicas* rs, const double* ladder, uint64_t seed)
{
    API_BEGIN
    require(ladder != nullptr, "null argument");
    tm_replicas& S = *rs;
    S.h_ladder.assign(ladder, ladder + S.R);
    for (int s = 1; s < S.R; s++) require(S.h_ladder[s] >= S.h_ladder[s - 1], "the ladder must be ascending");
    // the exchange rule min(1, exp(-dk dB / T)) assumes one temperature
    if (S.hmc_ready)
        for (int r = 1; r < S.R; r++)
            require(S.h_hmc[r].temperature == S.h_hmc[0].temperature,
                    "replica exchange over a kappa_b ladder needs one temperature for all replicas");
    S.ladder.alloc(S.R);
    S.owner.alloc(S.R);
    S.pt_round.alloc(1);
    S.swaps_acc.alloc(S.R);
    S.swaps_tried.alloc(S.R);
    std::vector<int> own(S.R);
    for (int s = 0; s < S.R; s++) own[s] = s;
    h2d(S.ladder.p, S.h_ladder.data(), sizeof(double) * S.R);
    h2d(S.owner.p, own.data(), sizeof(int) * S.R);
    HIPCHECK(hipMemsetAsync(S.pt_round.p, 0, sizeof(unsigned long long), g_rt.stream));
    HIPCHECK(hipMemsetAsync(S.swaps_acc.p, 0, sizeof(unsigned long long) * S.R, g_rt.stream));
    HIPCHECK(hipMemsetAsync(S.swaps_tried.p, 0, sizeof(unsigned long long) * S.R, g_rt.stream));
    S.pt_seed = seed;
    S.has_ladder = true;
    refresh_replica_args(S);
    API_END
}

int tm_replicas_swap(tm_replicas* rs)
{
    API_BEGIN
    tm_replicas& S = *rs;
    require(S.has_ladder && S.hmc_ready, "exchange needs a ladder and HMC parameters");
    // the exchange compares the bending of each replica's current state,
    // which an HMC step records
    require(S.steps_run > 0, "exchange needs at least one HMC step first");
    replicas_current(S);
    launch_pt_swap(S.d_args.p, S.d_hmc.p, S.owner.p, S.ladder.p, S.R, S.pt_seed, S.pt_round.p, S.swaps_acc.p,
                   S.swaps_tried.p, g_rt.stream);
    check_launch();
    API_END
}

int tm_replicas_hmc_run(tm_replicas* rs, int n_steps, int swap_every, int use_graph)
{
    API_BEGIN
    tm_replicas& S = *rs;
    require(S.hmc_ready, "tm_replicas_hmc_setup first");
    require(n_steps >= 0, "n_steps must be >= 0");
    require(swap_every <= 0 || S.has_ladder, "exchange needs a ladder");
    replicas_masks(S);
    if (use_graph && !S.graph_exec && n_steps > 0) {
        // the step reads every changing quantity (step counts, kappa_b, list
        // pointers) from device tables, so one capture serves all steps
        HIPCHECK(hipStreamBeginCapture(g_rt.stream, hipStreamCaptureModeThreadLocal));
        replicas_hmc_step(S);
        HIPCHECK(hipStreamEndCapture(g_rt.stream, &S.graph));
        HIPCHECK(hipGraphInstantiate(&S.graph_exec, S.graph, nullptr, nullptr, 0));
    }
    for (int k = 0; k < n_steps; k++) {
        if (use_graph) HIPCHECK(hipGraphLaunch(S.graph_exec, g_rt.stream));
        else replicas_hmc_step(S);
        check_launch();
        if (swap_every > 0 && (k + 1) % swap_every == 0)
            launch_pt_swap(S.d_args.p, S.d_hmc.p, S.owner.p, S.ladder.p, S.R, S.pt_seed, S.pt_round.p,
                           S.swaps_acc.p, S.swaps_tried.p, g_rt.stream);
    }
    check_launch();
    S.steps_run += n_steps;
    for (tm_mesh* M : S.meshes) M->device_ahead = true;
    API_END
}

int tm_replicas_stats(tm_replicas* rs, long long* accepted, long long* steps, int* slot_of, double* props,
                      long long* swaps_accepted, long long* swaps_tried)
{
    API_BEGIN
    tm_replicas& S = *rs;
    const int R = S.R;
    std::vector<HmcState> st(R);
    std::vector<int> own(R);
    std::vector<unsigned long long> sa(R, 0), stt(R, 0);
    if (S.hmc_ready) d2h(st.data(), S.states.p, sizeof(HmcState) * R);
    if (S.has_ladder) {
        d2h(own.data(), S.owner.p, sizeof(int) * R);
        d2h(sa.data(), S.swaps_acc.p, sizeof(unsigned long long) * R);
        d2h(stt.data(), S.swaps_tried.p, sizeof(unsigned long long) * R);
    }
    sync();
    for (int r = 0; r < R; r++) {
        if (accepted) accepted[r] = S.hmc_ready ? (long long)st[r].n_accepted : 0;
        if (steps) steps[r] = S.hmc_ready ? (long long)st[r].n_steps : 0;
        if (props)
            for (int k = 0; k < 6; k++) props[6 * r + k] = S.hmc_ready ? st[r].props[k] : 0.0;
        if (swaps_accepted) swaps_accepted[r] = (long long)sa[r];
        if (swaps_tried) swaps_tried[r] = (long long)stt[r];
    }
    if (slot_of)
        for (int s = 0; s < R; s++) slot_of[S.has_ladder ? own[s] : s] = s;
    API_END
}

int tm_replicas_update_repulsion(tm_replicas* rs)
{
    API_BEGIN
    tm_replicas& S = *rs;
    // each manager's list once, whatever the number of its memberships, on the
    // mesh of the last of them
    std::vector<NlistJob> jobs;
    const std::vector<char> last = last_members(S);
    for (int r = 0; r < S.R; r++) {
        upload_points(*S.meshes[r]);
        if (last[r]) jobs.push_back(NlistJob{&spare_nlist(*S.ems[r]), S.meshes[r]});
        if (jobs.size() == kBuildLists || r + 1 == S.R) {
            build_nlists(jobs, S.nl_tables);
            if (r + 1 < S.R) sync();    // the tables are used again
            jobs.clear();
        }
    }
    for (int r = 0; r < S.R; r++)
        if (last[r]) take_spare(*S.ems[r]);
    refresh_replica_args(S);
    API_END
}

}    // extern "C"

// ---- launch-shape autotuner ----
namespace {

Tuning from_c(const tm_tuning& c)
{
    Tuning t;
    t.rep_threads = c.rep_threads;
    t.rep_batch = c.rep_batch;
    t.p2_threads = c.pass2_threads;
    t.rep_fused = c.rep_fused;
    t.pair_cache = c.pair_cache;
    t.pflip_window = c.pflip_window;
    t.serial_window = c.serial_window;
    return t;
}

tm_tuning to_c(const Tuning& t)
{
    tm_tuning c{};
    c.rep_threads = t.rep_threads;
    c.rep_batch = t.rep_batch;
    c.pass2_threads = t.p2_threads;
    c.rep_fused = t.rep_fused;
    c.pair_cache = t.pair_cache;
    c.pflip_window = t.pflip_window;
    c.serial_window = t.serial_window;
    return c;
}

// mean time of `reps` launches of f after two untimed ones (ms)
template <class F>
double time_launches(F&& f, int reps)
{
    hipEvent_t a, b;
    HIPCHECK(hipEventCreate(&a));
    HIPCHECK(hipEventCreate(&b));
    f();
    f();
    HIPCHECK(hipEventRecord(a, g_rt.stream));
    for (int i = 0; i < reps; i++) f();
    HIPCHECK(hipEventRecord(b, g_rt.stream));
    check_launch();
    HIPCHECK(hipEventSynchronize(b));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return (double)ms / reps;
}

// Try every shape of the repulsion query and of pass 2 with launch(t) and
// keep the fastest of each; the two kernels are timed separately.  The query
// always has its own launch (rep_fused is kept at 0).
template <class RepF, class P2F>
Tuning search(Tuning base, bool has_rep, RepF&& rep, P2F&& p2, double* best_rep_ms, double* best_p2_ms)
{
    const int ths[4] = {64, 128, 256, 512}, bats[4] = {1, 2, 4, 8};
    Tuning best = base;
    double brep = 1e30, bp2 = 1e30;
    if (has_rep)
        for (int th : ths)
            for (int ba : bats) {
                Tuning t = best;
                t.rep_threads = th;
                t.rep_batch = ba;
                t.rep_fused = 0;
                const double ms = time_launches([&] { rep(t); }, 5);
                if (ms < brep) {
                    brep = ms;
                    best.rep_threads = th;
                    best.rep_batch = ba;
                }
            }
    best.rep_fused = 0;
    for (int th : ths) {
        Tuning t = best;
        t.p2_threads = th;
        const double ms = time_launches([&] { p2(t); }, 5);
        if (ms < bp2) {
            bp2 = ms;
            best.p2_threads = th;
        }
    }
    if (best_rep_ms) *best_rep_ms = has_rep ? brep : 0.0;
    if (best_p2_ms) *best_p2_ms = bp2;
    return best;
}

}    // namespace

extern "C" {

int tm_energy_set_tuning(tm_energy* em, const tm_tuning* t)
{
    API_BEGIN
    require(t != nullptr && tuning_valid(from_c(*t)), "invalid launch shape");
    em->tune = from_c(*t);
    API_END
}

int tm_energy_get_tuning(const tm_energy* em, tm_tuning* out)
{
    *out = to_c(em->tune);
    return TM_OK;
}

int tm_energy_autotune(tm_energy* em, tm_mesh* mesh, tm_tuning* out, double* ms_rep, double* ms_pass2)
{
    API_BEGIN
    tm_energy& E = *em;
    tm_mesh& M = *mesh;
    upload_points(M);
    // pass 2 reads q and the globals; the second pass 1 leaves the pair
    // cache in its steady state (recorded, displacement measured)
    run_pass1(E, M, E.precision, nullptr);
    run_pass1(E, M, E.precision, nullptr);
    const PassArgs a = pass_args(M.view(), E.nlist->view(), eparams_of(E), buffers(E, M), nullptr, E.grad.p);
    if (M.nv > 0)
        E.tune = search(
            E.tune, a.rep_v != nullptr, [&](const Tuning& t) { launch_rep(a, t, g_rt.stream); },
            [&](const Tuning& t) { launch_pass2_kernel(a, E.precision, t, g_rt.stream); }, ms_rep, ms_pass2);
    if (out) *out = to_c(E.tune);
    API_END
}

int tm_replicas_set_tuning(tm_replicas* rs, const tm_tuning* t)
{
    API_BEGIN
    require(t != nullptr && tuning_valid(from_c(*t)), "invalid launch shape");
    rs->drop_graph();
    const bool cache_on = from_c(*t).pair_cache && !rs->tune.pair_cache;
    set_group_shape(*rs, from_c(*t), cache_on);
    API_END
}

int tm_replicas_get_tuning(const tm_replicas* rs, tm_tuning* out)
{
    API_BEGIN
    require(out != nullptr, "null output");
    *out = to_c(rs->tune);
    API_END
}

int tm_replicas_autotune(tm_replicas* rs, tm_tuning* out, double* ms_rep, double* ms_pass2)
{
    API_BEGIN
    tm_replicas& S = *rs;
    replicas_masks(S);
    launch_pass1_grouped(S.group(), g_rt.stream);
    bool has_rep = false;
    for (const PassArgs& a : S.h_args) has_rep = has_rep || a.rep_v;
    // a new shape's tables are uploaded in the untimed warm-up launches
    auto shaped = [&](const Tuning& t) {
        if (t.rep_threads != S.tune.rep_threads || t.rep_batch != S.tune.rep_batch ||
            t.p2_threads != S.tune.p2_threads)
            set_group_shape(S, t, false);
        return S.group();
    };
    const Tuning best = search(
        S.tune, has_rep, [&](const Tuning& t) { launch_rep_grouped(shaped(t), g_rt.stream); },
        [&](const Tuning& t) { launch_pass2_grouped(shaped(t), g_rt.stream); }, ms_rep, ms_pass2);
    S.drop_graph();
    set_group_shape(S, best, false);
    if (out) *out = to_c(best);
    API_END
}

}    // extern "C"

// ---- surrogate force network ----
struct tm_surrogate {
    tm_mesh* mesh = nullptr;
    tm_energy* em = nullptr;
    int nv = 0;
    SgNorm norm{};
    float sigma_F = 1.0f;
    DevBuf<float> theta, grad, m1, m2;
    DevBuf<short> packed;
    SgPacked pk{};
    DevBuf<float> act;    // every activation and work array, carved below
    SgBuffers b{};
    DevBuf<float> geo_buf;
    SgGeom geo{};
    DevBuf<int> twin, err;
    // the feature pass: properties without repulsion, in buffers of its own
    DevBuf<double> q, gprops, vprops, partials, rep_v;
    DevBuf<unsigned> pass_count;
    DevBuf<int> pair_cnt;
    DevBuf<Globals> globals;
    DevBuf<double> neg_force, xsave;
    DevBuf<float> losses;
    std::vector<std::unique_ptr<DevBuf<double>>> snap_x, snap_g;
    int adam_step = 0;
    // plain-gradient fallback of tm_hmc_step_guarded
    int pol_window = 10;         // surrogate-driven outcomes counted together
    double pol_min_acc = 0.5;    // below this acceptance the exact gradient drives
    int pol_probe = 10;          // while it does: one surrogate-driven probe every pol_probe steps
    std::deque<int> recent;      // outcomes (1 accepted) of the last surrogate-driven steps
    bool fallback = false;
    int since_probe = 0;
    bool pending = false;        // the last guarded step was surrogate-driven, its outcome unread
    unsigned twin_topo = ~0u;    // topology of the twin table
    unsigned checked_topo = ~0u; // topology whose features were last checked
    bool topo_ok = false;        // ... and whether the network can take it (closed, valences 3..10)
    long long n_sg = 0, n_exact = 0, n_switch = 0;
};

namespace {

void sg_alloc(tm_surrogate& S)
{
    const size_t N = (size_t)S.nv;
    const size_t NW = N * kSgW;
    S.theta.alloc(kSgParams);
    S.grad.alloc(kSgParams);
    S.m1.alloc(kSgParams);
    S.m2.alloc(kSgParams);
    HIPCHECK(hipMemsetAsync(S.m1.p, 0, sizeof(float) * kSgParams, g_rt.stream));
    HIPCHECK(hipMemsetAsync(S.m2.p, 0, sizeof(float) * kSgParams, g_rt.stream));
    // packed weights
    const size_t np = (size_t)kSgW * kSgFeatPad + kSgLayers * (4 * kSgW * kSgW + 2 * kSgW * kSgW);
    S.packed.alloc(np);
    short* pp = S.packed.p;
    S.pk.in_t = pp;
    pp += kSgW * kSgFeatPad;
    for (int l = 0; l < kSgLayers; l++) {
        S.pk.u_t[l] = pp; pp += kSgW * kSgW;
        S.pk.wv_t[l] = pp; pp += 2 * kSgW * kSgW;
        S.pk.u_n[l] = pp; pp += kSgW * kSgW;
        S.pk.w_n[l] = pp; pp += kSgW * kSgW;
        S.pk.v_n[l] = pp; pp += kSgW * kSgW;
    }
    // activations
    const size_t nact = N * kSgFeatPad + (2 * (kSgLayers + 1) + 2 * kSgLayers + 3) * NW + 3 * N + sg_loss_rows(S.nv) +
                        1 + sg_partial_floats(S.nv);
    S.act.alloc(nact);
    float* a = S.act.p;
    S.b.f0 = a; a += N * kSgFeatPad;
    for (int l = 0; l <= kSgLayers; l++) { S.b.Z[l] = a; a += NW; S.b.H[l] = a; a += NW; }
    for (int l = 0; l < kSgLayers; l++) { S.b.P[l] = a; a += NW; S.b.M[l] = a; a += NW; }
    S.b.dH = a; a += NW;
    S.b.dP = a; a += NW;
    S.b.dM = a; a += NW;
    S.b.ghat = a; a += 3 * N;
    S.b.loss_partial = a; a += sg_loss_rows(S.nv);
    S.b.loss = a; a += 1;
    S.b.partial = a;
    S.geo_buf.alloc((size_t)kSgSlots * N * 5 + 3 * N);
    S.geo.eps = S.geo_buf.p;
    S.geo.ehat = S.geo_buf.p + (size_t)kSgSlots * N * 2;
    S.geo.nu = S.geo_buf.p + (size_t)kSgSlots * N * 5;
    S.twin.alloc((size_t)kSgSlots * N);
    S.err.alloc(1);
    S.q.alloc(N);
    S.gprops.alloc(6 * N);
    S.vprops.alloc(6 * N);
    S.partials.alloc((size_t)pass1_blocks(S.nv) * 6);
    alloc_pass_count(S.pass_count);
    S.rep_v.alloc(N);
    S.pair_cnt.alloc(N);
    S.globals.alloc(1);
    S.neg_force.alloc(3 * N);
    S.xsave.alloc(3 * N);
}

// properties without repulsion at the current positions into the
// surrogate's own buffers, then the input features
// exact_pass1: the energy manager's properties pass at these positions has just
// written S.vprops in the mixed precision, the same values
void sg_feature_pass(tm_surrogate& S, bool exact_pass1 = false)
{
    tm_mesh& M = *S.mesh;
    tm_energy& E = *S.em;
    EParams ep = eparams_of(E);
    ep.rep_lc1 = 0.0;    // no repulsion query: the features do not use it
    S.norm.ref[0] = ep.ref_area;
    S.norm.ref[1] = ep.ref_volume;
    S.norm.ref[2] = ep.ref_curvature;
    PassBuffers pb{};
    pb.q = S.q.p;
    pb.gprops = S.gprops.p;
    pb.pair_cnt = S.pair_cnt.p;
    pb.rep_v = S.rep_v.p;
    pb.partials = S.partials.p;
    pb.count = S.pass_count.p;
    pb.globals = S.globals.p;
    pb.list = M.generic.p;
    pb.nlist = 0;
    const Globals* globals = S.globals.p;
    if (exact_pass1) globals = E.globals.p;
    else launch_pass1(M.view(), E.nlist->view(), ep, 1, pb, S.vprops.p, g_rt.stream);
    sg_features(M.view(), S.vprops.p, globals, S.norm, S.geo, S.b.f0, S.err.p, g_rt.stream);
    check_launch();
}

void sg_check_err(tm_surrogate& S)
{
    int e = 0;
    d2h(&e, S.err.p, sizeof(int));
    sync();
    if (e) {
        HIPCHECK(hipMemsetAsync(S.err.p, 0, sizeof(int), g_rt.stream));
        throw TmError(TM_E_UNSUPPORTED, "surrogate needs a closed mesh with valences 3..10");
    }
}

// the loss and its parameter gradient after a forward pass with a target; the twin
// table follows the flips
void sg_gradient(tm_surrogate& S)
{
    const tm_mesh& M = *S.mesh;
    if (S.twin_topo != M.topo_version) {
        sg_twin(M.view(), S.twin.p, g_rt.stream);
        S.twin_topo = M.topo_version;
    }
    sg_backward(M.view(), S.b, S.geo, S.theta.p, S.pk, S.twin.p, S.grad.p, g_rt.stream);
}

// the exact gradient at the current positions (energy manager buffers)
void sg_exact_gradient(tm_surrogate& S, double* vprops = nullptr)
{
    run_pass1(*S.em, *S.mesh, S.em->precision, vprops);
    run_pass2(*S.em, *S.mesh, S.em->precision);
}

}    // namespace

extern "C" {

int tm_surrogate_create(tm_mesh* mesh, tm_energy* em, uint64_t seed, tm_surrogate** out)
{
    API_BEGIN
    require(mesh && em && out, "null argument");
    require(em->nlist && em->nlist->nv == mesh->nv, "mesh does not match the energy manager");
    tm_mesh& M = *mesh;
    upload_points(M);
    if (M.device_ahead) pull_points(M);    // host copies read below
    refresh_host_topology(M);
    require(M.nv > 0 && M.n_generic == 0, "surrogate needs a closed mesh");
    auto S = std::make_unique<tm_surrogate>();
    S->mesh = mesh;
    S->em = em;
    S->nv = M.nv;
    sg_alloc(*S);
    HIPCHECK(hipMemsetAsync(S->err.p, 0, sizeof(int), g_rt.stream));
    // mean edge length and raw features of the current state fix the
    // normalisation
    double lsum = 0.0;
    long ne = 0;
    for (int h = 0; h < M.nh; h += 2) {
        const int a = M.perm[M.he_to[h]], b = M.perm[M.he_to[h + 1]];
        const double* pa = M.points + 3 * a;
        const double* pb = M.points + 3 * b;
        lsum += std::sqrt((pa[0] - pb[0]) * (pa[0] - pb[0]) + (pa[1] - pb[1]) * (pa[1] - pb[1]) +
                          (pa[2] - pb[2]) * (pa[2] - pb[2]));
        ne++;
    }
    S->norm.lbar = ne ? lsum / ne : 1.0;
    for (int i = 0; i < kSgFeat; i++) {
        S->norm.mu[i] = 0.0;
        S->norm.sig[i] = 1.0;
    }
    sg_feature_pass(*S);
    sg_check_err(*S);
    std::vector<float> f((size_t)M.nv * kSgFeatPad);
    d2h(f.data(), S->b.f0, sizeof(float) * f.size());
    sync();
    for (int i = 0; i < kSgFeat; i++) {
        double m = 0.0, v = 0.0;
        for (int u = 0; u < M.nv; u++) m += f[(size_t)u * kSgFeatPad + i];
        m /= M.nv;
        for (int u = 0; u < M.nv; u++) {
            const double d = f[(size_t)u * kSgFeatPad + i] - m;
            v += d * d;
        }
        const double sd = std::sqrt(v / M.nv);
        if (i >= 4 && i <= 6) {    // global deviations: already dimensionless
            S->norm.mu[i] = 0.0;
            S->norm.sig[i] = 1.0;
        } else {
            S->norm.mu[i] = m;
            S->norm.sig[i] = sd > 1e-12 * std::fabs(m) + 1e-30 ? sd : 1.0;
        }
    }
    // force scale: rms of the exact force now
    sg_exact_gradient(*S);
    std::vector<double> g((size_t)3 * M.nv);
    d2h(g.data(), em->grad.p, sizeof(double) * g.size());
    sync();
    double ss = 0.0;
    for (double x : g) ss += x * x;
    S->sigma_F = (float)(ss > 0 ? std::sqrt(ss / g.size()) : 1.0);
    // Glorot-uniform weights, small output layer, zero biases
    std::vector<float> th(kSgParams, 0.0f);
    std::mt19937_64 rng(seed);
    auto fill = [&](int off, int fan_in, int fan_out, int count, float gain) {
        const float lim = gain * std::sqrt(6.0f / (float)(fan_in + fan_out));
        std::uniform_real_distribution<float> U(-lim, lim);
        for (int i = 0; i < count; i++) th[off + i] = U(rng);
    };
    fill(kSgOffWin, kSgFeat, kSgW, kSgFeatPad * kSgW, 1.0f);
    for (int i = kSgFeat * kSgW; i < kSgFeatPad * kSgW; i++) th[kSgOffWin + i] = 0.0f;
    for (int l = 0; l < kSgLayers; l++) {
        fill(sg_off_U(l), kSgW, kSgW, kSgW * kSgW, 1.0f);
        fill(sg_off_W(l), 2 * kSgW, kSgW, kSgW * kSgW, 0.5f);
        fill(sg_off_V(l), 2 * kSgW, kSgW, kSgW * kSgW, 0.5f);
        fill(sg_off_E(l), 2, kSgW, 2 * kSgW, 1.0f);
    }
    fill(kSgOffWs, kSgW, 1, kSgW, 0.1f);
    fill(kSgOffWt, kSgW, 1, kSgW, 0.1f);
    h2d(S->theta.p, th.data(), sizeof(float) * kSgParams);
    sg_pack(S->theta.p, S->pk, g_rt.stream);
    check_launch();
    sync();
    *out = S.release();
    API_END
}

int tm_surrogate_destroy(tm_surrogate* sg)
{
    delete sg;
    return TM_OK;
}

int tm_surrogate_params(tm_surrogate* sg, float* out, int* n)
{
    API_BEGIN
    if (n) *n = kSgParams;
    if (out) {
        d2h(out, sg->theta.p, sizeof(float) * kSgParams);
        sync();
    }
    API_END
}

int tm_surrogate_set_params(tm_surrogate* sg, const float* in)
{
    API_BEGIN
    require(in != nullptr, "null argument");
    h2d(sg->theta.p, in, sizeof(float) * kSgParams);
    sg_pack(sg->theta.p, sg->pk, g_rt.stream);
    check_launch();
    sync();
    API_END
}

int tm_surrogate_norm(tm_surrogate* sg, double* mu, double* sig, double* lbar, double* sigma_F)
{
    API_BEGIN
    for (int i = 0; i < kSgFeat; i++) {
        if (mu) mu[i] = sg->norm.mu[i];
        if (sig) sig[i] = sg->norm.sig[i];
    }
    if (lbar) *lbar = sg->norm.lbar;
    if (sigma_F) *sigma_F = sg->sigma_F;
    API_END
}

int tm_surrogate_forces(tm_surrogate* sg, double* forces)
{
    API_BEGIN
    tm_surrogate& S = *sg;
    upload_points(*S.mesh);
    sg_feature_pass(S);
    sg_forward(S.mesh->view(), S.b, S.geo, S.theta.p, S.pk, S.sigma_F, nullptr, S.neg_force.p, g_rt.stream);
    check_launch();
    sg_check_err(S);
    if (forces) {
        std::vector<double> g((size_t)3 * S.nv);
        download_rows(*S.mesh, S.neg_force.p, 3, g.data());
        for (size_t i = 0; i < g.size(); i++) forces[i] = -g[i];
    }
    API_END
}

int tm_surrogate_loss_grad(tm_surrogate* sg, double* loss, float* grad)
{
    API_BEGIN
    tm_surrogate& S = *sg;
    upload_points(*S.mesh);
    const bool mixed = S.em->precision == TM_PREC_MIXED;
    sg_exact_gradient(S, mixed ? S.vprops.p : nullptr);
    sg_feature_pass(S, mixed);
    sg_forward(S.mesh->view(), S.b, S.geo, S.theta.p, S.pk, S.sigma_F, S.em->grad.p, nullptr, g_rt.stream);
    sg_gradient(S);
    check_launch();
    float l = 0.0f;
    d2h(&l, S.b.loss, sizeof(float));
    std::vector<float> g(grad ? kSgParams : 0);    // a call that fails stores nothing
    d2h(g.data(), S.grad.p, sizeof(float) * g.size());
    sg_check_err(S);    // waits
    if (grad) std::copy(g.begin(), g.end(), grad);
    if (loss) *loss = l;
    API_END
}

int tm_surrogate_activations(tm_surrogate* sg, int which, float* out)
{
    API_BEGIN
    tm_surrogate& S = *sg;
    require(which >= 0 && which < 1 + (kSgLayers + 1) + kSgLayers, "unknown activation");
    const float* src;
    int w = kSgW;
    if (which == 0) {
        src = S.b.f0;
        w = kSgFeatPad;
    } else if (which <= kSgLayers + 1) {
        src = S.b.H[which - 1];
    } else {
        src = S.b.M[which - kSgLayers - 2];
    }
    std::vector<float> a((size_t)S.nv * w);
    d2h(a.data(), src, sizeof(float) * a.size());
    sync();
    for (int u = 0; u < S.nv; u++) {
        const int i = S.mesh->iperm[u];
        std::memcpy(out + (size_t)u * w, a.data() + (size_t)i * w, sizeof(float) * w);
    }
    API_END
}

int tm_surrogate_add_snapshot(tm_surrogate* sg)
{
    API_BEGIN
    tm_surrogate& S = *sg;
    upload_points(*S.mesh);
    sg_exact_gradient(S);
    auto x = std::make_unique<DevBuf<double>>();
    auto g = std::make_unique<DevBuf<double>>();
    x->alloc((size_t)3 * S.nv);
    g->alloc((size_t)3 * S.nv);
    HIPCHECK(hipMemcpyAsync(x->p, S.mesh->x.p, sizeof(double) * 3 * S.nv, hipMemcpyDeviceToDevice, g_rt.stream));
    HIPCHECK(hipMemcpyAsync(g->p, S.em->grad.p, sizeof(double) * 3 * S.nv, hipMemcpyDeviceToDevice, g_rt.stream));
    S.snap_x.push_back(std::move(x));
    S.snap_g.push_back(std::move(g));
    API_END
}

int tm_surrogate_num_snapshots(tm_surrogate* sg, int* n)
{
    *n = (int)sg->snap_x.size();
    return TM_OK;
}

int tm_surrogate_train(tm_surrogate* sg, int epochs, float lr, uint64_t seed, double* mean_loss)
{
    API_BEGIN
    tm_surrogate& S = *sg;
    const int ns = (int)S.snap_x.size();
    require(ns > 0, "no snapshots recorded");
    require(epochs >= 0, "epochs must be >= 0");
    tm_mesh& M = *S.mesh;
    upload_points(M);
    HIPCHECK(hipMemcpyAsync(S.xsave.p, M.x.p, sizeof(double) * 3 * S.nv, hipMemcpyDeviceToDevice, g_rt.stream));
    S.losses.alloc(std::max(ns, 1));
    std::vector<int> order(ns);
    std::iota(order.begin(), order.end(), 0);
    std::mt19937_64 rng(seed);
    for (int ep = 0; ep < epochs; ep++) {
        std::shuffle(order.begin(), order.end(), rng);
        for (int i = 0; i < ns; i++) {
            const int k = order[i];
            HIPCHECK(hipMemcpyAsync(M.x.p, S.snap_x[k]->p, sizeof(double) * 3 * S.nv, hipMemcpyDeviceToDevice,
                                    g_rt.stream));
            sg_feature_pass(S);
            sg_forward(M.view(), S.b, S.geo, S.theta.p, S.pk, S.sigma_F, S.snap_g[k]->p, nullptr, g_rt.stream);
            sg_gradient(S);
            sg_adam(kSgParams, S.theta.p, S.grad.p, S.m1.p, S.m2.p, lr, ++S.adam_step, g_rt.stream);
            sg_pack(S.theta.p, S.pk, g_rt.stream);
            HIPCHECK(hipMemcpyAsync(S.losses.p + i, S.b.loss, sizeof(float), hipMemcpyDeviceToDevice, g_rt.stream));
            check_launch();
        }
    }
    HIPCHECK(hipMemcpyAsync(M.x.p, S.xsave.p, sizeof(double) * 3 * S.nv, hipMemcpyDeviceToDevice, g_rt.stream));
    std::vector<float> ls(ns);
    d2h(ls.data(), S.losses.p, sizeof(float) * ns);
    sync();
    sg_check_err(S);
    if (mean_loss) {
        double a = 0.0;
        for (float x : ls) a += x;
        *mean_loss = epochs > 0 ? a / ns : 0.0;
    }
    API_END
}

// HMC step with the surrogate's forces along the trajectory and the exact
// energies at its two ends (hmc.py:133-158 with the force replaced)
int tm_hmc_step_surrogate(tm_hmc* hmc, tm_surrogate* sg, const tm_hmc_params* prm, double temperature,
                          const double* momenta, double uniform, uint64_t seed, uint64_t step)
{
    API_BEGIN
    require(hmc && sg && prm, "null argument");
    require(hmc->model == TM_HMC_ENERGY && hmc->em == sg->em && hmc->mesh == sg->mesh,
            "the HMC handle and the surrogate must share mesh and energy manager");
    require(prm->num_integration_steps >= 0, "num_integration_steps must be >= 0");
    tm_mesh& M = *hmc->mesh;
    tm_energy& E = *hmc->em;
    tm_surrogate& S = *sg;
    if (!M.device_ahead) push_points(M);
    const int n3 = hmc->n3;
    const double mass = prm->mass, dt = prm->time_step;
    const double dt2 = prm->time_step_sq != 0.0 ? prm->time_step_sq : dt * dt;
    const int L = prm->num_integration_steps;
    if (momenta) {
        upload_rows(M, momenta, hmc->p.p);
        check_launch();
        sync();
    }
    launch_hmc_begin(n3, M.x.p, hmc->x0.p, hmc->p.p, M.d_perm.p, momenta ? 0 : 1, seed, step,
                     std::sqrt(mass * temperature), hmc->kpart0.p, g_rt.stream);
    HmcState* st = hmc->state.p;
    run_pass1(E, M, E.precision, nullptr);    // exact E(x0), read by the first leap
    for (int i = 0; i <= L; i++) {
        sg_feature_pass(S);
        sg_forward(M.view(), S.b, S.geo, S.theta.p, S.pk, S.sigma_F, nullptr, S.neg_force.p, g_rt.stream);
        int mode = i == 0 ? kHmcFirst : kHmcKick;
        mode |= i < L ? kHmcDrift : kHmcLast;
        launch_hmc_leap(n3, M.x.p, hmc->p.p, hmc->a.p, S.neg_force.p, dt, dt2, mass, mode, E.globals.p, st,
                        hmc->kpart1.p, g_rt.stream);
        check_launch();
    }
    run_pass1(E, M, E.precision, nullptr);    // exact E(xn)
    launch_hmc_accept(n3, hmc->kpart0.p, hmc->kpart1.p, hmc->x0.p, M.x.p, 0, E.globals.p, mass, temperature,
                      uniform, seed, step, st, nullptr, g_rt.stream);
    launch_hmc_restore(n3, M.x.p, hmc->x0.p, st, g_rt.stream);
    check_launch();
    M.device_ahead = true;
    API_END
}

int tm_surrogate_set_policy(tm_surrogate* sg, int window, double min_acceptance, int probe_every)
{
    API_BEGIN
    require(sg != nullptr, "null argument");
    require(window >= 1 && probe_every >= 1, "window and probe_every must be >= 1");
    require(min_acceptance >= 0.0 && min_acceptance <= 1.0, "min_acceptance must be in [0, 1]");
    sg->pol_window = window;
    sg->pol_min_acc = min_acceptance;
    sg->pol_probe = probe_every;
    sg->recent.clear();
    sg->fallback = false;
    sg->since_probe = 0;
    API_END
}

int tm_surrogate_policy_state(tm_surrogate* sg, int* falling_back, long long* n_surrogate, long long* n_exact,
                              long long* n_switches, double* recent_acceptance)
{
    API_BEGIN
    require(sg != nullptr, "null argument");
    const tm_surrogate& S = *sg;
    if (falling_back) *falling_back = S.fallback;
    if (n_surrogate) *n_surrogate = S.n_sg;
    if (n_exact) *n_exact = S.n_exact;
    if (n_switches) *n_switches = S.n_switch;
    if (recent_acceptance) {
        double a = 0;
        for (int o : S.recent) a += o;
        *recent_acceptance = S.recent.empty() ? -1.0 : a / S.recent.size();
    }
    API_END
}

int tm_hmc_step_guarded(tm_hmc* hmc, tm_surrogate* sg, const tm_hmc_params* prm, double temperature,
                        const double* momenta, double uniform, uint64_t seed, uint64_t step, int* driver)
{
    API_BEGIN
    require(hmc && sg && prm, "null argument");
    tm_surrogate& S = *sg;
    tm_mesh& M = *hmc->mesh;
    // the outcome of the previous surrogate-driven step (waits for its
    // Metropolis kernel), then the switch in either direction
    if (S.pending) {
        HmcState st;
        d2h(&st, hmc->state.p, sizeof(HmcState));
        sync();
        S.pending = false;
        S.recent.push_back(st.accepted ? 1 : 0);
        while ((int)S.recent.size() > S.pol_window) S.recent.pop_front();
        if ((int)S.recent.size() == S.pol_window) {
            double a = 0;
            for (int o : S.recent) a += o;
            a /= S.pol_window;
            if (!S.fallback && a < S.pol_min_acc) {
                S.fallback = true;
                S.since_probe = 0;
                S.recent.clear();
                S.n_switch++;
            } else if (S.fallback && a >= S.pol_min_acc) {
                S.fallback = false;
                S.n_switch++;
            }
        }
    }
    bool use_sg = !S.fallback;
    if (S.fallback && ++S.since_probe >= S.pol_probe) {
        use_sg = true;
        S.since_probe = 0;
    }
    // the network takes closed meshes with valences 3..10 only; the topology
    // changes by flips between steps, so it is checked once per topology
    if (use_sg && S.checked_topo != M.topo_version) {
        if (!M.device_ahead) push_points(M);
        sg_feature_pass(S);
        int e = 0;
        d2h(&e, S.err.p, sizeof(int));
        sync();
        if (e) HIPCHECK(hipMemsetAsync(S.err.p, 0, sizeof(int), g_rt.stream));
        S.topo_ok = e == 0;
        S.checked_topo = M.topo_version;
    }
    use_sg = use_sg && S.topo_ok;
    int rc;
    if (use_sg) {
        rc = tm_hmc_step_surrogate(hmc, sg, prm, temperature, momenta, uniform, seed, step);
        S.pending = rc == TM_OK;
        S.n_sg++;
    } else {
        rc = tm_hmc_step(hmc, prm, temperature, momenta, uniform, seed, step);
        S.n_exact++;
    }
    if (rc != TM_OK) throw TmError(rc, tm_last_error());
    if (driver) *driver = use_sg ? 1 : 0;
    API_END
}

}    // extern "C"
