// tm_surrogate.hip -- a one-ring message-passing network that predicts the
// membrane forces, trained on the GPU from exact (positions, gradient) pairs.
//
// No counterpart in the reference.  The network drives HMC trajectories in
// place of the exact gradient; every trajectory is still accepted or rejected
// with the exact energy, so the chain samples the exact distribution (a
// position-dependent force field keeps the leapfrog map volume preserving and
// reversible, whether or not it is a gradient).
//
// Network (width W = 64, closed meshes, valence <= kSlots):
//   inputs   f_v   (8, normalised): vertex area, mean curvature c_v/a_v,
//                  valence, mean spoke length, the relative deviations of
//                  the global area, volume and curvature from their reference
//                  values, angle deficit; eps_vk (2): spoke length
//                  (l - lbar)/lbar and dihedral angle of edge (v, j_k)
//   layer 0  Z0 = f W_in + b_in,  H0 = silu(Z0)
//   layer l  P = H U_l,  M_v = (1/6) sum_k silu(P_{j_k} + eps_vk E_l),
//            Z = [H | M] [W_l; V_l] + b_l,  H <- H + silu(Z)       (l = 1..3)
//   output   s_vk = w_s . (H_v * H_{j_k}) + b_s,  t_v = w_t . H_v + b_t,
//            F_v = sigma_F (sum_k s_vk e_vk / |e_vk| + t_v nu_v)
// F is rotation equivariant (edge directions and the vertex normal nu_v carry
// all directions; every learned quantity is invariant) and s is symmetric in
// (v, j).  Dense products run on MFMA (bf16 operands, FP32 accumulation,
// v_mfma_f32_16x16x16_bf16); activations and all element-wise work are FP32.
// The training loss is mean |F/sigma_F - F*/sigma_F|^2 over vertices and
// components, F* = -dE/dx from the exact passes.
#include "tm_internal.h"
#include "tm_om.h"
#include "tm_surrogate.h"

namespace tmh {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// FP32 -> bf16, round to nearest even (finite inputs)
__device__ __forceinline__ short to_bf16(float f)
{
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}
__device__ __forceinline__ float silu(float x) { return x / (1.0f + __expf(-x)); }
__device__ __forceinline__ float silu_grad(float x)
{
    const float s = 1.0f / (1.0f + __expf(-x));
    return s * (1.0f + x * (1.0f - s));
}

// ------------------------------------------------------------ packing -----
// B operands of the GEMMs in bf16, as Bt[col][k] (k contiguous): forward
// products take W^T of the stored [k_in][c_out] weights, backward data
// products take the weights as stored.
__global__ void k_sg_pack(const float* __restrict__ theta, SgPacked pk)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    // input layer forward: in_t[c][k] = W_in[k][c]  (64 x 16)
    if (t < kSgW * kSgFeatPad) {
        const int c = t / kSgFeatPad, k = t % kSgFeatPad;
        pk.in_t[t] = to_bf16(theta[kSgOffWin + k * kSgW + c]);
    }
    for (int l = 0; l < kSgLayers; l++) {
        const float* U = theta + sg_off_U(l);
        const float* Wm = theta + sg_off_W(l);
        const float* V = theta + sg_off_V(l);
        if (t < kSgW * kSgW) {
            const int c = t / kSgW, k = t % kSgW;
            pk.u_t[l][t] = to_bf16(U[k * kSgW + c]);
            pk.u_n[l][t] = to_bf16(U[t]);
            pk.w_n[l][t] = to_bf16(Wm[t]);
            pk.v_n[l][t] = to_bf16(V[t]);
        }
        if (t < kSgW * 2 * kSgW) {
            const int c = t / (2 * kSgW), k = t % (2 * kSgW);
            pk.wv_t[l][t] = to_bf16(k < kSgW ? Wm[k * kSgW + c] : V[(k - kSgW) * kSgW + c]);
        }
    }
}

// --------------------------------------------------------------- GEMMs -----
// Y[n][c] = sum_k A[n][k] Bt[c][k] over K = KA + KB (A = [A1 | A2]), c < 64.
// Block: 4 waves, 64 rows, staged in LDS with the weights; wave w owns rows
// 16w..16w+15 and all 64 columns (four 16x16 tiles).  MFMA 16x16x16 operand lanes: A lane i holds row i % 16,
// k = 4 (i / 16) + 0..3; B lane i holds column i % 16, the same k; the
// accumulator lane i holds rows 4 (i / 16) + 0..3 of column i % 16.
// Epilogues: kSgStore Y = acc; kSgAccum Y += acc; kSgAct Z = acc + bias and
// H = (res ? res : 0) + silu(Z).
enum { kSgStore = 0, kSgAccum = 1, kSgAct = 2 };
template <int KA, int KB, int MODE>
__global__ void __launch_bounds__(256) k_sg_gemm(int N, const float* __restrict__ A1, const float* __restrict__ A2,
                                                 const short* __restrict__ Bt, const float* __restrict__ bias,
                                                 const float* __restrict__ res, float* __restrict__ Y,
                                                 float* __restrict__ H)
{
    constexpr int K = KA + KB;
    constexpr int KP = K + 8;    // padded LDS row (bf16): spreads the fragment reads over banks
    // the block's 64 rows of A and all of B, staged as bf16 with coalesced
    // 16-byte global loads
    __shared__ short s_a[64 * KP];
    __shared__ short s_b[64 * KP];
    const int row_base = blockIdx.x * 64;
    for (int q = threadIdx.x; q < 64 * (K / 4); q += 256) {
        const int r = q / (K / 4), k = 4 * (q % (K / 4));
        const int row = row_base + r;
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < N)
            x = k < KA ? *reinterpret_cast<const float4*>(A1 + (size_t)row * KA + k)
                       : *reinterpret_cast<const float4*>(A2 + (size_t)row * KB + (k - KA));
        short* d = s_a + r * KP + k;
        d[0] = to_bf16(x.x);
        d[1] = to_bf16(x.y);
        d[2] = to_bf16(x.z);
        d[3] = to_bf16(x.w);
    }
    for (int q = threadIdx.x; q < 64 * (K / 4); q += 256) {
        const int c = q / (K / 4), k = 4 * (q % (K / 4));
        const short4 x = *reinterpret_cast<const short4*>(Bt + c * K + k);
        short* d = s_b + c * KP + k;
        d[0] = x.x;
        d[1] = x.y;
        d[2] = x.z;
        d[3] = x.w;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int kq = 4 * (lane >> 4);
    const short* sa = s_a + (w * 16 + (lane & 15)) * KP + kq;
    floatx4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t] = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 16) {
        bf16x4 a;
#pragma unroll
        for (int i = 0; i < 4; i++) a[i] = sa[k0 + i];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const short* sb = s_b + (16 * t + (lane & 15)) * KP + kq + k0;
            bf16x4 b;
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = sb[i];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
        }
    }
    const int row0 = row_base + w * 16;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int col = 16 * t + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = row0 + kq + r;
            if (row >= N) continue;
            const size_t o = (size_t)row * kSgW + col;
            float y = acc[t][r];
            if (MODE == kSgStore) Y[o] = y;
            else if (MODE == kSgAccum) Y[o] += y;
            else {
                y += bias[col];
                Y[o] = y;
                H[o] = (res ? res[o] : 0.0f) + silu(y);
            }
        }
    }
}

// One layer's dense backward over 64-row tiles: with the incoming gradient D
// (kDz: D = dH silu'(Z), else D = dP as stored)
//   dH += D Wa^T                    (kGemms >= 1)
//   dM  = D Wb^T                    (kGemms == 2)
//   wpart[block] = [A1 | A2]^T D    (KF = KA + KB feature rows, 64 columns)
//   cpart[block] = column sums of D (kDz: the bias gradient)
// D is formed, rounded to bf16 and put into LDS once, by rows for the data
// products and by columns for the weight product, whose MFMA "k" dimension
// runs over the rows; wave w owns rows 16 w .. of the data products and column
// tile w of the weight product, which it accumulates in registers over all its
// block's tiles.  What bounds it is the traffic: D, its operands and dH once
// each.  At 40962 vertices one message-passing layer takes 22.4 us;
// silu', weight product, bias sums and the two data products as kernels of
// their own took 6.8 + 43.6 + 17.5 + 9.9 + 6.1 us.
constexpr int kSgTile = 64;
constexpr int kSgTrans = kSgTile + 4;    // padded row of a transposed tile (bf16)
template <int KA, int KB, bool kDz, int kGemms>
__global__ void __launch_bounds__(256) k_sg_layer_bwd(int N, const float* __restrict__ A1,
                                                      const float* __restrict__ A2, const float* Din,
                                                      const float* __restrict__ Z, const short* __restrict__ Wa,
                                                      const short* __restrict__ Wb, float* dH,
                                                      float* __restrict__ dM, float* __restrict__ wpart,
                                                      float* __restrict__ cpart)
{
    constexpr int KF = KA + KB, KT = KF / 16, KP = kSgW + 8;
    __shared__ __align__(16) short s_d[kGemms ? kSgTile * KP : 1];
    __shared__ __align__(16) short s_dt[kSgW * kSgTrans];
    __shared__ __align__(16) short s_ft[KF * kSgTrans];
    __shared__ __align__(16) short s_w[kGemms ? kGemms * kSgW * KP : 1];
    __shared__ float s_c[16][kSgW];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int l16 = lane & 15, kq = 4 * (lane >> 4);
    if constexpr (kGemms > 0)
        for (int q = tid; q < kGemms * kSgW * (kSgW / 4); q += 256) {
            const int g = q / (kSgW * kSgW / 4), c = (q / (kSgW / 4)) % kSgW, k = 4 * (q % (kSgW / 4));
            *reinterpret_cast<short4*>(s_w + (g * kSgW + c) * KP + k) =
                *reinterpret_cast<const short4*>((g ? Wb : Wa) + c * kSgW + k);
        }
    floatx4 acc[KT];
#pragma unroll
    for (int i = 0; i < KT; i++) acc[i] = floatx4{0, 0, 0, 0};
    float4 csum = make_float4(0.f, 0.f, 0.f, 0.f);
    const int tiles = (N + kSgTile - 1) / kSgTile;
    // a thread takes 4 x 4 blocks (four rows of four columns) of D, always in
    // the same columns, and of the features, so that a column's four rows go
    // to the transposed tile as one 8-byte write; the next tile's loads are in
    // flight while this one is multiplied
    constexpr int kQuads = KF / 4, kFeat = KF > 64 ? KF / 64 : 1;
    const int k = 4 * (tid & 15), rd = 4 * (tid >> 4);
    const int fq = tid % kQuads, rf = 4 * (tid / kQuads);
    const bool feat = rf < kSgTile;    // fewer features than columns: the first threads
    constexpr int kStep = kSgTile / kFeat;
    float4 d[4], z[kDz ? 4 : 1], x[kFeat][4];
    auto load = [&](int tile) {
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        const int base = tile * kSgTile;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = base + rd + i;
            d[i] = row < N ? *reinterpret_cast<const float4*>(Din + (size_t)row * kSgW + k) : zero;
            if constexpr (kDz) z[i] = row < N ? *reinterpret_cast<const float4*>(Z + (size_t)row * kSgW + k) : zero;
        }
#pragma unroll
        for (int u = 0; u < kFeat; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = base + rf + kStep * u + i, f = 4 * fq;
                x[u][i] = !feat || row >= N
                              ? zero
                              : (f < KA ? *reinterpret_cast<const float4*>(A1 + (size_t)row * KA + f)
                                        : *reinterpret_cast<const float4*>(A2 + (size_t)row * KB + (f - KA)));
            }
    };
    auto transpose = [&](short* t, int col, int row, const short4 (&b)[4]) {
        *reinterpret_cast<short4*>(t + (col + 0) * kSgTrans + row) = make_short4(b[0].x, b[1].x, b[2].x, b[3].x);
        *reinterpret_cast<short4*>(t + (col + 1) * kSgTrans + row) = make_short4(b[0].y, b[1].y, b[2].y, b[3].y);
        *reinterpret_cast<short4*>(t + (col + 2) * kSgTrans + row) = make_short4(b[0].z, b[1].z, b[2].z, b[3].z);
        *reinterpret_cast<short4*>(t + (col + 3) * kSgTrans + row) = make_short4(b[0].w, b[1].w, b[2].w, b[3].w);
    };
    load(blockIdx.x);
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int row_base = tile * kSgTile;
        short4 b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (kDz) {
                d[i].x *= silu_grad(z[i].x);
                d[i].y *= silu_grad(z[i].y);
                d[i].z *= silu_grad(z[i].z);
                d[i].w *= silu_grad(z[i].w);
                csum.x += d[i].x;
                csum.y += d[i].y;
                csum.z += d[i].z;
                csum.w += d[i].w;
            }
            b[i] = make_short4(to_bf16(d[i].x), to_bf16(d[i].y), to_bf16(d[i].z), to_bf16(d[i].w));
            if constexpr (kGemms > 0) *reinterpret_cast<short4*>(s_d + (rd + i) * KP + k) = b[i];
        }
        transpose(s_dt, k, rd, b);
#pragma unroll
        for (int u = 0; u < kFeat; u++) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                b[i] = make_short4(to_bf16(x[u][i].x), to_bf16(x[u][i].y), to_bf16(x[u][i].z), to_bf16(x[u][i].w));
            if (feat) transpose(s_ft, 4 * fq, rf + kStep * u, b);
        }
        __syncthreads();
        // dH of this tile as it was, then the next tile
        float old[kGemms ? 16 : 1];
        if constexpr (kGemms > 0)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = row_base + 16 * w + kq + r;
                    old[4 * t + r] = row < N ? dH[(size_t)row * kSgW + 16 * t + l16] : 0.0f;
                }
        if (tile + (int)gridDim.x < tiles) load(tile + gridDim.x);
        // weight product: column tile w, every feature tile
#pragma unroll
        for (int n0 = 0; n0 < kSgTile; n0 += 16) {
            const bf16x4 b = *reinterpret_cast<const bf16x4*>(s_dt + (16 * w + l16) * kSgTrans + n0 + kq);
#pragma unroll
            for (int i = 0; i < KT; i++) {
                const bf16x4 a = *reinterpret_cast<const bf16x4*>(s_ft + (16 * i + l16) * kSgTrans + n0 + kq);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[i], 0, 0, 0);
            }
        }
        // data products: rows 16 w .., four column tiles each
        if constexpr (kGemms > 0) {
#pragma unroll
            for (int g = 0; g < kGemms; g++) {
                floatx4 y[4];
#pragma unroll
                for (int t = 0; t < 4; t++) y[t] = floatx4{0, 0, 0, 0};
#pragma unroll
                for (int k0 = 0; k0 < kSgW; k0 += 16) {
                    const bf16x4 a = *reinterpret_cast<const bf16x4*>(s_d + (16 * w + l16) * KP + kq + k0);
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const bf16x4 b = *reinterpret_cast<const bf16x4*>(
                            s_w + (g * kSgW + 16 * t + l16) * KP + kq + k0);
                        y[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, y[t], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int row = row_base + 16 * w + kq + r;
                        const size_t o = (size_t)row * kSgW + 16 * t + l16;
                        if (row < N) {
                            if (g == 0) dH[o] = old[4 * t + r] + y[t][r];
                            else dM[o] = y[t][r];
                        }
                    }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < KT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            wpart[((size_t)blockIdx.x * KF + 16 * i + kq + r) * kSgW + 16 * w + l16] = acc[i][r];
    if constexpr (kDz) {
        float* c = &s_c[tid >> 4][4 * (tid & 15)];
        c[0] = csum.x;
        c[1] = csum.y;
        c[2] = csum.z;
        c[3] = csum.w;
        __syncthreads();
        if (tid < kSgW) {
            float a = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) a += s_c[i][tid];
            cpart[(size_t)blockIdx.x * kSgW + tid] = a;
        }
    }
}

// out[i] = sum over the blocks of partial[b][i], for every segment of the
// parameter gradient (and the loss) in one launch: a line of outputs per
// workgroup, 32 threads each, a fixed tree over those.  A chain of batches of
// loads: at 40962 vertices 18.9 us, with 8 threads for each output 27.4 us.
struct SgSegment {
    const float* partial;
    float* out;
    int rows, count;
};
constexpr int kSgSegments = 4 * kSgLayers + 4;
struct SgSegments {
    SgSegment s[kSgSegments];
    int block0[kSgSegments + 1];
};
constexpr int kSgRedOut = 32, kSgRedRows = 32;
__global__ void __launch_bounds__(kSgRedOut * kSgRedRows) k_sg_reduce(SgSegments g)
{
    __shared__ float s[kSgRedRows][kSgRedOut];
    int k = 0;
    while (k + 1 < kSgSegments && (int)blockIdx.x >= g.block0[k + 1]) k++;
    const SgSegment seg = g.s[k];
    const int o = threadIdx.x % kSgRedOut, b0 = threadIdx.x / kSgRedOut;
    const int i = ((int)blockIdx.x - g.block0[k]) * kSgRedOut + o;
    float a = 0.0f;
    if (i < seg.count) {
        constexpr int kBatch = 16;    // rows in flight
        for (int b = b0; b < seg.rows; b += kSgRedRows * kBatch) {
            float v[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int r = b + kSgRedRows * u;
                v[u] = r < seg.rows ? seg.partial[(size_t)r * seg.count + i] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) a += v[u];
        }
    }
    s[b0][o] = a;
    __syncthreads();
    if (b0 == 0 && i < seg.count) {
        float t[kSgRedRows];
#pragma unroll
        for (int u = 0; u < kSgRedRows; u++) t[u] = s[u][o];
#pragma unroll
        for (int w = kSgRedRows / 2; w > 0; w >>= 1)
#pragma unroll
            for (int u = 0; u < w; u++) t[u] += t[u + w];
        seg.out[i] = t[0];
    }
}

// ------------------------------------------------------------ features -----
// One thread per vertex: geometry of the ring (FP64 differences, FP32
// results), the normalised input features and the per-spoke edge data.
__global__ void k_sg_features(MeshView m, const double* __restrict__ vprops, const Globals* __restrict__ g,
                              SgNorm nrm, SgGeom geo, float* __restrict__ f0, int* __restrict__ err)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m.nv) return;
    const int N = m.nv;
    const int meta = m.meta[v];
    const int n = meta_valence(meta);
    if (meta_bslot(meta) >= 0 || n < 3 || n > kSgSlots) {
        atomicOr(err, 1);
        return;
    }
    const d3 xv = d3{m.x[3 * v], m.x[3 * v + 1], m.x[3 * v + 2]};
    // the whole ring in registers (slots past the valence: xv itself, unused),
    // each sector normal carried over to the slot it also bounds
    d3 e[kSgSlots];
#pragma unroll
    for (int k = 0; k < kSgSlots; k++) {
        const int j = k < n ? m.ring[k * N + v] : v;
        e[k] = d3{m.x[3 * j], m.x[3 * j + 1], m.x[3 * j + 2]} - xv;
    }
    d3 e_prev = e[kSgSlots - 1];
#pragma unroll
    for (int k = kSgSlots - 2; k >= 2; k--)
        if (k == n - 1) e_prev = e[k];
    d3 nk = cross(e[0], e_prev);                                 // face (v, j_0, j_{n-1})
    d3 nsum{0, 0, 0};
    double lsum = 0.0, angles = 0.0;
#pragma unroll
    for (int k = 0; k < kSgSlots; k++) {
        if (k < n) {
            const d3 e_next = k + 1 < n ? e[(k + 1) % kSgSlots] : e[0];
            const d3 nk1 = cross(e_next, e[k]);                  // face (v, j_{k+1}, j_k)
            nsum += nk;
            angles += atan2(sqrt(sqnorm(nk)), dot(e[k], e_prev));    // corner angle at v
            const double l = sqrt(sqnorm(e[k]));
            lsum += l;
            // dihedral of edge (v, j_k) between the two faces, signed by
            // (n_k x n_{k+1}) . e_k like the properties pass
            const float s = (float)(dot(cross(nk, nk1), e[k]) / l);
            const float c = (float)dot(nk, nk1);
            const int slot = k * N + v;
            geo.eps[2 * slot] = (float)((l - nrm.lbar) / nrm.lbar);
            geo.eps[2 * slot + 1] = atan2f(s, c);
            geo.ehat[3 * slot] = (float)(e[k].x / l);
            geo.ehat[3 * slot + 1] = (float)(e[k].y / l);
            geo.ehat[3 * slot + 2] = (float)(e[k].z / l);
            nk = nk1;
            e_prev = e[k];
        }
    }
    const double nn = sqrt(sqnorm(nsum));
    geo.nu[3 * v] = (float)(nsum.x / nn);
    geo.nu[3 * v + 1] = (float)(nsum.y / nn);
    geo.nu[3 * v + 2] = (float)(nsum.z / nn);
    const double a = vprops[6 * v], c = vprops[6 * v + 2];
    // relative deviations of the global area, volume and curvature from
    // their reference values (the penalty factors without their kappas), and
    // the angle deficit (the discrete Gaussian curvature of v)
    const double raw[kSgFeat] = {a, c / a, (double)n, lsum / n, g->props[0] / nrm.ref[0] - 1.0,
                                 g->props[1] / nrm.ref[1] - 1.0, g->props[2] / nrm.ref[2] - 1.0,
                                 6.283185307179586 - angles};
    for (int i = 0; i < kSgFeat; i++) f0[v * kSgFeatPad + i] = (float)((raw[i] - nrm.mu[i]) / nrm.sig[i]);
    for (int i = kSgFeat; i < kSgFeatPad; i++) f0[v * kSgFeatPad + i] = 0.0f;
}

// slot of v in the ring of its k-th neighbour (closed meshes)
__global__ void k_sg_twin(MeshView m, int* __restrict__ twin)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m.nv) return;
    const int N = m.nv;
    const int n = meta_valence(m.meta[v]);
    for (int k = 0; k < n && k < kSgSlots; k++) {
        const int j = m.ring[k * N + v];
        const int nj = meta_valence(m.meta[j]);
        int t = -1;
        for (int a = 0; a < nj && a < kSgSlots; a++)
            if (m.ring[a * N + j] == v) t = a;
        twin[k * N + v] = t;
    }
}

// ------------------------------------------------------------- messages -----
// The kernels below give a vertex a wave, lane = channel, four vertices per
// step.  Lane 4 k + i first loads what slot k of vertex i needs (one load for
// the step's ring, a few for its edge data); each neighbour's row is then
// requested with an index read off that lane, all rows of the four vertices
// in flight before the first is used.  One vertex at a time, each slot's index
// and edge data loaded by all lanes, left a chain of dependent loads per
// vertex.  The leading kRingPad slots are unrolled (ring columns past the
// valence hold -1), longer rings follow.
constexpr int kSgPer = 4;
static_assert(kSgPer * kRingPad <= 64, "a lane per slot of a step");

// The steps [first, last) of this workgroup of the `steps` steps of 16 vertices
// (4 waves of kSgPer): consecutive ones, and consecutive workgroups on one XCD,
// whose L2 then holds the rows of one compact part of the mesh.  Workgroups go
// round the 8 XCDs in turn; the grid is a multiple of 8.
struct SgSteps {
    int first, last;
};
__device__ __forceinline__ SgSteps sg_steps(int nv)
{
    const int chunk = gridDim.x / 8, lb = (blockIdx.x % 8) * chunk + blockIdx.x / 8;
    const int steps = (nv + 4 * kSgPer - 1) / (4 * kSgPer);
    const int per = (steps + (int)gridDim.x - 1) / (int)gridDim.x;
    return SgSteps{min(lb * per, steps), min((lb + 1) * per, steps)};
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ int at_lane(int x, int l) { return __builtin_amdgcn_readlane(x, l); }
__device__ __forceinline__ float at_lane(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// ring slots with edge data; a longer ring is refused by the feature kernel
__device__ __forceinline__ int sg_valence(int meta) { return min(meta_valence(meta), kSgSlots); }

// lane 4 k + i: slot k of vertex v0 + i (the last vertex past the end)
struct SgSlot {
    int v, s;    // vertex, index into the ring's columns
    int n;       // the vertex's valence
    int j;       // the neighbour (a valid row past the valence)
};
__device__ __forceinline__ SgSlot sg_slot(const MeshView& m, int v0)
{
    const int lane = threadIdx.x & 63, k = (lane / kSgPer) & (kRingPad - 1);
    SgSlot t;
    t.v = min(v0 + lane % kSgPer, m.nv - 1);
    t.s = k * m.nv + t.v;
    t.j = max(m.ring[t.s], 0);
    t.n = sg_valence(m.meta[t.v]);
    return t;
}

// M_v = (1/6) sum_k silu(P_{j_k} + eps_vk E).  At 40962 vertices 15.8 us,
// one vertex per wave 26.5 us.
__global__ void __launch_bounds__(256) k_sg_message(MeshView m, const float* __restrict__ P,
                                                    const float* __restrict__ eps, const float* __restrict__ E,
                                                    float* __restrict__ M)
{
    const int c = threadIdx.x & 63;
    const int N = m.nv;
    const SgSteps st = sg_steps(N);
    const int v0 = uniform((st.first * 4 + (threadIdx.x >> 6)) * kSgPer);    // one step per workgroup
    if (st.first >= st.last || v0 >= N) return;
    const float e0 = E[c], e1 = E[kSgW + c];
    const SgSlot t = sg_slot(m, v0);
    const float2 ex = reinterpret_cast<const float2*>(eps)[t.s];
    float p[kSgPer][kRingPad];
#pragma unroll
    for (int i = 0; i < kSgPer; i++)
#pragma unroll
        for (int k = 0; k < kRingPad; k++) p[i][k] = P[(size_t)at_lane(t.j, kSgPer * k + i) * kSgW + c];
#pragma unroll
    for (int i = 0; i < kSgPer; i++) {
        const int v = v0 + i, n = at_lane(t.n, i);
        if (v >= N) break;
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kRingPad; k++)
            if (k < n) {
                const int l = kSgPer * k + i;
                acc += silu(p[i][k] + at_lane(ex.x, l) * e0 + at_lane(ex.y, l) * e1);
            }
        for (int k = kRingPad; k < n; k++) {
            const int s = k * N + v, j = m.ring[s];
            acc += silu(P[(size_t)j * kSgW + c] + eps[2 * s] * e0 + eps[2 * s + 1] * e1);
        }
        M[(size_t)v * kSgW + c] = acc * (1.0f / 6.0f);
    }
}

// Pull form of the message backward: the spoke (u -> j) feeds M_u through
// P_j, so dP_j = sum over the neighbours u of j of (1/6) dM_u silu'(A_uj),
// A_uj = P_j + eps_uj E.  Each directed spoke is visited once, from j, so
// dE needs no atomics: per-block partials of sum dA eps.  At 40962 vertices
// 19.6 us, one vertex per wave 29.4 us.
__global__ void __launch_bounds__(256) k_sg_message_bwd(MeshView m, const int* __restrict__ twin,
                                                        const float* __restrict__ P, const float* __restrict__ eps,
                                                        const float* __restrict__ E, const float* __restrict__ dM,
                                                        float* __restrict__ dP, float* __restrict__ dE_partial)
{
    __shared__ float s_e[4][2 * kSgW];
    const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
    const int N = m.nv;
    const float e0 = E[c], e1 = E[kSgW + c];
    float de0 = 0.0f, de1 = 0.0f;
    const SgSteps st = sg_steps(N);
    for (int step = st.first; step < st.last; step++) {
        const int j0 = uniform((step * 4 + w) * kSgPer);
        const SgSlot t = sg_slot(m, j0);
        const bool in = t.s < t.n * N;    // slot below the valence: twin is set
        // the spoke (u -> j) in u's ring
        const float2 ex = reinterpret_cast<const float2*>(eps)[(in ? max(twin[t.s], 0) : 0) * N + t.j];
        float pj[kSgPer], d[kSgPer][kRingPad];
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            pj[i] = P[(size_t)min(j0 + i, N - 1) * kSgW + c];
#pragma unroll
            for (int k = 0; k < kRingPad; k++) d[i][k] = dM[(size_t)at_lane(t.j, kSgPer * k + i) * kSgW + c];
        }
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            const int j = j0 + i, n = at_lane(t.n, i);
            if (j >= N) break;
            float acc = 0.0f;
            auto spoke = [&](float dm, float y0, float y1) {
                const float da = (1.0f / 6.0f) * dm * silu_grad(pj[i] + y0 * e0 + y1 * e1);
                acc += da;
                de0 += da * y0;
                de1 += da * y1;
            };
#pragma unroll
            for (int k = 0; k < kRingPad; k++)
                if (k < n) spoke(d[i][k], at_lane(ex.x, kSgPer * k + i), at_lane(ex.y, kSgPer * k + i));
            for (int k = kRingPad; k < n; k++) {
                const int u = m.ring[k * N + j], s = max(twin[k * N + j], 0) * N + u;
                spoke(dM[(size_t)u * kSgW + c], eps[2 * s], eps[2 * s + 1]);
            }
            dP[(size_t)j * kSgW + c] = acc;
        }
    }
    s_e[w][c] = de0;
    s_e[w][kSgW + c] = de1;
    __syncthreads();
    if (w == 0) {
        float a0 = 0.0f, a1 = 0.0f;
        for (int q = 0; q < 4; q++) {
            a0 += s_e[q][c];
            a1 += s_e[q][kSgW + c];
        }
        dE_partial[(size_t)blockIdx.x * 2 * kSgW + c] = a0;
        dE_partial[(size_t)blockIdx.x * 2 * kSgW + kSgW + c] = a1;
    }
}

__device__ __forceinline__ float wave_sum(float x)
{
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// wave_sum of eight values at once, by the same additions: each of the first
// three steps leaves a lane half of the values it had, so ten lane moves do for
// all eight instead of six each.  Value k ends in the lanes whose bits 5, 4
// and 3 spell k; out[k] is uniform.
__device__ __forceinline__ void wave_sum8(const float (&x)[8], float (&out)[8])
{
    const int lane = threadIdx.x & 63;
    float a[4], b[2];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const bool up = lane & 32;
        a[i] = (up ? x[4 + i] : x[i]) + __shfl_xor(up ? x[i] : x[4 + i], 32, 64);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const bool up = lane & 16;
        b[i] = (up ? a[2 + i] : a[i]) + __shfl_xor(up ? a[i] : a[2 + i], 16, 64);
    }
    const bool up = lane & 8;
    float s = (up ? b[1] : b[0]) + __shfl_xor(up ? b[0] : b[1], 8, 64);
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
#pragma unroll
    for (int k = 0; k < 8; k++) out[k] = at_lane(s, 8 * k);
}

// --------------------------------------------------------------- output -----
// Per vertex s_vk, t_v, the force; with a target also the loss gradient
// g_v = d loss / d F_hat_v (F_hat = F / sigma_F) and per-block loss partials.
// The target is the exact gradient dE/dx (so F* = -target); the force is
// written as its negative (the gradient the HMC step expects).  At 40962
// vertices 19.4 us, one vertex per wave and a butterfly per spoke 36.7 us.
__global__ void __launch_bounds__(256) k_sg_output(MeshView m, const float* __restrict__ H, SgGeom geo,
                                                   const float* __restrict__ theta, float sigma_F,
                                                   const double* __restrict__ target, double* __restrict__ neg_force,
                                                   float* __restrict__ ghat, float* __restrict__ loss_partial,
                                                   float loss_scale)
{
    __shared__ float s_loss[4];
    const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
    const int N = m.nv;
    const float ws = theta[kSgOffWs + c], wt = theta[kSgOffWt + c], bs = theta[kSgOffBs], bt = theta[kSgOffBt];
    float lw = 0.0f;
    const SgSteps st = sg_steps(N);
    for (int step = st.first; step < st.last; step++) {
        const int v0 = uniform((step * 4 + w) * kSgPer);
        const SgSlot t = sg_slot(m, v0);
        const float* eh = geo.ehat + 3 * (size_t)t.s;
        const float ex = eh[0], ey = eh[1], ez = eh[2];
        const float nx = geo.nu[3 * t.v], ny = geo.nu[3 * t.v + 1], nz = geo.nu[3 * t.v + 2];
        float hv[kSgPer], hj[kSgPer][kRingPad];
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            hv[i] = H[(size_t)min(v0 + i, N - 1) * kSgW + c];
#pragma unroll
            for (int k = 0; k < kRingPad; k++) hj[i][k] = H[(size_t)at_lane(t.j, kSgPer * k + i) * kSgW + c];
        }
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            const int v = v0 + i, n = at_lane(t.n, i);
            if (v >= N) break;
            float x[kRingPad], sum[kRingPad];
#pragma unroll
            for (int k = 0; k < kRingPad; k++) x[k] = ws * hv[i] * hj[i][k];
            wave_sum8(x, sum);
            float F[3] = {0, 0, 0};
#pragma unroll
            for (int k = 0; k < kRingPad; k++)
                if (k < n) {
                    const float s = sum[k] + bs;
                    const int l = kSgPer * k + i;
                    F[0] += s * at_lane(ex, l);
                    F[1] += s * at_lane(ey, l);
                    F[2] += s * at_lane(ez, l);
                }
            for (int k = kRingPad; k < n; k++) {
                const int sl = k * N + v;
                const float s = wave_sum(ws * hv[i] * H[(size_t)m.ring[sl] * kSgW + c]) + bs;
                for (int q = 0; q < 3; q++) F[q] += s * geo.ehat[3 * sl + q];
            }
            const float tv = wave_sum(wt * hv[i]) + bt;
            F[0] += tv * at_lane(nx, i);
            F[1] += tv * at_lane(ny, i);
            F[2] += tv * at_lane(nz, i);
            if (c < 3) {
                const float f = c == 0 ? F[0] : (c == 1 ? F[1] : F[2]);
                if (neg_force) neg_force[3 * v + c] = -(double)sigma_F * f;
                if (target) {
                    const float r = f + (float)(target[3 * v + c] / sigma_F);
                    ghat[3 * v + c] = 2.0f * loss_scale * r;
                    lw += loss_scale * r * r;
                }
            }
        }
    }
    lw = wave_sum(lw);
    if (c == 0) s_loss[w] = lw;
    __syncthreads();
    if (threadIdx.x == 0 && loss_partial) loss_partial[blockIdx.x] = s_loss[0] + s_loss[1] + s_loss[2] + s_loss[3];
}

// Backward of the output layer:
//   dH_v = w_s * sum_k ((g_v - g_{j_k}) . e_vk) H_{j_k} + (g_v . nu_v) w_t
// (the spoke (j -> v) contributes through H_v with e_jv = -e_vj), and block
// partials of d w_s (64), d b_s, d w_t (64), d b_t.  At 40962 vertices
// 11.1 us, one vertex per wave 28.3 us.
__global__ void __launch_bounds__(256) k_sg_output_bwd(MeshView m, const float* __restrict__ H, SgGeom geo,
                                                       const float* __restrict__ theta,
                                                       const float* __restrict__ ghat, float* __restrict__ dH,
                                                       float* __restrict__ partial)
{
    __shared__ float s_p[4][kSgOutGrad];
    const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
    const int N = m.nv;
    const float ws = theta[kSgOffWs + c], wt = theta[kSgOffWt + c];
    float dws = 0.0f, dbs = 0.0f, dwt = 0.0f, dbt = 0.0f;
    const SgSteps st = sg_steps(N);
    for (int step = st.first; step < st.last; step++) {
        const int v0 = uniform((step * 4 + w) * kSgPer);
        const SgSlot t = sg_slot(m, v0);
        float hv[kSgPer], hj[kSgPer][kRingPad];
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            hv[i] = H[(size_t)min(v0 + i, N - 1) * kSgW + c];
#pragma unroll
            for (int k = 0; k < kRingPad; k++) hj[i][k] = H[(size_t)at_lane(t.j, kSgPer * k + i) * kSgW + c];
        }
        // g_v . e and g_j . e of the lane's slot, g_v . nu of its vertex
        const float gv0 = ghat[3 * t.v], gv1 = ghat[3 * t.v + 1], gv2 = ghat[3 * t.v + 2];
        auto along = [&](int sl, int j, float a, float b, float d, float& ds_v, float& ds_j) {
            const float ex = geo.ehat[3 * (size_t)sl], ey = geo.ehat[3 * (size_t)sl + 1],
                        ez = geo.ehat[3 * (size_t)sl + 2];
            ds_v = a * ex + b * ey + d * ez;
            ds_j = ghat[3 * j] * ex + ghat[3 * j + 1] * ey + ghat[3 * j + 2] * ez;
        };
        float sv, sj;
        along(t.s, t.j, gv0, gv1, gv2, sv, sj);
        const float sn = gv0 * geo.nu[3 * t.v] + gv1 * geo.nu[3 * t.v + 1] + gv2 * geo.nu[3 * t.v + 2];
#pragma unroll
        for (int i = 0; i < kSgPer; i++) {
            const int v = v0 + i, n = at_lane(t.n, i);
            if (v >= N) break;
            float acc = 0.0f;
            auto spoke = [&](float ds_v, float ds_j, float h) {
                acc += (ds_v - ds_j) * h;
                dws += ds_v * hv[i] * h;
                dbs += ds_v;
            };
#pragma unroll
            for (int k = 0; k < kRingPad; k++)
                if (k < n) spoke(at_lane(sv, kSgPer * k + i), at_lane(sj, kSgPer * k + i), hj[i][k]);
            for (int k = kRingPad; k < n; k++) {
                const int j = m.ring[k * N + v];
                float a, b;
                along(k * N + v, j, at_lane(gv0, i), at_lane(gv1, i), at_lane(gv2, i), a, b);
                spoke(a, b, H[(size_t)j * kSgW + c]);
            }
            const float dt = at_lane(sn, i);
            dH[(size_t)v * kSgW + c] = ws * acc + dt * wt;
            dwt += dt * hv[i];
            dbt += dt;
        }
    }
    // the parameter layout: w_s (64), b_s, w_t (64), b_t
    s_p[w][c] = dws;
    s_p[w][kSgW + 1 + c] = dwt;
    if (c == 0) {
        s_p[w][kSgW] = dbs;
        s_p[w][2 * kSgW + 1] = dbt;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kSgOutGrad; i += blockDim.x)
        partial[(size_t)blockIdx.x * kSgOutGrad + i] = s_p[0][i] + s_p[1][i] + s_p[2][i] + s_p[3][i];
}

// ------------------------------------------------------------------ Adam -----
__global__ void k_sg_adam(int n, float* __restrict__ theta, const float* __restrict__ grad, float* __restrict__ m1,
                          float* __restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = grad[i];
    const float a = b1 * m1[i] + (1.0f - b1) * g;
    const float b = b2 * m2[i] + (1.0f - b2) * g * g;
    m1[i] = a;
    m2[i] = b;
    theta[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// ------------------------------------------------------------ launchers -----
static inline int cdiv(int a, int b) { return (a + b - 1) / b; }
// workgroups of the vertex kernels (steps of 4 kSgPer vertices), a multiple of
// 8.  Those that leave partials take one step each up to 65536 vertices (fewer
// workgroups leave the last round of them uneven: a loss and gradient at 40962
// vertices takes 528 us with 2561 workgroups, 536 with 854 of three steps, 563
// with 1281 of two), and several above, where the partials would cost more.
static int vertex_blocks(int nv) { return cdiv(cdiv(nv, 4 * kSgPer), 8) * 8; }
static int partial_blocks(int nv) { return std::min(vertex_blocks(nv), 4096); }
// workgroups of the dense backward: as many tiles for each as for the others,
// at most one workgroup per CU
static int layer_blocks(int nv)
{
    const int tiles = cdiv(nv, kSgTile);
    return cdiv(tiles, cdiv(tiles, 256));
}

size_t sg_loss_rows(int nv) { return partial_blocks(nv); }
// partials of every segment of the parameter gradient
size_t sg_partial_floats(int nv)
{
    const size_t g = layer_blocks(nv), v = partial_blocks(nv);
    return g * (kSgLayers * (3 * kSgW * kSgW + kSgW) + kSgFeatPad * kSgW + kSgW) +
           v * (kSgLayers * 2 * kSgW + kSgOutGrad);
}

void sg_pack(const float* theta, const SgPacked& pk, hipStream_t s)
{
    hipLaunchKernelGGL(k_sg_pack, dim3(cdiv(kSgW * 2 * kSgW, 256)), dim3(256), 0, s, theta, pk);
}

void sg_features(const MeshView& m, const double* vprops, const Globals* g, const SgNorm& nrm, const SgGeom& geo,
                 float* f0, int* err, hipStream_t s)
{
    hipLaunchKernelGGL(k_sg_features, dim3(cdiv(m.nv, 128)), dim3(128), 0, s, m, vprops, g, nrm, geo, f0, err);
}

void sg_twin(const MeshView& m, int* twin, hipStream_t s)
{
    hipLaunchKernelGGL(k_sg_twin, dim3(cdiv(m.nv, 128)), dim3(128), 0, s, m, twin);
}

template <int KA, int KB, int MODE>
static void gemm(int N, const float* A1, const float* A2, const short* Bt, const float* bias, const float* res,
                 float* Y, float* H, hipStream_t s)
{
    hipLaunchKernelGGL((k_sg_gemm<KA, KB, MODE>), dim3(cdiv(N, 64)), dim3(256), 0, s, N, A1, A2, Bt, bias, res, Y,
                       H);
}

// Forward: features already in b.f0; with a target also the loss gradient.
void sg_forward(const MeshView& m, const SgBuffers& b, const SgGeom& geo, const float* theta, const SgPacked& pk,
                float sigma_F, const double* target, double* neg_force, hipStream_t s)
{
    const int N = m.nv;
    gemm<kSgFeatPad, 0, kSgAct>(N, b.f0, nullptr, pk.in_t, theta + kSgOffBin, nullptr, b.Z[0], b.H[0], s);
    for (int l = 0; l < kSgLayers; l++) {
        gemm<kSgW, 0, kSgStore>(N, b.H[l], nullptr, pk.u_t[l], nullptr, nullptr, b.P[l], nullptr, s);
        hipLaunchKernelGGL(k_sg_message, dim3(vertex_blocks(N)), dim3(256), 0, s, m, b.P[l], geo.eps,
                           theta + sg_off_E(l), b.M[l]);
        gemm<kSgW, kSgW, kSgAct>(N, b.H[l], b.M[l], pk.wv_t[l], theta + sg_off_b(l), b.H[l], b.Z[l + 1],
                                 b.H[l + 1], s);
    }
    const float loss_scale = 1.0f / (3.0f * (float)N);
    hipLaunchKernelGGL(k_sg_output, dim3(partial_blocks(N)), dim3(256), 0, s, m, b.H[kSgLayers], geo, theta,
                       sigma_F, target, neg_force, b.ghat, b.loss_partial, loss_scale);
}

// Backward after a forward with a target: the loss, and its parameter gradient
// into grad.
void sg_backward(const MeshView& m, const SgBuffers& b, const SgGeom& geo, const float* theta, const SgPacked& pk,
                 const int* twin, float* grad, hipStream_t s)
{
    const int N = m.nv, gv = partial_blocks(N), gl = layer_blocks(N);
    SgSegments seg{};
    int ns = 0;
    float* part = b.partial;
    // a segment of the reduction: `count` outputs from `rows` rows of partials
    auto segment = [&](float* out, int count, int rows) {
        float* p = part;
        seg.s[ns] = SgSegment{p, out, rows, count};
        seg.block0[ns + 1] = seg.block0[ns] + cdiv(count, kSgRedOut);
        ns++;
        part += (size_t)rows * count;
        return p;
    };
    const dim3 block(256);
    hipLaunchKernelGGL(k_sg_output_bwd, dim3(gv), block, 0, s, m, b.H[kSgLayers], geo, theta, b.ghat, b.dH,
                       segment(grad + kSgOffWs, kSgOutGrad, gv));
    // message-passing layers, last to first; b.dH holds dL/dH_l on entry
    for (int l = kSgLayers - 1; l >= 0; l--) {
        // residual: dH_l = dH_{l+1} + dZ W^T + dP U^T; the weights [W; V]
        float* wv = segment(grad + sg_off_W(l), 2 * kSgW * kSgW, gl);
        hipLaunchKernelGGL((k_sg_layer_bwd<kSgW, kSgW, true, 2>), dim3(gl), block, 0, s, N, b.H[l], b.M[l], b.dH,
                           b.Z[l + 1], pk.w_n[l], pk.v_n[l], b.dH, b.dM, wv, segment(grad + sg_off_b(l), kSgW, gl));
        hipLaunchKernelGGL(k_sg_message_bwd, dim3(gv), block, 0, s, m, twin, b.P[l], geo.eps, theta + sg_off_E(l),
                           b.dM, b.dP, segment(grad + sg_off_E(l), 2 * kSgW, gv));
        hipLaunchKernelGGL((k_sg_layer_bwd<kSgW, 0, false, 1>), dim3(gl), block, 0, s, N, b.H[l], nullptr, b.dP,
                           nullptr, pk.u_n[l], nullptr, b.dH, nullptr,
                           segment(grad + sg_off_U(l), kSgW * kSgW, gl), nullptr);
    }
    // input layer: H0 = silu(Z0)
    float* win = segment(grad + kSgOffWin, kSgFeatPad * kSgW, gl);
    hipLaunchKernelGGL((k_sg_layer_bwd<kSgFeatPad, 0, true, 0>), dim3(gl), block, 0, s, N, b.f0, nullptr, b.dH, b.Z[0],
                       nullptr, nullptr, nullptr, nullptr, win, segment(grad + kSgOffBin, kSgW, gl));
    const int nl = partial_blocks(N);
    seg.s[ns] = SgSegment{b.loss_partial, b.loss, nl, 1};
    seg.block0[ns + 1] = seg.block0[ns] + 1;
    hipLaunchKernelGGL(k_sg_reduce, dim3(seg.block0[ns + 1]), dim3(kSgRedOut * kSgRedRows), 0, s, seg);
}

void sg_adam(int n, float* theta, const float* grad, float* m1, float* m2, float lr, int step, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_sg_adam, dim3(cdiv(n, 256)), dim3(256), 0, s, n, theta, grad, m1, m2, lr, b1, b2, 1e-8f,
                       c1, c2);
}

}    // namespace tmh
