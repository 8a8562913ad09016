/*
 * Training of the MLP surrogate on the GPU with the project's own kernels
 * (it has no counterpart in the reference).  One step over a batch of B
 * samples (B a multiple of 64):
 *
 *   k_mlp_pack     BF16 A-layout tiles of the weights (forward) and of
 *                  their transposes (backward) from the masters, and the
 *                  sample indices of the step (counter-based hash of seed,
 *                  step, position)
 *   k_mlp_train    one block per 64 samples, one wave per 16 features:
 *                  forward pass as in inference (BF16 weights and
 *                  activations, FP32 accumulation), squared-error loss,
 *                  backward pass with the same MFMA product, per-block
 *                  partial gradients
 *   k_mlp_reduce   gradients = sum of the per-block partials in a fixed
 *                  order (deterministic), and Adam on the FP32 master
 *                  parameters
 *
 * Backward of layer l (Z_l = W_l H_{l-1} + b_l, H_l = gelu(Z_l); the
 * output layer Y = W_o H_L + b_o has no activation), loss = sum (Y - T)^2
 * over the batch and outputs, dY = 2 (Y - T) / (B (D + 2)):
 *   dZ_l = dH_l * gelu'(Z_l)          FP32, rounded to BF16 for the products
 *   db_l = sum over points of dZ_l    FP32
 *   dW_l = dZ_l H_{l-1}^T             BF16 x BF16, FP32 accumulation
 *   dH_{l-1} = W_l^T dZ_l             BF16 x BF16, FP32 accumulation
 * Z_l (FP32) of the forward pass is kept in global memory for the backward
 * pass (a lane reads back what it wrote), H_l (BF16) feature-major in LDS.  The loss reported is the mean squared error
 * over the batch and outputs.
 */
#include "mlp_common.hpp"

namespace fj {

/* Counter-based 64-bit hash (splitmix64 finaliser). */
__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

/* Where a training step's samples come from: `batch` positions into idx. */
struct BatchDraw {
    uint64_t seed;
    int64_t step, n;
    int32_t batch;
    int32_t* idx; /* null: nothing to draw */
};

/* One 16 x 16 tile of C[i][j] = sum_pt A[i][pt] B[j][pt], A and B
 * feature-major rows over K = 64 points. */
__device__ __forceinline__ f32x4 outer_tile(const __bf16* a_rows, const __bf16* b_rows, int lane)
{
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const int o = (lane & 15) * SROW + 8 * (lane >> 4);
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(a_rows + o + kc * 32),
                                                      *(const bf16x8*)(b_rows + o + kc * 32), acc, 0, 0, 0);
    return acc;
}

/* out[4 tiles of 16 points] = 16 features of W (A tiles wA, KC chunks of 32
 * inputs) x rows (point-major LDS rows). */
template <int KC>
__device__ __forceinline__ void layer_row(const bf16x8* __restrict__ wA, const __bf16* rows, f32x4 (&acc)[4], int lane)
{
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
        const bf16x8 a = wA[kc * 64 + lane];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a, *(const bf16x8*)(rows + (nt * 16 + (lane & 15)) * SROW + kc * 32 + 8 * (lane >> 4)), acc[nt], 0, 0,
                0);
    }
}

/* Sum over the 16 points of a tile row: every lane of the 16 gets it. */
__device__ __forceinline__ float points_sum(float v)
{
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

/* Feature e's dZ over the four point tiles: the rounded products' sum, or
 * with fused the second of the products rounded and the others added
 * unrounded.  Both are within FP32's rounding; which feature takes which is
 * fixed because a network trained from a seed is part of a run's set-up (a
 * last bit of a bias gradient moves trained pressures by 1e-3), so the
 * rounding of the sums is spelt out and the compiler may not fuse them as it
 * happens to schedule them. */
__device__ __forceinline__ float tiles_sum(bool fused, const f32x4 (&acc)[4], const float (&dg)[4][4],
                                           const float (&dz)[4][4], int e)
{
#pragma clang fp contract(off)
    if (fused) {
        const float s = fmaf(acc[0][e], dg[0][e], dz[1][e]);
        return fmaf(acc[3][e], dg[3][e], fmaf(acc[2][e], dg[2][e], s));
    }
    return dz[0][e] + dz[1][e] + dz[2][e] + dz[3][e];
}

/* LDS of k_mlp_train in BF16 values: point-major rows, feature-major dZ
 * rows, feature-major H_0 (16 rows) and H_1 .. H_L (64 rows each). */
constexpr int train_lds(int n_hidden) { return (64 + 64 + 16 + 64 * n_hidden) * SROW; }

/* One training pass over 64 samples per block.  Each of the four waves owns
 * 16 of the 64 features of every layer (of the output layer: 16 of the
 * points), so a layer is 4 or 8 matrix instructions of a wave between two
 * barriers instead of 16 or 32; with one wave to all 64 features, and H
 * read back from global memory value by value, a pass over 16384 samples (a
 * wave per CU, all latency) took 66 us.  Parameter offsets (row major, as
 * fjsph_set_surrogate takes them): W_1 [64][D], W_2..W_L [64][64], W_o
 * [D+2][64]; b_1..b_L [64], b_o [D+2]. */
template <int D>
__global__ __launch_bounds__(TPB) void k_mlp_train(MlpTrain m)
{
    constexpr int NO = D + 2;
    static_assert(NWAVE == 4, "a wave per 16 features");
    extern __shared__ __attribute__((aligned(16))) __bf16 lds[];
    __shared__ int32_t sidx[64];
    __shared__ float sloss[4], sdy[16][64];
    __bf16* const pm = lds;             /* point-major rows */
    __bf16* const fa = pm + 64 * SROW;  /* feature-major dZ */
    __bf16* const h0 = fa + 64 * SROW;  /* feature-major H_0, then H_1 .. H_L */
    __bf16* const h1 = h0 + 16 * SROW;
    const int lane = threadIdx.x & 63;
    const int q = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int L = m.n_hidden;
    const int64_t w = blockIdx.x;
    const int64_t base = w * 64;
    const int f0 = d_feature(q, lane, 0); /* the lane's four features of a 64-wide layer */
    const bf16x8* Wf = (const bf16x8*)m.wf;
    const bf16x8* Wt = (const bf16x8*)m.wt;
    const int64_t B = m.batch;
    /* ---- forward */
    {
        const int32_t my = m.idx[base + lane];
        if (q == 0) sidx[lane] = my;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = q * 8 + e;
            const __bf16 v = __bf16(k < D ? m.X[(int64_t)my * 4 + k] : 0.f);
            pm[lane * SROW + k] = v;
            if (k < 16) h0[k * SROW + lane] = v;
        }
    }
    __syncthreads();
    f32x4 acc[4];
    for (int l = 1; l <= L; ++l) {
        if (l == 1) layer_row<1>(Wf + q * 64, pm, acc, lane);
        else layer_row<2>(Wf + (size_t)(4 + (l - 2) * 8 + q * 2) * 64, pm, acc, lane);
        float* Z = m.Z + ((size_t)(l - 1) * B + base) * SW;
        __bf16* H = h1 + (size_t)(l - 1) * 64 * SROW;
        const float* bl = m.b + (l - 1) * SW + f0; /* the caller's array in the no-alloc entry: any alignment */
        const float4 b = make_float4(bl[0], bl[1], bl[2], bl[3]);
        __syncthreads(); /* every wave has read the rows */
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int pt = d_point(nt, lane);
            const float4 z = make_float4(acc[nt][0] + b.x, acc[nt][1] + b.y, acc[nt][2] + b.z, acc[nt][3] + b.w);
            *(float4*)(Z + pt * SW + f0) = z;
            bf16x4 hv;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                hv[e] = __bf16(gelu_erf((&z.x)[e]));
                H[(f0 + e) * SROW + pt] = hv[e];
            }
            *(bf16x4*)(pm + pt * SROW + f0) = hv;
        }
        __syncthreads();
    }
    /* ---- output layer, loss and dY: wave q has the points of tile q */
    {
        f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
        const bf16x8* wo = Wf + (size_t)(4 + (L - 1) * 8) * 64;
        const int pt = d_point(q, lane);
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
            y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wo[kc * 64 + lane], *(const bf16x8*)(pm + pt * SROW + kc * 32 + 8 * (lane >> 4)), y, 0, 0, 0);
        const float gscale = 2.0f / (float(B) * float(NO));
        float dy[4], lsum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int f = d_feature(0, lane, e);
            dy[e] = 0.f;
            if (f < NO) {
                const float diff = y[e] + m.bo[f] - m.T[(int64_t)sidx[pt] * 8 + f];
                lsum += diff * diff;
                dy[e] = gscale * diff;
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
        if (lane == 0) sloss[q] = lsum;
#pragma unroll
        for (int e = 0; e < 4; ++e) sdy[d_feature(0, lane, e)][pt] = dy[e];
        __syncthreads(); /* every wave has read the rows */
        /* dY as BF16: point-major rows (K = outputs, padded to 32) and
         * feature-major rows (outputs x points, padded to 16 rows) */
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = __bf16(dy[e]);
            fa[d_feature(0, lane, e) * SROW + pt] = v[e];
        }
        *(bf16x4*)(pm + pt * SROW + d_feature(0, lane, 0)) = v;
        *(bf16x4*)(pm + pt * SROW + 16 + d_feature(0, lane, 0)) = bf16x4{__bf16(0.f), __bf16(0.f), __bf16(0.f), __bf16(0.f)};
    }
    __syncthreads();
    float* dWp = m.dWp + (size_t)w * m.nw;
    float* dbp = m.dbp + (size_t)w * m.nb;
    if (threadIdx.x == 0) m.lossp[w] = sloss[0] + sloss[1] + sloss[2] + sloss[3];
    if (q == 0) {
        /* the output biases' gradients: the four tiles of a feature, then
         * their points, as in the hidden layers */
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int f = d_feature(0, lane, e), p0 = lane & 15;
            const float t = points_sum(sdy[f][p0] + sdy[f][16 + p0] + sdy[f][32 + p0] + sdy[f][48 + p0]);
            if (p0 == 0 && f < NO) dbp[(size_t)L * SW + f] = t;
        }
    }
    /* output layer: dW_o = dY H_L^T, dH_L = W_o^T dY */
    {
        const f32x4 g = outer_tile(fa, h1 + ((size_t)(L - 1) * 64 + q * 16) * SROW, lane);
        float* dW = dWp + (size_t)(SW * D + (L - 1) * SW * SW);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int fo = d_feature(0, lane, e);
            if (fo < NO) dW[fo * SW + d_point(q, lane)] = g[e];
        }
    }
    layer_row<1>(Wt + (size_t)((L - 1) * 8 + q) * 64, pm, acc, lane);
    /* hidden layers, last to first */
    for (int l = L; l >= 1; --l) {
        const float* Z = m.Z + ((size_t)(l - 1) * B + base) * SW;
        float4 z[4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) z[nt] = *(const float4*)(Z + d_point(nt, lane) * SW + f0);
        __syncthreads(); /* every wave has read the rows */
        float dz[4][4], dg[4][4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int pt = d_point(nt, lane);
            bf16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dg[nt][e] = gelu_erf_grad((&z[nt].x)[e]);
                dz[nt][e] = acc[nt][e] * dg[nt][e];
                v[e] = __bf16(dz[nt][e]);
                fa[(f0 + e) * SROW + pt] = v[e];
            }
            *(bf16x4*)(pm + pt * SROW + f0) = v;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float t = points_sum(tiles_sum(q == 0 && e == 0, acc, dg, dz, e));
            if ((lane & 15) == 0) dbp[(size_t)(l - 1) * SW + f0 + e] = t;
        }
        __syncthreads();
        float* dW = dWp + (l == 1 ? 0 : (size_t)(SW * D + (l - 2) * SW * SW));
        const __bf16* a = fa + q * 16 * SROW;
        if (l == 1) {
            const f32x4 g = outer_tile(a, h0, lane);
            const int fi = d_point(0, lane);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (fi < D) dW[(f0 + e) * D + fi] = g[e];
        } else {
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const f32x4 g = outer_tile(a, h1 + ((size_t)(l - 2) * 64 + nt * 16) * SROW, lane);
#pragma unroll
                for (int e = 0; e < 4; ++e) dW[(f0 + e) * SW + d_point(nt, lane)] = g[e];
            }
            layer_row<2>(Wt + (size_t)((l - 2) * 8 + q * 2) * 64, pm, acc, lane);
        }
    }
}

/* Sums over the blocks of k_mlp_train, in block order: the weight
 * gradients, the bias gradients and the squared error (columns 0 .. nw - 1,
 * nw .. nw + nb - 1, nw + nb), and with Adam (Kingma and Ba; bias
 * corrections 1/c1, 1/c2) the update of the parameters by them.  The
 * partials (13 MB for a batch of 16384) come in by eight waves to 64
 * columns, RCHUNK blocks at a time through LDS, and one wave adds them up
 * from there; a lane adding up its column from memory had a load in flight
 * at a time and took 45 us a launch, three launches a step. */
constexpr int RWAVES = 8, RCHUNK = 128;

template <bool ADAM>
__global__ __launch_bounds__(64 * RWAVES) void k_mlp_reduce(MlpTrain m, int64_t nblocks, float* __restrict__ gw,
                                                            float* __restrict__ gb, float* __restrict__ sse,
                                                            MlpAdam ad)
{
    __shared__ float part[RCHUNK][64];
    const int lane = threadIdx.x & 63, r = threadIdx.x >> 6;
    const int64_t k = blockIdx.x * (int64_t)64 + lane;
    const int64_t np = m.nw + m.nb;
    const float* src = k < m.nw ? m.dWp + k : k < np ? m.dbp + (k - m.nw) : m.lossp;
    const int64_t stride = k < m.nw ? m.nw : k < np ? m.nb : 1;
    float s = 0.f;
    for (int64_t b0 = 0; b0 < nblocks; b0 += RCHUNK) {
        if (b0 > 0) __syncthreads();
#pragma unroll
        for (int q = 0; q < RCHUNK / RWAVES; ++q) {
            const int64_t b = b0 + q * RWAVES + r;
            part[q * RWAVES + r][lane] = (b < nblocks && k <= np) ? src[b * stride] : 0.f;
        }
        __syncthreads();
        if (r == 0) {
            const int nb = int(min(int64_t(RCHUNK), nblocks - b0));
#pragma unroll 16
            for (int q = 0; q < nb; ++q) s += part[q][lane];
        }
    }
    if (r != 0 || k > np) return;
    if (k == np) {
        if (sse) *sse = s;
        return;
    }
    if constexpr (ADAM) {
        const float gk = s;
        const float a = ad.b1 * ad.m1[k] + (1.f - ad.b1) * gk;
        const float b = ad.b2 * ad.m2[k] + (1.f - ad.b2) * gk * gk;
        ad.m1[k] = a;
        ad.m2[k] = b;
        ad.p[k] -= ad.lr * (a / ad.c1) / (sqrtf(b / ad.c2) + ad.eps);
    } else {
        (k < m.nw ? gw[k] : gb[k - m.nw]) = s;
    }
}

/* BF16 A-layout tiles of the weights: forward tiles (layer 1: 4 tiles of
 * W_1 padded to 64 x 32; hidden: 8 tiles each; output: 2 tiles of W_o
 * padded to 16 x 64), then backward tiles of the transposes (hidden l >= 2:
 * 8 tiles of W_l^T; output: 4 tiles of W_o^T padded to 64 x 32).  One
 * thread per (tile, lane); the threads after those draw the batch. */
template <int D>
__global__ __launch_bounds__(TPB) void k_mlp_pack(const float* __restrict__ w, int32_t n_hidden, bf16x8* __restrict__ wf,
                                                  bf16x8* __restrict__ wt, BatchDraw draw)
{
    constexpr int NO = D + 2;
    const int L = n_hidden;
    const int nf = 4 + (L - 1) * 8 + 2, nb = (L - 1) * 8 + 4;
    const int64_t gid = blockIdx.x * (int64_t)TPB + threadIdx.x;
    if (gid >= int64_t(nf + nb) * 64) {
        const int64_t j = gid - int64_t(nf + nb) * 64;
        if (draw.idx && j < draw.batch) {
            const uint64_t h = mix64(draw.seed ^ mix64(uint64_t(draw.step) * 0x100000001b3ull + uint64_t(j)));
            draw.idx[j] = int32_t(h % uint64_t(draw.n));
        }
        return;
    }
    const int tile = int(gid / 64), lane = int(gid % 64);
    const int i = lane & 15, k0 = 8 * (lane >> 4);
    bf16x8 v;
    if (tile < nf) {
        /* forward: A[i][k] = W[mt*16 + i][kc*32 + k] */
        int mt, kc, nout, nin;
        size_t off;
        if (tile < 4) {
            mt = tile; kc = 0; nout = SW; nin = D; off = 0;
        } else if (tile < 4 + (L - 1) * 8) {
            const int l = (tile - 4) / 8, t = (tile - 4) % 8;
            mt = t / 2; kc = t % 2; nout = SW; nin = SW; off = size_t(SW) * D + size_t(l) * SW * SW;
        } else {
            mt = 0; kc = tile - 4 - (L - 1) * 8; nout = NO; nin = SW; off = size_t(SW) * D + size_t(L - 1) * SW * SW;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int r = mt * 16 + i, c = kc * 32 + k0 + e;
            v[e] = __bf16(r < nout && c < nin ? w[off + size_t(r) * nin + c] : 0.f);
        }
        wf[gid] = v;
    } else {
        /* backward: A[i][k] = W^T[mt*16 + i][kc*32 + k] = W[kc*32 + k][mt*16 + i] */
        const int tb = tile - nf;
        int mt, kc, nout, nin;
        size_t off;
        if (tb < (L - 1) * 8) {
            const int l = tb / 8, t = tb % 8;
            mt = t / 2; kc = t % 2; nout = SW; nin = SW; off = size_t(SW) * D + size_t(l) * SW * SW;
        } else {
            mt = tb - (L - 1) * 8; kc = 0; nout = NO; nin = SW; off = size_t(SW) * D + size_t(L - 1) * SW * SW;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int r = kc * 32 + k0 + e, c = mt * 16 + i; /* W[r][c], r < nout, c < nin */
            v[e] = __bf16(r < nout && c < nin ? w[off + size_t(r) * nin + c] : 0.f);
        }
        wt[gid - int64_t(nf) * 64] = v;
    }
}

hipError_t launch_mlp_train(int dim, const MlpTrain& m, hipStream_t st)
{
    const dim3 g((unsigned)(m.batch / 64)), b(TPB);
    const size_t lds = size_t(train_lds(m.n_hidden)) * sizeof(__bf16);
    const auto k = dim == 2 ? k_mlp_train<2> : k_mlp_train<3>;
    /* more than the default 64 KiB from five hidden layers on */
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 int(train_lds(8) * sizeof(__bf16)));
        if (e != hipSuccess) return e;
    }
    MlpTrain arg = m;
    void* args[] = {&arg};
    return hipLaunchKernel((const void*)k, g, b, args, lds, st);
}

void launch_mlp_reduce(const MlpTrain& m, float* gw, float* gb, float* sse, hipStream_t st)
{
    const int64_t cols = m.nw + m.nb + 1;
    hipLaunchKernelGGL(k_mlp_reduce<false>, dim3((unsigned)((cols + 63) / 64)), dim3(64 * RWAVES), 0, st, m,
                       int64_t(m.batch / 64), gw, gb, sse, MlpAdam{});
}

void launch_mlp_reduce_adam(const MlpTrain& m, float* sse, const MlpAdam& ad, hipStream_t st)
{
    const int64_t cols = m.nw + m.nb + 1;
    hipLaunchKernelGGL(k_mlp_reduce<true>, dim3((unsigned)((cols + 63) / 64)), dim3(64 * RWAVES), 0, st, m,
                       int64_t(m.batch / 64), (float*)nullptr, (float*)nullptr, sse, ad);
}

int64_t mlp_tiles_fwd(int n_hidden) { return 4 + int64_t(n_hidden - 1) * 8 + 2; }
int64_t mlp_tiles_bwd(int n_hidden) { return int64_t(n_hidden - 1) * 8 + 4; }

static void pack(int dim, const float* w, int32_t n_hidden, void* wf, void* wt, const BatchDraw& draw, hipStream_t st)
{
    const int64_t n = (mlp_tiles_fwd(n_hidden) + mlp_tiles_bwd(n_hidden)) * 64 + (draw.idx ? draw.batch : 0);
    const auto k = dim == 2 ? k_mlp_pack<2> : k_mlp_pack<3>;
    hipLaunchKernelGGL(k, dim3(grid_of(n)), dim3(TPB), 0, st, w, n_hidden, (bf16x8*)wf, (bf16x8*)wt, draw);
}

void launch_mlp_pack(int dim, const float* w, int32_t n_hidden, void* wf, void* wt, hipStream_t st)
{
    pack(dim, w, n_hidden, wf, wt, BatchDraw{}, st);
}

void launch_mlp_pack_draw(int dim, const float* w, int32_t n_hidden, void* wf, void* wt, uint64_t seed, int64_t step,
                          int64_t n, int32_t batch, int32_t* idx, hipStream_t st)
{
    pack(dim, w, n_hidden, wf, wt, BatchDraw{seed, step, n, batch, idx}, st);
}

}  // namespace fj
