// Training of the voxel embedding MLP on gfx950, FP32 throughout.
//
// One step over A anchors with K = NH^3 window offsets each, V = A (K + 1)
// voxel slots (the anchor's target voxel, then the atlas voxel at every
// offset):
//   train_forward    embeddings of all slots, 16 slots a wave at a time, every
//                    layer on FP32 MFMA.
//   train_loss       one workgroup per anchor: teacher SSD and student
//                    distance for every offset, both log-softmaxes, the KL
//                    term, and the gradient with respect to every embedding
//                    of the anchor.
//   train_backward   per 16 slots: the hidden layers again, their gradients,
//                    and the products that make the parameter gradients,
//                    summed in accumulators over the wave's slots, then over
//                    the workgroup's waves in order.
//   grad_reduce      the workgroups' sums in a fixed order: the gradient does
//                    not depend on scheduling.
//   adam_step        Adam on the FP32 master parameters.
// Only embeddings and their gradients (16 floats a slot each) go through
// memory: the hidden activations of 3.4e5 slots would be 0.4 GB a step, and
// computing them twice costs 30 us of matrix time.
// No counterpart in the reference program.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "pct_internal.h"
#include "pct_mlp.h"
#include "pct_tiled.h"

namespace pct {

constexpr int kMaxWindow = 15; // NH

struct TrainArgs {
    const float* img;
    const float* atlas;       // [n][N]
    long long N;
    int nx, ny, nz, hw;
    const int* anchors;       // [A][4] z, x, y, atlas
    int n_anchors;
    int K;                    // NH^3
    int inside;               // 1: every window lies inside the volume with a margin of 1, and
                              // offsets to a neighbour fit 32 bits
    long long V;              // A * (K + 1)
    const float* params;      // device copy of the parameter vector
    float* emb;               // [V][16] embeddings
    float* demb;              // [V][16] d loss / d embedding
    float* loss;              // [A]
    float mu, inv_sd;
    float teacher_t, tau;
};

// ---------------------------------------------------------------------------
// MFMA layout
// ---------------------------------------------------------------------------
//
// All products are v_mfma_f32_16x16x4_f32, D(16x16) += A(16x4) B(4x16): lane
// (n = lane & 15, g = lane >> 4) holds A[n][g], B[g][n] and, in four registers
// i, D[4 g + i][n].  The layers run transposed (units x slots): register i of
// one layer's output tile, as it lies, is the B operand of a step whose four
// contraction indices are 4 g + i, so the next layer takes it without moving
// data, with its weights laid out to match.  The parameter gradients contract
// over slots instead: the rows go through an LDS tile [row][slot], from which a
// lane reads four slots 4 g + i of its row, operands of four steps.

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The first layer's contraction index (step s, group g): a feature, 30 for the
// constant 1 whose weight is the bias, 31 for nothing.  The central differences
// sit in lanes that hold their two patch values.
__device__ const unsigned char kFeatOf[4][8] = {{0, 1, 2, 3, 5, 6, 7, 8},
                                                {9, 11, 13, 15, 17, 18, 19, 20},
                                                {12, 14, 21, 23, 24, 25, 26, 29},
                                                {4, 22, 10, 16, 27, 28, 30, 31}};
constexpr int kFeatOne = 30, kFeatNone = 31;

// Weight of feature f (0 .. 31 as above) to hidden unit m.
__device__ __forceinline__ float first_weight(const float* __restrict__ p, int f, int m) {
    return f < kFeat ? p[kOffW1 + f * kHid + m] : f == kFeatOne ? p[kOffB1 + m] : 0.f;
}

// Patch index of the lane's slot s (the centre where the slot holds none).
__device__ __forceinline__ int patch_of(int g, int s) {
    const int f = kFeatOf[g][s];
    return f < 27 ? f : 13;
}

// Offsets of the lane's eight patch values from its voxel (used where a.inside).
__device__ __forceinline__ void patch_offsets(const TrainArgs& a, int g, int (&off)[8]) {
    const int plane = a.inside ? a.nx * a.ny : 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int p = patch_of(g, s);
        off[s] = (p / 9 - 1) * plane + ((p / 3) % 3 - 1) * a.ny + (p % 3 - 1);
    }
}

// The raw patch values of slot 16 tile + n, and whether the slot exists (a slot
// past the end reads the first anchor's voxel).
__device__ __forceinline__ void load_patch(const TrainArgs& a, long long tile, int n, int g,
                                           const int (&off)[8], float (&raw)[8], bool* ok) {
    const long long v0 = tile * 16;
    long long i = v0 / (a.K + 1);
    int k = (int)(v0 - i * (a.K + 1)) + n;
    while (k > a.K) {
        k -= a.K + 1;
        ++i;
    }
    *ok = v0 + n < a.V;
    if (!*ok) i = k = 0;
    const int4 an = reinterpret_cast<const int4*>(a.anchors)[i];   // z, x, y, atlas
    int z = an.x, x = an.y, y = an.z;
    const float* __restrict__ vol = a.img;
    if (k > 0) {
        const int c = k - 1, nw = 2 * a.hw + 1;
        z += c / (nw * nw) - a.hw;
        x += (c / nw) % nw - a.hw;
        y += c % nw - a.hw;
        vol = a.atlas + (long long)an.w * a.N;
    }
    if (a.inside) {   // uniform
        const float* __restrict__ p = vol + ((long long)z * a.nx + x) * a.ny + y;
#pragma unroll
        for (int s = 0; s < 8; ++s) raw[s] = p[off[s]];
    } else {
        // g(u) = 0 outside the volume, where the raw value would be mu
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int p = patch_of(g, s);
            const int zz = z + p / 9 - 1, xx = x + (p / 3) % 3 - 1, yy = y + p % 3 - 1;
            const bool in = zz >= 0 && zz < a.nz && xx >= 0 && xx < a.nx && yy >= 0 && yy < a.ny;
            raw[s] = in ? vol[((long long)zz * a.nx + xx) * a.ny + yy] : a.mu;
        }
    }
}

// The lane's eight first-layer inputs from its raw patch values.
__device__ __forceinline__ void features(const TrainArgs& a, int g, bool ok,
                                         const float (&raw)[8], float (&x)[8]) {
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = (raw[s] - a.mu) * a.inv_sd;
    const float d01 = 0.5f * (x[1] - x[0]), d23 = 0.5f * (x[3] - x[2]);
    if (g == 2) x[7] = d01;
    if (g == 3) {
        x[4] = d01;
        x[5] = d23;
        x[6] = 1.f;
        x[7] = 0.f;
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) x[s] = ok ? x[s] : 0.f;
}

__device__ __forceinline__ v4f relu(v4f v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = fmaxf(v[i], 0.f);
    return v;
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------

// Bound by the matrix pipe: 112 products of 32 cycles for 16 slots, 31 us at
// 3.4e5 slots (60 us measured, with the fragments' loads; 181 us with one thread
// per slot and the hidden activations written out).  Each wave keeps the 112
// weight fragments in registers and takes a run of consecutive tiles; the next
// tile's patch loads are in flight during the products.  Fetching the parameters
// through LDS changes nothing.
constexpr int kFwdWaves = 4;
constexpr int kWaves = 2048;   // waves that share the tiles (two per SIMD)
__global__ __launch_bounds__(kFwdWaves * 64, 2) void train_forward(TrainArgs a, long long tiles,
                                                                   long long chunk) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long t0 = ((long long)blockIdx.x * kFwdWaves + wv) * chunk;
    const long long t1 = min(tiles, t0 + chunk);
    if (t0 >= t1) return;   // per wave; no barrier below
    const float* __restrict__ p = a.params;
    float w1[4][8], w2[4][16], w3[16];
    v4f b2[4], b3;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
#pragma unroll
        for (int s = 0; s < 8; ++s) w1[m][s] = first_weight(p, kFeatOf[g][s], 16 * m + n);
#pragma unroll
        for (int q = 0; q < 16; ++q)
            w2[m][q] = p[kOffW2 + (16 * (q >> 2) + 4 * g + (q & 3)) * kHid + 16 * m + n];
#pragma unroll
        for (int i = 0; i < 4; ++i) b2[m][i] = p[kOffB2 + 16 * m + 4 * g + i];
    }
#pragma unroll
    for (int q = 0; q < 16; ++q)
        w3[q] = p[kOffW3 + (16 * (q >> 2) + 4 * g + (q & 3)) * kEmb + n];
#pragma unroll
    for (int i = 0; i < 4; ++i) b3[i] = p[kOffB3 + 4 * g + i];
    int off[8];
    patch_offsets(a, g, off);
    bool ok;
    float raw[8];
    load_patch(a, t0, n, g, off, raw, &ok);
    for (long long t = t0; t < t1; ++t) {
        float x[8];
        features(a, g, ok, raw, x);
        const bool ok_now = ok;
        load_patch(a, min(t + 1, t1 - 1), n, g, off, raw, &ok);
        v4f h1[4], h2[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) h1[m] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int m = 0; m < 4; ++m) h1[m] = mfma4(w1[m][s], x[s], h1[m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            h1[m] = relu(h1[m]);
            h2[m] = b2[m];
        }
#pragma unroll
        for (int q = 0; q < 16; ++q)
#pragma unroll
            for (int m = 0; m < 4; ++m) h2[m] = mfma4(w2[m][q], h1[q >> 2][q & 3], h2[m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) h2[m] = relu(h2[m]);
        v4f e[4] = {b3, (v4f){0.f, 0.f, 0.f, 0.f}, (v4f){0.f, 0.f, 0.f, 0.f},
                    (v4f){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int m = 0; m < 4; ++m) e[m] = mfma4(w3[4 * m + i], h2[m][i], e[m]);
        if (ok_now)
            *reinterpret_cast<v4f*>(a.emb + (t * 16 + n) * kEmb + 4 * g) =
                (e[0] + e[1]) + (e[2] + e[3]);
    }
}

// ---------------------------------------------------------------------------
// loss
// ---------------------------------------------------------------------------

constexpr int kLossThreads = 512;
constexpr int kLossWaves = kLossThreads / 64;

// Workgroup sum and maximum in a fixed order: within the waves, then over them.
__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();   // red's last readers are done
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int w = 1; w < kLossWaves; ++w) r += red[w];
    return r;
}
__device__ __forceinline__ float block_max(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int w = 1; w < kLossWaves; ++w) r = fmaxf(r, red[w]);
    return r;
}

__global__ __launch_bounds__(kLossThreads) void train_loss(TrainArgs a) {
    extern __shared__ float sh[];
    float* lp = sh;                                 // [K] teacher logits
    float* lq = sh + a.K;                           // [K] student logits
    float* gsum = sh + 2 * a.K;                     // [kLossThreads][kEmb + 1]
    __shared__ float red[kLossWaves];
    __shared__ float eT[kEmb];
    __shared__ float tp[27];                        // target patch
    const int i = blockIdx.x;
    const long long base = (long long)i * (a.K + 1);
    const float* __restrict__ E = a.emb + base * kEmb;
    float* __restrict__ D = a.demb + base * kEmb;
    const int* an = a.anchors + 4 * i;
    const int z = an[0], x = an[1], y = an[2];
    const float* __restrict__ A = a.atlas + (long long)an[3] * a.N;
    const long long plane = (long long)a.nx * a.ny;
    if (threadIdx.x < kEmb) eT[threadIdx.x] = E[threadIdx.x];
    if (threadIdx.x < 27) {
        const int p = threadIdx.x;
        tp[p] = a.img[(z + p / 9 - 1) * plane + (long long)(x + (p / 3) % 3 - 1) * a.ny +
                      (y + p % 3 - 1)];
    }
    __syncthreads();
    const int nw = 2 * a.hw + 1;
    float mp = -__builtin_huge_valf(), mq = -__builtin_huge_valf();
    for (int c = threadIdx.x; c < a.K; c += kLossThreads) {
        // inside by a margin of 1 (only an even NH has offsets beyond it)
        const int zc = min(max(z + c / (nw * nw) - a.hw, 1), a.nz - 2),
                  xc = min(max(x + (c / nw) % nw - a.hw, 1), a.nx - 2),
                  yc = min(max(y + c % nw - a.hw, 1), a.ny - 2);
        const float* __restrict__ q = A + zc * plane + (long long)xc * a.ny + yc;
        float ssd = 0.f;
#pragma unroll
        for (int p = 0; p < 27; ++p) {
            const float d = tp[p] - q[(p / 9 - 1) * plane + (long long)((p / 3) % 3 - 1) * a.ny +
                                      (p % 3 - 1)];
            ssd = fmaf(d, d, ssd);
        }
        const v4f* e = reinterpret_cast<const v4f*>(E + (long long)(1 + c) * kEmb);
        float dist = 0.f;
#pragma unroll
        for (int j = 0; j < kEmb; ++j) {
            const float d = eT[j] - e[j >> 2][j & 3];
            dist = fmaf(d, d, dist);
        }
        lp[c] = -ssd / a.teacher_t;
        lq[c] = -dist / a.tau;
        mp = fmaxf(mp, lp[c]);
        mq = fmaxf(mq, lq[c]);
    }
    mp = block_max(mp, red);
    mq = block_max(mq, red);
    float zp = 0.f, zq = 0.f;
    for (int c = threadIdx.x; c < a.K; c += kLossThreads) {
        zp += expf(lp[c] - mp);
        zq += expf(lq[c] - mq);
    }
    zp = block_sum(zp, red);
    zq = block_sum(zq, red);
    const float lzp = mp + logf(zp), lzq = mq + logf(zq);
    const float gscale = 1.f / (a.tau * (float)a.n_anchors);
    float kl = 0.f;
    float gT[kEmb];
#pragma unroll
    for (int j = 0; j < kEmb; ++j) gT[j] = 0.f;
    for (int c = threadIdx.x; c < a.K; c += kLossThreads) {
        const float lpn = lp[c] - lzp, lqn = lq[c] - lzq;
        const float p = expf(lpn), q = expf(lqn);
        kl = fmaf(p, lpn - lqn, kl);
        const float g = (p - q) * gscale;   // d loss / d dist_c
        const v4f* e = reinterpret_cast<const v4f*>(E + (long long)(1 + c) * kEmb);
        v4f* d = reinterpret_cast<v4f*>(D + (long long)(1 + c) * kEmb);
#pragma unroll
        for (int q4 = 0; q4 < kEmb / 4; ++q4) {
            const v4f ev = e[q4];
            v4f dv;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float diff = eT[4 * q4 + j] - ev[j];
                gT[4 * q4 + j] = fmaf(2.f * g, diff, gT[4 * q4 + j]);
                dv[j] = -2.f * g * diff;
            }
            d[q4] = dv;
        }
    }
    kl = block_sum(kl, red);
    // the target's gradient: thread (j, part) adds 16 of dimension j's terms,
    // then the 32 parts
#pragma unroll
    for (int j = 0; j < kEmb; ++j) gsum[threadIdx.x * (kEmb + 1) + j] = gT[j];
    __syncthreads();
    {
        constexpr int kParts = kLossThreads / kEmb;
        static_assert(kParts == 32, "one half wave per dimension");
        const int j = threadIdx.x / kParts, part = threadIdx.x % kParts;
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < kLossThreads / kParts; ++r)
            sum += gsum[(part + r * kParts) * (kEmb + 1) + j];
#pragma unroll
        for (int o = kParts / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kParts);
        if (part == 0) D[j] = sum;
    }
    if (threadIdx.x == 0) a.loss[i] = kl / (float)a.n_anchors;
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

// Bound by the matrix pipe: 288 products for 16 slots (96 for the hidden layers
// again, 80 for their gradients, 112 for the parameters'), 80 us at 3.4e5
// slots; the LDS reads of the fragments and rows take 60 % of that beside it.
// 163 us measured, against 168 us for the activations' gradients and 487 us for
// the parameters' from 0.4 GB of activations.  Eight waves share the weight
// fragments in LDS (176 of them; the 112 registers of parameter-gradient
// accumulators leave no room for them) and have an LDS tile each for the
// transposed rows.
constexpr int kBwdWaves = 8;
constexpr int kRowX = 128;   // rows of the inputs in a wave's tile
constexpr int kTileRows = kRowX + 32, kTileStride = 20;   // 16 slots, padded: no bank is hit twice
constexpr int kFrag1 = 0, kFrag2 = 2048, kFrag3 = 6144, kFrag2T = 7168, kBias2 = 11264,
              kFragEnd = 11328;
constexpr int kBwdLds = (kFragEnd + kBwdWaves * kTileRows * kTileStride) * 4;
static_assert(kNetParams <= kFragEnd, "the gradient's sum reuses the fragments' LDS");

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// D tile (16 rows from `row`) of 16 slots into the LDS tile.
__device__ __forceinline__ void put_rows(float* tile, int row, int n, int g, v4f v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) tile[(row + 4 * g + i) * kTileStride + n] = v[i];
}
// Operands of four steps over the 16 slots, rows from `row`.
__device__ __forceinline__ v4f get_rows(const float* tile, int row, int n, int g) {
    return *reinterpret_cast<const v4f*>(tile + (row + n) * kTileStride + 4 * g);
}

__global__ __launch_bounds__(kBwdWaves * 64, 2) void train_backward(TrainArgs a, long long tiles,
                                                                    long long chunk,
                                                                    float* partial) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    {
        const float* __restrict__ p = a.params;
        // fragment f of a section: float4 [f][lane], component i = step 4 f + i
        for (int e = threadIdx.x; e < kFragEnd; e += kBwdWaves * 64) {
            const int i = e & 3, l = (e >> 2) & 63, ln = l & 15, lg = l >> 4;
            float w;
            if (e < kFrag2) {
                const int f = e >> 8, m = f >> 1, st = 4 * (f & 1) + i;
                w = first_weight(p, kFeatOf[lg][st], 16 * m + ln);
            } else if (e < kFrag3) {
                const int f = (e - kFrag2) >> 8, m = f >> 2, kt = f & 3;
                w = p[kOffW2 + (16 * kt + 4 * lg + i) * kHid + 16 * m + ln];
            } else if (e < kFrag2T) {
                const int m = (e - kFrag3) >> 8;
                w = p[kOffW3 + (16 * m + ln) * kEmb + 4 * lg + i];
            } else if (e >= kBias2) {
                w = p[kOffB2 + e - kBias2];
            } else {
                const int f = (e - kFrag2T) >> 8, m = f >> 2, kt = f & 3;
                w = p[kOffW2 + (16 * m + ln) * kHid + 16 * kt + 4 * lg + i];
            }
            lds[e] = w;
        }
    }
    __syncthreads();
    float* tile = lds + kFragEnd + wv * kTileRows * kTileStride;
    auto frag = [&](int section, int f) {
        return *reinterpret_cast<const v4f*>(lds + section + (f * 64 + lane) * 4);
    };
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f g1[2][4], g2[4][4], g3[4];   // gradients of W1 (and b1), W2, W3
    float gb2[4], gb3 = 0.f;         // and of b2, b3: row 16 m + n, slots 4 g .. 4 g + 3
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        g1[0][m] = g1[1][m] = g3[m] = zero;
        gb2[m] = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) g2[k][m] = zero;
    }
    int off[8];
    patch_offsets(a, g, off);
    const long long t0 = ((long long)blockIdx.x * kBwdWaves + wv) * chunk;
    const long long t1 = min(tiles, t0 + chunk);
    if (t0 < t1) {   // uniform over the wave; no workgroup barrier inside
        bool ok;
        float raw[8];
        load_patch(a, t0, n, g, off, raw, &ok);
        v4f de_next = ok ? *reinterpret_cast<const v4f*>(a.demb + (t0 * 16 + n) * kEmb + 4 * g)
                         : zero;
        for (long long t = t0; t < t1; ++t) {
            float x[8];
            features(a, g, ok, raw, x);
#pragma unroll
            for (int s = 0; s < 8; ++s) tile[(kRowX + 8 * g + s) * kTileStride + n] = x[s];
            const v4f de = de_next;
            const long long tn = min(t + 1, t1 - 1);
            load_patch(a, tn, n, g, off, raw, &ok);
            de_next = ok ? *reinterpret_cast<const v4f*>(a.demb + (tn * 16 + n) * kEmb + 4 * g)
                         : zero;
            v4f h1[4], h2[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) h1[m] = zero;
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const v4f w = frag(kFrag1, 2 * m + f);
#pragma unroll
                    for (int i = 0; i < 4; ++i) h1[m] = mfma4(w[i], x[4 * f + i], h1[m]);
                }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                h1[m] = relu(h1[m]);
                h2[m] = *reinterpret_cast<const v4f*>(lds + kBias2 + 16 * m + 4 * g);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const v4f w = frag(kFrag2, 4 * m + k);
#pragma unroll
                    for (int i = 0; i < 4; ++i) h2[m] = mfma4(w[i], h1[k][i], h2[m]);
                }
            // through the third layer and its input's ReLU
            v4f d2[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                h2[m] = relu(h2[m]);
                const v4f w = frag(kFrag3, m);
                d2[m] = zero;
#pragma unroll
                for (int i = 0; i < 4; ++i) d2[m] = mfma4(w[i], de[i], d2[m]);
#pragma unroll
                for (int i = 0; i < 4; ++i) d2[m][i] = h2[m][i] > 0.f ? d2[m][i] : 0.f;
            }
            // W2: h1 (rows 0 .. 63) with d2 (rows 64 .. 127)
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                put_rows(tile, 16 * m, n, g, h1[m]);
                put_rows(tile, 64 + 16 * m, n, g, d2[m]);
            }
            // through the second layer meanwhile
            v4f d1[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) d1[m] = zero;
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const v4f w = frag(kFrag2T, 4 * m + k);
#pragma unroll
                    for (int i = 0; i < 4; ++i) d1[m] = mfma4(w[i], d2[k][i], d1[m]);
                }
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) d1[m][i] = h1[m][i] > 0.f ? d1[m][i] : 0.f;
            wave_lds_sync();
            {
                v4f rb[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    rb[m] = get_rows(tile, 64 + 16 * m, n, g);
                    gb2[m] += (rb[m][0] + rb[m][1]) + (rb[m][2] + rb[m][3]);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const v4f ra = get_rows(tile, 16 * k, n, g);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int m = 0; m < 4; ++m) g2[k][m] = mfma4(ra[i], rb[m][i], g2[k][m]);
                }
            }
            wave_lds_sync();
            // W3: h2 (rows 0 .. 63) with de (rows 64 .. 79)
#pragma unroll
            for (int m = 0; m < 4; ++m) put_rows(tile, 16 * m, n, g, h2[m]);
            put_rows(tile, 64, n, g, de);
            wave_lds_sync();
            {
                const v4f rb = get_rows(tile, 64, n, g);
                gb3 += (rb[0] + rb[1]) + (rb[2] + rb[3]);
                v4f ra[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) ra[k] = get_rows(tile, 16 * k, n, g);
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = 0; k < 4; ++k) g3[k] = mfma4(ra[k][i], rb[i], g3[k]);
            }
            wave_lds_sync();
            // W1: x (row 8 g + s of its own rows) with d1 (rows 64 .. 127)
#pragma unroll
            for (int m = 0; m < 4; ++m) put_rows(tile, 64 + 16 * m, n, g, d1[m]);
            wave_lds_sync();
            {
                v4f rb[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) rb[m] = get_rows(tile, 64 + 16 * m, n, g);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const v4f ra = get_rows(tile, kRowX + 16 * k, n, g);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int m = 0; m < 4; ++m) g1[k][m] = mfma4(ra[i], rb[m][i], g1[k][m]);
                }
            }
            wave_lds_sync();   // the rows are rewritten next
        }
    }
    // biases: the sum over the four groups of slots
#pragma unroll
    for (int o = 32; o > 8; o >>= 1) {
#pragma unroll
        for (int m = 0; m < 4; ++m) gb2[m] += __shfl_xor(gb2[m], o);
        gb3 += __shfl_xor(gb3, o);
    }
    // the workgroup's gradient: its waves' sums in wave order
    __syncthreads();
    for (int e = threadIdx.x; e < kNetParams; e += kBwdWaves * 64) lds[e] = 0.f;
    for (int w = 0; w < kBwdWaves; ++w) {
        __syncthreads();
        if (wv != w) continue;   // uniform over the wave; the barriers are shared
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int r = 16 * k + 4 * g + i, f = kFeatOf[r >> 3][r & 7];
                    if (f != kFeatNone)
                        lds[(f == kFeatOne ? kOffB1 : kOffW1 + f * kHid) + 16 * m + n] +=
                            g1[k][m][i];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    lds[kOffW2 + (16 * k + 4 * g + i) * kHid + 16 * m + n] += g2[k][m][i];
                lds[kOffW3 + (16 * m + 4 * g + i) * kEmb + n] += g3[m][i];
            }
        }
        if (g == 0) {
#pragma unroll
            for (int m = 0; m < 4; ++m) lds[kOffB2 + 16 * m + n] += gb2[m];
            lds[kOffB3 + n] += gb3;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kNetParams; e += kBwdWaves * 64)
        partial[(long long)blockIdx.x * kNetParams + e] = lds[e];
}

// Sums the workgroups' gradients: thread (p, part) every fourth of them, then
// the four parts.  Up to 256 partial vectors of 29 KB: 5 us, where one thread
// per parameter over 666 of them, one dependent load after another, took 157.
constexpr int kReduceParts = 4;
__global__ __launch_bounds__(256) void grad_reduce(const float* __restrict__ partial, int nblk,
                                                   float* __restrict__ grad) {
    __shared__ float sh[kReduceParts][64];
    const int c = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + c;
    float s = 0.f;
    if (p < kNetParams) {
#pragma unroll 8
        for (int b = part; b < nblk; b += kReduceParts) s += partial[(long long)b * kNetParams + p];
    }
    sh[part][c] = s;
    __syncthreads();
    if (part == 0 && p < PCT_MLP_NPARAMS) grad[p] = (sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c]);
}

__global__ void adam_step(float* __restrict__ params, float* __restrict__ m1,
                          float* __restrict__ m2, const float* __restrict__ grad, float lr,
                          float bc1, float bc2) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= kNetParams) return;
    const float g = grad[p];
    const float a = 0.9f * m1[p] + 0.1f * g;
    const float b = 0.999f * m2[p] + 0.001f * g * g;
    m1[p] = a;
    m2[p] = b;
    params[p] -= lr * (a / bc1) / (sqrtf(b / bc2) + 1e-8f);
}

// Device buffers of one training run, carved from the library workspace, and
// the split of the slots' tiles over waves and workgroups.
struct TrainPlan {
    int K = 0, n_anchors = 0, nblk = 0, fwd_blk = 0;
    long long V = 0, tiles = 0, chunk = 0;
    size_t o_params = 0, o_m1 = 0, o_m2 = 0, o_grad = 0, o_anchors = 0, o_emb = 0, o_demb = 0,
           o_loss = 0, o_partial = 0, bytes = 0;
};

static TrainPlan plan_training(int nh, int n_anchors) {
    TrainPlan t;
    t.K = nh * nh * nh;
    t.n_anchors = n_anchors;
    t.V = (long long)n_anchors * (t.K + 1);
    t.tiles = (t.V + 15) / 16;
    t.chunk = (t.tiles + kWaves - 1) / kWaves;
    const long long waves = (t.tiles + t.chunk - 1) / t.chunk;
    t.fwd_blk = (int)((waves + kFwdWaves - 1) / kFwdWaves);
    t.nblk = (int)((waves + kBwdWaves - 1) / kBwdWaves);
    auto align = [](size_t v) { return (v + 255) & ~(size_t)255; };
    size_t off = 0;
    t.o_params = off; off = align(off + 4 * PCT_MLP_NPARAMS);
    t.o_anchors = off; off = align(off + 16 * (size_t)n_anchors);   // copied with the parameters
    t.o_m1 = off; off = align(off + 4 * PCT_MLP_NPARAMS);
    t.o_m2 = off; off = align(off + 4 * PCT_MLP_NPARAMS);
    t.o_grad = off; off = align(off + 4 * PCT_MLP_NPARAMS);
    t.o_emb = off; off = align(off + 4 * (size_t)kEmb * t.V);
    t.o_demb = off; off = align(off + 4 * (size_t)kEmb * t.V);
    t.o_loss = off; off = align(off + 4 * (size_t)n_anchors);
    t.o_partial = off; off = align(off + 4 * (size_t)t.nblk * kNetParams);
    t.bytes = off;
    return t;
}

static int check_train_problem(const pct_problem* pb) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (pb->nh > kMaxWindow || pb->patch != 3) return PCT_ERR_UNSUPPORTED;
    const int r = (pb->nh - 1) / 2 + 1;
    if (pb->nx <= 2 * r || pb->ny <= 2 * r || pb->nz <= 2 * r) return PCT_ERR_DIMS;
    return PCT_OK;
}

// Pinned host memory of a device through which one gradient call at a time
// exchanges its small inputs and results: one asynchronous copy in, and the last
// kernels write the loss and the gradient straight into it.  A call with four
// copies from and to pageable memory, two of which the host waits for in turn,
// takes 319 us, this 264 (96x96x64, n = 3, NH = 11, 256 anchors; 250 of them in the
// kernels).  A call that finds it in use, needs more than kExchangeBytes or cannot
// have pinned memory makes those copies.  Given back by release_train_buffers.
constexpr size_t kExchangeBytes = (size_t)1 << 20;
struct ExchangeBuffer {
    std::mutex mu;   // held by the call that uses it
    char *host = nullptr, *dev = nullptr;
};
static ExchangeBuffer g_exchange[64];

struct Exchange {
    char *host = nullptr, *dev = nullptr;
    std::unique_lock<std::mutex> lk;
    Exchange(int device, size_t bytes) {
        if (device < 0 || device >= 64 || bytes > kExchangeBytes) return;
        ExchangeBuffer& b = g_exchange[device];
        lk = std::unique_lock<std::mutex>(b.mu, std::try_to_lock);
        if (!lk.owns_lock()) return;
        if (!b.host) {
            void *h = nullptr, *d = nullptr;
            if (hipHostMalloc(&h, kExchangeBytes, hipHostMallocMapped) != hipSuccess) {
                (void)hipGetLastError();
                return;
            }
            if (hipHostGetDevicePointer(&d, h, 0) != hipSuccess) {
                (void)hipGetLastError();
                (void)hipHostFree(h);
                return;
            }
            b.host = static_cast<char*>(h);
            b.dev = static_cast<char*>(d);
        }
        host = b.host;
        dev = b.dev;
    }
};

void release_train_buffers() {
    for (auto& b : g_exchange) {
        std::lock_guard<std::mutex> lk(b.mu);   // waits for a call that uses it
        if (b.host) (void)hipHostFree(b.host);
        b.host = b.dev = nullptr;
    }
}

// Enqueues forward, loss, backward and the gradient into `grad` (device or
// mapped host memory).
static int enqueue_step(const TrainPlan& t, const TrainArgs& a, char* w, float* grad,
                        hipStream_t s) {
    hipLaunchKernelGGL(train_forward, dim3(t.fwd_blk), dim3(kFwdWaves * 64), 0, s, a, t.tiles,
                       t.chunk);
    const size_t loss_lds = sizeof(float) * (2 * (size_t)t.K + kLossThreads * (kEmb + 1));
    hipLaunchKernelGGL(train_loss, dim3(t.n_anchors), dim3(kLossThreads), loss_lds, s, a);
    float* partial = reinterpret_cast<float*>(w + t.o_partial);
    hipLaunchKernelGGL(train_backward, dim3(t.nblk), dim3(kBwdWaves * 64), kBwdLds, s, a, t.tiles,
                       t.chunk, partial);
    hipLaunchKernelGGL(grad_reduce, dim3((PCT_MLP_NPARAMS + 63) / 64), dim3(256), 0, s, partial,
                       t.nblk, grad);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

// Lets the kernels with more than 64 KiB of LDS have it on the current device.
static int allow_train_lds(const TrainPlan& t) {
    const size_t loss_lds = sizeof(float) * (2 * (size_t)t.K + kLossThreads * (kEmb + 1));
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(train_backward),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kBwdLds) != hipSuccess ||
        hipFuncSetAttribute(reinterpret_cast<const void*>(train_loss),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)loss_lds) != hipSuccess)
        return PCT_ERR_HIP;
    return PCT_OK;
}

static TrainArgs make_train_args(const pct_problem* pb, const TrainPlan& t, const float* params,
                                 float tau, float teacher_t, const float* d_img,
                                 const float* d_atlas, char* w) {
    TrainArgs a;
    a.img = d_img;
    a.atlas = d_atlas;
    a.N = (long long)pb->nx * pb->ny * pb->nz;
    a.nx = pb->nx;
    a.ny = pb->ny;
    a.nz = pb->nz;
    a.hw = (pb->nh - 1) / 2;
    a.anchors = reinterpret_cast<const int*>(w + t.o_anchors);
    a.n_anchors = t.n_anchors;
    a.K = t.K;
    // anchors lie hw + 1 inside; an even NH has more offsets than its window
    a.inside = (pb->nh & 1) && (long long)pb->nx * pb->ny < (1LL << 30);
    a.V = t.V;
    a.params = reinterpret_cast<const float*>(w + t.o_params);
    a.emb = reinterpret_cast<float*>(w + t.o_emb);
    a.demb = reinterpret_cast<float*>(w + t.o_demb);
    a.loss = reinterpret_cast<float*>(w + t.o_loss);
    a.mu = params[kOffMu];
    a.inv_sd = params[kOffSd];
    a.teacher_t = teacher_t > 0.f ? teacher_t : (float)problem_divisor(pb);
    a.tau = tau;
    return a;
}

}  // namespace pct

using namespace pct;

extern "C" int pct_mlp_loss_grad_dev(const pct_problem* pb, const float* params,
                                     const int* anchors, int n_anchors, float tau,
                                     float teacher_t, const float* d_img, const float* d_atlas,
                                     double* loss, float* grad, pct_stream_t stream) {
    int rc = check_train_problem(pb);
    if (rc) return rc;
    if (!params || !anchors || n_anchors < 1 || !(tau > 0.f) || !d_img || !d_atlas || !loss ||
        !grad)
        return PCT_ERR_INVALID;
    const int r = (pb->nh - 1) / 2 + 1;
    for (int i = 0; i < n_anchors; ++i) {
        const int* an = anchors + 4 * i;
        if (an[0] < r || an[0] >= pb->nz - r || an[1] < r || an[1] >= pb->nx - r || an[2] < r ||
            an[2] >= pb->ny - r || an[3] < 0 || an[3] >= pb->n_atlas)
            return PCT_ERR_INVALID;
    }
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const TrainPlan t = plan_training(pb->nh, n_anchors);
    void* ws = nullptr;
    rc = ensure_workspace(dev, t.bytes, &ws);
    if (rc) return rc;
    rc = allow_train_lds(t);
    if (rc) return rc;
    char* w = static_cast<char*>(ws);
    TrainArgs a = make_train_args(pb, t, params, tau, teacher_t, d_img, d_atlas, w);
    const size_t in_bytes = t.o_anchors - t.o_params + 16 * (size_t)n_anchors;
    Exchange x(dev, in_bytes + 4 * (size_t)(PCT_MLP_NPARAMS + n_anchors));
    if (x.host) {
        std::memcpy(x.host, params, 4 * PCT_MLP_NPARAMS);
        std::memcpy(x.host + t.o_anchors - t.o_params, anchors, 16 * (size_t)n_anchors);
        float* h_grad = reinterpret_cast<float*>(x.host + in_bytes);
        float* d_grad = reinterpret_cast<float*>(x.dev + in_bytes);
        a.loss = d_grad + PCT_MLP_NPARAMS;
        rc = hipMemcpyAsync(w + t.o_params, x.host, in_bytes, hipMemcpyHostToDevice, s) ==
                     hipSuccess
                 ? enqueue_step(t, a, w, d_grad, s)
                 : PCT_ERR_HIP;
        // also after an error: the buffer is free once nothing uses it
        if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = PCT_ERR_HIP;
        if (rc) return rc;
        std::memcpy(grad, h_grad, 4 * PCT_MLP_NPARAMS);
        double sum = 0.0;
        for (int i = 0; i < n_anchors; ++i) sum += h_grad[PCT_MLP_NPARAMS + i];
        *loss = sum;
        return PCT_OK;
    }
    if (hipMemcpyAsync(w + t.o_params, params, 4 * PCT_MLP_NPARAMS, hipMemcpyHostToDevice, s) !=
            hipSuccess ||
        hipMemcpyAsync(w + t.o_anchors, anchors, 16 * (size_t)n_anchors, hipMemcpyHostToDevice,
                       s) != hipSuccess)
        return PCT_ERR_HIP;
    rc = enqueue_step(t, a, w, reinterpret_cast<float*>(w + t.o_grad), s);
    if (rc) return rc;
    std::vector<float> lv(n_anchors);
    if (hipMemcpyAsync(grad, w + t.o_grad, 4 * PCT_MLP_NPARAMS, hipMemcpyDeviceToHost, s) !=
            hipSuccess ||
        hipMemcpyAsync(lv.data(), w + t.o_loss, 4 * (size_t)n_anchors, hipMemcpyDeviceToHost,
                       s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return PCT_ERR_HIP;
    double sum = 0.0;
    for (float v : lv) sum += v;
    *loss = sum;
    return PCT_OK;
}

extern "C" int pct_mlp_train_dev(const pct_problem* pb, float* params,
                                 const pct_train_opts* opts, const float* d_img,
                                 const float* d_atlas, float* loss_trace, pct_stream_t stream) {
    int rc = check_train_problem(pb);
    if (rc) return rc;
    if (!params || !opts || opts->steps < 0 || opts->anchors < 1 || !(opts->tau > 0.f) ||
        !(opts->lr > 0.f) || !d_img || !d_atlas)
        return PCT_ERR_INVALID;
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const TrainPlan t = plan_training(pb->nh, opts->anchors);
    void* ws = nullptr;
    rc = ensure_workspace(dev, t.bytes, &ws);
    if (rc) return rc;
    rc = allow_train_lds(t);
    if (rc) return rc;
    char* w = static_cast<char*>(ws);
    float* d_params = reinterpret_cast<float*>(w + t.o_params);
    if (hipMemcpyAsync(d_params, params, 4 * PCT_MLP_NPARAMS, hipMemcpyHostToDevice, s) !=
            hipSuccess ||
        hipMemsetAsync(w + t.o_m1, 0, 4 * PCT_MLP_NPARAMS, s) != hipSuccess ||
        hipMemsetAsync(w + t.o_m2, 0, 4 * PCT_MLP_NPARAMS, s) != hipSuccess)
        return PCT_ERR_HIP;
    const TrainArgs a =
        make_train_args(pb, t, params, opts->tau, opts->teacher_t, d_img, d_atlas, w);
    const int r = (pb->nh - 1) / 2 + 1;
    const int iz = pb->nz - 2 * r, ix = pb->nx - 2 * r, iy = pb->ny - 2 * r;
    uint64_t st = opts->seed ^ 0x9E3779B97F4A7C15ULL;
    std::vector<int> anc(4 * (size_t)opts->anchors);
    std::vector<float> lv(opts->anchors);
    double b1 = 1.0, b2 = 1.0;
    for (int step = 0; step < opts->steps; ++step) {
        for (int i = 0; i < opts->anchors; ++i) {
            anc[4 * i + 0] = r + (int)(splitmix64(st) % (uint64_t)iz);
            anc[4 * i + 1] = r + (int)(splitmix64(st) % (uint64_t)ix);
            anc[4 * i + 2] = r + (int)(splitmix64(st) % (uint64_t)iy);
            anc[4 * i + 3] = (int)(splitmix64(st) % (uint64_t)pb->n_atlas);
        }
        if (hipMemcpyAsync(w + t.o_anchors, anc.data(), 16 * (size_t)opts->anchors,
                           hipMemcpyHostToDevice, s) != hipSuccess)
            return PCT_ERR_HIP;
        rc = enqueue_step(t, a, w, reinterpret_cast<float*>(w + t.o_grad), s);
        if (rc) return rc;
        b1 *= 0.9;
        b2 *= 0.999;
        hipLaunchKernelGGL(adam_step, dim3((kNetParams + 255) / 256), dim3(256), 0, s, d_params,
                           reinterpret_cast<float*>(w + t.o_m1),
                           reinterpret_cast<float*>(w + t.o_m2),
                           reinterpret_cast<const float*>(w + t.o_grad), opts->lr,
                           (float)(1.0 - b1), (float)(1.0 - b2));
        if (hipGetLastError() != hipSuccess) return PCT_ERR_HIP;
        // the anchor vector is rewritten next step and the loss is read now
        if (hipMemcpyAsync(lv.data(), w + t.o_loss, 4 * (size_t)opts->anchors,
                           hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return PCT_ERR_HIP;
        if (loss_trace) {
            double sum = 0.0;
            for (float v : lv) sum += v;
            loss_trace[step] = (float)sum;
        }
    }
    if (hipMemcpyAsync(params, d_params, 4 * kNetParams, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return PCT_ERR_HIP;
    return PCT_OK;
}
