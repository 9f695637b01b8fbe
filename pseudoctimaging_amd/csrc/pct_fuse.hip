// Plain FP32 multi-atlas patch fusion for gfx950 (MI355X).
//
// Semantics follow the reference fusion loop (src/CPU/NewPatchedBrainPureC.cpp:
// 1184-1212 PatchSimilarity, 1350-1449 the OpenMP loop nest; the CUDA kernels
// src/GPU/PatchBasedPseudoCT.cu:162-641 compute the same function).  The
// design is new:
//
//  * Tiled kernel (EXEC_CHOICE SM).  For a fixed atlas a and offset d the
//    27-term SSD of every target voxel is a 3x3x3 box sum of the squared
//    difference D_d(u) = (T(u) - A_a(u+d))^2, so it is computed separably:
//    x by register pairs, z by register pairs, y across lanes with two DPP
//    adds (wave_shr:1 / wave_shl:1).  Lanes map to consecutive y (coalesced
//    global and conflict-free LDS accesses); each lane owns a BZ x BX block
//    of outputs in (z, x) and keeps the scaled target patch of that block in
//    VGPRs.  Per (atlas, dz) the workgroup stages the atlas MRI planes it
//    needs (BZ+2 planes) and the CT planes (BZ planes) for its tile in LDS;
//    the (dx, dy) loop then reads LDS at compile-time offsets.  MRI values are
//    pre-scaled by sqrt(log2(e)/div) so the weight is exp2(-SSD') with no
//    multiply.  A work item is (tile, group of atlases); it writes per-group
//    float partial sums P, S, and a finalize kernel adds the groups in a fixed
//    order and applies the reference's NaN rule (cpp:1437-1443), so results
//    are deterministic.
//  * Direct kernel (EXEC_CHOICE GM / GM2).  One lane per voxel, the 27-term
//    SSD per candidate straight from global memory, FP32.  An independent
//    GPU implementation used as the GM/GM2 surface and as a cross-check.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "pct_internal.h"

#include "pct_tiled.h"

namespace pct {

// P and S of COUNT partials from g on added in order, all their loads in flight
// at once.
template <int COUNT>
__device__ __forceinline__ void add_partials(const float* __restrict__ at, long long N, float& P,
                                             float& S) {
    float p[COUNT], q[COUNT];
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        p[k] = at[(2 * k) * N];
        q[k] = at[(2 * k + 1) * N];
    }
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        P += p[k];
        S += q[k];
    }
}

// Sum of the per-group partials in group order; border voxels get 0
// (the reference zeroes its output, cu:1693 / cpp:1606).  A large volume is bound
// by the partials' bytes, a small one by the latency of one load after another
// and by launching waves: hence eight partials at a time, and a wave per 64 voxels
// of a row.  30x34x22, n = 2, NH = 7 (14 partials): 5.2 -> 3.9 us, the call 18.0 ->
// 15.1; 64x64x32: 34.6 -> 32.3; 222x222x112, n = 10: 85 -> 83 us (442 MB).
constexpr int kFinRows = 4;
__global__ __launch_bounds__(64 * kFinRows) void fuse_finalize(const float* __restrict__ ws,
                                                               int n_groups, long long N, int nx,
                                                               int ny, int nz, int r,
                                                               float* __restrict__ out) {
    const int y = blockIdx.x * 64 + (threadIdx.x & 63);
    const int x = blockIdx.y * kFinRows + (threadIdx.x >> 6);
    const int z = blockIdx.z;
    if (y >= ny || x >= nx) return;
    const long long idx = ((long long)z * nx + x) * ny + y;
    const bool interior = z >= r && z < nz - r && x >= r && x < nx - r && y >= r && y < ny - r;
    float v = 0.f;
    if (interior) {
        float P = 0.f, S = 0.f;
        const float* __restrict__ at = ws + idx;
        int g = n_groups;
        for (; g >= 8; g -= 8, at += 16 * N) add_partials<8>(at, N, P, S);
        if (g & 4) {
            add_partials<4>(at, N, P, S);
            at += 8 * N;
        }
        if (g & 2) {
            add_partials<2>(at, N, P, S);
            at += 4 * N;
        }
        if (g & 1) add_partials<1>(at, N, P, S);
        v = fused_value(P, S);
    }
    out[idx] = v;
}

// Adds the n partial sums after the first to it, in order, as the finalize pass
// would (see launch_rounds).
__global__ __launch_bounds__(256) void fold_partials(float* __restrict__ ws, int n,
                                                     long long floats) {
    const long long i = blockIdx.x * 256LL + threadIdx.x;
    if (i >= floats) return;
    float v = ws[i];
    for (int j = 1; j <= n; ++j) v += ws[j * floats + i];
    ws[i] = v;
}

// ---------------------------------------------------------------------------
// direct kernel (GM / GM2 surface)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void fuse_direct(const float* __restrict__ img,
                                                   const float* __restrict__ atlas,
                                                   const float* __restrict__ label, long long N,
                                                   int nx, int ny, int nz, int hw, int n_atlas,
                                                   float k, float* __restrict__ out) {
    const int y = blockIdx.x * blockDim.x + threadIdx.x;
    const int x = blockIdx.y;
    const int z = blockIdx.z;
    if (y >= ny) return;
    const int r = hw + 1;
    const long long plane = (long long)nx * ny;
    const long long idx = z * plane + (long long)x * ny + y;
    if (!(z >= r && z < nz - r && x >= r && x < nx - r && y >= r && y < ny - r)) {
        out[idx] = 0.f;
        return;
    }
    float t[27];
#pragma unroll
    for (int p = 0; p < 27; ++p)
        t[p] = img[idx + (p / 9 - 1) * plane + (long long)((p / 3) % 3 - 1) * ny + (p % 3 - 1)];
    float P = 0.f, S = 0.f;
    for (int a = 0; a < n_atlas; ++a) {
        const float* __restrict__ A = atlas + (long long)a * N;
        const float* __restrict__ L = label + (long long)a * N;
        for (int dz = -hw; dz <= hw; ++dz)
            for (int dx = -hw; dx <= hw; ++dx)
                for (int dy = -hw; dy <= hw; ++dy) {
                    const long long c = idx + dz * plane + (long long)dx * ny + dy;
                    float ssd = 0.f;
#pragma unroll
                    for (int p = 0; p < 27; ++p) {
                        const float df =
                            t[p] - A[c + (p / 9 - 1) * plane + (long long)((p / 3) % 3 - 1) * ny +
                                     (p % 3 - 1)];
                        ssd = fmaf(df, df, ssd);
                    }
                    const float w = __builtin_amdgcn_exp2f(-ssd * k);
                    P = fmaf(w, L[c], P);
                    S += w;
                }
    }
    out[idx] = fused_value(P, S);
}

// The cross-term pairs of every voxel of atlases [0, n_atlas): with AA the
// 3x3x3 sum of (scale * A)^2 (zero outside the volume) and E = 2^-AA, the
// pair (L * E, E), or (+inf, E) where the CT value L lies beyond
// kXtLabelBound or is not a number, which the slab staging flags.  A
// workgroup owns 64 y x 4 x columns of one chunk of zc planes and sweeps it
// in z: the in-plane 3x3 sums of each plane's (4+2) x (64+2) tile, staged
// through LDS, enter a running sum over three planes.  Four planes are
// loaded per step (eight loads in flight per lane, issued with the step's
// CT loads before the previous step's sums), and chunking z
// (two halo planes per chunk) gives the grid enough workgroups to hide HBM
// latency on a single subject.  Every AA is ((s(z-1) + s(z)) + s(z+1)) with
// each in-plane sum in (dx, dy) order, whatever the chunking.
constexpr int kSqBoxY = 64, kSqBoxX = 4, kSqStep = 4;
constexpr int kSqThreads = kSqBoxY * kSqBoxX;
constexpr int kSqTile = (kSqBoxX + 2) * (kSqBoxY + 2);
constexpr int kSqLoads = (kSqTile + kSqThreads - 1) / kSqThreads;
constexpr int kSqMinChunk = 8;
__global__ __launch_bounds__(kSqThreads) void atlas_sq_box(const float* __restrict__ atlas,
                                                           const float* __restrict__ label,
                                                           long long N, int nx, int ny, int nz,
                                                           int n_atlas, int zc, int n_chunks,
                                                           float scale,
                                                           f32x2* __restrict__ le) {
    __shared__ float tile[kSqStep * kSqTile];
    const int ly = threadIdx.x % kSqBoxY, lx = threadIdx.x / kSqBoxY;
    const int y0 = blockIdx.x * kSqBoxY, x0 = blockIdx.y * kSqBoxX;
    const long long plane = (long long)nx * ny;
    const int y = y0 + ly, x = x0 + lx;
    // the lane's tile elements: in-plane offset, and whether they lie in the plane
    long long off[kSqLoads];
    bool in[kSqLoads];
#pragma unroll
    for (int j = 0; j < kSqLoads; ++j) {
        const int e = threadIdx.x + j * kSqThreads;
        const int rx = e / (kSqBoxY + 2), cy = e - rx * (kSqBoxY + 2);
        const int xx = x0 - 1 + rx, yy = y0 - 1 + cy;
        in[j] = e < kSqTile && xx >= 0 && xx < nx && yy >= 0 && yy < ny;
        off[j] = in[j] ? (long long)xx * ny + yy : 0;
    }
    const int n_work = n_atlas * n_chunks;
    for (int wi = blockIdx.z; wi < n_work; wi += gridDim.z) {
        const int at = wi / n_chunks, ck = wi - at * n_chunks;
        const int zs = ck * zc, ze = min(nz, zs + zc);   // output planes [zs, ze)
        const float* __restrict__ A = atlas + (long long)at * N;
        const float* __restrict__ L = label + (long long)at * N;
        f32x2* __restrict__ out = le + (long long)at * N;
        const bool col_in = x < nx && y < ny;
        const long long col = col_in ? (long long)x * ny + y : 0;
        float s_prev = 0.f, s_cur = 0.f;   // in-plane sums of planes q-2 and q-1
        // raw values of planes p .. p+3 at the lane's tile elements, loaded
        // from clamped planes (always inside the volume) so that all of a
        // step's loads are in flight together; the step that stores them
        // zeroes the positions outside the volume and past the chunk's last
        // plane ze, and scales the rest
        float v[kSqStep][kSqLoads];
        auto load_step = [&](int p) {
#pragma unroll
            for (int k = 0; k < kSqStep; ++k) {
                const long long qo = (long long)clampi(p + k, nz) * plane;
#pragma unroll
                for (int j = 0; j < kSqLoads; ++j) v[k][j] = A[qo + off[j]];
            }
        };
        // CT values of output planes p-1 .. p+2 (plane q completes output
        // q-1), read only for the outputs the step writes
        float lab[kSqStep];
        auto load_labels = [&](int p) {
#pragma unroll
            for (int k = 0; k < kSqStep; ++k)
                lab[k] = L[(long long)clampi(p + k - 1, nz) * plane + col];
        };
        load_step(zs - 1);
        load_labels(zs - 1);
        // planes zs-1 .. ze: plane q completes output plane q-1
        for (int p = zs - 1; p <= ze; p += kSqStep) {
            __syncthreads();   // the previous step's reads of the tiles are done
            // the loads are used only here, after the barrier: the compiler
            // would otherwise move each under its own branch and wait for it
#pragma unroll
            for (int k = 0; k < kSqStep; ++k)
#pragma unroll
                for (int j = 0; j < kSqLoads; ++j) asm volatile("" : "+v"(v[k][j]));
#pragma unroll
            for (int k = 0; k < kSqStep; ++k) {
                const int q = p + k;
                const bool qin = q >= 0 && q < nz && q <= ze;
#pragma unroll
                for (int j = 0; j < kSqLoads; ++j) {
                    const int e = threadIdx.x + j * kSqThreads;
                    if (e < kSqTile) tile[k * kSqTile + e] = (qin && in[j]) ? v[k][j] * scale : 0.f;
                }
            }
            __syncthreads();
            float lab_now[kSqStep];
#pragma unroll
            for (int k = 0; k < kSqStep; ++k) lab_now[k] = lab[k];
            // the next step's loads are in flight during this step's sums
            if (p + kSqStep <= ze) {
                load_step(p + kSqStep);
                load_labels(p + kSqStep);
            }
#pragma unroll
            for (int k = 0; k < kSqStep; ++k) {
                const int q = p + k;
                if (q > ze) break;
                const float* t = tile + k * kSqTile;
                float s = 0.f;
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                    for (int dy = 0; dy < 3; ++dy) {
                        const float w = t[(lx + dx) * (kSqBoxY + 2) + ly + dy];
                        s = fmaf(w, w, s);
                    }
                if (q - 1 >= zs && col_in) {
                    const float e = __builtin_amdgcn_exp2f(-((s_prev + s_cur) + s));
                    const float l = lab_now[k];
                    out[(q - 1) * plane + col] =
                        f32x2{fabsf(l) <= kXtLabelBound ? l * e : __builtin_inff(), e};
                }
                s_prev = s_cur;
                s_cur = s;
            }
        }
    }
}

// cpp:1583-1593, float32, same operation order.
__global__ void normalize_labels_kernel(float* __restrict__ v, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        v[i] = 255.0f * ((v[i] + 1024.0f) / 4095.0f);
}

// ---------------------------------------------------------------------------
// host side: configuration table, geometry, launches
// ---------------------------------------------------------------------------

using TiledFn = void (*)(TiledArgs);

struct TiledEntry {
    TileShape shape;
    int hw;
    TiledFn fn;
    int lds_bytes;
    // resident workgroups per CU reported by the runtime (registers and LDS);
    // 0 until a gfx950 device has been seen
    mutable int occupancy;
};

template <int W, int BX, int BZ, int NW, int HW, int FORM>
TiledEntry make_entry() {
    using C = TiledCfg<W, BX, BZ, NW, HW>;
    if constexpr (FORM == 1)
        return TiledEntry{{W, BX, BZ, NW, 1}, HW, &fuse_tiled_xt<W, BX, BZ, NW, HW>,
                          XtCfg<C>::LDS_BYTES, 0};
    else
        return TiledEntry{{W, BX, BZ, NW, 0}, HW, &fuse_tiled<W, BX, BZ, NW, HW>, C::LDS_BYTES, 0};
}

template <int W, int BX, int BZ, int NW, int FORM = 0>
void add_shape(std::vector<TiledEntry>& v) {
    v.push_back(make_entry<W, BX, BZ, NW, 1, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 2, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 3, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 4, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 5, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 6, FORM>());
    v.push_back(make_entry<W, BX, BZ, NW, 7, FORM>());
}

// The shapes compiled into the library (index = pct_tile_config.id).
const std::vector<TileShape>& shapes() {
    static const std::vector<TileShape> s = {
        {64, 4, 8, 4},   // 0: one 62-wide y segment per wave, 16 x rows per workgroup
        {32, 4, 8, 4},   // 1: two 30-wide y segments per wave, 32 x rows
        {32, 4, 4, 2},   // 2: small LDS footprint, several workgroups per CU
        {32, 2, 8, 4},   // 3: 16 x rows, 8 planes
        {64, 4, 4, 4},   // 4: 16 x rows, 4 planes
        {32, 4, 4, 4},   // 5: 32 x rows, 4 planes; two workgroups per CU up to NH=11
        {32, 2, 6, 4},   // 6: 16 x rows, 6 planes; two workgroups per CU up to NH=11
        {32, 2, 4, 4},   // 7: 16 x rows, 4 planes; three workgroups per CU up to NH=11
        {32, 4, 2, 4},   // 8: 32 x rows, 2 planes; three workgroups per CU up to NH=11
        {64, 2, 4, 4},   // 9: 8 x rows of 62-wide segments, 4 planes
        {32, 2, 2, 8},   // 10: 32 x rows, 2 planes, eight waves share one slab
        {32, 2, 2, 4},   // 11: 16 x rows, 2 planes; five workgroups per CU up to NH=11
        {32, 2, 2, 2},   // 12: 8 x rows, 2 planes, two waves; eight workgroups per CU
        {32, 2, 4, 8},   // 13: 32 x rows, 4 planes, eight waves
        {32, 4, 2, 8},   // 14: 64 x rows, 2 planes, eight waves
        // cross-term form (slab: BZ + 2 MRI planes and BZ planes of (L~, E) pairs)
        {32, 2, 4, 4, 1},   // 15: 16 x rows, 4 planes; two workgroups per CU up to NH=11
        {32, 2, 2, 4, 1},   // 16: 16 x rows, 2 planes; four workgroups per CU up to NH=11
        {32, 2, 2, 8, 1},   // 17: 32 x rows, 2 planes, eight waves
        {32, 4, 2, 4, 1},   // 18: 32 x rows, 2 planes
        {64, 2, 2, 4, 1},   // 19: 8 x rows of 62-wide segments, 2 planes
    };
    return s;
}

static const std::vector<TiledEntry>& entries() {
    static const std::vector<TiledEntry> e = [] {
        std::vector<TiledEntry> v;
        add_shape<64, 4, 8, 4>(v);
        add_shape<32, 4, 8, 4>(v);
        add_shape<32, 4, 4, 2>(v);
        add_shape<32, 2, 8, 4>(v);
        add_shape<64, 4, 4, 4>(v);
        add_shape<32, 4, 4, 4>(v);
        add_shape<32, 2, 6, 4>(v);
        add_shape<32, 2, 4, 4>(v);
        add_shape<32, 4, 2, 4>(v);
        add_shape<64, 2, 4, 4>(v);
        add_shape<32, 2, 2, 8>(v);
        add_shape<32, 2, 2, 4>(v);
        add_shape<32, 2, 2, 2>(v);
        add_shape<32, 2, 4, 8>(v);
        add_shape<32, 4, 2, 8>(v);
        add_shape<32, 2, 4, 4, 1>(v);
        add_shape<32, 2, 2, 4, 1>(v);
        add_shape<32, 2, 2, 8, 1>(v);
        add_shape<32, 4, 2, 4, 1>(v);
        add_shape<64, 2, 2, 4, 1>(v);
        return v;
    }();
    return e;
}

static const TiledEntry* find_entry(int shape_id, int hw) {
    if (shape_id < 0 || shape_id >= (int)shapes().size()) return nullptr;
    if (hw < 1 || hw > kMaxTiledHalfWindow) return nullptr;
    const auto& e = entries()[shape_id * kMaxTiledHalfWindow + (hw - 1)];
    return &e;
}

int validate_problem(const pct_problem* pb) {
    if (!pb) return PCT_ERR_INVALID;
    if (pb->nx < 1 || pb->ny < 1 || pb->nz < 1 || pb->n_atlas < 1) return PCT_ERR_INVALID;
    if (pb->nh < 1 || pb->patch != 3) return PCT_ERR_INVALID;
    if (!(pb->div >= 0.0) || !std::isfinite(pb->div)) return PCT_ERR_INVALID;
    if (pb->div == 0.0) {
        if (!(pb->sigma > 0.0) || !(pb->beta > 0.0)) return PCT_ERR_INVALID;
        if (!std::isfinite(pb->sigma) || !std::isfinite(pb->beta)) return PCT_ERR_INVALID;
    }
    const long long N = (long long)pb->nx * pb->ny * pb->nz;
    if (pb->nx > 65535 || pb->ny > 65535 || pb->nz > 65535) return PCT_ERR_TOO_LARGE;
    if (N * (long long)pb->n_atlas > (1LL << 40)) return PCT_ERR_TOO_LARGE;
    return PCT_OK;
}

double problem_divisor(const pct_problem* pb) {
    return pb->div > 0.0 ? pb->div : pct_weight_divisor(pb->sigma, pb->beta);
}

static int interior(int n, int r) { return std::max(0, n - 2 * r); }

bool make_geometry(const pct_problem* pb, int shape_id, int group, TileGeometry* g, int split) {
    const int hw = (pb->nh - 1) / 2;
    const TiledEntry* e = find_entry(shape_id, hw);
    if (!e) return false;
    const TileShape& s = e->shape;
    if (e->lds_bytes > kLdsPerCu) return false;
    const int S = 64 / s.seg_width;
    const int WX = s.waves * S * s.bx;
    const int OY = s.seg_width - 2;
    g->hw = hw;
    g->r = hw + 1;
    const int iy = interior(pb->ny, g->r), ix = interior(pb->nx, g->r), iz = interior(pb->nz, g->r);
    g->tiles_y = (iy + OY - 1) / OY;
    g->tiles_x = (ix + WX - 1) / WX;
    g->tiles_z = (iz + s.bz - 1) / s.bz;
    g->n_tiles = (long long)g->tiles_y * g->tiles_x * g->tiles_z;
    g->group = std::max(1, std::min(group, pb->n_atlas));
    g->n_groups = (pb->n_atlas + g->group - 1) / g->group;
    // more parts than dz: a multiple of them, with squared differences only
    const int nw = 2 * hw + 1;
    if (s.form == 1) split = std::min(split, nw);
    g->n_split = split <= nw ? std::max(1, split) : nw * std::min(split / nw, nw);
    g->slots = 0;
    g->n_items = g->n_tiles * g->n_parts();
    g->lds_bytes = e->lds_bytes;
    const int by_lds = kLdsPerCu / e->lds_bytes;
    const int by_waves = 32 / s.waves;  // 8 waves per SIMD slot budget, 4 SIMDs
    g->wg_per_cu = e->occupancy > 0 ? e->occupancy : std::max(1, std::min(by_lds, by_waves));
    return g->n_items < INT_MAX;
}

// ---- cost model -------------------------------------------------------------
//
// Time of one fusion call with a tile shape, atlas group and split of the
// window, in microseconds.  The form is the kernel's: per candidate a wave
// issues `plain` FP32 instructions, which pair between waves, 2 BZ BX DPP adds
// and BZ BX exps; per slab it copies rows; an item runs its candidates at the
// rate one wave alone reaches (latency) or at the SIMD's, whichever is slower for
// the waves resident; a grid runs floor(items / slots) rounds and a tail.  The
// coefficients are a least-squares fit on MI355X to 5492 timed (problem, shape,
// group, split) points of 66 problems: random sizes from 24 to 256 voxels, 1 to
// 10 atlases, NH 3 to 15, times from 9 us to 15 ms, squared-difference shapes
// also on data out of the cross-term range.  RMS error 7 %; the configuration
// the model picks is within 3.3 % of the fastest one timed on average (worst
// 20 %, at 15 us), where a fixed shape per window and one part were 1.0 to 3.9
// times slower, the more the smaller the problem.
namespace model {
constexpr double kPlain = 5.389, kExp = 2.013;        // cycles, SIMD saturated
constexpr double kAlone = 5.902, kAlone0 = 42.3;      // cycles per instruction and candidate, one wave
constexpr double kRow = 53.1, kSlab = 596.0;          // cycles per copied plane row, per slab
constexpr double kRound = 1003.0;                     // latency of one batch of copies
constexpr double kWaves = 0.698;                      // exponent of the resident waves
constexpr double kTail = 0.229;                       // part of a round the last items add
constexpr double kMhz = 2350.0;
constexpr double kLaunch = 6.5 + 4.3;                 // kernel and finalize launches
constexpr double kFinalize = 1.264 * 4 / 4e6;         // per float read or written
constexpr double kFinalRound = 0.6;                   // latency of eight partials
constexpr double kPairs0 = 7.3, kPairs = 1.532 * 16 / 4e6;   // pair pre-pass
// measured over modelled, by shape
constexpr double kShape[] = {1.12, 1.12, 1.02, 1.05, 0.96, 0.96, 0.99, 0.96, 0.88, 0.95,
                             1.00, 0.97, 0.96, 0.99, 0.88, 1.04, 1.07, 1.11, 1.01, 1.06};
}   // namespace model

// Microseconds one item takes with `wgs` workgroups resident per CU.
static double item_time(int shape_id, const TileGeometry& g, double wgs) {
    using namespace model;
    const TileShape& s = shapes()[shape_id];
    const double bx = s.bx, bz = s.bz, nh = 2 * g.hw + 1;
    const bool xt = s.form == 1, moves = !xt || s.bz == 2;   // slabs keep shared planes
    const double sums = s.bx == 2 && s.bz == 2 ? 20 : 2 * (bz + 2) * bx + 1.5 * bz * bx;
    const double plain = (xt ? 0 : (bz + 2) * (bx + 2)) + sums + 2 * bz * bx;
    const double busy = kPlain * plain + kExp * bz * bx;
    const double alone = kAlone * (plain + 2 * bz * bx) + kExp * bz * bx + kAlone0;
    const int segs = 64 / s.seg_width;
    const double rows = (double)(s.waves * segs * s.bx + 2 + 2 * g.hw) / s.waves *
                        ((s.seg_width + 2 * g.hw + 63) / 64);
    const double whole = rows * (xt ? 3 * bz + 2 : 2 * bz + 2);
    const double next = moves ? rows * (xt ? 3 : 2) : whole;
    const double batches = xt ? 1.5 * bz + 1 : bz + 1;
    const double slabs = std::ceil(nh / g.n_split);
    const double lines = g.n_split > nh ? std::ceil(nh * nh / g.n_split) : nh;   // dy
    const double copies = kRow * (whole + (slabs - 1) * next) + kSlab * slabs;
    const double latency = kRound * (batches + (slabs - 1) * (moves ? 1 : batches));
    const double waves = std::max(wgs * s.waves / 4.0, 0.25);   // resident per SIMD
    const double cycles =
        g.group * std::max(slabs * lines * nh * alone + copies + latency,
                           std::pow(waves, kWaves) * (slabs * lines * nh * busy + copies));
    return cycles / kMhz * kShape[shape_id];
}

static double model_cost(const pct_problem* pb, int shape_id, int group, TileGeometry* geo,
                         int split = 1) {
    using namespace model;
    TileGeometry g;
    if (!make_geometry(pb, shape_id, group, &g, split)) return -1;
    static_assert(sizeof(kShape) / sizeof(kShape[0]) == 20, "one factor per shape");
    if (geo) *geo = g;
    const double N = (double)pb->nx * pb->ny * pb->nz;
    const double per_cu = (double)g.n_items / kNumCu, slots = g.wg_per_cu;
    const double kernel =
        per_cu <= slots ? item_time(shape_id, g, std::max(1.0, std::ceil(per_cu)))
                        : (per_cu / slots + kTail) * item_time(shape_id, g, slots);
    double us = kernel + kLaunch + kFinalize * N * (1 + 2 * g.n_parts()) +
                kFinalRound * (g.n_parts() / 8);
    if (shapes()[shape_id].form == 1) us += kPairs0 + kPairs * N * pb->n_atlas;
    return us;
}

double model_class_cost(const std::vector<const pct_problem*>& pbs, int shape_id, int group) {
    using namespace model;
    std::vector<TileGeometry> geo(pbs.size());
    double items = 0, us = 0, slots = 1;
    for (size_t i = 0; i < pbs.size(); ++i) {
        if (!make_geometry(pbs[i], shape_id, std::min(group, pbs[i]->n_atlas), &geo[i])) return -1;
        items += (double)geo[i].n_items;
        slots = geo[i].wg_per_cu;
    }
    const double wgs = std::min(slots, std::max(1.0, std::ceil(items / kNumCu)));
    double rounds = 0, longest = 0;
    for (size_t i = 0; i < pbs.size(); ++i) {
        const double t = item_time(shape_id, geo[i], wgs);
        rounds += (double)geo[i].n_items / (kNumCu * wgs) * t;
        longest = std::max(longest, t);
        const double N = (double)pbs[i]->nx * pbs[i]->ny * pbs[i]->nz;
        us += kFinalize * N * (1 + 2 * geo[i].n_parts());
        if (shapes()[shape_id].form == 1) us += kPairs0 + kPairs * N * pbs[i]->n_atlas;
    }
    return us + std::max(longest, rounds + kTail * longest);
}

// Whether MRI values of about unit range lie in the cross-term range.  The
// library cannot know the values when it picks a shape; outside the range the
// cross-term shapes fall back to squared differences item by item, slower than
// the squared-difference shapes made for them (128x128x64, n=4, NH 5, sigma 0.25:
// 241 us against 169).
static bool unit_range_in_bound(const pct_problem* pb) {
    return std::sqrt(1.4426950408889634 / problem_divisor(pb)) <= (double)kXtBound;
}

// Whether the model may pick a cross-term shape.  Below NH 7 it never does: the
// candidates are too few to pay for the pair pre-pass.  Written down because the
// size of a caller's workspace depends on it.
static bool may_take_xterm(const pct_problem* pb) {
    return (pb->nh - 1) / 2 >= 3 && unit_range_in_bound(pb);
}

// Candidate splits of the window: whole, halves, thirds, pairs of dz, single ones,
// and halves, thirds, fifths and single dy of each.  The partial sums of a split may not need more memory than 256 MiB (or
// than the groups alone).  Groups are of one atlas: several to an item save up to
// 2 % from NH 7 on and 9 % at NH 3 (fewer partial sums), but one sum over ten
// atlases rounds five times as far off, and a host-buffer call copies the next
// group while one runs.
static std::vector<int> candidate_splits(const pct_problem* pb, int group) {
    const int nh = 2 * ((pb->nh - 1) / 2) + 1;
    const double per_part = 8.0 * pb->nx * pb->ny * pb->nz *
                            ((pb->n_atlas + group - 1) / group);
    std::vector<int> out;
    for (int s : {1, 2, 3, (nh + 1) / 2, nh, 2 * nh, 3 * nh, 5 * nh, nh * nh})
        if (s <= nh * nh && (s > 3 || s <= nh) && (out.empty() || s > out.back()) && (s == 1 || s * per_part <= 268435456.0))
            out.push_back(s);
    return out;
}

struct ShapeKey {
    int nx, ny, nz, n, nh;
    bool operator<(const ShapeKey& o) const {
        return std::tie(nx, ny, nz, n, nh) < std::tie(o.nx, o.ny, o.nz, o.n, o.nh);
    }
};

struct Config {
    int shape_id = -1, group = 1, split = 1;
};

static std::mutex g_cfg_mutex;
static std::map<ShapeKey, Config> g_tuned;
// the model's choices, so that a call costs a lookup and not 100 evaluations
// (about 10 us); cleared when it holds kPlanned of them
static std::map<std::pair<ShapeKey, bool>, Config> g_planned;
constexpr size_t kPlanned = 256;
static int g_forced_id = -1, g_forced_group = 0;

static Config model_choice(const pct_problem* pb, bool xt, bool* known) {
    Config best;
    double best_us = -1;
    *known = true;
    for (int sid = 0; sid < (int)shapes().size(); ++sid) {
        if (!xt && shapes()[sid].form == 1) continue;
        for (int sp : candidate_splits(pb, 1)) {
            const double us = model_cost(pb, sid, 1, nullptr, sp);
            if (us < 0) continue;
            if (best_us < 0 || us < best_us * 0.999) {
                best_us = us;
                best = Config{sid, 1, sp};
            }
        }
    }
    if (best.shape_id >= 0) *known = find_entry(best.shape_id, (pb->nh - 1) / 2)->occupancy > 0;
    return best;
}

// The forced or tuned configuration of a problem, if there is one (g_cfg_mutex held).
static bool fixed_config(const pct_problem* pb, Config* c) {
    if (g_forced_id >= 0) {
        *c = Config{g_forced_id, g_forced_group > 0 ? g_forced_group : 1, 1};
        return true;
    }
    const auto it = g_tuned.find(ShapeKey{pb->nx, pb->ny, pb->nz, pb->n_atlas, pb->nh});
    if (it == g_tuned.end()) return false;
    *c = it->second;
    return true;
}

// The configuration of a problem: forced, tuned, or the model's.
static bool choose(const pct_problem* pb, int* shape_id, double* cost, TileGeometry* geo) {
    Config c;
    {
        std::lock_guard<std::mutex> lk(g_cfg_mutex);
        if (!fixed_config(pb, &c)) {
            const bool xt = may_take_xterm(pb);
            const auto key =
                std::make_pair(ShapeKey{pb->nx, pb->ny, pb->nz, pb->n_atlas, pb->nh}, xt);
            const auto pl = g_planned.find(key);
            if (pl != g_planned.end()) {
                c = pl->second;
            } else {
                bool known = false;   // whether a device's occupancy went into it
                c = model_choice(pb, xt, &known);
                if (known) {
                    if (g_planned.size() >= kPlanned) g_planned.clear();
                    g_planned.emplace(key, c);
                }
            }
        }
    }
    if (c.shape_id < 0) return false;
    *shape_id = c.shape_id;
    if (!cost) return make_geometry(pb, c.shape_id, c.group, geo, c.split);
    *cost = model_cost(pb, c.shape_id, c.group, geo, c.split);
    return *cost >= 0;
}

// ---------------------------------------------------------------------------
// device / workspace management
// ---------------------------------------------------------------------------

struct DeviceState {
    bool checked = false;
    bool ok = false;
    void* ws = nullptr;
    size_t ws_bytes = 0;
    bool recorded = false;       // a graph runs in `ws` in rounds (see fuse_workspace)
    std::vector<void*> kept;     // such workspaces since outgrown
};

static std::mutex g_dev_mutex;
static std::map<int, DeviceState> g_dev;

int check_device(int* dev_out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return PCT_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lk(g_dev_mutex);
    DeviceState& st = g_dev[dev];
    if (!st.checked) {
        hipDeviceProp_t prop;
        st.checked = true;
        st.ok = hipGetDeviceProperties(&prop, dev) == hipSuccess &&
                std::strncmp(prop.gcnArchName, "gfx950", 6) == 0;
        if (st.ok) {
            for (const auto& e : entries()) {
                if (e.lds_bytes > kLdsPerCu) continue;
                (void)hipFuncSetAttribute(reinterpret_cast<const void*>(e.fn),
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          e.lds_bytes);
                int n = 0;
                if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                        &n, reinterpret_cast<const void*>(e.fn), e.shape.waves * 64,
                        (size_t)e.lds_bytes) == hipSuccess && n > 0)
                    e.occupancy = n;
                else
                    (void)hipGetLastError();
            }
        }
    }
    if (dev_out) *dev_out = dev;
    return st.ok ? PCT_OK : PCT_ERR_NO_DEVICE;
}

int ensure_workspace(int dev, size_t bytes, void** ptr) {
    std::lock_guard<std::mutex> lk(g_dev_mutex);
    DeviceState& st = g_dev[dev];
    if (st.ws_bytes < bytes) {
        if (st.ws) {
            if (hipDeviceSynchronize() != hipSuccess) return PCT_ERR_HIP;
            if (st.recorded)
                st.kept.push_back(st.ws);
            else
                (void)hipFree(st.ws);
            st.recorded = false;
            st.ws = nullptr;
            st.ws_bytes = 0;
        }
        if (hipMalloc(&st.ws, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return PCT_ERR_NO_MEMORY;
        }
        st.ws_bytes = bytes;
    }
    *ptr = st.ws;
    return PCT_OK;
}

bool is_xterm_shape(int shape_id) {
    return shape_id >= 0 && shape_id < (int)shapes().size() && shapes()[shape_id].form == 1;
}

size_t tiled_le_offset(const pct_problem* pb, int n_slots) {
    const size_t N = (size_t)pb->nx * pb->ny * pb->nz;
    return ((2 * (size_t)n_slots * N * sizeof(float)) + 255) & ~(size_t)255;
}

static size_t pairs_bytes(const pct_problem* pb) {
    const size_t N = (size_t)pb->nx * pb->ny * pb->nz;
    return ((size_t)pb->n_atlas * N * sizeof(f32x2) + 255) & ~(size_t)255;
}

size_t tiled_ws_bytes(const pct_problem* pb, int n_slots, int shape_id) {
    return tiled_le_offset(pb, n_slots) + (is_xterm_shape(shape_id) ? pairs_bytes(pb) : 0);
}

// Workspace that the configuration `choose` takes can run in: the partial sums of
// whole windows, and the pairs where the model may pick a cross-term shape.  It
// depends on the problem alone (not on what the model picks, nor on the device),
// grows with every extent and the atlases, and touches no GPU.
static size_t least_ws_bytes(const pct_problem* pb) {
    Config c;
    std::unique_lock<std::mutex> lk(g_cfg_mutex);
    const bool fixed = fixed_config(pb, &c);
    lk.unlock();
    if (!fixed)
        return tiled_le_offset(pb, pb->n_atlas) + (may_take_xterm(pb) ? pairs_bytes(pb) : 0);
    TileGeometry g;
    if (!make_geometry(pb, c.shape_id, c.group, &g)) return 0;
    return tiled_ws_bytes(pb, g.n_groups, c.shape_id);
}

// Workspaces that the geometry can run in: with all partial sums in memory, with
// those of whole windows, with one.
static std::vector<size_t> workspace_sizes(const pct_problem* pb, int shape_id,
                                           const TileGeometry& g) {
    std::vector<size_t> v;
    for (int slots : {g.n_parts(), g.n_groups, 1}) {
        const size_t bytes = tiled_ws_bytes(pb, slots, shape_id);
        if (v.empty() || bytes < v.back()) v.push_back(bytes);
    }
    return v;
}

// The library's workspace for a fusion: grown to the first of workspace_sizes that
// there is memory for.  Nothing grows while the stream is recorded into a graph, so a
// workspace that earlier calls left between them is used as it is; it is then kept
// for the graph when a later call outgrows it, until pct_release.
static int fuse_workspace(int dev, const pct_problem* pb, int shape_id, const TileGeometry& g,
                          hipStream_t stream, void** ptr, size_t* bytes) {
    std::vector<size_t> sizes;
    {
        std::lock_guard<std::mutex> lk(g_dev_mutex);
        DeviceState& st = g_dev[dev];
        *ptr = st.ws;
        *bytes = st.ws_bytes;
        if (st.ws_bytes >= tiled_ws_bytes(pb, g.n_parts(), shape_id)) return PCT_OK;
        sizes = workspace_sizes(pb, shape_id, g);
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (st.ws_bytes >= sizes.back()) {
            if (hipStreamIsCapturing(stream, &status) != hipSuccess) (void)hipGetLastError();
            if (status == hipStreamCaptureStatusActive) {
                st.recorded = true;
                return PCT_OK;
            }
        }
    }
    int rc = PCT_ERR_NO_MEMORY;
    for (size_t k = 0; k < sizes.size() && rc == PCT_ERR_NO_MEMORY; ++k) {
        *bytes = sizes[k];
        rc = ensure_workspace(dev, sizes[k], ptr);
    }
    return rc;
}

// Lets the geometry keep as many partial sums as fit `bytes`; false where not one does.
static bool fit_slots(const pct_problem* pb, int shape_id, size_t bytes, TileGeometry* g) {
    g->slots = 0;
    if (tiled_ws_bytes(pb, g->n_parts(), shape_id) <= bytes) return true;
    const size_t N = (size_t)pb->nx * pb->ny * pb->nz;
    const size_t fixed = is_xterm_shape(shape_id) ? pairs_bytes(pb) : 0;
    if (bytes < fixed) return false;
    // the sums end on a multiple of 256 bytes
    const size_t most = ((bytes - fixed) & ~(size_t)255) / (8 * N);
    g->slots = (int)std::min<size_t>(most, (size_t)g->n_parts() - 1);
    return g->slots > 0;
}

int launch_atlas_pairs(const pct_problem* pb, const float* atlas, const float* label,
                       int n_atlas, float scale, f32x2* le, hipStream_t stream) {
    if (n_atlas <= 0) return PCT_OK;
    const long long N = (long long)pb->nx * pb->ny * pb->nz;
    const int gy = (pb->ny + kSqBoxY - 1) / kSqBoxY, gx = (pb->nx + kSqBoxX - 1) / kSqBoxX;
    // z chunks: about 8192 workgroups (eight per CU, four waves each), chunks
    // of at least kSqMinChunk planes
    const long long base = (long long)gy * gx * n_atlas;
    int n_chunks = (int)std::min<long long>((8192 + base - 1) / base,
                                            std::max(1, pb->nz / kSqMinChunk));
    n_chunks = std::max(1, n_chunks);
    const int zc = (pb->nz + n_chunks - 1) / n_chunks;
    n_chunks = (pb->nz + zc - 1) / zc;
    const dim3 grid(gy, gx, (unsigned)std::min<long long>((long long)n_atlas * n_chunks, 65535));
    hipLaunchKernelGGL(atlas_sq_box, grid, dim3(kSqThreads), 0, stream, atlas, label, N, pb->nx,
                       pb->ny, pb->nz, n_atlas, zc, n_chunks, scale, le);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

static bool valid_choice(int choice) {
    return choice == PCT_CHOICE_GM || choice == PCT_CHOICE_GM2 || choice == PCT_CHOICE_SM ||
           choice == PCT_CHOICE_DIRECT;
}

// GM, GM2 and SM run the tiled kernel where it is instantiated; DIRECT and
// other window sizes run the direct kernel.
static bool is_tiled_choice(const pct_problem* pb, int choice) {
    return choice != PCT_CHOICE_DIRECT && (pb->nh - 1) / 2 <= kMaxTiledHalfWindow &&
           (pb->nh - 1) / 2 >= 1;
}

int launch_finalize(const pct_problem* pb, const TileGeometry& g, const float* ws, float* out,
                    hipStream_t stream) {
    const long long N = (long long)pb->nx * pb->ny * pb->nz;
    const dim3 fb(64 * kFinRows),
        fgrid((pb->ny + 63) / 64, (pb->nx + kFinRows - 1) / kFinRows, pb->nz);
    // parts that ran in rounds are one sum by now
    const int n = g.n_items <= 0 ? 0 : g.slots ? 1 : g.n_parts();
    hipLaunchKernelGGL(fuse_finalize, fgrid, fb, 0, stream, ws, n, N, pb->nx, pb->ny, pb->nz, g.r,
                       out);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

TiledArgs make_tiled_args(const pct_problem* pb, const TileGeometry& g, const float* img,
                          const float* atlas, const float* label, float* ws) {
    TiledArgs a;
    a.img = img;
    a.atlas = atlas;
    a.label = label;
    a.ws = ws;
    a.N = (long long)pb->nx * pb->ny * pb->nz;
    a.nx = pb->nx;
    a.ny = pb->ny;
    a.nz = pb->nz;
    a.r = g.r;
    a.tiles_y = g.tiles_y;
    a.tiles_x = g.tiles_x;
    a.n_tiles = (int)g.n_tiles;
    a.n_items = (int)g.n_items;
    a.n_atlas = pb->n_atlas;
    a.group = g.group;
    a.n_split = g.n_split;
    a.parts = g.n_split;
    a.first_part = 0;
    a.add = 0;
    const double div = problem_divisor(pb);
    a.scale = (float)std::sqrt(1.4426950408889634 / div);
    a.only = nullptr;
    a.le = nullptr;
    return a;
}

// Launches the single-problem tiled kernel of `shape_id` over the items
// described by `a` (no finalize pass).
int launch_tiled_items(const TiledArgs& a, int shape_id, int hw, hipStream_t stream) {
    const TiledEntry* e = find_entry(shape_id, hw);
    if (!e) return PCT_ERR_UNSUPPORTED;
    if (is_xterm_shape(shape_id) && !a.le) return PCT_ERR_INVALID;   // pair pass not run
    if (a.n_items <= 0) return PCT_OK;
    TiledArgs copy = a;
    void* kargs[] = {&copy};
    if (hipLaunchKernel(reinterpret_cast<const void*>(e->fn), dim3((unsigned)a.n_items),
                        dim3(e->shape.waves * 64), kargs, (size_t)e->lds_bytes,
                        stream) != hipSuccess)
        return PCT_ERR_HIP;
    return PCT_OK;
}

// Optional per-launch HIP events around the fusion kernels and the pruned
// kernel (see pct_kernel_timing).  Events are created once and reused.
struct KernelTimer {
    std::mutex mu;
    bool enabled = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> pool;
    size_t used = 0;
    static constexpr size_t kMax = 4096;

    // Returns the event pair to record around the next launch, or nulls.
    std::pair<hipEvent_t, hipEvent_t> next() {
        std::lock_guard<std::mutex> lk(mu);
        if (!enabled || used >= kMax) return {nullptr, nullptr};
        if (used == pool.size()) {
            hipEvent_t a = nullptr, b = nullptr;
            if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess)
                return {nullptr, nullptr};
            pool.emplace_back(a, b);
        }
        return pool[used++];
    }
};
static KernelTimer g_timer;

TimedLaunch::TimedLaunch(hipStream_t st) : s(st) {
    const auto ev = g_timer.next();
    begin = ev.first;
    end = ev.second;
    if (begin) (void)hipEventRecord(begin, s);
}

TimedLaunch::~TimedLaunch() {
    if (end) (void)hipEventRecord(end, s);
}

// The items of `a` where the workspace holds fewer partial sums than there are
// parts: as many consecutive parts a launch (whole groups, or parts of one) as it
// holds, each round's sums added to the first one, which the next round's first
// item goes on from.  The partial sums are added one after another in the order of
// the finalize pass, so the output has the same bits as with all of them in memory.
// In the least workspace 30x34x22, n = 2, NH = 7 takes 95 us (15 with all 14 parts in
// memory), 60x60x60, n = 1, NH = 15 473 us (127) and 40x66x30, n = 3, NH = 9 129 us (45);
// items of whole windows in the same memory took 83, 498 and 151.
static int launch_rounds(const TiledArgs& all, const TileGeometry& g, int shape_id,
                         hipStream_t stream) {
    const int groups = std::max(1, g.slots / g.n_split);   // a launch
    const int parts = std::min(g.slots, g.n_split);
    for (int g0 = 0; g0 < g.n_groups; g0 += groups)
        for (int first = 0; first < g.n_split; first += parts) {
            const int ng = std::min(groups, g.n_groups - g0);
            const int a0 = g0 * g.group, a1 = std::min(all.n_atlas, (g0 + ng) * g.group);
            TiledArgs a = all;
            a.atlas += (long long)a0 * a.N;
            a.label += (long long)a0 * a.N;
            if (a.le) a.le += (long long)a0 * a.N;
            a.n_atlas = a1 - a0;
            a.first_part = first;
            a.parts = std::min(parts, g.n_split - first);
            a.add = g0 > 0 || first > 0;
            a.n_items = (int)(g.n_tiles * ng * a.parts);
            const int rc = launch_tiled_items(a, shape_id, g.hw, stream);
            if (rc) return rc;
            if (ng * a.parts > 1) {
                hipLaunchKernelGGL(fold_partials, dim3((unsigned)((2 * a.N + 255) / 256)),
                                   dim3(256), 0, stream, a.ws, ng * a.parts - 1, 2 * a.N);
                if (hipGetLastError() != hipSuccess) return PCT_ERR_HIP;
            }
        }
    return PCT_OK;
}

static int launch_tiled(const pct_problem* pb, const float* img, const float* atlas,
                        const float* label, float* out, void* ws, size_t ws_bytes,
                        int shape_id, const TileGeometry& g, hipStream_t stream) {
    if (ws_bytes < tiled_ws_bytes(pb, g.n_slots(), shape_id)) return PCT_ERR_INVALID;
    TiledArgs a = make_tiled_args(pb, g, img, atlas, label, static_cast<float*>(ws));
    if (is_xterm_shape(shape_id) && g.n_items > 0) {
        f32x2* le = reinterpret_cast<f32x2*>(static_cast<char*>(ws) +
                                             tiled_le_offset(pb, g.n_slots()));
        const int rc = launch_atlas_pairs(pb, atlas, label, pb->n_atlas, a.scale, le, stream);
        if (rc) return rc;
        a.le = le;
    }
    if (g.n_items > 0) {
        TimedLaunch timed(stream);
        const int rc = g.slots ? launch_rounds(a, g, shape_id, stream)
                               : launch_tiled_items(a, shape_id, g.hw, stream);
        if (rc) return rc;
    }
    return launch_finalize(pb, g, static_cast<const float*>(ws), out, stream);
}

int launch_direct(const pct_problem* pb, const float* img, const float* atlas,
                         const float* label, float* out, hipStream_t stream) {
    const long long N = (long long)pb->nx * pb->ny * pb->nz;
    const int hw = (pb->nh - 1) / 2;
    const double div = problem_divisor(pb);
    const float k = (float)(1.4426950408889634 / div);
    const dim3 block(256), grid((pb->ny + 255) / 256, pb->nx, pb->nz);
    TimedLaunch timed(stream);
    hipLaunchKernelGGL(fuse_direct, grid, block, 0, stream, img, atlas, label, N, pb->nx, pb->ny,
                       pb->nz, hw, pb->n_atlas, k, out);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

}  // namespace pct

extern "C" int pct_kernel_timing(int enable) {
    pct::KernelTimer& t = pct::g_timer;
    std::lock_guard<std::mutex> lk(t.mu);
    t.enabled = enable != 0;
    if (t.enabled) t.used = 0;
    return PCT_OK;
}

extern "C" int pct_kernel_timing_read(double* total_ms, int* launches) {
    if (!total_ms || !launches) return PCT_ERR_INVALID;
    pct::KernelTimer& t = pct::g_timer;
    std::lock_guard<std::mutex> lk(t.mu);
    double sum = 0;
    for (size_t i = 0; i < t.used; ++i) {
        if (hipEventSynchronize(t.pool[i].second) != hipSuccess) return PCT_ERR_HIP;
        float ms = 0;
        if (hipEventElapsedTime(&ms, t.pool[i].first, t.pool[i].second) != hipSuccess)
            return PCT_ERR_HIP;
        sum += ms;
    }
    *total_ms = sum;
    *launches = (int)t.used;
    return PCT_OK;
}

// ---------------------------------------------------------------------------
// C ABI (GPU part)
// ---------------------------------------------------------------------------

using namespace pct;

extern "C" int pct_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return n;
}

extern "C" int pct_set_device(int device) {
    if (device < 0 || device >= pct_device_count()) return PCT_ERR_NO_DEVICE;
    if (hipSetDevice(device) != hipSuccess) {
        (void)hipGetLastError();
        return PCT_ERR_NO_DEVICE;
    }
    return check_device(nullptr);
}

extern "C" int pct_normalize_labels_dev(float* d_label, size_t n, pct_stream_t stream) {
    if (!d_label && n) return PCT_ERR_INVALID;
    int rc = check_device(nullptr);
    if (rc) return rc;
    if (n == 0) return PCT_OK;
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(normalize_labels_kernel, dim3(blocks), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), d_label, (long long)n);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

extern "C" size_t pct_fuse_workspace_size(const pct_problem* pb, int choice) {
    if (validate_problem(pb) != PCT_OK) return 0;
    if (!is_tiled_choice(pb, choice)) return 0;
    int sid = 0;
    TileGeometry g;
    if (!choose(pb, &sid, nullptr, &g)) return 0;
    return least_ws_bytes(pb);
}

static int fuse_dev_impl(const pct_problem* pb, const float* img, const float* atlas,
                         const float* label, float* out, int choice, void* ws, size_t ws_bytes,
                         bool own_ws, hipStream_t stream) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (!img || !atlas || !label || !out) return PCT_ERR_INVALID;
    if (!valid_choice(choice)) return PCT_ERR_INVALID;
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    if (!is_tiled_choice(pb, choice)) return launch_direct(pb, img, atlas, label, out, stream);
    int sid = 0;
    TileGeometry g;
    if (!choose(pb, &sid, nullptr, &g)) return PCT_ERR_UNSUPPORTED;
    if (own_ws) {
        rc = fuse_workspace(dev, pb, sid, g, stream, &ws, &ws_bytes);
        if (rc) return rc;
    } else if (!ws || ws_bytes < least_ws_bytes(pb) || (reinterpret_cast<uintptr_t>(ws) & 255)) {
        return PCT_ERR_INVALID;
    }
    if (!fit_slots(pb, sid, ws_bytes, &g)) return PCT_ERR_INVALID;
    return launch_tiled(pb, img, atlas, label, out, ws, ws_bytes, sid, g, stream);
}

extern "C" int pct_fuse_dev(const pct_problem* pb, const float* d_img, const float* d_atlas,
                            const float* d_label, float* d_out, int choice, pct_stream_t stream) {
    return fuse_dev_impl(pb, d_img, d_atlas, d_label, d_out, choice, nullptr, 0, true,
                         reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pct_fuse_dev_ws(const pct_problem* pb, const float* d_img, const float* d_atlas,
                               const float* d_label, float* d_out, int choice, void* d_ws,
                               size_t ws_bytes, pct_stream_t stream) {
    return fuse_dev_impl(pb, d_img, d_atlas, d_label, d_out, choice, d_ws, ws_bytes, false,
                         reinterpret_cast<hipStream_t>(stream));
}

// ---- allocation-free variant of pct_fuse_dev --------------------------------
//
// The partial sums live in `scratch`, a file-scope device array of fixed size
// that every GPU holds from module load to process end.  Its address on a
// device comes from hipGetSymbolAddress (the array's name in host code is
// only a stand-in), fetched once per device with that device current.  The
// run uses one atlas group (every item sums all atlases, so the partials are
// 2 N floats and every interior voxel is written by exactly one item before
// the finalize pass reads it: nothing needs clearing) and the
// squared-difference kernels, which need no cross-term pairs.

constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mutex;
static std::map<int, void*> g_scratch_ptr;   // device -> address of `scratch`

static int scratch_address(int dev, void** ptr) {
    std::lock_guard<std::mutex> lk(g_scratch_mutex);
    auto it = g_scratch_ptr.find(dev);
    if (it == g_scratch_ptr.end()) {
        void* p = nullptr;
        // `dev` is current: check_device read it with hipGetDevice
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return PCT_ERR_HIP;
        }
        it = g_scratch_ptr.emplace(dev, p).first;
    }
    *ptr = it->second;
    return PCT_OK;
}

// The squared-difference shape the model picks for one atlas group.
static bool choose_noalloc(const pct_problem* pb, int* shape_id, TileGeometry* geo) {
    double best = -1;
    for (int sid = 0; sid < (int)shapes().size(); ++sid) {
        if (is_xterm_shape(sid)) continue;
        TileGeometry g;
        const double c = model_cost(pb, sid, pb->n_atlas, &g);
        if (c >= 0 && (best < 0 || c < best * 0.999)) {
            best = c;
            *shape_id = sid;
            *geo = g;
        }
    }
    return best >= 0;
}

extern "C" int pct_fuse_dev_noalloc(const pct_problem* pb, const float* d_img, const float* d_atlas,
                                    const float* d_label, float* d_out, int choice,
                                    pct_stream_t stream) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (!d_img || !d_atlas || !d_label || !d_out) return PCT_ERR_INVALID;
    if (!valid_choice(choice)) return PCT_ERR_INVALID;
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (!is_tiled_choice(pb, choice))   // the direct kernel uses no scratch
        return launch_direct(pb, d_img, d_atlas, d_label, d_out, s);
    int sid = -1;
    TileGeometry g;
    if (!choose_noalloc(pb, &sid, &g)) return PCT_ERR_UNSUPPORTED;
    const size_t need = tiled_ws_bytes(pb, g.n_parts(), sid);
    if (need > kNoAllocScratchBytes) return PCT_ERR_TOO_LARGE;
    void* ws = nullptr;
    rc = scratch_address(dev, &ws);
    if (rc) return rc;
    TiledArgs a = make_tiled_args(pb, g, d_img, d_atlas, d_label, static_cast<float*>(ws));
    rc = launch_tiled_items(a, sid, g.hw, s);
    if (rc) return rc;
    return launch_finalize(pb, g, static_cast<const float*>(ws), d_out, s);
}

// Device buffers, streams and events of the host-buffer entry points, kept
// per device between calls (grown on demand, freed by pct_release).  One
// host-buffer call at a time runs on a device.
constexpr int kCopyChunks = 10;  // atlas chunks whose copies overlap the fusion
// Host buffers are staged through a ring of pinned buffers: the host
// threads copy one piece into a pinned buffer while the DMA engine moves
// the earlier pieces, which is about twice the rate of a copy from pageable
// memory.
constexpr int kPinBufs = 4;
constexpr size_t kPinBytes = (size_t)16 << 20;
struct HostCallState {
    std::mutex mu;
    float *img = nullptr, *atlas = nullptr, *label = nullptr, *out = nullptr;
    size_t n_cap = 0, na_cap = 0;
    // workspace of the host-buffer calls (partial sums, cross-term pairs, post-chain
    // lists): their own, so that they never share memory with device-buffer
    // calls still running on the caller's streams
    void* ws = nullptr;
    size_t ws_cap = 0;
    // chunk kernels alternate between two compute streams, so that the tail
    // of one chunk overlaps the start of the next
    hipStream_t compute = nullptr, compute2 = nullptr, copy = nullptr;
    hipEvent_t ev[kCopyChunks] = {};
    hipEvent_t join = nullptr;
    void* pin[kPinBufs] = {};          // pinned staging ring (all or none)
    hipEvent_t pin_ev[kPinBufs] = {};  // last transfer that used each buffer
    bool pin_busy[kPinBufs] = {};
    int pin_next = 0;
};
static std::mutex g_host_mutex;
static std::map<int, HostCallState*> g_host_state;

static HostCallState& host_state(int dev) {
    std::lock_guard<std::mutex> lk(g_host_mutex);
    HostCallState*& st = g_host_state[dev];
    if (!st) st = new HostCallState();
    return *st;
}

static void free_pinned(HostCallState& st) {
    for (int b = 0; b < kPinBufs; ++b) {
        if (st.pin[b]) (void)hipHostFree(st.pin[b]);
        if (st.pin_ev[b]) (void)hipEventDestroy(st.pin_ev[b]);
        st.pin[b] = nullptr;
        st.pin_ev[b] = nullptr;
    }
}

// Host -> device through the pinned ring, in pieces of kPinBytes on stream
// cs.  Without the ring (pinned memory refused) a plain pageable copy.
static int stage_h2d(HostCallState& st, void* d_dst, const void* h_src, size_t bytes,
                     hipStream_t cs) {
    if (!st.pin[0])
        return hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, cs) == hipSuccess
                   ? PCT_OK
                   : PCT_ERR_HIP;
    for (size_t o = 0; o < bytes; o += kPinBytes) {
        const size_t len = std::min(kPinBytes, bytes - o);
        const int b = st.pin_next;
        st.pin_next = (b + 1) % kPinBufs;
        if (st.pin_busy[b] && hipEventSynchronize(st.pin_ev[b]) != hipSuccess) return PCT_ERR_HIP;
        parallel_copy(st.pin[b], static_cast<const char*>(h_src) + o, len);
        if (hipMemcpyAsync(static_cast<char*>(d_dst) + o, st.pin[b], len, hipMemcpyHostToDevice,
                           cs) != hipSuccess ||
            hipEventRecord(st.pin_ev[b], cs) != hipSuccess)
            return PCT_ERR_HIP;
        st.pin_busy[b] = true;
    }
    return PCT_OK;
}

// Device -> host through the pinned ring on stream s: up to kPinBufs pieces
// in flight, each copied out by the host threads as it lands.  Returns when
// the host buffer holds the data.
static int stage_d2h(HostCallState& st, void* h_dst, const void* d_src, size_t bytes,
                     hipStream_t s) {
    if (!st.pin[0]) {
        if (hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return PCT_ERR_HIP;
        return PCT_OK;
    }
    const size_t pieces = (bytes + kPinBytes - 1) / kPinBytes;
    auto piece_len = [&](size_t i) { return std::min(kPinBytes, bytes - i * kPinBytes); };
    auto drain = [&](size_t i) {
        const int b = (int)(i % kPinBufs);
        if (hipEventSynchronize(st.pin_ev[b]) != hipSuccess) return PCT_ERR_HIP;
        parallel_copy(static_cast<char*>(h_dst) + i * kPinBytes, st.pin[b], piece_len(i));
        return PCT_OK;
    };
    for (size_t i = 0; i < pieces; ++i) {
        const int b = (int)(i % kPinBufs);
        if (i >= (size_t)kPinBufs) {
            const int rc = drain(i - kPinBufs);
            if (rc) return rc;
        } else if (st.pin_busy[b] && hipEventSynchronize(st.pin_ev[b]) != hipSuccess) {
            return PCT_ERR_HIP;
        }
        if (hipMemcpyAsync(st.pin[b], static_cast<const char*>(d_src) + i * kPinBytes,
                           piece_len(i), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipEventRecord(st.pin_ev[b], s) != hipSuccess)
            return PCT_ERR_HIP;
        st.pin_busy[b] = true;
    }
    for (size_t i = pieces > (size_t)kPinBufs ? pieces - kPinBufs : 0; i < pieces; ++i) {
        const int rc = drain(i);
        if (rc) return rc;
    }
    return PCT_OK;
}

static void free_host_buffers(HostCallState& st) {
    if (st.img) (void)hipFree(st.img);
    if (st.atlas) (void)hipFree(st.atlas);
    if (st.label) (void)hipFree(st.label);
    if (st.out) (void)hipFree(st.out);
    if (st.ws) (void)hipFree(st.ws);
    st.img = st.atlas = st.label = st.out = nullptr;
    st.ws = nullptr;
    st.n_cap = st.na_cap = st.ws_cap = 0;
}

// Grows the host-call workspace to `bytes` (the previous call drained every
// stream, so nothing still uses it).
static int host_workspace(HostCallState& st, size_t bytes, void** ws) {
    if (st.ws_cap < bytes) {
        if (st.ws) (void)hipFree(st.ws);
        st.ws = nullptr;
        st.ws_cap = 0;
        if (hipMalloc(&st.ws, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return PCT_ERR_NO_MEMORY;
        }
        st.ws_cap = bytes;
    }
    *ws = st.ws;
    return PCT_OK;
}

static int prepare_host_state(HostCallState& st, size_t N, size_t NA) {
    if (!st.compute) {
        if (hipStreamCreateWithFlags(&st.compute, hipStreamNonBlocking) != hipSuccess ||
            hipStreamCreateWithFlags(&st.compute2, hipStreamNonBlocking) != hipSuccess ||
            hipStreamCreateWithFlags(&st.copy, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&st.join, hipEventDisableTiming) != hipSuccess)
            return PCT_ERR_HIP;
        for (auto& e : st.ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
                return PCT_ERR_HIP;
        bool pinned = true;
        for (int b = 0; b < kPinBufs && pinned; ++b)
            pinned = hipHostMalloc(&st.pin[b], kPinBytes, hipHostMallocDefault) == hipSuccess &&
                     hipEventCreateWithFlags(&st.pin_ev[b], hipEventDisableTiming) == hipSuccess;
        if (!pinned) {
            // the pageable copies still work, only slower
            (void)hipGetLastError();
            free_pinned(st);
        }
    }
    // the previous call drained every stream
    for (int b = 0; b < kPinBufs; ++b) st.pin_busy[b] = false;
    st.pin_next = 0;
    if (st.n_cap < N || st.na_cap < NA) {
        free_host_buffers(st);   // the workspace too; host_workspace regrows it
        if (hipMalloc(&st.img, N * 4) != hipSuccess || hipMalloc(&st.atlas, NA * 4) != hipSuccess ||
            hipMalloc(&st.label, NA * 4) != hipSuccess || hipMalloc(&st.out, N * 4) != hipSuccess) {
            (void)hipGetLastError();
            free_host_buffers(st);
            return PCT_ERR_NO_MEMORY;
        }
        st.n_cap = N;
        st.na_cap = NA;
    }
    return PCT_OK;
}

// Host buffers in and out around the device fusion (cu:1687-1744); with
// `post`, the NaN fill, rounding and HU rescale run on the device before the
// copy back.  For the tiled kernel the atlases are copied in chunks of whole
// atlas groups on a copy stream, and each chunk's work items run on one of
// two compute streams as soon as its copy has landed, so the copies of the
// later chunks overlap the fusion of the earlier ones.  Every item writes the same
// partial sums as in one launch, and the finalize pass adds the groups in
// their fixed order: the output is that of pct_fuse_dev bit for bit.
static int fuse_host_impl(const pct_problem* pb, const float* img, const float* atlas,
                          const float* label, float* out, int choice, bool post) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (!img || !atlas || !label || !out) return PCT_ERR_INVALID;
    if (!valid_choice(choice)) return PCT_ERR_INVALID;
    const size_t N = (size_t)pb->nx * pb->ny * pb->nz;
    if (post && N >= (size_t)INT_MAX) return PCT_ERR_TOO_LARGE;   // device post chain's limit
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    const size_t NA = N * pb->n_atlas;
    HostCallState& st = host_state(dev);
    std::lock_guard<std::mutex> lk(st.mu);
    rc = prepare_host_state(st, N, NA);
    if (rc) return rc;
    hipStream_t s = st.compute, cs = st.copy;
    int sid = 0;
    TileGeometry g;
    const bool tiled = is_tiled_choice(pb, choice) && choose(pb, &sid, nullptr, &g);
    void* ws = nullptr;
    {
        const size_t post_need =
            std::max<size_t>(post ? postprocess_ws_bytes(pb->nh, pb->nx, pb->ny, pb->nz) : 0, 256);
        std::vector<size_t> sizes = {post_need};
        if (tiled) sizes = workspace_sizes(pb, sid, g);
        rc = PCT_ERR_NO_MEMORY;
        for (size_t k = 0; k < sizes.size() && rc == PCT_ERR_NO_MEMORY; ++k) {
            rc = host_workspace(st, std::max(post_need, sizes[k]), &ws);
            if (!rc && tiled) fit_slots(pb, sid, sizes[k], &g);
        }
    }
    f32x2* le = tiled && is_xterm_shape(sid)
                    ? reinterpret_cast<f32x2*>(static_cast<char*>(ws) +
                                               tiled_le_offset(pb, g.n_slots()))
                    : nullptr;
    // cu:1687-1699: host->device copies
    if (!rc) rc = stage_h2d(st, st.img, img, N * 4, cs);
    if (!rc && tiled) {
        // rounds go through all atlases in order, so they wait for all copies
        const int chunks = g.slots ? 1 : std::min(g.n_groups, kCopyChunks);
        for (int c = 0; c < chunks && !rc; ++c) {
            const int g0 = (int)((long long)c * g.n_groups / chunks);
            const int g1 = (int)((long long)(c + 1) * g.n_groups / chunks);
            const int a0 = g0 * g.group, a1 = std::min(pb->n_atlas, g1 * g.group);
            const size_t off = (size_t)a0 * N, len = (size_t)(a1 - a0) * N;
            rc = stage_h2d(st, st.atlas + off, atlas + off, len * 4, cs);
            if (!rc) rc = stage_h2d(st, st.label + off, label + off, len * 4, cs);
            if (rc) break;
            if (hipEventRecord(st.ev[c], cs) != hipSuccess ||
                hipStreamWaitEvent((c & 1) ? st.compute2 : s, st.ev[c], 0) != hipSuccess) {
                rc = PCT_ERR_HIP;
                break;
            }
            // the items of groups g0 .. g1-1: pointers offset to the chunk
            TiledArgs a = make_tiled_args(pb, g, st.img, st.atlas + off, st.label + off,
                                          static_cast<float*>(ws) + 2 * (size_t)(g0 * g.n_split) * N);
            a.n_atlas = a1 - a0;
            a.n_items = (int)(g.n_tiles * (g1 - g0) * g.n_split);
            hipStream_t cstream = (c & 1) ? st.compute2 : s;
            if (le) {
                // pairs of the chunk's atlases, computed as the single launch does
                rc = launch_atlas_pairs(pb, st.atlas + off, st.label + off, a1 - a0, a.scale,
                                        le + off, cstream);
                a.le = le + off;
            }
            if (!rc)
                rc = g.slots ? launch_rounds(a, g, sid, cstream)
                             : launch_tiled_items(a, sid, g.hw, cstream);
        }
        if (!rc && (hipEventRecord(st.join, st.compute2) != hipSuccess ||
                    hipStreamWaitEvent(s, st.join, 0) != hipSuccess))
            rc = PCT_ERR_HIP;
        if (!rc) rc = launch_finalize(pb, g, static_cast<const float*>(ws), st.out, s);
    } else if (!rc) {
        rc = stage_h2d(st, st.atlas, atlas, NA * 4, cs);
        if (!rc) rc = stage_h2d(st, st.label, label, NA * 4, cs);
        if (!rc && (hipEventRecord(st.ev[0], cs) != hipSuccess ||
                    hipStreamWaitEvent(s, st.ev[0], 0) != hipSuccess))
            rc = PCT_ERR_HIP;
        if (!rc) rc = fuse_dev_impl(pb, st.img, st.atlas, st.label, st.out, choice, ws,
                                    st.ws_cap, false, s);
    }
    if (!rc && post) rc = postprocess_dev_ws(pb->nh, pb->nx, pb->ny, pb->nz, st.out, ws, s);
    if (!rc) rc = stage_d2h(st, out, st.out, N * 4, s);
    // every stream is drained before returning, also after an error
    if (hipStreamSynchronize(cs) != hipSuccess && !rc) rc = PCT_ERR_HIP;
    if (hipStreamSynchronize(st.compute2) != hipSuccess && !rc) rc = PCT_ERR_HIP;
    if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = PCT_ERR_HIP;
    if (rc) (void)hipGetLastError();
    return rc;
}

namespace pct {
void release_host_buffers() {
    std::lock_guard<std::mutex> lk(g_host_mutex);
    for (auto& kv : g_host_state) {
        HostCallState* st = kv.second;
        {
            // waits for a call still running on this device; released
            // before the state (and its mutex) is deleted
            std::lock_guard<std::mutex> lk2(st->mu);
            int cur = 0;
            (void)hipGetDevice(&cur);
            (void)hipSetDevice(kv.first);
            if (st->compute) (void)hipStreamSynchronize(st->compute);
            if (st->compute2) (void)hipStreamSynchronize(st->compute2);
            if (st->copy) (void)hipStreamSynchronize(st->copy);
            free_host_buffers(*st);
            free_pinned(*st);
            for (auto& e : st->ev)
                if (e) (void)hipEventDestroy(e);
            if (st->join) (void)hipEventDestroy(st->join);
            if (st->compute) (void)hipStreamDestroy(st->compute);
            if (st->compute2) (void)hipStreamDestroy(st->compute2);
            if (st->copy) (void)hipStreamDestroy(st->copy);
            (void)hipSetDevice(cur);
        }
        delete st;
    }
    g_host_state.clear();
}
}  // namespace pct

extern "C" int pct_fuse_host(const pct_problem* pb, const float* img, const float* atlas,
                             const float* label, float* out, int choice) {
    return fuse_host_impl(pb, img, atlas, label, out, choice, false);
}

extern "C" int pct_pseudo_ct_host(const pct_problem* pb, const float* img, const float* atlas,
                                  const float* label, float* out_hu, int choice) {
    return fuse_host_impl(pb, img, atlas, label, out_hu, choice, true);
}

extern "C" int pct_tile_config_count(void) { return (int)shapes().size(); }

static void fill_config(int sid, double cost, const TileGeometry& g, pct_tile_config* out) {
    const TileShape& s = shapes()[sid];
    out->id = sid;
    out->seg_width = s.seg_width;
    out->bx = s.bx;
    out->bz = s.bz;
    out->waves = s.waves;
    out->atlas_group = g.group;
    out->lds_bytes = g.lds_bytes;
    out->items = g.n_items;
    out->est_cost = cost;
    out->measured_ms = -1;
    out->form = s.form;
}

extern "C" int pct_tile_config_choose(const pct_problem* pb, pct_tile_config* out) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (!out) return PCT_ERR_INVALID;
    int sid = 0;
    double cost = 0;
    TileGeometry g;
    if (!choose(pb, &sid, &cost, &g)) return PCT_ERR_UNSUPPORTED;
    fill_config(sid, cost, g, out);
    return PCT_OK;
}

extern "C" int pct_tile_config_force(int id, int atlas_group) {
    if (id >= (int)shapes().size()) return PCT_ERR_INVALID;
    std::lock_guard<std::mutex> lk(g_cfg_mutex);
    g_forced_id = id < 0 ? -1 : id;
    g_forced_group = atlas_group;
    return PCT_OK;
}

extern "C" int pct_autotune(const pct_problem* pb, const float* d_img, const float* d_atlas,
                            const float* d_label, float* d_out, int reps, pct_stream_t stream,
                            pct_tile_config* best) {
    int rc = validate_problem(pb);
    if (rc) return rc;
    if (!d_img || !d_atlas || !d_label || !d_out) return PCT_ERR_INVALID;
    int dev = 0;
    rc = check_device(&dev);
    if (rc) return rc;
    if ((pb->nh - 1) / 2 < 1 || (pb->nh - 1) / 2 > kMaxTiledHalfWindow) return PCT_ERR_UNSUPPORTED;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (reps < 1) reps = 1;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) return PCT_ERR_HIP;
    double best_ms = -1;
    Config best_c;
    TileGeometry best_g;
    // per shape: groups of one atlas and of all, and the model's split
    for (int sid = 0; sid < (int)shapes().size(); ++sid) {
        std::vector<Config> tries = {{sid, 1, 1}};
        if (pb->n_atlas > 1) tries.push_back({sid, pb->n_atlas, 1});
        double bc = -1;
        Config m;
        for (int sp : candidate_splits(pb, 1)) {
            const double c = model_cost(pb, sid, 1, nullptr, sp);
            if (c >= 0 && (bc < 0 || c < bc * 0.999)) {
                bc = c;
                m = Config{sid, 1, sp};
            }
        }
        if (bc < 0) continue;
        if (m.split != 1) tries.push_back(m);
        for (const Config& t : tries) {
            TileGeometry g;
            if (!make_geometry(pb, t.shape_id, t.group, &g, t.split)) continue;
            void* ws = nullptr;
            const size_t need = tiled_ws_bytes(pb, g.n_parts(), sid);
            rc = ensure_workspace(dev, need, &ws);
            if (rc == PCT_ERR_NO_MEMORY && t.split > 1) {
                rc = PCT_OK;   // the shape's other candidates need less
                continue;
            }
            if (rc) break;
            // warm-up
            rc = launch_tiled(pb, d_img, d_atlas, d_label, d_out, ws, need, sid, g, s);
            if (rc) break;
            (void)hipEventRecord(e0, s);
            for (int i = 0; i < reps && !rc; ++i)
                rc = launch_tiled(pb, d_img, d_atlas, d_label, d_out, ws, need, sid, g, s);
            (void)hipEventRecord(e1, s);
            if (hipEventSynchronize(e1) != hipSuccess) rc = PCT_ERR_HIP;
            if (rc) break;
            float ms = 0;
            (void)hipEventElapsedTime(&ms, e0, e1);
            ms /= reps;
            if (best_ms < 0 || ms < best_ms) {
                best_ms = ms;
                best_c = t;
                best_g = g;
            }
        }
        if (rc) break;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (best_c.shape_id < 0) return PCT_ERR_UNSUPPORTED;
    {
        std::lock_guard<std::mutex> lk(g_cfg_mutex);
        g_tuned[ShapeKey{pb->nx, pb->ny, pb->nz, pb->n_atlas, pb->nh}] = best_c;
    }
    if (best) {
        fill_config(best_c.shape_id,
                    model_cost(pb, best_c.shape_id, best_c.group, nullptr, best_c.split), best_g,
                    best);
        best->measured_ms = best_ms;
    }
    return PCT_OK;
}

extern "C" void pct_release(void) {
    release_batch_graphs();
    release_learned_models();
    release_train_buffers();
    release_host_buffers();
    std::lock_guard<std::mutex> lk(g_dev_mutex);
    for (auto& kv : g_dev) {
        DeviceState& st = kv.second;
        if (st.ws) st.kept.push_back(st.ws);
        if (!st.kept.empty()) {
            int cur = 0;
            (void)hipGetDevice(&cur);
            (void)hipSetDevice(kv.first);
            (void)hipDeviceSynchronize();
            for (void* p : st.kept) (void)hipFree(p);
            (void)hipSetDevice(cur);
        }
        st.kept.clear();
        st.ws = nullptr;
        st.ws_bytes = 0;
        st.recorded = false;
    }
}
