// Post-fusion chain on the GPU: NaN fill by the median of the 3x3x3
// neighbourhood, rounding, and the HU rescale, with the reference's order
// of operations (src/CPU/NewPatchedBrainPureC.cpp:1020-1106 Median and
// RegularizationStep, 1221-1227 RoundMatrix, 1725-1739 the HU rescale).
//
// RegularizationStep sweeps the interior in z, x, y order and overwrites each
// NaN voxel in place, so a voxel sees the values filled earlier in the same
// sweep.  Only NaN voxels ever change, and a NaN voxel's median reads its
// neighbours: those before it in scan order as this sweep left them, those
// after it as the previous sweep did (a NaN one after it is still NaN when
// it is reached).  With the wavefront index t = 4z + 2x + y every neighbour
// before a voxel in scan order has a smaller t and every neighbour after it
// a larger one (the steepest neighbours differ by (0, 0, +-1), (0, +-1, -+1)
// and (+-1, -+1, -+1): t steps of 1, 1 and 1).  Filling the sweep's NaN
// voxels in increasing t, all voxels of one t at once, therefore gives the
// sequential sweep's values bit for bit.
//
// The first sweep runs in tiles over the whole chip (fill_tiles_kernel).  It
// leaves NaN only where a voxel has no value around it at its turn; those
// voxels go through the later sweeps in one workgroup (nan_fill_levels_kernel:
// a counting sort of the list by t, then the levels in increasing t with a
// barrier after each non-empty one, one voxel per thread), until none is left
// or a sweep fills nothing.  Medians follow the std::stable_sort of cpp:1035,
// signed zeros included.  Rounding and the rescale are elementwise.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "pct_internal.h"
#include "pct_tiled.h"

namespace pct {

constexpr int kFillThreads = 1024;

// Comparators of Batcher's merge-exchange sorting network for 27 inputs
// (Knuth, TAOCP vol. 3, 5.2.2 Algorithm M; valid for any input count):
// 155 (min, max) pairs, built at compile time.
struct SortNet27 {
    int n = 0;
    unsigned char lo[160] = {}, hi[160] = {};
};
constexpr SortNet27 merge_exchange27() {
    SortNet27 L{};
    constexpr int N = 27;
    int t = 0;
    while ((1 << t) < N) ++t;
    for (int p = 1 << (t - 1); p > 0; p >>= 1) {
        int q = 1 << (t - 1), r = 0, d = p;
        for (;;) {
            for (int i = 0; i < N - d; ++i)
                if ((i & p) == r) {
                    L.lo[L.n] = (unsigned char)i;
                    L.hi[L.n] = (unsigned char)(i + d);
                    ++L.n;
                }
            if (q == p) break;
            d = q - p;
            q >>= 1;
            r = p;
        }
    }
    return L;
}
constexpr SortNet27 kSortNet27 = merge_exchange27();
static_assert(kSortNet27.n == 155, "merge exchange for 27 inputs");

// Order-preserving integer key of a float that is not NaN (an involution:
// applied to a key it gives the float's bits back).  -0 sorts before +0.
__device__ __forceinline__ int float_key(float f) {
    const int u = __float_as_int(f);
    return u ^ (int)((unsigned)(u >> 31) >> 1);
}

// Median of the non-NaN values among `cnt` of v[27] by stable ranks: the
// std::stable_sort of cpp:1035, equal values in their gathered order.
__device__ __forceinline__ float median_by_ranks(const float (&v)[27], int cnt) {
    const int hi = cnt / 2, lo_rank = cnt / 2 - 1;
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int i = 0; i < 27; ++i) {
        if (isnan(v[i])) continue;
        int rank = 0;
#pragma unroll
        for (int j = 0; j < 27; ++j)
            rank += (!isnan(v[j]) && (v[j] < v[i] || (v[j] == v[i] && j < i))) ? 1 : 0;
        if (rank == hi) b = v[i];
        if (rank == lo_rank) a = v[i];
    }
    if (cnt % 2 == 0) return (float)(((double)a + (double)b) / 2);
    return b;
}

// Median of the 3x3x3 neighbourhood of voxel `id` over its non-NaN values
// (cpp:1020-1043): the middle value, or the float64 mean of the two middle
// values, of their stable sort; NaN when all 27 are NaN.  Values that compare
// equal have the same bits except -0 and +0, so unless both signed zeros
// occur, any sort of the values gives the stable sort's bits: a sorting
// network of integer min/max pairs over order-preserving keys (NaN keyed
// last), 155 pairs against 27 x 27 rank comparisons.  With both signed zeros
// the ranks decide.
__device__ __forceinline__ float neighbourhood_median(const float* arr, int id, int pl, int ny) {
    float v[27];
#pragma unroll
    for (int k = 0; k < 27; ++k)
        v[k] = __hip_atomic_load(arr + id + (k / 9 - 1) * pl + ((k / 3) % 3 - 1) * ny + (k % 3 - 1),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    int cnt = 0;
    bool neg_zero = false, pos_zero = false;
    int key[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const bool nan = isnan(v[k]);
        cnt += nan ? 0 : 1;
        const int u = __float_as_int(v[k]);
        neg_zero |= u == (int)0x80000000;
        pos_zero |= u == 0;
        key[k] = nan ? INT_MAX : float_key(v[k]);
    }
    if (cnt == 0) return __builtin_nanf("");
    if (neg_zero && pos_zero) return median_by_ranks(v, cnt);
#pragma unroll
    for (int c = 0; c < kSortNet27.n; ++c) {
        const int i = kSortNet27.lo[c], j = kSortNet27.hi[c];
        const int mn = min(key[i], key[j]);
        key[j] = max(key[i], key[j]);
        key[i] = mn;
    }
    const int hi = cnt / 2, lo_rank = cnt / 2 - 1;
    int ka = 0, kb = 0;
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        kb = k == hi ? key[k] : kb;
        ka = k == lo_rank ? key[k] : ka;
    }
    const float a = __int_as_float(float_key(__int_as_float(ka))), b = __int_as_float(float_key(__int_as_float(kb)));
    if (cnt % 2 == 0) return (float)(((double)a + (double)b) / 2);
    return b;
}

// ---------------------------------------------------------------------------
// first sweep: tiles in dependency order
// ---------------------------------------------------------------------------
//
// With interior coordinates (z, x, y) and the skewed ones
//     Z = z,  X = x + z,  Y = y + x + 2 z     (t = Z + X + Y up to a constant)
// every neighbour before a voxel in scan order has no larger Z, X and Y, and
// every one after it no smaller.  The skewed space is cut into tiles of kTZ x
// kTX x kTY; tile (i, j, k) may run once the tiles of (i - {0,1}, j - {0,1},
// k - {0,1}) that hold NaN voxels are done: what it reads of earlier voxels is
// then final, and no later voxel it reads has changed, since those tiles wait
// for this one.  A workgroup takes the next tile from a list ordered by i + j +
// k, waits for the tiles before it, copies the tile and its halo into LDS as
// order-preserving integer keys, and runs the tile's levels of t with a
// workgroup barrier after each.  A tile is handed out only after all tiles it
// waits for, to workgroups that are already running, so every wait ends.
//
// What bounds it is the chain of tiles: a tile starts when all levels of the ones
// before it are done, so its kTileLevels levels and one hand-over between workgroups
// (flag, LDS copy) come once per diagonal (at 222x222x112, NH = 3: 107 diagonals of
// up to 213 tiles, 2782 levels in a row where the volume has 1080).  Hence small
// tiles, eight lanes to a voxel (about 130 instructions to a median instead of 900
// for one lane sorting 27 values), and an LDS copy that starts before the wait with
// what no tile before it changes.  222x222x112 with 4.2e6 NaN voxels: 48.2 ms for
// the one-workgroup sweep (45 us a level), 1.53 ms here, 1.48 of it in
// fill_tiles_kernel: 14 us a diagonal.  Of those 33000 cycles the levels take 21000
// (810 each), the copy after the wait 1900 and the release 1700; what the other
// 9000 go to has not been measured.  Tiles of
// {4, 8, 32} took 2.7 ms (before the early copy), {4, 8, 8} 2.04, {8, 8, 8}
// 2.22, {4, 16, 8} 2.56; 512 workgroups 1.70.  Polling with acquire loads,
// which invalidate the caches each time, took 4.6-6.2 ms.
constexpr int kTZ = 4, kTX = 8, kTY = 16;
constexpr int kTileLanes = 8;                              // lanes per voxel
constexpr int kTileThreads = kTZ * kTX * kTileLanes;       // one voxel per (Z, X) and level
constexpr int kTileLevels = kTZ + kTX + kTY - 2;
constexpr int kSZ = kTZ + 2, kSX = kTX + 4, kSY = kTY + 8; // with the halo
constexpr int kStage = kSZ * kSX * kSY;
// the staged elements: the tile and its halo after it (known before the tiles
// before it are done), then the halo before it
constexpr int kAfter = (kSZ - 1) * (kSX - 2) * (kSY - 4), kBefore = kStage - kAfter;
constexpr int kAfterLoads = (kAfter + kTileThreads - 1) / kTileThreads;
constexpr int kBeforeLoads = (kBefore + kTileThreads - 1) / kTileThreads;
constexpr int kTileWgs = 256;                              // workgroups that take tiles
constexpr int kWaitStores = 0x0f70;                        // s_waitcnt vmcnt(0), no other counter
static_assert(kTileLevels <= 32, "one mask bit per level");
static_assert(kTX % 4 == 0 && kTY >= 4 && kTX >= 2 && kTZ >= 1, "neighbours lie in adjacent tiles");

// The tiles that can hold interior voxels.  Row i spans X from kTZ i, and
// (i, j) spans Y from kTZ i + kTX j, so j and k are counted from there.
struct FillTiles {
    int nx, ny, nz, lo;   // volume, first interior coordinate
    int iz, ix, iy;       // interior extents
    int ni, nj, nk;       // tiles per axis of the compact numbering
    int n_tiles, n_diag;  // n_diag: bound of i + j + k
};

__host__ __device__ __forceinline__ int tile_j0(int i) { return kTZ * i / kTX; }
__host__ __device__ __forceinline__ int tile_k0(int i, int j) { return (kTZ * i + kTX * j) / kTY; }

__device__ __forceinline__ void tile_coords(const FillTiles& f, int tile, int* i, int* j, int* k) {
    const int kk = tile % f.nk, ij = tile / f.nk;
    *i = ij / f.nj;
    *j = tile_j0(*i) + ij % f.nj;
    *k = tile_k0(*i, *j) + kk;
}

// Index of tile (i, j, k), or -1 where it holds no interior voxel.
__device__ __forceinline__ int tile_index(const FillTiles& f, int i, int j, int k) {
    if (i < 0) return -1;
    const int jj = j - tile_j0(i);
    if (jj < 0 || jj >= f.nj) return -1;
    const int kk = k - tile_k0(i, j);
    if (kk < 0 || kk >= f.nk) return -1;
    return (i * f.nj + jj) * f.nk + kk;
}

// Counters and the diagonals' histogram of one fill.
struct FillState {
    int* next;        // tiles handed out
    int* n_busy;      // tiles with NaN voxels
    int* left;        // voxels still NaN after the first sweep
    int* done;        // [n_tiles] 1: nothing (more) to do
    int* order;       // [n_tiles] busy tiles by diagonal
    int* diag;        // [n_diag + 1] tiles per diagonal, then their places
};

// Whether tile (i, j, k) holds an interior NaN voxel; one wave per tile.
__device__ __forceinline__ bool tile_has_nan(const float* __restrict__ arr, const FillTiles& f,
                                             int i, int j, int k) {
    const int lane = threadIdx.x & 63;
    constexpr int kLoads = kTZ * kTX * kTY / 64;
    bool nan = false;
#pragma unroll 8
    for (int q = 0; q < kLoads; ++q) {
        const int e = q * 64 + lane;
        const int Z = kTZ * i + e / (kTX * kTY), X = kTX * j + (e / kTY) % kTX,
                  Y = kTY * k + e % kTY;
        const int z = Z, x = X - Z, y = Y - X - Z;
        const bool in = z < f.iz && x >= 0 && x < f.ix && y >= 0 && y < f.iy;
        const long long id =
            ((long long)(f.lo + z) * f.nx + (f.lo + x)) * f.ny + (f.lo + y);
        const float v = arr[in ? id : 0];
        nan |= in && isnan(v);
    }
    return __ballot(nan) != 0;
}

// The tiles with work, listed by diagonal.  Up to kPlanDiags diagonals and
// kPlanTiles tiles one workgroup does it with the histogram in LDS, after a scan
// kernel or, for up to kPlanScan tiles, with the scan as well: the chain then
// takes 4 launches on the smallest volumes and 5 on others, where clearing,
// counting, placing and listing as kernels of their own make it 7 (28x26x24, 0.2 %
// NaN: 28.0 -> 21.2 us; 222x222x112, 4.2e6 NaN: 1.62 -> 1.56 ms, with 0.2 % NaN 112.5
// -> 113.6 us; 128x128x64, 0.2 %: 54.5 -> 52.6).  Past that one workgroup would be
// the slower one (330x320x200, 45000 tiles, 0.2 %: 350 against 357 us) or its LDS too
// small, and those kernels run.
constexpr int kPlanDiags = 4096, kPlanTiles = 1 << 16, kPlanScan = 256, kPlanThreads = 1024;

// The general path: the counters, the scan with its histogram, the places of the
// diagonals and the list.
__global__ void fill_clear_kernel(FillState st, int n_diag) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t <= n_diag) st.diag[t] = 0;
    if (t == 0) *st.next = *st.n_busy = *st.left = 0;
}

constexpr int kScanWaves = 4;
template <bool COUNT>   // COUNT: into the histogram too
__global__ __launch_bounds__(kScanWaves * 64) void fill_scan_kernel(
    const float* __restrict__ arr, FillTiles f, FillState st) {
    const int tile = blockIdx.x * kScanWaves + (threadIdx.x >> 6);
    if (tile >= f.n_tiles) return;   // per wave; no barrier below
    int i, j, k;
    tile_coords(f, tile, &i, &j, &k);
    const bool busy = tile_has_nan(arr, f, i, j, k);
    if ((threadIdx.x & 63) == 0) {
        st.done[tile] = busy ? 0 : 1;
        if (COUNT && busy) atomicAdd(st.diag + (i + j + k), 1);
    }
}

// Exclusive prefix of the n counts at `diag` by a workgroup of kPlanThreads, in
// place; returns the total.
__device__ __forceinline__ int diagonal_places(int* diag, int n) {
    __shared__ int wtot[kPlanThreads / 64];
    const int seg = (n + kPlanThreads - 1) / kPlanThreads;
    const int b0 = min(n, (int)threadIdx.x * seg), b1 = min(n, b0 + seg);
    int own = 0;
    for (int b = b0; b < b1; ++b) own += diag[b];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o);
        if (lane >= o) incl += v;
    }
    if (lane == 63) wtot[w] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int j = 0; j < kPlanThreads / 64; ++j) {
        before += j < w ? wtot[j] : 0;
        total += wtot[j];
    }
    int run = before + incl - own;
    for (int b = b0; b < b1; ++b) {
        const int c = diag[b];
        diag[b] = run;
        run += c;
    }
    return total;
}

__global__ __launch_bounds__(kPlanThreads) void fill_places_kernel(FillState st, int n_diag) {
    const int total = diagonal_places(st.diag, n_diag);
    if (threadIdx.x == 0) *st.n_busy = total;
}

// Busy tiles into the list by diagonal (any order within one).
__global__ void fill_order_kernel(FillTiles f, FillState st) {
    const int tile = blockIdx.x * blockDim.x + threadIdx.x;
    if (tile >= f.n_tiles || st.done[tile]) return;
    int i, j, k;
    tile_coords(f, tile, &i, &j, &k);
    st.order[atomicAdd(st.diag + (i + j + k), 1)] = tile;
}

// The whole plan in one workgroup (n_diag <= kPlanDiags).  SCAN: f.n_tiles <=
// kPlanScan tiles are scanned here; otherwise fill_scan_kernel left the flags.
template <bool SCAN>
__global__ __launch_bounds__(kPlanThreads) void fill_plan_kernel(const float* __restrict__ arr,
                                                                 FillTiles f, FillState st) {
    __shared__ int diag[kPlanDiags];
    __shared__ int busy[SCAN ? kPlanScan : 1];
    for (int d = threadIdx.x; d < f.n_diag; d += kPlanThreads) diag[d] = 0;
    if (SCAN)
        for (int t = threadIdx.x >> 6; t < f.n_tiles; t += kPlanThreads / 64) {
            int i, j, k;
            tile_coords(f, t, &i, &j, &k);
            const bool nan = tile_has_nan(arr, f, i, j, k);
            if ((threadIdx.x & 63) == 0) {
                busy[t] = nan ? 1 : 0;
                st.done[t] = nan ? 0 : 1;
            }
        }
    __syncthreads();
    // the thread's busy tiles: bit 8 i + k is tile 8192 i + 8 threadIdx.x + k (SCAN:
    // bit 0, tile threadIdx.x)
    constexpr int kRound = 8 * kPlanThreads;
    static_assert(kPlanTiles <= 8 * kRound, "one bit per tile");
    unsigned long long mine = 0;
    if (SCAN) {
        mine = (int)threadIdx.x < f.n_tiles && busy[threadIdx.x] ? 1 : 0;
    } else {
        for (int i = 0; i * kRound < f.n_tiles; ++i) {
            const int t0 = i * kRound + 8 * threadIdx.x;
            if (t0 >= f.n_tiles) break;
            // up to 7 flags past the last tile's are read: the array is a multiple
            // of 64 long
            const int4* p = reinterpret_cast<const int4*>(st.done + t0);
            const int4 lo = p[0], hi = p[1];
            const int v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (t0 + k < f.n_tiles && v[k] == 0) mine |= 1ull << (8 * i + k);
        }
    }
    auto each = [&](auto use) {   // the busy tiles' (tile, diagonal)
        for (unsigned long long m = mine; m; m &= m - 1) {
            const int bit = __ffsll((long long)m) - 1;
            const int t = SCAN ? threadIdx.x : (bit >> 3) * kRound + 8 * threadIdx.x + (bit & 7);
            int i, j, k;
            tile_coords(f, t, &i, &j, &k);
            use(t, i + j + k);
        }
    };
    each([&](int, int d) { atomicAdd(&diag[d], 1); });
    __syncthreads();
    const int total = diagonal_places(diag, f.n_diag);
    __syncthreads();
    each([&](int t, int d) { st.order[atomicAdd(&diag[d], 1)] = t; });
    if (threadIdx.x == 0) {
        *st.next = *st.left = 0;
        *st.n_busy = total;
    }
}

// Lane exchanges within the eight lanes of a voxel.
template <int CTRL>
__device__ __forceinline__ int lane_swap(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
constexpr int kSwap1 = 0xB1;    // lane ^ 1 (quad_perm 1, 0, 3, 2)
constexpr int kSwap2 = 0x4E;    // lane ^ 2 (quad_perm 2, 3, 0, 1)
constexpr int kSwap3 = 0x1B;    // lane ^ 3 (quad_perm 3, 2, 1, 0)
constexpr int kSwap7 = 0x141;   // lane ^ 7 (row_half_mirror)

// The value of the lane before (within a row of 16).
__device__ __forceinline__ int lane_before(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
}

__device__ __forceinline__ int med3i(int a, int b, int c) {
    return max(min(a, b), min(max(a, b), c));
}

__device__ __forceinline__ void order2(int& a, int& b) {
    const int mn = min(a, b);
    b = max(a, b);
    a = mn;
}

// Each lane keeps the smaller (bound INT_MIN) or the larger (INT_MAX) of its
// slots and another lane's: slot s against slot s, or against 3 - s (REV).
template <int CTRL, bool REV>
__device__ __forceinline__ void lane_split(int (&k)[4], int bound) {
    int o[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) o[s] = lane_swap<CTRL>(k[REV ? 3 - s : s]);
#pragma unroll
    for (int s = 0; s < 4; ++s) k[s] = med3i(k[s], o[s], bound);
}

// Sorts a lane's four slots when they form a bitonic sequence.
__device__ __forceinline__ void bitonic4(int (&k)[4]) {
    order2(k[0], k[2]);
    order2(k[1], k[3]);
    order2(k[0], k[1]);
    order2(k[2], k[3]);
}

// Sorts the 32 keys of eight lanes: afterwards lane q holds ranks 4 q .. 4 q + 3.
// b1, b2, b4: INT_MIN where bit 0, 1, 2 of the lane is 0, else INT_MAX.
__device__ __forceinline__ void sort8x4(int (&k)[4], int b1, int b2, int b4) {
    order2(k[0], k[1]);
    order2(k[2], k[3]);
    order2(k[0], k[2]);
    order2(k[1], k[3]);
    order2(k[1], k[2]);
    lane_split<kSwap1, true>(k, b1);
    bitonic4(k);
    lane_split<kSwap3, true>(k, b2);
    lane_split<kSwap1, false>(k, b1);
    bitonic4(k);
    lane_split<kSwap7, true>(k, b4);
    lane_split<kSwap2, false>(k, b2);
    lane_split<kSwap1, false>(k, b1);
    bitonic4(k);
}

__global__ __launch_bounds__(kTileThreads) void fill_tiles_kernel(float* arr, FillTiles f,
                                                                  FillState st, int* left_list) {
    __shared__ int key[kStage];
    __shared__ int s_ticket;
    __shared__ unsigned s_levels;      // levels of the tile with NaN voxels
    __shared__ int s_neg_zero;         // a -0 may occur in the tile
    const int tid = threadIdx.x;
    const int q = tid & (kTileLanes - 1), v = tid / kTileLanes;
    const int vz = v / kTX, vx = v % kTX;
    const int b1 = (q & 1) ? INT_MAX : INT_MIN, b2 = (q & 2) ? INT_MAX : INT_MIN,
              b4 = (q & 4) ? INT_MAX : INT_MIN;
    // LDS offsets of the lane's neighbours q, q + 8, ... of the 27 (the last
    // slot of lanes 3 .. 7 is empty: none_if raises it to INT_MAX)
    auto offset = [](int n) {
        const int dz = n / 9 - 1, dx = (n / 3) % 3 - 1, dy = n % 3 - 1;
        return (dz * kSX + (dx + dz)) * kSY + dy + dx + 2 * dz;
    };
    int off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = opaque(offset(min(q + 8 * s, 26)));
    const int none_if = q < 3 ? INT_MIN : INT_MAX;
    // the staged elements of the thread, as (sz, sx, sy) packed in bytes, -1
    // for none; element (0, 0, 0) lies at Z - 1, X - 2, Y - 4 of the tile's origin
    int after[kAfterLoads], before[kBeforeLoads];
    auto pack = [](int sz, int sx, int sy) { return (sz << 16) | (sx << 8) | sy; };
#pragma unroll
    for (int l = 0; l < kAfterLoads; ++l) {
        const int e = tid + l * kTileThreads;
        constexpr int W = kSY - 4, H = kSX - 2;
        after[l] = e < kAfter ? pack(1 + e / (H * W), 2 + (e / W) % H, 4 + e % W) : -1;
    }
#pragma unroll
    for (int l = 0; l < kBeforeLoads; ++l) {
        // plane sz = 0, then rows sx < 2, then columns sy < 4
        int e = tid + l * kTileThreads;
        int c = -1;
        if (e < kSX * kSY) {
            c = pack(0, e / kSY, e % kSY);
        } else if ((e -= kSX * kSY) < (kSZ - 1) * 2 * kSY) {
            c = pack(1 + e / (2 * kSY), (e / kSY) % 2, e % kSY);
        } else if ((e -= (kSZ - 1) * 2 * kSY) < (kSZ - 1) * (kSX - 2) * 4) {
            c = pack(1 + e / ((kSX - 2) * 4), 2 + (e / 4) % (kSX - 2), e % 4);
        }
        before[l] = c;
    }
    const int n_busy = *st.n_busy;
    for (;;) {
        __syncthreads();   // the previous tile is done with the shared state
        if (tid == 0) {
            s_ticket = atomicAdd(st.next, 1);
            s_levels = 0;
            s_neg_zero = 0;
        }
        __syncthreads();
        const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
        if (ticket >= n_busy) return;   // uniform; every tile has been handed out
        const int tile = st.order[ticket];
        int i, j, k;
        tile_coords(f, tile, &i, &j, &k);
        // volume coordinates of element (0, 0, 0)
        const int Z0 = kTZ * i - 1, X0 = kTX * j - 2, Y0 = kTY * k - 4;
        auto load = [&](int c, bool* in) {
            const int Z = Z0 + (c >> 16), X = X0 + ((c >> 8) & 255), Y = Y0 + (c & 255);
            const int z = f.lo + Z, x = f.lo + X - Z, y = f.lo + Y - X - Z;
            *in = c >= 0 && (unsigned)z < (unsigned)f.nz && (unsigned)x < (unsigned)f.nx &&
                  (unsigned)y < (unsigned)f.ny;
            return arr[*in ? ((long long)z * f.nx + x) * f.ny + y : 0];
        };
        bool neg = false;
        auto store = [&](int c, bool in, float v) {   // INT_MAX: NaN or outside the volume
            const int kv = in && !isnan(v) ? float_key(v) : INT_MAX;
            neg |= kv == -1;
            if (c >= 0) key[((c >> 16) * kSX + ((c >> 8) & 255)) * kSY + (c & 255)] = kv;
            return kv;
        };
        {
            float raw[kAfterLoads];
            bool in[kAfterLoads];
#pragma unroll
            for (int l = 0; l < kAfterLoads; ++l) raw[l] = load(after[l], &in[l]);
            unsigned levels = 0;
#pragma unroll
            for (int l = 0; l < kAfterLoads; ++l) {
                const int c = after[l];
                const int kv = store(c, in[l], raw[l]);
                const int zl = (c >> 16) - 1, xl = ((c >> 8) & 255) - 2, yl = (c & 255) - 4;
                const int Z = kTZ * i + zl, X = kTX * j + xl, Y = kTY * k + yl;
                const int x = X - Z, y = Y - X - Z;
                if (in[l] && kv == INT_MAX && zl < kTZ && xl < kTX && yl < kTY && Z < f.iz &&
                    x >= 0 && x < f.ix && y >= 0 && y < f.iy)
                    levels |= 1u << (zl + xl + yl);
            }
            if (levels) atomicOr(&s_levels, levels);
        }
        if (tid >= 1 && tid < 8) {
            const int p = tile_index(f, i - (tid & 1), j - ((tid >> 1) & 1), k - (tid >> 2));
            if (p >= 0)
                while (__hip_atomic_load(st.done + p, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) == 0)
                    __builtin_amdgcn_s_sleep(1);
        }
        // one acquire after the waits, by the wave that waited (an acquire in
        // the loop would invalidate the caches at every poll)
        if (tid < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();
        {
            float raw[kBeforeLoads];
            bool in[kBeforeLoads];
#pragma unroll
            for (int l = 0; l < kBeforeLoads; ++l) raw[l] = load(before[l], &in[l]);
#pragma unroll
            for (int l = 0; l < kBeforeLoads; ++l) store(before[l], in[l], raw[l]);
        }
        if (neg) s_neg_zero = 1;
        __syncthreads();

        // the lane's voxel at level l is (vz, vx, l - vz - vx); y runs over
        // the interior for local Y in [y_lo, y_hi)
        const int Z = kTZ * i + vz, X = kTX * j + vx;
        const int x = X - Z;
        const bool row_in = Z < f.iz && x >= 0 && x < f.ix;
        const int y_base = X + Z - kTY * k;   // local Y of interior y = 0
        const int y_lo = max(0, y_base), y_hi = row_in ? min(kTY, y_base + f.iy) : 0;
        const long long row_id =
            ((long long)(f.lo + Z) * f.nx + (f.lo + x)) * f.ny + f.lo - y_base;
        const int* const row_key = key + ((vz + 1) * kSX + vx + 2) * kSY + 4;
        unsigned todo = (unsigned)__builtin_amdgcn_readfirstlane((int)s_levels);
        while (todo) {   // uniform
            const int l = __builtin_ctz(todo);
            todo &= todo - 1;
            const int yl = l - vz - vx;
            const int* const at = row_key + min(max(yl, 0), kTY - 1);
            const int centre = at[0];
            int kk[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) kk[s] = at[off[s]];
            kk[3] = max(kk[3], none_if);
            const bool valid = yl >= y_lo && yl < y_hi && centre == INT_MAX;
            if (__ballot(valid)) {   // uniform over the wave
                int cnt = 0;
#pragma unroll
                for (int s = 0; s < 4; ++s) cnt += kk[s] != INT_MAX ? 1 : 0;
                cnt += lane_swap<kSwap1>(cnt);
                cnt += lane_swap<kSwap2>(cnt);
                cnt += lane_swap<kSwap7>(cnt);
                sort8x4(kk, b1, b2, b4);
                // the lane that holds rank cnt / 2 (slot hs) forms the median:
                // the rank before it is its slot before, or the last of the
                // lane before
                const int hi = cnt >> 1, hs = hi & 3;
                const int prev = lane_before(kk[3]);
                const int kb = hs & 2 ? (hs & 1 ? kk[3] : kk[2]) : (hs & 1 ? kk[1] : kk[0]);
                const int ka = hs & 2 ? (hs & 1 ? kk[2] : kk[1]) : (hs & 1 ? kk[0] : prev);
                const float b = __int_as_float(float_key(__int_as_float(kb)));
                const float a = __int_as_float(float_key(__int_as_float(ka)));
                float res = (cnt & 1) ? b : (float)(((double)a + (double)b) / 2);
                if (s_neg_zero) {   // -0 and +0 may meet: the stable ranks decide
                    float ra = 0.f, rb = 0.f;
#pragma unroll 1
                    for (int m = 0; m < 27; ++m) {
                        const int km = at[offset(m)];
                        if (km == INT_MAX) continue;
                        const float fm = __int_as_float(float_key(__int_as_float(km)));
                        int rank = 0;
#pragma unroll 1
                        for (int n = 0; n < 27; ++n) {
                            const int kn = at[offset(n)];
                            const float fn = __int_as_float(float_key(__int_as_float(kn)));
                            rank += kn != INT_MAX && (fn < fm || (fn == fm && n < m)) ? 1 : 0;
                        }
                        if (rank == hi) rb = fm;
                        if (rank == hi - 1) ra = fm;
                    }
                    res = (cnt & 1) ? rb : (float)(((double)ra + (double)rb) / 2);
                }
                if (valid && q == (hi >> 2)) {
                    if (cnt == 0) res = __builtin_nanf("");
                    const long long id = row_id + yl;
                    arr[id] = res;
                    if (isnan(res)) {   // no value around it, or infinities of both signs
                        left_list[atomicAdd(st.left, 1)] = (int)id;
                    } else {
                        const int rk = float_key(res);
                        key[at - key] = rk;
                        if (rk == -1) s_neg_zero = 1;
                    }
                }
            }
            __syncthreads();
        }
        // The release below waits for the stores of its own wave alone (and a
        // workgroup barrier for none in memory), so each wave waits here for the
        // values it stored: they are in the L2 before the barrier, and the release
        // writes that back before the flag.
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitStores);
        __syncthreads();
        if (tid == 0)
            __hip_atomic_store(st.done + tile, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// the other sweeps
// ---------------------------------------------------------------------------

// The sweeps of RegularizationStep over the listed voxels, in one workgroup.
// hist has t_count + 1 ints; sorted and the lists hold `interior` ints.
// Every thread that reads or writes these buffers during the fill belongs to
// this one workgroup (the inputs come from earlier launches on the stream),
// so values and list entries go through workgroup-scope atomics and every
// level ends with a workgroup barrier, whose workgroup-scope release and
// acquire let a level see the ones before it.  Agent-scope fences would
// write back and invalidate the L2 at every level.  The level histogram is
// built by atomics performed in L2 and read back with agent-scope loads.
__global__ __launch_bounds__(kFillThreads) void nan_fill_levels_kernel(
    float* __restrict__ arr, int* list_a, int* list_b, int* sorted, int* hist,
    const int* count0, int nx, int ny, int t_count, int* sweeps_out) {
    __shared__ int s_n, s_next, s_filled;
    __shared__ int s_end[kFillThreads];   // level ends of one chunk of levels
    const int pl = nx * ny;
    int* cur = list_a;
    int* nxt = list_b;
    if (threadIdx.x == 0) s_n = __hip_atomic_load(count0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    int n = s_n;
    int sweeps = 0;
    while (n > 0) {
        ++sweeps;
        // counting sort of the list by t = 4 z + 2 x + y
        for (int t = threadIdx.x; t <= t_count; t += kFillThreads) hist[t] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kFillThreads) {
            const int id = cur[i];
            const int z = id / pl, x = (id - z * pl) / ny, y = id - z * pl - x * ny;
            atomicAdd(hist + 4 * z + 2 * x + y, 1);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            // exclusive prefix of the counts; hist[t] becomes the level start.
            // The counts come from atomics performed in L2: read them with
            // agent-scope loads, which do not use the CU's L1, 16 at a time.
            int run = 0;
            for (int t0 = 0; t0 <= t_count; t0 += 16) {
                int c[16];
#pragma unroll
                for (int k = 0; k < 16; ++k)
                    c[k] = t0 + k <= t_count ? __hip_atomic_load(hist + t0 + k, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT)
                                             : 0;
#pragma unroll
                for (int k = 0; k < 16; ++k)
                    if (t0 + k <= t_count) {
                        hist[t0 + k] = run;
                        run += c[k];
                    }
            }
            s_next = 0;
            s_filled = 0;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kFillThreads) {
            const int id = cur[i];
            const int z = id / pl, x = (id - z * pl) / ny, y = id - z * pl - x * ny;
            sorted[atomicAdd(hist + 4 * z + 2 * x + y, 1)] = id;
        }
        __syncthreads();
        // hist[t] is now the end of level t; levels in increasing t, their
        // ends read into LDS a chunk at a time
        int begin = 0;
        for (int t0 = 0; t0 < t_count; t0 += kFillThreads) {
            if (t0 + (int)threadIdx.x < t_count)
                s_end[threadIdx.x] = __hip_atomic_load(hist + t0 + threadIdx.x, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);   // L2 atomics
            __syncthreads();
            const int tn = min(kFillThreads, t_count - t0);
            for (int k = 0; k < tn; ++k) {
                const int end = s_end[k];
                if (end == begin) continue;   // uniform: an empty level
                for (int i = begin + (int)threadIdx.x; i < end; i += kFillThreads) {
                    const int id = __hip_atomic_load(sorted + i, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP);
                    const float res = neighbourhood_median(arr, id, pl, ny);
                    __hip_atomic_store(arr + id, res, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (isnan(res))
                        __hip_atomic_store(nxt + atomicAdd(&s_next, 1), id, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                    else
                        atomicAdd(&s_filled, 1);
                }
                __syncthreads();
                begin = end;
            }
            __syncthreads();   // s_end is rewritten for the next chunk
        }
        const int m = s_next, filled = s_filled;
        __syncthreads();   // every thread read the counters
        if (m == 0 || filled == 0) break;
        int* tmp = cur;
        cur = nxt;
        nxt = tmp;
        n = m;
    }
    if (threadIdx.x == 0 && sweeps_out) *sweeps_out = sweeps;
}

// RoundMatrix (cpp:1221-1227) then round(4095 * (v / 255)) - 1024 in float
// (cpp:1732-1738); `round` rounds halves away from zero on both sides.
__global__ void round_hu_kernel(float* __restrict__ arr, long long n, int to_hu) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        float v = roundf(arr[i]);
        if (to_hu) v = roundf(4095.0f * (v / 255.0f)) - 1024.0f;
        arr[i] = v;
    }
}

static int post_checks(int nh, int nx, int ny, int nz, const float* d_arr) {
    if (!d_arr || nh < 1 || nx < 1 || ny < 1 || nz < 1) return PCT_ERR_INVALID;
    if ((long long)nx * ny * nz >= INT_MAX) return PCT_ERR_TOO_LARGE;
    return PCT_OK;
}

// Interior voxel count of the post chain's NaN fill.
static long long fill_interior(int nh, int nx, int ny, int nz) {
    const int lo = (nh - 1) / 2 + 1;
    const long long iz = nz - 2 * lo, ix = nx - 2 * lo, iy = ny - 2 * lo;
    return (iz > 0 && ix > 0 && iy > 0) ? iz * ix * iy : 0;
}

// Wavefront levels of a volume: t = 4 z + 2 x + y ranges over [0, t_count).
static long long fill_levels(int nx, int ny, int nz) {
    return 4LL * (nz - 1) + 2LL * (nx - 1) + (ny - 1) + 1;
}

// The fill's tiles (a volume below 2^31 voxels with interior voxels).
static FillTiles fill_tiles(int nh, int nx, int ny, int nz) {
    FillTiles f;
    f.nx = nx;
    f.ny = ny;
    f.nz = nz;
    f.lo = (nh - 1) / 2 + 1;
    f.iz = nz - 2 * f.lo;
    f.ix = nx - 2 * f.lo;
    f.iy = ny - 2 * f.lo;
    f.ni = (f.iz + kTZ - 1) / kTZ;
    f.nj = (kTZ + f.ix - 2) / kTX + 2;
    f.nk = (kTZ + kTX + f.iy - 3) / kTY + 2;
    f.n_tiles = f.ni * f.nj * f.nk;
    const int j_end = tile_j0(f.ni - 1) + f.nj;
    f.n_diag = f.ni + j_end + tile_k0(f.ni - 1, j_end) + f.nk;
    return f;
}

// Workspace of the NaN fill: counters, three voxel lists (two sweeps' and the
// sorted one), the level histogram, the tiles' states and order, and the
// diagonals' histogram.
struct FillLayout {
    size_t list, hist, done, order, diag, bytes;
};
static FillLayout fill_layout(int nh, int nx, int ny, int nz) {
    auto align = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const long long interior = fill_interior(nh, nx, ny, nz);
    FillLayout w{};
    w.list = align((size_t)interior * 4);
    w.hist = 256 + 3 * w.list;
    w.done = w.hist + align((size_t)(fill_levels(nx, ny, nz) + 1) * 4);
    if (!interior) {
        w.bytes = w.done;
        return w;
    }
    const FillTiles f = fill_tiles(nh, nx, ny, nz);
    w.order = w.done + align((size_t)f.n_tiles * 4);
    w.diag = w.order + align((size_t)f.n_tiles * 4);
    w.bytes = w.diag + align((size_t)(f.n_diag + 1) * 4);
    return w;
}

static int enqueue_fill(int nh, int nx, int ny, int nz, float* d_arr, void* ws, hipStream_t s) {
    if (fill_interior(nh, nx, ny, nz) == 0) return PCT_OK;
    const FillLayout lay = fill_layout(nh, nx, ny, nz);
    const FillTiles f = fill_tiles(nh, nx, ny, nz);
    char* w = static_cast<char*>(ws);
    int* counters = reinterpret_cast<int*>(w);
    int* la = reinterpret_cast<int*>(w + 256);
    int* lb = reinterpret_cast<int*>(w + 256 + lay.list);
    int* srt = reinterpret_cast<int*>(w + 256 + 2 * lay.list);
    int* hist = reinterpret_cast<int*>(w + lay.hist);
    FillState st;
    st.next = counters;
    st.n_busy = counters + 16;
    st.left = counters + 32;
    st.done = reinterpret_cast<int*>(w + lay.done);
    st.order = reinterpret_cast<int*>(w + lay.order);
    st.diag = reinterpret_cast<int*>(w + lay.diag);
    const dim3 scan_grid((unsigned)((f.n_tiles + kScanWaves - 1) / kScanWaves));
    if (f.n_diag > kPlanDiags || f.n_tiles > kPlanTiles) {
        hipLaunchKernelGGL(fill_clear_kernel, dim3((unsigned)(f.n_diag / 256 + 1)), dim3(256), 0,
                           s, st, f.n_diag);
        hipLaunchKernelGGL(fill_scan_kernel<true>, scan_grid, dim3(kScanWaves * 64), 0, s, d_arr,
                           f, st);
        hipLaunchKernelGGL(fill_places_kernel, dim3(1), dim3(kPlanThreads), 0, s, st, f.n_diag);
        hipLaunchKernelGGL(fill_order_kernel, dim3((unsigned)((f.n_tiles + 255) / 256)),
                           dim3(256), 0, s, f, st);
    } else if (f.n_tiles > kPlanScan) {
        hipLaunchKernelGGL(fill_scan_kernel<false>, scan_grid, dim3(kScanWaves * 64), 0, s, d_arr,
                           f, st);
        hipLaunchKernelGGL(fill_plan_kernel<false>, dim3(1), dim3(kPlanThreads), 0, s, d_arr, f,
                           st);
    } else {
        hipLaunchKernelGGL(fill_plan_kernel<true>, dim3(1), dim3(kPlanThreads), 0, s, d_arr, f,
                           st);
    }
    hipLaunchKernelGGL(fill_tiles_kernel, dim3((unsigned)std::min(f.n_tiles, kTileWgs)),
                       dim3(kTileThreads), 0, s, d_arr, f, st, la);
    hipLaunchKernelGGL(nan_fill_levels_kernel, dim3(1), dim3(kFillThreads), 0, s, d_arr, la, lb,
                       srt, hist, st.left, nx, ny, (int)fill_levels(nx, ny, nz), (int*)nullptr);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

// The fill on the library's per-device workspace.
static int enqueue_fill_lib(int nh, int nx, int ny, int nz, float* d_arr, hipStream_t s) {
    int dev = 0;
    int rc = check_device(&dev);
    if (rc) return rc;
    const long long interior = fill_interior(nh, nx, ny, nz);
    if (interior == 0) return PCT_OK;
    void* ws = nullptr;
    rc = ensure_workspace(dev, fill_layout(nh, nx, ny, nz).bytes, &ws);
    if (rc) return rc;
    return enqueue_fill(nh, nx, ny, nz, d_arr, ws, s);
}

static int enqueue_round_hu(int nx, int ny, int nz, float* d_arr, hipStream_t s) {
    const long long n = (long long)nx * ny * nz;
    const unsigned blocks = (unsigned)std::min<long long>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(round_hu_kernel, dim3(blocks), dim3(256), 0, s, d_arr, n, 1);
    return hipGetLastError() == hipSuccess ? PCT_OK : PCT_ERR_HIP;
}

size_t postprocess_ws_bytes(int nh, int nx, int ny, int nz) {
    return fill_layout(nh, nx, ny, nz).bytes;
}

int postprocess_dev_ws(int nh, int nx, int ny, int nz, float* d_arr, void* ws, hipStream_t s) {
    int rc = post_checks(nh, nx, ny, nz, d_arr);
    if (rc) return rc;
    rc = enqueue_fill(nh, nx, ny, nz, d_arr, ws, s);
    if (rc) return rc;
    return enqueue_round_hu(nx, ny, nz, d_arr, s);
}

}  // namespace pct

using namespace pct;

extern "C" int pct_regularize_dev(int nh, int nx, int ny, int nz, float* d_arr,
                                  pct_stream_t stream) {
    const int rc = post_checks(nh, nx, ny, nz, d_arr);
    if (rc) return rc;
    return enqueue_fill_lib(nh, nx, ny, nz, d_arr, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pct_postprocess_dev(int nh, int nx, int ny, int nz, float* d_arr,
                                   pct_stream_t stream) {
    int rc = post_checks(nh, nx, ny, nz, d_arr);
    if (rc) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    rc = enqueue_fill_lib(nh, nx, ny, nz, d_arr, s);
    if (rc) return rc;
    return enqueue_round_hu(nx, ny, nz, d_arr, s);
}
