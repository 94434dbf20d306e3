// Neighbour search for the sSSA-SDPD engine on gfx950.
//
// Replaces buildKDTree + Particle::find_neighbors + add_to_neighbor_list
// (ENG/src/simulate_threads.cpp:80-108, ENG/src/particle.cpp:150-294) and the
// ANN kd-tree fixed-radius search they call (ANN/src/kd_fix_rad_search.cpp).
//
//  * The neighbour SET and the r^2 bits come from counting-sort cell binning:
//    tree points are binned into cells of side >= h, candidates in the 3^d
//    surrounding cells are tested with ANN's exact acceptance rule
//    (r2 = ((0 + t0^2) + t1^2) + t2^2 with t = q - p in FP64, r2 <= h^2,
//    r2 != 0 (no self match, ANN.h:235), sqrt(r2) <= h (particle.cpp:162)).
//  * The list ORDER is ANN's: ascending r2, ties in the kd-tree's depth-first
//    visit order (pr_queue_k.h:100-116, kd_fix_rad_search.cpp:100-140).  Ties
//    are ranked through the lowest common ancestor of the two leaves in a
//    sliding-midpoint kd-tree built on the GPU level by level
//    (kd_tree.cpp:314-405, kd_split.cpp:146-213, kd_util.cpp:291-319): the
//    point on the query's side of that node's cut is visited first.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "engine.hpp"

namespace ssa {

// ---------------------------------------------------------------------------
// Order-preserving map of doubles to unsigned 64-bit keys (for atomic min/max).
__device__ __forceinline__ unsigned long long dkey(double x) {
    unsigned long long b = (unsigned long long)__double_as_longlong(x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ULL);
}
__device__ __forceinline__ double dkey_inv(unsigned long long k) {
    unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFULL) : ~k;
    return __longlong_as_double((long long)b);
}

// ---------------------------------------------------------------------------
// Exclusive scan of int32 counts (3-phase: block reduce, scan of block sums,
// add) into T: int where the total has a known bound, int64_t for the rows of
// the stand-alone search, whose lists together may pass 2^31 entries.
constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

template <class T> __device__ T block_exclusive_scan(T v, T *lds, T &total) {
    // v: thread partial; returns exclusive prefix within the block
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    T x = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        T y = __shfl_up(x, o, WAVE);
        if (lane >= o) x += y;
    }
    if (lane == WAVE - 1) lds[w] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        T acc = 0;
        for (int i = 0; i < SCAN_BLOCK / WAVE; i++) { T t = lds[i]; lds[i] = acc; acc += t; }
        lds[SCAN_BLOCK / WAVE] = acc;
    }
    __syncthreads();
    total = lds[SCAN_BLOCK / WAVE];
    T r = x - v + lds[w];
    __syncthreads();
    return r;
}

template <class I, class T> __global__ void k_scan_tiles(const I *in, T *out, long long n, T *tile_sums) {
    __shared__ T lds[SCAN_BLOCK / WAVE + 1];
    long long base = (long long)blockIdx.x * SCAN_TILE + (long long)threadIdx.x * SCAN_ITEMS;
    T v[SCAN_ITEMS];
    T s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        v[k] = (base + k < n) ? (T)in[base + k] : (T)0;
        s += v[k];
    }
    T total;
    T pre = block_exclusive_scan(s, lds, total);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        if (base + k < n) out[base + k] = pre;
        pre += v[k];
    }
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

template <class T> __global__ void k_scan_add(T *out, long long n, const T *tile_pre) {
    long long i = (long long)blockIdx.x * SCAN_TILE + threadIdx.x;
    T add = tile_pre[blockIdx.x];
    for (int k = 0; k < SCAN_ITEMS; k++, i += SCAN_BLOCK)
        if (i < n) out[i] += add;
}

template <class I, class T> __global__ void k_scan_fix(const I *in, T *out, long long n) {
    if (threadIdx.x == 0) out[n] = n > 0 ? out[n - 1] + (T)in[n - 1] : (T)0;
}

// bytes of tmp for sums of `elem` bytes
size_t scan_tmp_bytes(long long n, size_t elem) {
    size_t b = 0;
    long long m = n + 1;
    for (;;) {
        long long tiles = (m + SCAN_TILE - 1) / SCAN_TILE;
        b += (size_t)(2 * tiles + 4) * elem;
        if (tiles <= 1) break;
        m = tiles + 1;
    }
    return b + 256;
}

// out[i] = sum(in[0..i-1]); out must have n+1 entries (out[n] = total).
template <class I, class T> static void exclusive_scan(hipStream_t s, const I *in, T *out, long long n, void *tmp) {
    // scan n+1 elements where in[n] is treated as 0
    long long m = n + 1;
    long long tiles = (m + SCAN_TILE - 1) / SCAN_TILE;
    T *sums = (T *)tmp;
    T *pre = sums + tiles + 1;
    // in[n] may be out of bounds: run the tile scan on n elements and fix the
    // last entry with the tile total
    hipLaunchKernelGGL((k_scan_tiles<I, T>), dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, s, in, out, n, sums);
    if (tiles > 1) {
        exclusive_scan<T, T>(s, sums, pre, tiles, (void *)(pre + tiles + 1));
        hipLaunchKernelGGL(k_scan_add<T>, dim3((unsigned)tiles), dim3(SCAN_BLOCK), 0, s, out, n, pre);
    }
    // out[n] = out[n-1] + in[n-1]
    hipLaunchKernelGGL((k_scan_fix<I, T>), dim3(1), dim3(1), 0, s, in, out, n);
}
void exclusive_scan_i32(hipStream_t s, const int *in, int *out, long long n, void *tmp) {
    exclusive_scan<int, int>(s, in, out, n, tmp);
}
void exclusive_scan_i64(hipStream_t s, const int *in, int64_t *out, long long n, void *tmp) {
    exclusive_scan<int, int64_t>(s, in, out, n, tmp);
}

// ---------------------------------------------------------------------------
// Bounding box of the points (annEnclRect, ANN/src/kd_util.cpp:73-90).
__global__ void k_bbox_init(unsigned long long *t) {
    int i = threadIdx.x;
    if (i < 3) { t[i] = ~0ULL; t[3 + i] = 0ULL; }
}
__global__ void k_bbox(const double *pts, int n, int dim, unsigned long long *t) {
    __shared__ unsigned long long smin[3][4], smax[3][4];
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    for (int d = 0; d < dim; d++) {
        unsigned long long kmin = ~0ULL, kmax = 0;
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
            unsigned long long k = dkey(pts[(size_t)d * n + i]);
            kmin = k < kmin ? k : kmin;
            kmax = k > kmax ? k : kmax;
        }
        for (int o = WAVE / 2; o > 0; o >>= 1) {
            unsigned long long a = __shfl_down(kmin, o, WAVE), b = __shfl_down(kmax, o, WAVE);
            kmin = a < kmin ? a : kmin;
            kmax = b > kmax ? b : kmax;
        }
        if (lane == 0) { smin[d][w] = kmin; smax[d][w] = kmax; }
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)dim) {
        int d = threadIdx.x;
        unsigned long long a = smin[d][0], b = smax[d][0];
        for (int k = 1; k < 4; k++) { a = smin[d][k] < a ? smin[d][k] : a; b = smax[d][k] > b ? smax[d][k] : b; }
        atomicMin(&t[d], a);
        atomicMax(&t[3 + d], b);
    }
}
__global__ void k_bbox_fin(const unsigned long long *t, double *bb, int dim) {
    int d = threadIdx.x;
    if (d < 3) {
        bb[2 * d] = d < dim ? dkey_inv(t[d]) : 0.0;
        bb[2 * d + 1] = d < dim ? dkey_inv(t[3 + d]) : 0.0;
    }
}
void compute_bbox(hipStream_t s, const double *pts, int n, int dim, double *d_bbox, unsigned long long *tmp) {
    hipLaunchKernelGGL(k_bbox_init, dim3(1), dim3(64), 0, s, tmp);
    unsigned nb = (unsigned)std::min<long long>((n + 255) / 256, 512);
    hipLaunchKernelGGL(k_bbox, dim3(nb), dim3(256), 0, s, pts, n, dim, tmp);
    hipLaunchKernelGGL(k_bbox_fin, dim3(1), dim3(64), 0, s, tmp, d_bbox, dim);
}

// Cell grid with side >= h over the bounding box bb[6] (host values).
// Counts are formed in double: a point far from the rest (a bounding box of
// 1e7 cells per side) must coarsen the grid, not wrap an integer product.
// A non-finite extent (NaN/Inf positions, reported by the state check) gets
// one cell.
void grid_setup(const double *bb, int n, int dim, double h, Grid &g) {
    const double limit = (double)std::max<long long>(4LL * n, 1 << 20);
    double cell = h * 1.01;
    g.open = false;
    for (int d = 0; d < dim && d < 3; d++) g.open = g.open || !std::isfinite(bb[2 * d + 1] - bb[2 * d]);
    for (;;) {
        double tot = 1.0, c[3] = {1.0, 1.0, 1.0};
        for (int d = 0; d < dim && d < 3; d++) {
            const double ext = bb[2 * d + 1] - bb[2 * d];
            c[d] = (std::isfinite(ext) && ext > 0.0) ? std::floor(ext / cell) + 1.0 : 1.0;
            tot *= c[d];
        }
        if (tot <= limit || !std::isfinite(cell)) {
            long long t = 1;
            for (int d = 0; d < 3; d++) {
                g.dims[d] = d < dim ? (int)std::min(c[d], limit) : 1;
                g.origin[d] = d < dim ? bb[2 * d] : 0.0;
                g.tile[d] = g.ntile[d] = 0;
                t *= g.dims[d];
            }
            g.ncell = t;
            break;
        }
        cell *= 1.5;
    }
    g.inv_cell = 1.0 / cell;
}

__device__ __forceinline__ int cell_coord(double x, double o, double inv, int dimc) {
    double c = floor((x - o) * inv);
    if (c < -1.0) c = -1.0;
    if (c > (double)dimc) c = (double)dimc;
    return (int)c;
}

// Tiles of 4 x 4 x 4 cells in 3D, 8 x 8 in 2D, 64 in 1D (a few hundred
// points each at the search's cell size), narrower where the grid is.
void grid_tile(Grid &g, int dim) {
    const int T = dim >= 3 ? 4 : (dim == 2 ? 8 : 64);
    long long k = 1;
    for (int d = 0; d < 3; d++) {
        g.tile[d] = d < dim ? std::max(1, std::min(T, g.dims[d])) : 1;
        g.ntile[d] = (g.dims[d] + g.tile[d] - 1) / g.tile[d];
        k *= (long long)g.ntile[d] * g.tile[d];
    }
    g.ncell = k;
}

__device__ __forceinline__ int cell_key(const int c[3], const Grid &g) {
    if (g.tile[0] == 0) return (c[2] * g.dims[1] + c[1]) * g.dims[0] + c[0];
    const int t = (c[2] / g.tile[2] * g.ntile[1] + c[1] / g.tile[1]) * g.ntile[0] + c[0] / g.tile[0];
    const int w = ((c[2] % g.tile[2]) * g.tile[1] + c[1] % g.tile[1]) * g.tile[0] + c[0] % g.tile[0];
    return t * (g.tile[0] * g.tile[1] * g.tile[2]) + w;
}

// A position in units of the cells' side from the grid's corner, in single
// precision (see near_limit).
__device__ __forceinline__ float4 in_cells(const double x[3], int dim, const Grid &g) {
    float u[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 3; d++)
        if (d < dim) u[d] = (float)((x[d] - g.origin[d]) * g.inv_cell);
    return make_float4(u[0], u[1], u[2], 0.f);
}

// crowded: raised to a cell's count when it passes FR_MAX_CELL
__global__ void k_cell_count(const double *pts, int n, int dim, Grid g, int *cell_of, int *count, int *crowded) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int c[3] = {0, 0, 0};
    for (int d = 0; d < dim; d++) {
        int v = cell_coord(pts[(size_t)d * n + i], g.origin[d], g.inv_cell, g.dims[d]);
        c[d] = min(max(v, 0), g.dims[d] - 1);
    }
    const int cell = cell_key(c, g);
    cell_of[i] = cell;
    const int k = atomicAdd(&count[cell], 1) + 1;
    if (crowded && k > FR_MAX_CELL) atomicMax(crowded, k);
}

__global__ void k_cell_scatter(const double *pts, int n, int dim, Grid g, const int *cell_of, const int *start,
                               int *fill, int *sorted, double *spts, float4 *near) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int c = cell_of[i];
    int p = start[c] + atomicAdd(&fill[c], 1);
    sorted[p] = i;
    // one 32-byte record per point (x, y, z, its index): a candidate is two
    // 16-byte loads
    double x[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < dim; d++) x[d] = pts[(size_t)d * n + i];
    double2 *o = (double2 *)(spts + 4 * (size_t)p);
    o[0] = make_double2(x[0], x[1]);
    o[1] = make_double2(x[2], __longlong_as_double(i));
    if (near) near[p] = in_cells(x, dim, g);
}

void bin_points(hipStream_t s, const double *pts, int n, int dim, const Grid &g, int *cell_of, int *cell_count,
                int *cell_start, int *cell_fill, int *sorted, double *spts, void *scan_tmp, int *crowded, float4 *near) {
    HIP_OK(hipMemsetAsync(cell_count, 0, sizeof(int) * g.ncell, s));
    HIP_OK(hipMemsetAsync(cell_fill, 0, sizeof(int) * g.ncell, s));
    hipLaunchKernelGGL(k_cell_count, dim3((n + 255) / 256), dim3(256), 0, s, pts, n, dim, g, cell_of, cell_count,
                       crowded);
    exclusive_scan_i32(s, cell_count, cell_start, g.ncell, scan_tmp);
    hipLaunchKernelGGL(k_cell_scatter, dim3((n + 255) / 256), dim3(256), 0, s, pts, n, dim, g, cell_of, cell_start,
                       cell_fill, sorted, spts, near);
}

// One thread per cell: insertion sort of the cell's indices (cells hold a
// few tens of points; this runs only when particles are renumbered).  A cell
// past FR_MAX_CELL is left as it is: the search of that step reports it.
__global__ void k_cell_order(const int *start, long long ncell, int *sorted) {
    const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const int b = start[c], e = start[c + 1];
    if (e - b > FR_MAX_CELL) return;
    for (int i = b + 1; i < e; i++) {
        const int v = sorted[i];
        int j = i - 1;
        while (j >= b && sorted[j] > v) { sorted[j + 1] = sorted[j]; j--; }
        sorted[j + 1] = v;
    }
}

void cell_order_by_index(hipStream_t s, const int *cell_start, long long ncell, int *sorted) {
    if (ncell <= 0) return;
    hipLaunchKernelGGL(k_cell_order, dim3((unsigned)((ncell + 255) / 256)), dim3(256), 0, s, cell_start, ncell, sorted);
}

// ---------------------------------------------------------------------------
// GPU kd-tree (ANN sliding-midpoint rule, bucket size 1), built level by
// level.  The split of each cell follows sl_midpt_split exactly, and the
// two-pass partition reproduces annPlaneSplit's permutation: in each pass the
// k-th misplaced element from the left is swapped with the k-th misplaced
// element from the right, which is what the two-pointer loop does
// (ANN/src/kd_util.cpp:291-319).
struct KdWork {
    int *perm, *seg, *flags, *scan, *WL, *WR;
    int *s_start, *s_n, *s_node, *s_cd, *s_mode, *s_br1, *s_nlo, *s_clo, *s_chi;
    double *s_cv, *s_lo, *s_hi;                 // boxes [3][cap]
    unsigned long long *s_min, *s_max;          // [3][cap]
    int *n_start, *n_n, *n_node;                // next level
    double *n_lo, *n_hi;                        // [3][cap]
    // (cells that one workgroup finishes are kept at the far end of the n_
    // arrays, from cap - 1 down: a level has at most n / 1025 others)
    int *counters;                              // [0] next segs, [1] nodes, [2] cells kept for k_kd_local, [3] a cell had no split
    void *scan_tmp;
};

static size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

// Cells of up to this many points are split down to single points by one
// workgroup (k_kd_local), a point per thread.  A level over the whole array is
// 27 launches and a wait for the host, about 100 us however small its cells
// are, and a tree has some log2(n) + 4 levels: with the last ten of them in one
// launch the tree of 64,000 points takes 1.0 instead of 1.9 ms, of 121 points
// 0.13 instead of 0.72 ms.  1,024: the most a workgroup holds with a point per
// thread, at 85 KB of LDS.
constexpr int KD_LOCAL = 1024;

size_t kd_work_bytes(int n) {
    size_t cap = (size_t)n + 1;
    size_t b = 0;
    b += align_up(sizeof(int) * cap) * 6;                      // perm seg flags WL WR + spare
    b += align_up(sizeof(int) * (cap + 1));                    // scan
    b += align_up(sizeof(int) * cap) * 9;                      // s_* ints
    b += align_up(sizeof(double) * cap) * 7;                   // s_cv, s_lo[3], s_hi[3]
    b += align_up(sizeof(unsigned long long) * cap) * 6;       // s_min, s_max
    b += align_up(sizeof(int) * cap) * 3;                      // n_start n_n n_node
    b += align_up(sizeof(double) * cap) * 6;                   // n_lo n_hi
    b += align_up(sizeof(int) * 16);
    b += align_up(scan_tmp_bytes(cap + 1));
    return b + 4096;
}

static KdWork carve(void *base, int n) {
    size_t cap = (size_t)n + 1;
    char *p = (char *)base;
    auto take = [&](size_t bytes) { void *r = p; p += align_up(bytes); return r; };
    KdWork w;
    w.perm = (int *)take(sizeof(int) * cap);
    w.seg = (int *)take(sizeof(int) * cap);
    w.flags = (int *)take(sizeof(int) * cap);
    w.WL = (int *)take(sizeof(int) * cap);
    w.WR = (int *)take(sizeof(int) * cap);
    take(sizeof(int) * cap);
    w.scan = (int *)take(sizeof(int) * (cap + 1));
    w.s_start = (int *)take(sizeof(int) * cap);
    w.s_n = (int *)take(sizeof(int) * cap);
    w.s_node = (int *)take(sizeof(int) * cap);
    w.s_cd = (int *)take(sizeof(int) * cap);
    w.s_mode = (int *)take(sizeof(int) * cap);
    w.s_br1 = (int *)take(sizeof(int) * cap);
    w.s_nlo = (int *)take(sizeof(int) * cap);
    w.s_clo = (int *)take(sizeof(int) * cap);
    w.s_chi = (int *)take(sizeof(int) * cap);
    w.s_cv = (double *)take(sizeof(double) * cap);
    w.s_lo = (double *)take(sizeof(double) * cap * 3);
    w.s_hi = (double *)take(sizeof(double) * cap * 3);
    w.s_min = (unsigned long long *)take(sizeof(unsigned long long) * cap * 3);
    w.s_max = (unsigned long long *)take(sizeof(unsigned long long) * cap * 3);
    w.n_start = (int *)take(sizeof(int) * cap);
    w.n_n = (int *)take(sizeof(int) * cap);
    w.n_node = (int *)take(sizeof(int) * cap);
    w.n_lo = (double *)take(sizeof(double) * cap * 3);
    w.n_hi = (double *)take(sizeof(double) * cap * 3);
    w.counters = (int *)take(sizeof(int) * 16);
    w.scan_tmp = take(scan_tmp_bytes(cap + 1));
    return w;
}

__global__ void k_kd_init(int n, int *perm, int *seg, KdDev kd) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { perm[i] = i; seg[i] = 0; }
}

__global__ void k_kd_root(const double *bb, int n, int dim, KdWork w, KdDev kd, int cap) {
    if (threadIdx.x != 0) return;
    w.s_start[0] = 0;
    w.s_n[0] = n;
    w.s_node[0] = 0;
    for (int d = 0; d < 3; d++) {
        // A box from -inf to +inf has no middle to cut at: its cut would put
        // every point on the upper side and leave that child's lower bound NaN,
        // after which no cell is cut there again (lengths that do not compare
        // lose against the others).  The root starts so: its one child would
        // only add a level above all the points.  Dimension 0 is the one that
        // others are compared with, so there the tree is refused.
        const bool endless = d > 0 && bb[2 * d] == -INFINITY && bb[2 * d + 1] == INFINITY;
        w.s_lo[(size_t)d * cap] = endless ? NAN : bb[2 * d];
        w.s_hi[(size_t)d * cap] = bb[2 * d + 1];
    }
    kd.parent[0] = -1;
    kd.depth[0] = 0;
    kd.is_hi[0] = 0;
    kd.cd[0] = 0;
    kd.cv[0] = 0.0;
    w.counters[1] = 1;
    if (n == 1) kd.leaf_of[0] = 0;
    // a tree of one workgroup's points: the root is the one cell kept for it
    // (the box was read above: with n = 1 the arrays' ends are their starts)
    if (n > 1 && n <= KD_LOCAL) {
        w.n_start[cap - 1] = 0;
        w.n_n[cap - 1] = n;
        w.n_node[cap - 1] = 0;
        for (int d = 0; d < 3; d++) {
            w.n_lo[(size_t)d * cap + cap - 1] = w.s_lo[(size_t)d * cap];
            w.n_hi[(size_t)d * cap + cap - 1] = w.s_hi[(size_t)d * cap];
        }
    }
}

__global__ void k_kd_mm_init(int nseg, unsigned long long *mn, unsigned long long *mx, int cap) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nseg)
        for (int d = 0; d < 3; d++) { mn[(size_t)d * cap + i] = ~0ULL; mx[(size_t)d * cap + i] = 0ULL; }
}

// Segmented min/max over positions: a wave combines lanes of the same
// segment before one lane per segment run issues the atomics.
__global__ void k_kd_minmax(const double *pts, int n, int dim, const int *perm, const int *seg,
                            unsigned long long *mn, unsigned long long *mx, int cap) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    int lane = threadIdx.x & (WAVE - 1);
    int s = p < n ? seg[p] : -1;
    int sp = __shfl_up(s, 1, WAVE);
    bool head = (lane == 0) || (sp != s);
    for (int d = 0; d < dim; d++) {
        unsigned long long a = ~0ULL, b = 0ULL;
        if (s >= 0) a = b = dkey(pts[(size_t)d * n + perm[p]]);
        for (int o = 1; o < WAVE; o <<= 1) {
            unsigned long long oa = __shfl_down(a, o, WAVE), ob = __shfl_down(b, o, WAVE);
            int os = __shfl_down(s, o, WAVE);
            if (lane + o < WAVE && os == s) { a = oa < a ? oa : a; b = ob > b ? ob : b; }
        }
        if (head && s >= 0) {
            atomicMin(&mn[(size_t)d * cap + s], a);
            atomicMax(&mx[(size_t)d * cap + s], b);
        }
    }
}

// sl_midpt_split's choice of cut dimension and value (kd_split.cpp:146-188)
// for the box lo, hi and the points' extent mn, mx; mode 1 (2): the cut slid
// to the least (largest) coordinate.
__device__ __forceinline__ void kd_choose(const double lo[3], const double hi[3], const double mn[3],
                                          const double mx[3], int dim, int &cut_dim, double &cv, int &mode) {
    const double ERR = 0.001;
    double max_length = hi[0] - lo[0];
    for (int d = 1; d < dim; d++) {
        double length = hi[d] - lo[d];
        if (length > max_length) max_length = length;
    }
    double max_spread = -1, c_lo = lo[0], c_hi = hi[0], c_mn = mn[0], c_mx = mx[0];
    cut_dim = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (d < dim && (hi[d] - lo[d]) >= (1 - ERR) * max_length) {
            double spr = mx[d] - mn[d];
            if (spr > max_spread) {
                max_spread = spr;
                cut_dim = d;
                c_lo = lo[d]; c_hi = hi[d]; c_mn = mn[d]; c_mx = mx[d];
            }
        }
    }
    const double ideal = (c_lo + c_hi) / 2;
    mode = 0;
    if (ideal < c_mn) { cv = c_mn; mode = 1; }
    else if (ideal > c_mx) { cv = c_mx; mode = 2; }
    else cv = ideal;
}
// n_lo rule (kd_split.cpp:208-212)
__device__ __forceinline__ int kd_n_lo(int mode, int cnt, int br1, int br2) {
    if (mode == 1) return 1;
    if (mode == 2) return cnt - 1;
    if (br1 > cnt / 2) return br1;
    if (br2 < cnt / 2) return br2;
    return cnt / 2;
}

__global__ void k_kd_choose(int nseg, int dim, KdWork w, int cap) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    double lo[3], hi[3], mn[3], mx[3];
    for (int d = 0; d < 3; d++) {
        lo[d] = w.s_lo[(size_t)d * cap + s];
        hi[d] = w.s_hi[(size_t)d * cap + s];
        mn[d] = d < dim ? dkey_inv(w.s_min[(size_t)d * cap + s]) : 0.0;
        mx[d] = d < dim ? dkey_inv(w.s_max[(size_t)d * cap + s]) : 0.0;
    }
    int cut_dim, mode;
    double cv;
    kd_choose(lo, hi, mn, mx, dim, cut_dim, cv, mode);
    w.s_cd[s] = cut_dim;
    w.s_cv[s] = cv;
    w.s_mode[s] = mode;
}

// pass 0: flag v < cv on the whole segment; pass 1: flag v <= cv on
// [start+br1, end).
__global__ void k_kd_flags(const double *pts, int n, const int *perm, const int *seg, KdWork w, int pass) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int s = seg[p];
    int f = 0;
    if (s >= 0) {
        double v = pts[(size_t)w.s_cd[s] * n + perm[p]];
        double cv = w.s_cv[s];
        if (pass == 0) f = v < cv;
        else f = (p >= w.s_start[s] + w.s_br1[s]) && (v <= cv);
    }
    w.flags[p] = f;
}

// Ranks of misplaced elements and the swap (both passes).  Range of the pass:
// [b, e) with b = start (+br1 for pass 1); C = number of flagged elements.
__global__ void k_kd_rank(int n, const int *perm, const int *seg, KdWork w, int pass) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int s = seg[p];
    if (s < 0) return;
    int b = w.s_start[s] + (pass ? w.s_br1[s] : 0);
    int e = w.s_start[s] + w.s_n[s];
    if (p < b) return;
    const int *A = w.scan;
    int C = A[e] - A[b];
    int f = w.flags[p];
    if (p < b + C && !f) {
        int k = (p - b) - (A[p] - A[b]);
        w.WL[b + k] = perm[p];
    } else if (p >= b + C && f) {
        int k = A[e] - A[p + 1];
        w.WR[b + k] = perm[p];
    }
}
__global__ void k_kd_swap(int n, int *perm, const int *seg, KdWork w, int pass) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int s = seg[p];
    if (s < 0) return;
    int b = w.s_start[s] + (pass ? w.s_br1[s] : 0);
    int e = w.s_start[s] + w.s_n[s];
    if (p < b) return;
    const int *A = w.scan;
    int C = A[e] - A[b];
    int f = w.flags[p];
    if (p < b + C && !f) {
        int k = (p - b) - (A[p] - A[b]);
        perm[p] = w.WR[b + k];
    } else if (p >= b + C && f) {
        int k = A[e] - A[p + 1];
        perm[p] = w.WL[b + k];
    }
}
__global__ void k_kd_br1(int nseg, KdWork w) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    int b = w.s_start[s], e = b + w.s_n[s];
    w.s_br1[s] = w.scan[e] - w.scan[b];
}

// Node records and the next level.
__global__ void k_kd_children(int nseg, KdWork w, KdDev kd, const int *perm, int cap) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    int b = w.s_start[s], cnt = w.s_n[s];
    int br1 = w.s_br1[s];
    int br2 = br1 + (w.scan[b + cnt] - w.scan[b + br1]);
    int mode = w.s_mode[s];
    int n_lo = kd_n_lo(mode, cnt, br1, br2);
    if (n_lo < 1 || n_lo >= cnt) {      // coordinates that do not compare (NaN)
        w.counters[3] = 1;
        n_lo = cnt / 2;
    }
    w.s_nlo[s] = n_lo;
    int node = w.s_node[s];
    int cd = w.s_cd[s];
    double cv = w.s_cv[s];
    kd.cd[node] = cd;
    kd.cv[node] = cv;
    int c0 = atomicAdd(&w.counters[1], 2);
    int dep = kd.depth[node] + 1;
    for (int side = 0; side < 2; side++) {
        int child = c0 + side;
        int cstart = side ? b + n_lo : b;
        int cn = side ? cnt - n_lo : n_lo;
        kd.parent[child] = node;
        kd.depth[child] = dep;
        kd.is_hi[child] = side;
        kd.cd[child] = 0;
        kd.cv[child] = 0.0;
        int nseg_id = -1;
        if (cn == 1) {
            kd.leaf_of[perm[cstart]] = child;
        } else if (cn > 1) {
            int at;
            if (cn > KD_LOCAL) at = nseg_id = atomicAdd(&w.counters[0], 1);
            else at = cap - 1 - atomicAdd(&w.counters[2], 1);
            w.n_start[at] = cstart;
            w.n_n[at] = cn;
            w.n_node[at] = child;
            for (int d = 0; d < 3; d++) {
                double lo = w.s_lo[(size_t)d * cap + s], hi = w.s_hi[(size_t)d * cap + s];
                if (d == cd) {
                    if (side == 0) hi = cv;
                    else lo = cv;
                }
                w.n_lo[(size_t)d * cap + at] = lo;
                w.n_hi[(size_t)d * cap + at] = hi;
            }
        }
        if (side == 0) w.s_clo[s] = nseg_id;
        else w.s_chi[s] = nseg_id;
    }
}

__global__ void k_kd_reseg(int n, int *seg, KdWork w) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int s = seg[p];
    if (s < 0) return;
    seg[p] = (p - w.s_start[s] < w.s_nlo[s]) ? w.s_clo[s] : w.s_chi[s];
}

__global__ void k_kd_promote(int nseg, KdWork w, int cap) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    w.s_start[s] = w.n_start[s];
    w.s_n[s] = w.n_n[s];
    w.s_node[s] = w.n_node[s];
    for (int d = 0; d < 3; d++) {
        w.s_lo[(size_t)d * cap + s] = w.n_lo[(size_t)d * cap + s];
        w.s_hi[(size_t)d * cap + s] = w.n_hi[(size_t)d * cap + s];
    }
}

// One workgroup splits one kept cell down to single points, level by level as
// the kernels above do: thread p holds the point at position p of the cell,
// the range [b, e) of its present sub-cell and that one's box and node.
__global__ void __launch_bounds__(KD_LOCAL)
k_kd_local(const double *__restrict__ pts, int n, int dim, KdWork w, KdDev kd, int cap) {
    __shared__ double x[3][KD_LOCAL];                        // by place in the cell at the start
    __shared__ unsigned long long s_mn[3][KD_LOCAL], s_mx[3][KD_LOCAL];   // by b
    __shared__ int A[KD_LOCAL + 1], WL[KD_LOCAL], WR[KD_LOCAL], w_tot[KD_LOCAL / WAVE], s_base;
    const int seg = cap - 1 - (int)blockIdx.x;
    const int start = w.n_start[seg], m = w.n_n[seg];
    const int p = threadIdx.x, lane = p & (WAVE - 1), wv = p / WAVE;
    const bool live = p < m;
    // exclusive prefix of a flag over the threads into A; the total
    auto scan = [&](bool f) {
        const unsigned long long h = __ballot(f);
        if (lane == 0) w_tot[wv] = (int)__popcll(h);
        __syncthreads();
        int pre = 0, all = 0;
        for (int u = 0; u < KD_LOCAL / WAVE; u++) {
            if (u == wv) pre = all;
            all += w_tot[u];
        }
        A[p] = pre + (int)__popcll(h & ((1ULL << lane) - 1ULL));
        if (p == 0) A[KD_LOCAL] = all;
        __syncthreads();
        return all;
    };
    int id = p;                                              // place at the start of the point held now
    const int g0 = live ? w.perm[start + p] : 0;             // its index
    for (int d = 0; d < 3; d++) x[d][p] = live && d < dim ? pts[(size_t)d * n + g0] : 0.0;
    int b = 0, e = m, node = w.n_node[seg];
    int depth = kd.depth[node];
    double lo[3], hi[3];
    for (int d = 0; d < 3; d++) {
        lo[d] = w.n_lo[(size_t)d * cap + seg];
        hi[d] = w.n_hi[(size_t)d * cap + seg];
    }
    // a cell of m points has 2m - 2 nodes below its own
    if (p == 0) s_base = atomicAdd(&w.counters[1], 2 * m - 2);
    __syncthreads();
    int base = s_base;
    bool on = live && m > 1;
    // every level splits every sub-cell of two or more points
    while (__syncthreads_or(on)) {
        if (on && p == b)
            for (int d = 0; d < dim; d++) { s_mn[d][b] = ~0ULL; s_mx[d][b] = 0ULL; }
        __syncthreads();
        const int tag = on ? b : -1, up = __shfl_up(tag, 1, WAVE);
        const bool head = on && (lane == 0 || up != tag);
        for (int d = 0; d < dim; d++) {
            unsigned long long mn = ~0ULL, mx = 0ULL;
            if (on) mn = mx = dkey(x[d][id]);
            for (int o = 1; o < WAVE; o <<= 1) {
                const unsigned long long on_ = __shfl_down(mn, o, WAVE), ox = __shfl_down(mx, o, WAVE);
                const int ot = __shfl_down(tag, o, WAVE);
                if (lane + o < WAVE && ot == tag) { mn = on_ < mn ? on_ : mn; mx = ox > mx ? ox : mx; }
            }
            if (head) {
                atomicMin(&s_mn[d][b], mn);
                atomicMax(&s_mx[d][b], mx);
            }
        }
        __syncthreads();
        int cd = 0, mode = 0;
        double cv = 0.0;
        if (on) {
            double mn[3], mx[3];
            for (int d = 0; d < 3; d++) {
                mn[d] = d < dim ? dkey_inv(s_mn[d][b]) : 0.0;
                mx[d] = d < dim ? dkey_inv(s_mx[d][b]) : 0.0;
            }
            kd_choose(lo, hi, mn, mx, dim, cd, cv, mode);
        }
        // annPlaneSplit's two passes: v < cv over the sub-cell, then v <= cv
        // over what is left of it
        int br[2] = {0, 0};
        for (int pass = 0; pass < 2; pass++) {
            const int from = b + (pass ? br[0] : 0);
            const double v = on ? x[cd][id] : 0.0;
            const bool f = on && p >= from && (pass ? v <= cv : v < cv);
            scan(f);
            const int C = on ? A[e] - A[from] : 0;
            br[pass] = C;
            const bool left = on && p >= from && p < from + C && !f, right = on && p >= from + C && f;
            const int kl = left ? (p - from) - (A[p] - A[from]) : 0;
            const int kr = right ? A[e] - A[p + 1] : 0;
            if (left) WL[from + kl] = id;
            if (right) WR[from + kr] = id;
            __syncthreads();
            if (left) id = WR[from + kl];
            if (right) id = WL[from + kr];
            __syncthreads();
        }
        int n_lo = on ? kd_n_lo(mode, e - b, br[0], br[0] + br[1]) : 0;
        if (on && (n_lo < 1 || n_lo >= e - b)) {   // coordinates that do not compare (NaN)
            w.counters[3] = 1;
            n_lo = (e - b) / 2;
        }
        // two nodes for each sub-cell, in the order of the sub-cells
        const bool lead = on && p == b;
        const int segs = scan(lead);
        if (on) {
            const int c0 = base + 2 * A[b];
            if (lead) {
                kd.cd[node] = cd;
                kd.cv[node] = cv;
                for (int side = 0; side < 2; side++) {
                    kd.parent[c0 + side] = node;
                    kd.depth[c0 + side] = depth + 1;
                    kd.is_hi[c0 + side] = side;
                    kd.cd[c0 + side] = 0;
                    kd.cv[c0 + side] = 0.0;
                }
            }
            const int side = p - b >= n_lo ? 1 : 0;
            node = c0 + side;
            depth++;
#pragma unroll
            for (int d = 0; d < 3; d++)
                if (d == cd) {
                    if (side) lo[d] = cv;
                    else hi[d] = cv;
                }
            if (side) b += n_lo;
            else e = b + n_lo;
            if (e - b == 1) {
                kd.leaf_of[w.perm[start + id]] = node;
                on = false;
            }
        }
        base += 2 * segs;
    }
}

void kd_build(hipStream_t st, const double *pts, int n, int dim, KdDev &kd, void *work, size_t work_bytes) {
    (void)work_bytes;
    KdWork w = carve(work, n);
    int cap = n + 1;
    const int B = 256;
    unsigned gn = (unsigned)((n + B - 1) / B);
    // root box = bounding rectangle of the points
    double *d_bb = (double *)w.n_lo;   // scratch for the 6 bbox values
    compute_bbox(st, pts, n, dim, d_bb, (unsigned long long *)w.s_min);
    hipLaunchKernelGGL(k_kd_init, dim3(gn), dim3(B), 0, st, n, w.perm, w.seg, kd);
    HIP_OK(hipMemsetAsync(w.counters, 0, sizeof(int) * 16, st));
    hipLaunchKernelGGL(k_kd_root, dim3(1), dim3(64), 0, st, d_bb, n, dim, w, kd, cap);
    int nseg = n > KD_LOCAL ? 1 : 0, local = n > 1 && n <= KD_LOCAL ? 1 : 0;
    int levels = 0;
    while (nseg > 0) {
        unsigned gs = (unsigned)((nseg + B - 1) / B);
        hipLaunchKernelGGL(k_kd_mm_init, dim3(gs), dim3(B), 0, st, nseg, w.s_min, w.s_max, cap);
        hipLaunchKernelGGL(k_kd_minmax, dim3(gn), dim3(B), 0, st, pts, n, dim, w.perm, w.seg, w.s_min, w.s_max, cap);
        hipLaunchKernelGGL(k_kd_choose, dim3(gs), dim3(B), 0, st, nseg, dim, w, cap);
        // pass 1: < cv
        hipLaunchKernelGGL(k_kd_flags, dim3(gn), dim3(B), 0, st, pts, n, w.perm, w.seg, w, 0);
        exclusive_scan_i32(st, w.flags, w.scan, n, w.scan_tmp);
        hipLaunchKernelGGL(k_kd_rank, dim3(gn), dim3(B), 0, st, n, w.perm, w.seg, w, 0);
        hipLaunchKernelGGL(k_kd_swap, dim3(gn), dim3(B), 0, st, n, w.perm, w.seg, w, 0);
        hipLaunchKernelGGL(k_kd_br1, dim3(gs), dim3(B), 0, st, nseg, w);
        // pass 2: <= cv on [start+br1, end)
        hipLaunchKernelGGL(k_kd_flags, dim3(gn), dim3(B), 0, st, pts, n, w.perm, w.seg, w, 1);
        exclusive_scan_i32(st, w.flags, w.scan, n, w.scan_tmp);
        hipLaunchKernelGGL(k_kd_rank, dim3(gn), dim3(B), 0, st, n, w.perm, w.seg, w, 1);
        hipLaunchKernelGGL(k_kd_swap, dim3(gn), dim3(B), 0, st, n, w.perm, w.seg, w, 1);
        HIP_OK(hipMemsetAsync(w.counters, 0, sizeof(int), st));
        hipLaunchKernelGGL(k_kd_children, dim3(gs), dim3(B), 0, st, nseg, w, kd, w.perm, cap);
        hipLaunchKernelGGL(k_kd_reseg, dim3(gn), dim3(B), 0, st, n, w.seg, w);
        int cnt[3] = {0, 0, 0};
        HIP_OK(hipMemcpyAsync(cnt, w.counters, sizeof(cnt), hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        const int next = cnt[0];
        local = cnt[2];
        if (next > 0) {
            hipLaunchKernelGGL(k_kd_promote, dim3((unsigned)((next + B - 1) / B)), dim3(B), 0, st, next, w, cap);
        }
        nseg = next;
        if (++levels > n + 2) throw HipError("kd_build: no progress", hipErrorUnknown, __FILE__, __LINE__);
    }
    if (local > 0)
        hipLaunchKernelGGL(k_kd_local, dim3((unsigned)local), dim3(KD_LOCAL), 0, st, pts, n, dim, w, kd, cap);
    int bad = 0;
    HIP_OK(hipMemcpyAsync(&bad, w.counters + 3, sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    if (bad) throw HipError("kd_build: no progress", hipErrorUnknown, __FILE__, __LINE__);
    kd.n_nodes = 2 * n - 1;
    kd.valid = true;
}

// ---------------------------------------------------------------------------
// Fixed-radius search.

// Each lane of the search builds and sorts its list in SLOTS LDS slots
// (slot-major, one column per lane of a one-wavefront block) and writes it
// out once.  A list that outgrows them moves to the output arrays (entries
// in visit order, then the later hits) and is sorted there, one global
// round trip per step of the insertion sort, which stalls the whole
// wavefront: the launch picks the smallest of 12, 16, 24 or 32 slots that
// holds the longest list of the previous search (fewer slots keep more
// wavefronts resident for the gathers; a lattice at h = 1.3 spacing holds 6
// neighbours per list, a flowing one 9 on average and up to ~20).
constexpr int FR_SLOT_CHOICES[4] = {12, 16, 24, 32};

struct KdView {
    const int *parent, *depth, *cd, *is_hi, *leaf_of;
    const double *cv;
    int valid;
};

// true when tree point a is visited before tree point b by ANN's search from
// query q (nearer child first: cut_diff < 0 visits the low child first,
// kd_fix_rad_search.cpp:106-136).
__device__ bool kd_before(const KdView &kd, int a, int b, const double *q) {
    if (!kd.valid) return a < b;
    int na = kd.leaf_of[a], nb = kd.leaf_of[b];
    int da = kd.depth[na], db = kd.depth[nb];
    while (da > db) { na = kd.parent[na]; da--; }
    while (db > da) { nb = kd.parent[nb]; db--; }
    while (kd.parent[na] != kd.parent[nb]) { na = kd.parent[na]; nb = kd.parent[nb]; }
    int p = kd.parent[na];
    double cut_diff = q[kd.cd[p]] - kd.cv[p];
    int near_hi = cut_diff < 0 ? 0 : 1;
    return kd.is_hi[na] == near_hi;
}

// Insertion sort of a list of cnt entries by (r2, ANN visit order); I and D
// return references to entry k's index and r2.
template <class IA, class DA>
__device__ __forceinline__ void sort_list(IA I, DA D, int cnt, const KdView &kd, const double *qp) {
    for (int i = 1; i < cnt; i++) {
        int ji = I(i);
        double ri = D(i);
        int k = i - 1;
        while (k >= 0) {
            double rk = D(k);
            int jk = I(k);
            bool after = rk > ri || (rk == ri && kd_before(kd, ji, jk, qp));
            if (!after) break;
            I(k + 1) = jk;
            D(k + 1) = rk;
            k--;
        }
        I(k + 1) = ji;
        D(k + 1) = ri;
    }
}

// D_ij of one edge (add_to_neighbor_list, particle.cpp:160-187): the 3-D
// constant of wfd in every dimension, operation for operation.
__device__ __forceinline__ double edge_dij(double mi, double ri, double mj, double rj, double rr2, double rr,
                                           double h) {
    double ih = 1.0 / h;
    double ihsq = ih * ih;
    double dhr = h - rr;
    double wfd = -25.066903536973515383e0 * dhr * dhr * ihsq * ihsq * ihsq * ih;
    const double m = Den<double>(mi + mj).div(-2.0 * (mi * mj));
    const double D = Den<double>(rr2 + 0.01 * h * h).div(Den<double>(ri * rj).div(m * (ri + rj)) * rr2 * wfd);
    if (D == D) return D;
    // a divisor of 0: the plain divisions tell inf and NaN apart
    return -2.0 * (mi * mj) / (mi + mj) * (ri + rj) / (ri * rj) * rr2 * wfd / (rr2 + 0.01 * h * h);
}

// SLOTS 0: the lists' lengths only.
// NEAR: of the candidates in a query's 27 cells (57 for 9 neighbours) most are
// told apart by their single-precision positions in units of a cell (near,
// 16 bytes each), with room for those positions' rounding (see near_limit);
// only what remains is loaded and compared in double precision.  What bounds
// the search is the address unit and L1 (a wavefront's 64 queries load from 64
// different lines at each candidate, three loads each before: 212 million
// accesses for a million queries, 136 now); a query with more than SLOTS such
// candidates takes the plain way.  Cylinder: 0.62 -> 0.54 ms at 1,000,000
// particles, 70 -> 63 us at 64,000 (the binning, which writes near, +11 us at a
// million).  Also tried: rows of cells staged in LDS (0.68 ms: queries go in the
// particles' order, in which few runs of cells join up), and the event loop's
// rows written four lanes to a row (0.56 ms: no gain).
template <int SLOTS, bool NEAR>
__global__ void __launch_bounds__(WAVE)
k_fr_search(const double *__restrict__ q, int m, const double *__restrict__ spts, const float4 *__restrict__ near,
            float lim_near, const int *__restrict__ cell_start, int n, int dim, double h, Grid g, KdView kd, int W,
            int *__restrict__ out_idx, double *__restrict__ out_r2, int *__restrict__ deg, DevErr *err,
            const int *__restrict__ order, FinishArgs fin, int has_fin) {
    __shared__ int l_idx[SLOTS > 0 ? SLOTS * WAVE : 1];
    __shared__ double l_r2[SLOTS > 0 ? SLOTS * WAVE : 1];
    __shared__ double s_dm[FIN_MAX_DMAT];
    const int tl = (int)threadIdx.x;
    if (has_fin && fin.Ddiag) {
        for (int k = tl; k < fin.S * fin.T; k += WAVE) s_dm[k] = fin.Dmat[k];
        __syncthreads();
    }
    const int chunk = xcd_chunk((m + WAVE - 1) / WAVE);
    if (chunk < 0) return;
    int t = chunk * WAVE + tl;
    // lanes past the end stay for the wave's reduction of the degree
    const bool live = t < m;
    int qi = live ? (order ? order[t] : t) : 0;
    int cnt = 0;
    if (err->crowded > 0) {
        // the binning put more than FR_MAX_CELL points in one cell (a point
        // far from the rest coarsened the grid): no lists, and the step
        // reports it instead of scanning those cells for every query
        if (live) deg[qi] = 0;
        if (t == 0) atomicCAS(&err->code, 0, (int)SSASDPD_ERR_CAPACITY);
        return;
    }
    if (live) {
        auto LI = [&](int k) -> int & { return l_idx[k * WAVE + tl]; };
        auto LD = [&](int k) -> double & { return l_r2[k * WAVE + tl]; };
        auto GI = [&](int k) -> int & { return out_idx[(size_t)k * m + qi]; };
        auto GD = [&](int k) -> double & { return out_r2[(size_t)k * m + qi]; };
        const int L = W < SLOTS ? W : SLOTS;   // LDS slots in use
        double qp[3] = {0.0, 0.0, 0.0};
        for (int d = 0; d < dim; d++) qp[d] = q[(size_t)d * m + qi];
        int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
        for (int d = 0; d < 3; d++) {
            if (d < dim) {
                const int c = cell_coord(qp[d], g.origin[d], g.inv_cell, g.dims[d]);
                lo[d] = max(c - 1, 0);
                hi[d] = min(c + 1, g.dims[d] - 1);
            }
        }
        // a point at squared distance d belongs to the list if d <= h * h, d != 0
        // and sqrt(d) <= h; the root is monotone, so that is one comparison
        // with the largest such d
        double lim = h * h;
        while (sqrt(lim) > h) lim = __longlong_as_double(__double_as_longlong(lim) - 1);
        // the candidate rows' bounds, all loaded before the first is used
        int rb[9], re[9], nrow = 0;
        for (int cz = lo[2]; cz <= hi[2]; cz++)
            for (int cy = lo[1]; cy <= hi[1]; cy++) {
                const int row = (cz * g.dims[1] + cy) * g.dims[0];
                rb[nrow] = cell_start[row + lo[0]];
                re[nrow] = cell_start[row + hi[0] + 1];
                nrow++;
            }
        auto accept = [&](int j, double dist) {
            if constexpr (SLOTS == 0) {
                cnt++;
                return;
            }
            if (cnt < L) {
                LI(cnt) = j;
                LD(cnt) = dist;
            } else {
                if (cnt == L)   // the list moves to the output arrays
                    for (int k = 0; k < L; k++) { GI(k) = LI(k); GD(k) = LD(k); }
                if (cnt < W) { GI(cnt) = j; GD(cnt) = dist; }
            }
            cnt++;
        };
        auto exact = [&](const double2 &a, const double2 &b) {
            double dist = 0.0;
            double t0 = qp[0] - a.x;
            dist = dist + t0 * t0;
            if (dim > 1) { double t1 = qp[1] - a.y; dist = dist + t1 * t1; }
            if (dim > 2) { double t2 = qp[2] - b.x; dist = dist + t2 * t2; }
            if (dist <= lim && dist != 0.0) accept((int)__double_as_longlong(b.y), dist);
        };
        // candidates in visit order, fetched CB at a time so one round trip
        // serves CB of them
        constexpr int CB = 4, CN = 8;
        bool plain = true;
        if constexpr (NEAR) {
            const float4 qn = in_cells(qp, dim, g);
            int found = 0;
            for (int r = 0; r < nrow; r++) {
                const int pe = re[r];
                for (int p0 = rb[r]; p0 < pe; p0 += CN) {
                    float4 c[CN];
#pragma unroll
                    for (int u = 0; u < CN; u++) c[u] = near[p0 + u < pe ? p0 + u : p0];
#pragma unroll
                    for (int u = 0; u < CN; u++) {
                        const float dx = qn.x - c[u].x, dy = qn.y - c[u].y, dz = qn.z - c[u].z;
                        // (not a number: left to the exact test)
                        if (p0 + u < pe && !(dx * dx + dy * dy + dz * dz > lim_near)) {
                            if (found < SLOTS) LI(found) = p0 + u;
                            found++;
                        }
                    }
                }
            }
            plain = found > SLOTS;
            if (!plain) {
                for (int k0 = 0; k0 < found; k0 += CB) {
                    double2 a[CB], b[CB];
#pragma unroll
                    for (int u = 0; u < CB; u++) {
                        const double2 *sp = (const double2 *)(spts + 4 * (size_t)LI(k0 + u < found ? k0 + u : k0));
                        a[u] = sp[0];
                        b[u] = sp[1];
                    }
                    // (the list grows behind the places read)
#pragma unroll
                    for (int u = 0; u < CB; u++)
                        if (k0 + u < found) exact(a[u], b[u]);
                }
            }
        }
        if (plain) {
            for (int r = 0; r < nrow; r++) {
                const int pe = re[r];
                for (int p0 = rb[r]; p0 < pe; p0 += CB) {
                    double2 a[CB], b[CB];
#pragma unroll
                    for (int u = 0; u < CB; u++) {
                        const double2 *sp = (const double2 *)(spts + 4 * (size_t)(p0 + u < pe ? p0 + u : p0));
                        a[u] = sp[0];
                        b[u] = sp[1];
                    }
#pragma unroll
                    for (int u = 0; u < CB; u++)
                        if (p0 + u < pe) exact(a[u], b[u]);
                }
            }
        }
        if (SLOTS == 0) {
            deg[qi] = cnt;
        } else if (cnt > W) {
            atomicExch(&err->overflow, 1);
            deg[qi] = 0;
        } else {
            deg[qi] = cnt;
            if (cnt <= L) {
                sort_list(LI, LD, cnt, kd, qp);
                // with the finish, r2 is only the spill area of long lists
                for (int k = 0; k < cnt; k++) {
                    GI(k) = LI(k);
                    if (!has_fin) GD(k) = LD(k);
                }
            } else {
                sort_list(GI, GD, cnt, kd, qp);
            }
            if (has_fin) {
                // r, D_ij, the neighbour's type and the voxel-major row, in
                // list order; the neighbours' records are fetched FB at a
                // time ahead of the stores (the compiler cannot move a load
                // above a store through these pointers)
                const double mi = fin.mass[qi], ri = fin.rho[qi];
                double dd[FIN_MAX_SPECIES] = {};
                constexpr int FB = 4;
                for (int k0 = 0; k0 < cnt; k0 += FB) {
                    int jj[FB], tj[FB];
                    double rr2[FB], rj[FB], mj[FB];
#pragma unroll
                    for (int u = 0; u < FB; u++) {
                        const int k = k0 + u < cnt ? k0 + u : k0;
                        jj[u] = cnt <= L ? LI(k) : GI(k);
                        rr2[u] = cnt <= L ? LD(k) : GD(k);
                        if (fin.rec) {
                            const PRec *pj = fin.rec + jj[u];
                            const double2 rm = *(const double2 *)&pj->rho;
                            rj[u] = rm.x;
                            mj[u] = rm.y;
                            tj[u] = pj->type;
                        } else {
                            mj[u] = fin.mass[jj[u]];
                            rj[u] = fin.rho[jj[u]];
                            tj[u] = fin.type[jj[u]];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < FB; u++) {
                        const int k = k0 + u;
                        if (k >= cnt) break;
                        const double rr = sqrt(rr2[u]);
                        const double D = edge_dij(mi, ri, mj[u], rj[u], rr2[u], rr, h);
                        if (D != D) {
                            atomicCAS(&err->code, 0, (int)SSASDPD_ERR_NAN_DIJ);
                            atomicMin(&err->particle, qi);
                        }
                        const size_t e = (size_t)k * m + qi;
                        fin.r[e] = rr;
                        if (fin.Dij) fin.Dij[e] = D;
                        if (fin.ntype) fin.ntype[e] = tj[u];
                        fin.erow[(size_t)qi * W + k] = EdgeRec{jj[u], tj[u], D};
                        if (fin.Ddiag) {
#pragma unroll
                            for (int s2 = 0; s2 < FIN_MAX_SPECIES; s2++)
                                if (s2 < fin.S) dd[s2] += s_dm[s2 * fin.T + (tj[u] - 1)] * D;
                        }
                    }
                }
                if (fin.Ddiag) {
#pragma unroll
                    for (int s2 = 0; s2 < FIN_MAX_SPECIES; s2++)
                        if (s2 < fin.S) fin.Ddiag[(size_t)qi * fin.S + s2] = dd[s2];
                }
            }
        }
    }
    // one atomic per wavefront for the longest list
    int mx = cnt;
    for (int o = WAVE / 2; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, WAVE));
    if (tl == 0) atomicMax(&err->max_deg, mx);
}

// The squared distance, in cells and single precision, past which a point is
// farther than h for certain.  Of two positions at most `span` cells from the
// corner each component is off by at most 2^-24 span, their difference by
// 2^-23 span and one rounding, the distance by sqrt(3) times that and 1e-6 of
// itself: 4 2^-23 span + 1e-5 covers it.  (A span past 2^20 leaves the filter
// little to tell apart, and it lets everything through; so does a grid with an
// open dimension, whose one cell says nothing about the positions in it.)
static float near_limit(const Grid &g, double h) {
    if (g.open) return INFINITY;
    const double span = 2.0 + std::max({g.dims[0], g.dims[1], g.dims[2]});
    const double r = h * g.inv_cell + 1e-5 + 4.0 * 1.1920928955078125e-7 * span;
    return (float)(r * r * 1.00001);
}
template <int SLOTS>
static void launch_search(hipStream_t s, const double *q, int m, const double *spts, const float4 *near,
                          const int *cell_start, int n, int dim, double h, const Grid &g, const KdView &v, int W,
                          int *out_idx, double *out_r2, int *deg, DevErr *err, const int *order, const FinishArgs *fin) {
    const FinishArgs f = fin ? *fin : FinishArgs{};
    const dim3 grid = xcd_grid((m + WAVE - 1) / WAVE);
    if constexpr (SLOTS > 0) {
        if (near) {
            hipLaunchKernelGGL((k_fr_search<SLOTS, true>), grid, dim3(WAVE), 0, s, q, m, spts, near, near_limit(g, h),
                               cell_start, n, dim, h, g, v, W, out_idx, out_r2, deg, err, order, f, fin ? 1 : 0);
            return;
        }
    }
    hipLaunchKernelGGL((k_fr_search<SLOTS, false>), grid, dim3(WAVE), 0, s, q, m, spts, nullptr, 0.f, cell_start, n,
                       dim, h, g, v, W, out_idx, out_r2, deg, err, order, f, fin ? 1 : 0);
}

void fr_search(hipStream_t s, const double *q, int m, const double *spts, const float4 *near, const int *cell_start,
               int n, int dim, double h, const Grid &g, const KdDev *kd, int W, int *out_idx, double *out_r2,
               int *deg, DevErr *err, const int *order, const FinishArgs *fin, int slots_hint) {
    KdView v{};
    if (kd && kd->valid) {
        v.parent = kd->parent; v.depth = kd->depth; v.cd = kd->cd; v.is_hi = kd->is_hi;
        v.leaf_of = kd->leaf_of; v.cv = kd->cv; v.valid = 1;
    }
    // a query that is a point finds itself among the near candidates; an
    // engine's hint is the longest list of a step before, which few reach
    const int want = slots_hint + (near && !fin ? 1 : 0);
    // lists past every choice, or close to the last: their near candidates (the
    // lists and a few more) do not fit either, and the query walks its cells twice
    // (60,000 particles, lists of up to 30: 211 us, 185 without the first pass;
    // lists of up to 27: 125 us with it, 144 without)
    if (want > FR_SLOT_CHOICES[3] - 4) near = nullptr;
    if (want <= FR_SLOT_CHOICES[0])
        launch_search<12>(s, q, m, spts, near, cell_start, n, dim, h, g, v, W, out_idx, out_r2, deg, err, order, fin);
    else if (want <= FR_SLOT_CHOICES[1])
        launch_search<16>(s, q, m, spts, near, cell_start, n, dim, h, g, v, W, out_idx, out_r2, deg, err, order, fin);
    else if (want <= FR_SLOT_CHOICES[2])
        launch_search<24>(s, q, m, spts, near, cell_start, n, dim, h, g, v, W, out_idx, out_r2, deg, err, order, fin);
    else
        launch_search<32>(s, q, m, spts, near, cell_start, n, dim, h, g, v, W, out_idx, out_r2, deg, err, order, fin);
}

void fr_count(hipStream_t s, const double *q, int m, const double *spts, const int *cell_start, int n, int dim,
              double h, const Grid &g, int *deg, DevErr *err) {
    launch_search<0>(s, q, m, spts, nullptr, cell_start, n, dim, h, g, KdView{}, 0, nullptr, nullptr, deg, err,
                     nullptr, nullptr);
}

// ---------------------------------------------------------------------------
// Host layouts: particle-major points to component-major, column-major lists to
// rows.
__global__ void k_soa3(const double *aos, int n, double *soa) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int d = 0; d < 3; d++) soa[(size_t)d * n + i] = aos[3 * (size_t)i + d];
}
__global__ void k_csr(int m, int W, const int *deg, const int64_t *row, const int *oi, const double *orr, int *ci,
                      double *cr) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int d = deg[i];
    const int64_t o = row[i];
    for (int k = 0; k < d && k < W; k++) {
        ci[o + k] = oi[(size_t)k * m + i];
        cr[o + k] = orr[(size_t)k * m + i];
    }
}
void soa3(hipStream_t s, const double *aos, int n, double *soa) {
    if (n > 0) hipLaunchKernelGGL(k_soa3, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, aos, n, soa);
}
void csr_lists(hipStream_t s, int m, int W, const int *deg, const int64_t *row, const int *oi, const double *orr,
               int *ci, double *cr) {
    if (m > 0)
        hipLaunchKernelGGL(k_csr, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, m, W, deg, row, oi, orr, ci, cr);
}

}  // namespace ssa
