// GPU-resident NSM (next-subvolume method) for the sSSA part.
//
//   rdme_rates        nsm_core__initialize_rxn_propensities and
//                     nsm_core__initialize_diff_propensities
//                     (ENG/src/simulate_rdme.cpp:113-152)
//   rdme_queue_build  nsm_core__initialize_heap + NRMConstant_v5::build
//                     (simulate_rdme.cpp:155-195, NRMConstant_v5.cpp:27-85)
//   rdme_take_step    nsm_core__take_step (simulate_rdme.cpp:211-472)
//
// The event queue is an indexed min-tree over the voxels' firing times:
// F0 = 64*PL voxels under each level-1 node, 64 nodes under each node above
// (one wavefront reduces one node).  The levels above the voxels live in LDS
// while the event loop runs.  The reference's time-binned hash
// table always yields the global minimum among firing times inside its
// current window [L, U] and rebuilds the window when that set is empty
// (NRMConstant_v5.cpp:156-281); the window scalars are kept here with the
// same update rules, so the min-tree returns the same event sequence (up to
// exactly equal firing times, which the table breaks by bin order).
//
// One 64-lane workgroup runs one trajectory's event loop; every lane
// executes the scalar logic (uniform control flow, broadcast loads), lanes
// split the min-tree node reductions and the neighbour-row loads.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <cmath>

#include "engine.hpp"
#include "rng.hpp"
#include "vm.hpp"
#include "window.hpp"

namespace ssa {

constexpr int MAXS = 16;
constexpr int MAXR = 16;

// Mass-action propensities (generated functions, solver.py:344-373).
__device__ __forceinline__ double propensity(const Rxn &re, const uint32_t *xv, double vol, int tp) {
    if (re.mask && !((re.mask >> tp) & 1ULL)) return 0.0;
    const int *xs = (const int *)xv;
    switch (re.kind) {
    case 0: return re.k * vol;
    case 1: return re.k * xs[re.a];
    case 2: return ((re.k * xs[re.a]) * xs[re.b]) / vol;
    default: return ((re.k * xs[re.a]) * (xs[re.a] - 1)) / vol;
    }
}

// ---------------------------------------------------------------------------
// Rates (simulate_rdme.cpp:113-152), one thread per voxel.  VM: kind-4
// reactions through the expression VM.
template <bool VM>
__global__ void k_rates(RdmeArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    int i = chunk * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int b = blockIdx.y;
    uint32_t *xx = a.xx + b * a.bs_xx;
    double *rrate = a.rrate + b * a.bs_rr, *srrate = a.srrate + b * a.bs_n, *sdrate = a.sdrate + b * a.bs_n;
    const int S = a.S, R = a.R;
    uint32_t xv[MAXS];
    for (int s = 0; s < S; s++) xv[s] = xx[(size_t)i * S + s];
    double sr = 0.0;
    const double *df = a.data_fn ? a.data_fn + (size_t)i * a.n_df : nullptr;
    // mass / rho of this step, formed by the particle phase (simulate_rdme.cpp:123)
    const double vol = a.vol[i];
    for (int j = 0; j < R; j++) {
        const Rxn re = a.rx[j];
        double p;
        if (VM && re.kind == 4)   // simulate_rdme.cpp:124 evaluates at t = 0.0
            p = (re.mask && !((re.mask >> a.type[i]) & 1ULL))
                    ? 0.0 : vm_eval_u32(a.vm_code, re.a, a.vm_k, xx + (size_t)i * S, vol, 0.0, df);
        else
            p = propensity(re, xv, vol, a.type[i]);
        rrate[(size_t)i * R + j] = p;
        sr += p;
    }
    srrate[i] = sr;
    double sd = 0.0;
    for (int s = 0; s < S; s++) sd += a.Ddiag[(size_t)i * S + s] * xv[s];
    sdrate[i] = sd;
}
// The per-species diffusion sums over the neighbour row (Ddiag) of models
// with more species than the search's finish forms, shared by every
// trajectory, from this step's lists; the particle phase runs it (beside
// the previous step's event loop when a look-ahead runs it).
__global__ void k_diag(RdmeArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    const int i = chunk * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int dg = a.deg[i];
    for (int s = 0; s < a.S; s++) {
        double dd = 0.0;
        for (int k = 0; k < dg; k++) {
            const size_t e = (size_t)k * a.n + i;
            const double dc = a.Dmat[(size_t)s * a.T + (a.ntype[e] - 1)];   // ntype[e] = type of neighbour e
            dd += dc * a.Dij[e];
        }
        a.Ddiag[(size_t)i * a.S + s] = dd;
    }
}
void rdme_diag(hipStream_t s, const RdmeArgs &a) {
    hipLaunchKernelGGL(k_diag, xcd_grid((a.n + 255) / 256), dim3(256), 0, s, a);
}
void rdme_rates(hipStream_t s, const RdmeArgs &a, int n_traj) {
    const dim3 g(xcd_grid((a.n + 255) / 256).x, n_traj);
    if (a.vm_ncode > 0) hipLaunchKernelGGL(k_rates<true>, g, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(k_rates<false>, g, dim3(256), 0, s, a);
}

// ---------------------------------------------------------------------------
// prop, nonzero flags
__global__ void k_qprop(RdmeArgs a, double *prop, int *nz, int *act) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    double p = a.srrate[i] + a.sdrate[i];
    prop[i] = p;
    nz[i] = p != 0.0;
    act[i] = p > 0;
}

// Partial sums for the fast (seeded) mode: fixed block/lane order, so the
// result is deterministic.
constexpr int QSUM_BLOCKS = 256;
__global__ void k_qsum_part(const double *prop, int n, double *part) {
    __shared__ double w[4];
    double s = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) s += prop[i];
    for (int o = WAVE / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) w[threadIdx.x / WAVE] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((w[0] + w[1]) + w[2]) + w[3];
}

// propensitySum (simulate_rdme.cpp:167-179) and the first time window.
// exact: added in voxel order by one wavefront (bit-identical to the
// reference's loop); otherwise the block partials are added in order.
__global__ void k_qsum(RdmeArgs a, const double *prop, const int *act_scan, int exact, const double *part) {
    const int lane = threadIdx.x;
    double s = 0.0;
    if (exact) {
        for (int base = 0; base < a.n; base += WAVE) {
            double v = base + lane < a.n ? prop[base + lane] : 0.0;
            int m = min(WAVE, a.n - base);
            for (int k = 0; k < m; k++) s += __shfl(v, k, WAVE);
        }
    } else {
        for (int k = 0; k < QSUM_BLOCKS; k++) s += part[k];
    }
    if (lane == 0) {
        QueueState q = *a.qs;
        q.endTime = a.endTime;
        long long active = act_scan[a.n];
        q.active = (unsigned long long)active;
        int ok = 0;
        if (a.S > 0 && s > 0.0) ok = set_bins(q, a.t0, s, active) ? 1 : 0;
        q.initialized = ok ? 2 : 0;   // 2: draws pending
        q.rxnCount = 0;
        *a.qs = q;
        *a.psum_out = s;
    }
}

// Firing times in voxel order (NRMConstant_v5.cpp:52-71): the k-th voxel with
// non-zero propensity takes the k-th exponential of the build.
__global__ void k_qtimes(RdmeArgs a, const double *prop, const int *nz_scan) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const QueueState *q = a.qs;
    if (q->initialized != 2) return;
    double p = prop[i];
    double t;
    if (p == 0.0) {
        t = INFINITY;
    } else {
        unsigned long long idx = q->rng_pos + (unsigned long long)nz_scan[i];
        double e;
        if (a.rng_kind == 1) e = idx < a.n_words ? a.expo[idx] : NAN;
        else e = word_expo(philox64(a.seed, a.stream_id, idx));
        t = e / p + a.t0;
    }
    a.qtime[i] = t;
}

__global__ void k_qfinish(RdmeArgs a, const int *nz_scan) {
    if (threadIdx.x != 0) return;
    QueueState q = *a.qs;
    if (q.initialized == 2) {
        unsigned long long cnt = (unsigned long long)nz_scan[a.n];
        if (a.rng_kind == 1 && q.rng_pos + cnt > a.n_words) q.err = SSASDPD_ERR_REPLAY_EXHAUSTED;
        q.rng_pos += cnt;
        q.initialized = (cnt == q.active) ? 1 : 0;
    }
    *a.qs = q;
}

// The event loop's nodes: the least firing time of every 64*pl voxels, one
// wavefront per node.
__global__ void k_node_min(const double *qt, int n, int pl, double *node_min, int nodes) {
    const int node = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    const int lane = threadIdx.x & (WAVE - 1);
    if (node >= nodes) return;
    double t = INFINITY;
    for (int p = 0; p < pl; p++) {
        const int c = (node * pl + p) * WAVE + lane;
        if (c < n) t = fmin(t, qt[c]);
    }
    for (int o = WAVE / 2; o > 0; o >>= 1) t = fmin(t, __shfl_xor(t, o, WAVE));
    if (lane == 0) node_min[node] = t;
}

void rdme_queue_build(hipStream_t s, const RdmeArgs &a, void *scan_tmp, int *work) {
    // work: prop (n doubles) | nz (n+1) | act (n+1) | nz_scan (n+1) | act_scan (n+1) | part
    double *prop = (double *)work;
    int *nz = (int *)(prop + a.n);
    int *act = nz + a.n + 1;
    int *nz_scan = act + a.n + 1;
    int *act_scan = nz_scan + a.n + 1;
    double *part = (double *)(((uintptr_t)(act_scan + a.n + 1) + 15) & ~(uintptr_t)15);
    unsigned g = (unsigned)((a.n + 255) / 256);
    const bool exact = a.rng_kind == 1;
    hipLaunchKernelGGL(k_qprop, dim3(g), dim3(256), 0, s, a, prop, nz, act);
    exclusive_scan_i32(s, nz, nz_scan, a.n, scan_tmp);
    exclusive_scan_i32(s, act, act_scan, a.n, scan_tmp);
    if (!exact) hipLaunchKernelGGL(k_qsum_part, dim3(QSUM_BLOCKS), dim3(256), 0, s, prop, a.n, part);
    hipLaunchKernelGGL(k_qsum, dim3(1), dim3(WAVE), 0, s, a, prop, act_scan, exact ? 1 : 0, part);
    hipLaunchKernelGGL(k_qtimes, dim3(g), dim3(256), 0, s, a, prop, nz_scan);
    hipLaunchKernelGGL(k_qfinish, dim3(1), dim3(64), 0, s, a, nz_scan);
    tree_rebuild(s, a);
}

void tree_rebuild(hipStream_t s, const RdmeArgs &a) {
    hipLaunchKernelGGL(k_node_min, dim3((unsigned)((a.tree_nodes + 3) / 4)), dim3(256), 0, s, a.qtime, a.n, a.pl,
                       a.tmin, a.tree_nodes);
}

// The expression VM over m argument sets (ssasdpd_vm_eval).
__global__ void k_vm_eval(const uint32_t *code, int start, const double *K, int x_is_double, int n_x, int n_df,
                          int m, const double *xd, const uint32_t *xu, const double *vol, const double *t,
                          const double *df, double *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const double *dfi = n_df > 0 ? df + (size_t)i * n_df : nullptr;
    out[i] = x_is_double ? vm_eval_f64(code, start, K, xd + (size_t)i * n_x, vol[i], t[i], dfi)
                         : vm_eval_u32(code, start, K, xu + (size_t)i * n_x, vol[i], t[i], dfi);
}
void vm_eval_batch(hipStream_t s, const uint32_t *code, int start, const double *K, int x_is_double, int n_x,
                   int n_df, int m, const double *xd, const uint32_t *xu, const double *vol, const double *t,
                   const double *df, double *out) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_vm_eval, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, code, start, K, x_is_double,
                       n_x, n_df, m, xd, xu, vol, t, df, out);
}

// What the library accepts as an event-loop model: the tables of its chemistry
// and programs beside a tree of tree_nodes (time, voxel) pairs, up to 64 KiB.
size_t ssa_lds_bytes(int tree_nodes, int S, int R, int T, int nnzN, int nnzG, int n_code, int n_consts) {
    auto a16 = [](size_t x) { return (x + 15) & ~(size_t)15; };
    size_t off = 0;
    off = a16(off + sizeof(double) * tree_nodes);
    off = a16(off + sizeof(int) * tree_nodes);
    off = a16(off + sizeof(Rxn) * R);
    off = a16(off + sizeof(double) * S * T);
    off = a16(off + sizeof(int) * (R + 1));
    off = a16(off + sizeof(int) * nnzN);
    off = a16(off + sizeof(int) * nnzN);
    off = a16(off + sizeof(int) * (S + R + 1));
    off = a16(off + sizeof(int) * nnzG);
    if (n_code > 0) {
        off = a16(off + sizeof(uint32_t) * n_code);
        off = a16(off + sizeof(double) * n_consts);
        off = a16(off + sizeof(uint32_t) * 64);
    }
    return off;
}

}  // namespace ssa
