// Rates and event queue of the NSM (next-subvolume method), the sSSA part; the
// event loop is in nsm.hip.
//
//   rdme_queue_build  nsm_core__initialize_rxn_propensities,
//                     nsm_core__initialize_diff_propensities and
//                     nsm_core__initialize_heap + NRMConstant_v5::build
//                     (ENG/src/simulate_rdme.cpp:113-195,
//                     NRMConstant_v5.cpp:27-85), for all trajectories of a
//                     batch in three launches or four
//   rdme_diag         the diffusion sums over the neighbour rows
//   tree_rebuild      the queue's node bounds after a change of their width
//
// The queue is the voxels' firing times and the minimum of every node of
// 64*pl voxels.  The reference's time-binned hash table always yields the
// global minimum among the firing times inside its current window [L, U] and
// rebuilds the window when that set is empty (NRMConstant_v5.cpp:156-281); the
// window's scalars are kept with the same update rules (window.hpp), so the
// event sequence is the same (up to exactly equal firing times, which the
// table breaks by bin order).
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
// The work space of the queue build, per trajectory: the blocks' counts and
// their running sum, the partial propensity sums and what the last kernel
// needs to know.
constexpr int QBLOCK = 256;        // voxels per block
constexpr int QSUM_BLOCKS = 256;   // partial sums of the propensities
struct QWork {
    int *count, *before;           // [blocks]
    double *part;                  // [QSUM_BLOCKS]
    unsigned long long *first;     // [2] the build's first random word; whether it draws
};
__host__ __device__ __forceinline__ int q_blocks(int n) { return (n + QBLOCK - 1) / QBLOCK; }
size_t q_work_bytes(int n) {
    return ((sizeof(int) * 2 * (size_t)q_blocks(n) + 15) & ~(size_t)15) + sizeof(double) * QSUM_BLOCKS + 16;
}
__device__ __forceinline__ QWork q_work(const RdmeArgs &a, size_t b) {
    char *p = a.qwork + b * a.bs_qwork;
    const int nb = q_blocks(a.n);
    QWork w;
    w.count = (int *)p;
    w.before = w.count + nb;
    w.part = (double *)(p + ((sizeof(int) * 2 * (size_t)nb + 15) & ~(size_t)15));
    w.first = (unsigned long long *)(w.part + QSUM_BLOCKS);
    return w;
}

// Rates (simulate_rdme.cpp:113-152), one thread per voxel.  VM: kind-4
// reactions through the expression VM.
template <bool VM>
__global__ void __launch_bounds__(QBLOCK) k_rates(RdmeArgs a) {
    __shared__ double w_sum[QBLOCK / WAVE];
    __shared__ int w_cnt[QBLOCK / WAVE];
    const int nb = q_blocks(a.n);
    const int chunk = xcd_chunk(nb);
    if (chunk < 0) return;
    const int b = blockIdx.y, i = chunk * QBLOCK + threadIdx.x;
    if (a.only_new && a.qs[b].initialized == 1) return;
    double p = 0.0;
    if (i < a.n) {
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
            double pr;
            if (VM && re.kind == 4)   // simulate_rdme.cpp:124 evaluates at t = 0.0
                pr = (re.mask && !((re.mask >> a.type[i]) & 1ULL))
                         ? 0.0 : vm_eval_u32(a.vm_code, re.a, a.vm_k, xx + (size_t)i * S, vol, 0.0, df);
            else
                pr = propensity(re, xv, vol, a.type[i]);
            rrate[(size_t)i * R + j] = pr;
            sr += pr;
        }
        srrate[i] = sr;
        double sd = 0.0;
        for (int s = 0; s < S; s++) sd += a.Ddiag[(size_t)i * S + s] * xv[s];
        sdrate[i] = sd;
        p = sr + sd;
    }
    // the queue build's sums over this block: voxels whose propensity is not
    // zero (low half) and is positive (high half), and the propensities
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    const int c = (int)__popcll(__ballot(p != 0.0)) | (int)__popcll(__ballot(p > 0.0)) << 16;
    double sum = p;
    for (int o = WAVE / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, WAVE);
    if (lane == 0) {
        w_cnt[w] = c;
        w_sum[w] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const QWork q = q_work(a, b);
        q.count[chunk] = ((w_cnt[0] + w_cnt[1]) + w_cnt[2]) + w_cnt[3];
        if (nb <= QSUM_BLOCKS) q.part[chunk] = ((w_sum[0] + w_sum[1]) + w_sum[2]) + w_sum[3];
    }
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

// ---------------------------------------------------------------------------
// Partial sums for the fast (seeded) mode: fixed block/lane order, so the
// result is deterministic.  With at most QSUM_BLOCKS blocks of voxels k_rates
// has formed them already.
__global__ void __launch_bounds__(QBLOCK) k_qsum_part(RdmeArgs a) {
    __shared__ double w[4];
    const int b = blockIdx.y;
    if (a.only_new && a.qs[b].initialized == 1) return;
    const double *sr = a.srrate + b * a.bs_n, *sd = a.sdrate + b * a.bs_n;
    double s = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x) s += sr[i] + sd[i];
    for (int o = WAVE / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0) w[threadIdx.x / WAVE] = s;
    __syncthreads();
    if (threadIdx.x == 0) q_work(a, b).part[blockIdx.x] = ((w[0] + w[1]) + w[2]) + w[3];
}

// One workgroup per trajectory: the running sum of the blocks' counts, the
// propensity sum (simulate_rdme.cpp:167-179) and the first time window.
// exact: the sum is added in voxel order by one wavefront (bit-identical to
// the reference's loop); otherwise the partial sums are added in order.  The
// draws of the build are taken from the stream here.
constexpr int QSCAN = 1024;
__global__ void __launch_bounds__(QSCAN) k_qstate(RdmeArgs a, int exact) {
    __shared__ int w_sum[QSCAN / WAVE];
    __shared__ double l_part[QSUM_BLOCKS];
    const int b = blockIdx.y, tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    QueueState *const qs = a.qs + b;
    const QWork q = q_work(a, b);
    if (a.only_new && qs->initialized == 1) {
        if (tid == 0) q.first[1] = 0;      // no times to draw
        return;
    }
    const int nb = q_blocks(a.n);
    // voxels that draw (low 32 bits) and active ones, over all blocks
    unsigned long long carry = 0;
    for (int c0 = 0; c0 < nb; c0 += QSCAN) {
        const int k = c0 + tid;
        const int v = k < nb ? q.count[k] : 0;
        const int mine = v & 0xFFFF;
        int x = mine, act = v >> 16;
        for (int o = 1; o < WAVE; o <<= 1) {
            const int y = __shfl_up(x, o, WAVE);
            if (lane >= o) x += y;
        }
        for (int o = WAVE / 2; o > 0; o >>= 1) act += __shfl_xor(act, o, WAVE);
        __syncthreads();
        if (lane == WAVE - 1) w_sum[w] = x;
        __syncthreads();
        int pre = 0, tot = 0;
        for (int u = 0; u < QSCAN / WAVE; u++) {
            if (u == w) pre = tot;
            tot += w_sum[u];
        }
        if (k < nb) q.before[k] = (int)(carry & 0xFFFFFFFFULL) + pre + x - mine;
        __syncthreads();
        if (lane == 0) w_sum[w] = act;
        __syncthreads();
        int all = 0;
        for (int u = 0; u < QSCAN / WAVE; u++) all += w_sum[u];
        carry += (unsigned long long)(unsigned)tot + ((unsigned long long)(unsigned)all << 32);
    }
    if (!exact) {
        const int np = nb < QSUM_BLOCKS ? nb : QSUM_BLOCKS;
        if (tid < QSUM_BLOCKS) l_part[tid] = tid < np ? q.part[tid] : 0.0;
    }
    __syncthreads();
    if (w != 0) return;
    double s = 0.0;
    if (exact) {
        const double *sr = a.srrate + b * a.bs_n, *sd = a.sdrate + b * a.bs_n;
        for (int base = 0; base < a.n; base += WAVE) {
            const double v = base + lane < a.n ? sr[base + lane] + sd[base + lane] : 0.0;
            const int m = min(WAVE, a.n - base);
            for (int k = 0; k < m; k++) s += __shfl(v, k, WAVE);
        }
    } else {
        for (int k = 0; k < QSUM_BLOCKS; k++) s += l_part[k];
    }
    if (lane == 0) {
        QueueState st = *qs;
        const unsigned long long cnt = carry & 0xFFFFFFFFULL, active = carry >> 32;
        st.endTime = a.endTime;
        st.active = active;
        bool ok = false;
        if (a.S > 0 && s > 0.0) ok = set_bins(st, a.t0, s, (long long)active);
        st.initialized = 0;
        st.rxnCount = 0;
        q.first[0] = st.rng_pos;
        q.first[1] = ok ? 1 : 0;
        if (ok) {
            if (a.rng_kind == 1 && st.rng_pos + cnt > a.n_words) st.err = SSASDPD_ERR_REPLAY_EXHAUSTED;
            st.rng_pos += cnt;
            st.initialized = cnt == active ? 1 : 0;
        }
        *qs = st;
    }
}

// Firing times in voxel order (NRMConstant_v5.cpp:52-71): the k-th voxel with
// non-zero propensity takes the k-th exponential of the build.  Nodes of up
// to a block's voxels get their minimum at once.
__global__ void __launch_bounds__(QBLOCK) k_qtimes(RdmeArgs a, int nodes_here) {
    __shared__ int w_cnt[QBLOCK / WAVE];
    __shared__ double w_min[QBLOCK / WAVE];
    const int chunk = xcd_chunk(q_blocks(a.n));
    if (chunk < 0) return;
    const int b = blockIdx.y, i = chunk * QBLOCK + threadIdx.x;
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    const QWork q = q_work(a, b);
    if (!q.first[1]) return;
    const double p = i < a.n ? a.srrate[b * a.bs_n + i] + a.sdrate[b * a.bs_n + i] : 0.0;
    const unsigned long long nz = __ballot(p != 0.0);
    if (lane == 0) w_cnt[w] = (int)__popcll(nz);
    __syncthreads();
    double t = INFINITY;
    if (i < a.n) {
        if (p != 0.0) {
            int k = q.before[chunk] + (int)__popcll(nz & ((1ULL << lane) - 1ULL));
            for (int u = 0; u < w; u++) k += w_cnt[u];
            const unsigned long long idx = q.first[0] + (unsigned long long)k;
            double e;
            if (a.rng_kind == 1) e = idx < a.n_words ? a.expo[idx] : NAN;
            else e = word_expo(philox64(a.seeds ? a.seeds[b] : a.seed, a.stream_id, idx));
            t = e / p + a.t0;
        }
        a.qtime[b * a.bs_n + i] = t;
    }
    if (!nodes_here) return;
    for (int o = WAVE / 2; o > 0; o >>= 1) t = fmin(t, __shfl_xor(t, o, WAVE));
    if (lane == 0) w_min[w] = t;
    __syncthreads();
    if (threadIdx.x < QBLOCK / WAVE && threadIdx.x % a.pl == 0) {
        const int node = (chunk * (QBLOCK / WAVE) + (int)threadIdx.x) / a.pl;
        if (node < a.tree_nodes) {
            double m = INFINITY;
            for (int u = 0; u < a.pl; u++) m = fmin(m, w_min[threadIdx.x + u]);
            a.tmin[b * a.bs_tree + node] = m;
        }
    }
}

// The event loop's nodes: the least firing time of every 64*pl voxels, one
// wavefront per node.
__global__ void k_node_min(RdmeArgs a) {
    const int n = a.n, pl = a.pl, nodes = a.tree_nodes;
    const double *qt = a.qtime + blockIdx.y * a.bs_n;
    double *node_min = a.tmin + blockIdx.y * a.bs_tree;
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

// Rates, propensity sum, window, firing times and node minima of n_traj
// trajectories: three launches (four past 65,536 voxels), where one scan per
// trajectory and array took seventeen each: launches, not their work, were
// what the build took (64,000 particles 53 -> 23 us a step, 400 trajectories
// of 121 voxels 14.7 -> 0.04 ms).
void rdme_queue_build(hipStream_t s, const RdmeArgs &all, int n_traj) {
    constexpr int MOST = 32768;            // trajectories of one launch (grid.y)
    if (n_traj > MOST) {
        rdme_queue_build(s, all, MOST);
        RdmeArgs r = all;
        r.xx += MOST * r.bs_xx;
        r.rrate += MOST * r.bs_rr;
        r.srrate += MOST * r.bs_n;
        r.sdrate += MOST * r.bs_n;
        r.qtime += MOST * r.bs_n;
        r.tmin += MOST * r.bs_tree;
        r.qwork += MOST * r.bs_qwork;
        r.qs += MOST;
        if (r.seeds) r.seeds += MOST;
        rdme_queue_build(s, r, n_traj - MOST);
        return;
    }
    const RdmeArgs &a = all;
    const int nb = q_blocks(a.n);
    const dim3 g(xcd_grid(nb).x, n_traj);
    if (a.vm_ncode > 0) hipLaunchKernelGGL(k_rates<true>, g, dim3(QBLOCK), 0, s, a);
    else hipLaunchKernelGGL(k_rates<false>, g, dim3(QBLOCK), 0, s, a);
    const bool exact = a.rng_kind == 1;
    if (!exact && nb > QSUM_BLOCKS)
        hipLaunchKernelGGL(k_qsum_part, dim3(QSUM_BLOCKS, n_traj), dim3(QBLOCK), 0, s, a);
    hipLaunchKernelGGL(k_qstate, dim3(1, n_traj), dim3(QSCAN), 0, s, a, exact ? 1 : 0);
    const bool nodes_here = WAVE * a.pl <= QBLOCK;
    hipLaunchKernelGGL(k_qtimes, g, dim3(QBLOCK), 0, s, a, nodes_here ? 1 : 0);
    if (!nodes_here) tree_rebuild(s, a, n_traj);
}

void tree_rebuild(hipStream_t s, const RdmeArgs &a, int n_traj) {
    hipLaunchKernelGGL(k_node_min, dim3((unsigned)((a.tree_nodes + 3) / 4), n_traj), dim3(256), 0, s, a);
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

// What the library accepts as an event-loop model, up to 64 KiB: the tables of
// its chemistry and programs beside tree_nodes (time, voxel) pairs, as a tree of
// them once stood in LDS.  (What the loop uses now is nsm_lds_bytes.)
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
