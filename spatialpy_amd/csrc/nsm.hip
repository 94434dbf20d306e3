// The NSM event loop (nsm_core__take_step, ENG/src/simulate_rdme.cpp:211-472,
// with the queue of NRMConstant_v5.cpp:89-281) on gfx950: one wavefront per
// trajectory, up to 64 consecutive events at a time, one per lane.
//
// What bounds it.  Taken one by one, every event is a chain of two dependent
// memory round trips (its voxel, then its destination) and about a thousand
// instructions, 3-4 us, with one lane's worth of work in a 64-lane wavefront.
// But consecutive events rarely touch each other: of the next 64 events in
// firing order, those before the first one that shares a voxel with an
// earlier one (26 on average on a 2D dam break with 1,000 molecules, 51 on a
// 64,000-voxel lattice, 6 on 121 voxels) can be carried out side by side.
// So each round
//   1. takes the earliest voxels of the queue, one per lane, in firing order;
//   2. loads their states together (one round trip for all of them);
//   3. hands out the random words: how many an event draws depends on what it
//      is, so each lane's position in the stream is the prefix sum of the
//      earlier lanes' draws, iterated until it no longer changes;
//   4. chooses every lane's reaction or hop, loads the destinations together,
//      and forms the new counts, rates and firing times;
//   5. keeps the longest prefix of lanes that no earlier lane of the round
//      interferes with (a voxel touched before, a new firing time that comes
//      before the lane's own, a draw count that was not the expected one) and
//      stores it; the others stay in the queue for the next round.
// Operations, their order and the random words are those of the one-by-one
// loop, so every result has the same bits.  Events that leave the common
// path (a selection that ran past the last reaction, species or neighbour,
// a hop into the voxel itself, the end of a replay stream) are carried out
// only as the first lane of a round.
//
// Where consecutive events do interfere (a few voxels, or one that holds nearly
// all molecules) a round keeps one or two of them, and costs as much as one that
// keeps sixty, the more the more species and reactions its lanes carry.  There
// events go one by one instead (event_alone), a lane per species and per reaction
// of the voxel: nsm_alone chooses the kernel that can do both, and that one goes
// by what its last rounds kept.
//
// The queue.  Firing times of all voxels are in memory (qtime).  Three sets,
// divided by two horizons, hold every voxel with a finite time once: the
// `front`, at most 64 voxels sorted by (time, voxel), one per lane, up to the
// first horizon; the near list, unsorted in LDS, up to the second; and nodes
// of 64*pl voxels, of whose remaining voxels LDS keeps a lower bound of the
// times.  A new time goes into the set its horizon says (a node's bound is
// lowered).  A front that runs low takes the near list's earliest and moves
// the first horizon on; a near list that runs low scans the nodes whose bound
// lies under the next second horizon, and those nodes get the exact minimum
// of the rest.  The steps in time follow the mean gap between the entries the
// last ones brought.  No tree is repaired after an event, and a scan of the
// nodes brings hundreds of events.
//
// Measured (MI355X, time per event, the one-by-one loop with its event tree
// against the rounds): 40^3 lattice, 200,000 molecules 3.7 -> 0.36 us; 256 of
// those trajectories at once 14.7 -> 1.6 ns; 2D dam break 3.6 -> 0.42 us; 1M
// cylinder, 860 events a step, 2.8 -> 0.45 us; 121 voxels 3.5 -> 1.5 us;
// custom propensities on 144 voxels 30 -> 5.2 us; 4 voxels 3.6 -> 5.5 us in
// rounds, 3.0 us one by one (16 voxels with 16 species and 16 reactions 4.3 ->
// 16.4 and 3.7 us).  A round takes 20,000 to 50,000 cycles, most of them
// latencies (two round trips, LDS, dependent FP64 operations) of a single
// wavefront.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <cmath>
#include <type_traits>

#include "engine.hpp"
#include "rng.hpp"
#include "vm.hpp"
#include "window.hpp"

namespace ssa {

namespace {

constexpr int FRONT_LOW = 40;      // refill the front below this many entries
constexpr int FRONT_FILL = 56;     // entries that aims at
constexpr int NEAR = 512;          // entries of the near list
constexpr int NEAR_LOW = 32;       // refill the near list below this many
constexpr int NEAR_FILL = 350;     // entries that aims at, at most
constexpr int GROUP = 32;          // nodes a wavefront scans together (2 lanes each)
constexpr int WAVES = 4;           // wavefronts of a workgroup, at most
constexpr int ROW = 8;             // neighbour entries fetched together
constexpr int POOL = 512;          // uniforms kept ready (a ring)
constexpr int CLAIMS = 2048;       // slots of each claim table

// ---------------------------------------------------------------------------
// Cross-lane moves (DPP).
template <int CTRL, int RMASK> __device__ __forceinline__ int dpp_i(int old, int x) {
    return __builtin_amdgcn_update_dpp(old, x, CTRL, RMASK, 0xF, false);
}
template <int CTRL, int RMASK> __device__ __forceinline__ double dpp_d(double old, double x) {
    return __hiloint2double(dpp_i<CTRL, RMASK>(__double2hiint(old), __double2hiint(x)),
                            dpp_i<CTRL, RMASK>(__double2loint(old), __double2loint(x)));
}
__device__ __forceinline__ int rl_i(int x, int lane) { return __builtin_amdgcn_readlane(x, lane); }
__device__ __forceinline__ double rl_d(double x, int lane) {
    return __hiloint2double(rl_i(__double2hiint(x), lane), rl_i(__double2loint(x), lane));
}
// inclusive sum over the lanes
__device__ __forceinline__ int scan_add(int x) {
    x += dpp_i<0x111, 0xF>(0, x);   // row_shr 1, 2, 4, 8
    x += dpp_i<0x112, 0xF>(0, x);
    x += dpp_i<0x114, 0xF>(0, x);
    x += dpp_i<0x118, 0xF>(0, x);
    x += dpp_i<0x142, 0xA>(0, x);   // row_bcast15 into rows 1, 3
    x += dpp_i<0x143, 0xC>(0, x);   // row_bcast31 into rows 2, 3
    return x;
}
// inclusive minimum over the lanes
__device__ __forceinline__ double scan_min(double x) {
    const double inf = INFINITY;
    x = fmin(x, dpp_d<0x111, 0xF>(inf, x));
    x = fmin(x, dpp_d<0x112, 0xF>(inf, x));
    x = fmin(x, dpp_d<0x114, 0xF>(inf, x));
    x = fmin(x, dpp_d<0x118, 0xF>(inf, x));
    x = fmin(x, dpp_d<0x142, 0xA>(inf, x));
    x = fmin(x, dpp_d<0x143, 0xC>(inf, x));
    return x;
}
__device__ __forceinline__ double wave_min(double x) { return rl_d(scan_min(x), WAVE - 1); }
// lane l gets lane l-1's value, lane 0 gets `first`
__device__ __forceinline__ double shift_up(double first, double x) { return dpp_d<0x138, 0xF>(first, x); }

__device__ __forceinline__ int first_lane(unsigned long long m) { return m ? (int)__builtin_ctzll(m) : WAVE; }
__device__ __forceinline__ int last_lane(unsigned long long m) { return 63 - (int)__builtin_clzll(m); }
__device__ __forceinline__ unsigned long long below(int n) { return n >= WAVE ? ~0ULL : (1ULL << n) - 1ULL; }

// (t, v) before (t2, v2): by time, ties to the lower voxel
// (bitwise: no branches)
__device__ __forceinline__ bool before(double t, int v, double t2, int v2) {
    return (t < t2) | ((t == t2) & (v < v2));
}

// LDS ordering inside the wavefront (and, for memory, what it stored before
// what it loads next)
__device__ __forceinline__ void sync_wave() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }

// Times are never negative, so their bits order like the times.
__device__ __forceinline__ void lds_min(double *p, double t) {
    atomicMin((unsigned long long *)p, (unsigned long long)__double_as_longlong(t));
}

struct __attribute__((packed, aligned(8))) Pair { double a, b; };   // a 16-byte load at 8-byte alignment

// The workgroup's LDS.
struct Lds {
    double *lb;            // [nodes] lower bounds
    double *pool;          // [POOL] uniforms of words (base + k) & (POOL - 1)
    double *epool;         // [POOL] their exponential variates
    double *qt;            // [NEAR] the near list's times
    int *qv;               // [NEAR] and voxels
    double *ht;            // [NEAR] times on their way into the front
    int *hv;               // [NEAR] and voxels
    int *nodes;            // [WAVES][GROUP] nodes to scan (and 64 places while ranks are checked)
    unsigned *claim;       // [2][CLAIMS] (in the same place as ht, hv)
    Rxn *rx;               // [R]
    double *Dmat;          // [S][T]
    int *dN;               // [R][MS] stoichiometry, dense
    unsigned *dep;         // [S + R] dependency columns as reaction bitmasks
    unsigned *tot;         // [S] species totals
    struct Scan {          // a scan of the nodes, shared by the wavefronts
        double to, far_t, drop;
        int far_v, count, stop, pad[3];
    } *scan;
    uint32_t *vmx;         // [S][64] counts staged for the VM
    uint32_t *vcode;
    double *vk;
};

size_t a16(size_t x) { return (x + 15) & ~(size_t)15; }

}  // namespace

// LDS bytes of the event loop (the layout of ssa_run below).
size_t nsm_lds_bytes(int nodes, int S, int R, int T, int n_code, int n_consts) {
    size_t o = a16(sizeof(double) * nodes);
    o += sizeof(double) * 2 * POOL + (sizeof(double) + sizeof(int)) * NEAR + sizeof(int) * WAVES * GROUP;
    o += sizeof(unsigned) * 2 * CLAIMS + sizeof(Lds::Scan);
    o += a16(sizeof(Rxn) * R) + a16(sizeof(double) * S * T) + a16(sizeof(int) * R * 16) + a16(sizeof(unsigned) * (S + R));
    o += a16(sizeof(unsigned) * S);
    static_assert(sizeof(Lds::Scan) % 16 == 0, "keeps the next array aligned");
    if (n_code > 0)
        o += sizeof(uint32_t) * WAVE * S + a16(sizeof(uint32_t) * n_code) + a16(sizeof(double) * n_consts);
    return o;
}

namespace {

// Snapshot k of one trajectory: its counts [n][S] and its species totals.
__device__ __noinline__ void snapshot_counts(const uint32_t *xx, uint32_t *snap_xx, uint32_t *snap_tot, size_t nsS,
                                             int S, int k, const unsigned *tot, int lane) {
    sync_wave();
    if (snap_xx) {
        uint32_t *dst = snap_xx + (size_t)k * nsS;
        for (size_t i = lane; i < nsS; i += WAVE) dst[i] = xx[i];
    }
    if (snap_tot && lane < S) snap_tot[(size_t)k * S + lane] = tot[lane];
}

// x[i] of a small register array at a wave-uniform or lane index
template <int M, class X> __device__ __forceinline__ X pick(const X (&x)[M], int i) {
    X r = x[0];
#pragma unroll
    for (int k = 1; k < M; k++) {
        const X v = x[k];      // (a conditional load would put x in memory)
        r = i == k ? v : r;
    }
    return r;
}

// One lane's view of a voxel: counts, propensities, their sums.
template <int MS, int MR> struct Voxel {
    uint32_t x[MS];
    double r[MR];
    double sr, sd;
};

// Everything the rounds share (uniform over the wavefront unless noted).
template <int MS, int MR, bool VM> struct Loop {
    const RdmeArgs &a;
    Lds L;
    uint32_t *xx;
    double *rrate, *srrate, *sdrate, *qtime;
    int waves;                            // of the workgroup
    int lane, n, S, R, T, W, nn, nv, nvs;   // nn nodes of nv = 2^nvs voxels
    uint64_t seed;
    // the random stream: next word, words in the pool up to
    unsigned long long pos, fill, n_words;
    // the front: lane l holds entry l (+inf past cnt), up to the horizon
    double ft;
    int fv, cnt;
    double tau_t;
    int tau_v;
    // the near list's count and its horizon
    int nc;
    double far_t;
    int far_v;
    double gap;                           // mean time between the queue's entries
    int near_fill;                        // entries a refill of the near list aims at
    // the reactions of models of up to 8, kept out of LDS: kind, reactants
    static constexpr bool HELD = MR <= 8 && !VM;
    int ri[HELD ? MR : 1];
    double rk[HELD ? MR : 1];
    uint64_t rm[HELD ? MR : 1];
    double guess_empty;                   // VM models: a hop empties a lone molecule's voxel (0 / 1)

    __device__ explicit Loop(const RdmeArgs &args) : a(args) {}

    // ---- propensities -----------------------------------------------------
    // Propensity of reaction j (uniform) for this lane's counts: the
    // operations of the generated functions (solver.py:344-373).  TABLE: the
    // reaction from LDS at any j, otherwise from registers at a constant one.
    template <bool TABLE>
    __device__ __forceinline__ double prop(int j, const uint32_t (&x)[MS], double vol, int tp, double t,
                                           const double *df) const {
        int kind, ia, ib;
        double k;
        uint64_t mask;
        if constexpr (HELD && !TABLE) {
            kind = ri[j] & 255;
            ia = (ri[j] >> 8) & 255;
            ib = ri[j] >> 16;
            k = rk[j];
            mask = rm[j];
        } else {
            const Rxn *re = L.rx + j;
            kind = __builtin_amdgcn_readfirstlane(re->kind);
            ia = __builtin_amdgcn_readfirstlane(re->a);
            ib = __builtin_amdgcn_readfirstlane(re->b);
            k = re->k;
            mask = re->mask;
        }
        double p;
        if (VM && kind == 4) {
            p = vm_run<uint32_t, WAVE, true>(L.vcode, ia, L.vk, L.vmx + lane, vol, t, df);
        } else if (kind == 0) {
            p = k * vol;
        } else {
            const int xa = (int)pick(x, ia);
            p = k * xa;
            if (kind != 1) p = (p * (kind == 2 ? (int)pick(x, ib) : xa - 1)) / vol;
        }
        return (mask && !((mask >> tp) & 1ULL)) ? 0.0 : p;
    }
    // the VM reads a lane's counts from LDS
    __device__ __forceinline__ void stage(const uint32_t (&x)[MS]) const {
        if (VM && L.vmx) {
            sync_wave();
#pragma unroll
            for (int s = 0; s < MS; s++)
                if (s < S) L.vmx[s * WAVE + lane] = x[s];
            sync_wave();
        }
    }
    // The propensities of the reactions in this lane's column `dep` after a
    // change of counts, the changes added in the column's order; lanes' masks
    // differ, so every reaction of any lane's column is evaluated.  (Models
    // without custom propensities.)
    __device__ __forceinline__ double update(Voxel<MS, MR> &vx, unsigned dep, double vol, int tp, double t,
                                             const double *df, bool active) const {
        double rd = 0.0;
#pragma unroll
        for (int j = 0; j < MR; j++) {
            const bool on = active && ((dep >> j) & 1u);   // j < R: dep has R bits
            if (!__ballot(on)) continue;
            const double p = prop<false>(j, vx.x, vol, tp, t, df);
            if (on) {
                rd += p - vx.r[j];
                vx.r[j] = p;
            }
        }
        return rd;
    }

    // ---- the random stream --------------------------------------------------
    __device__ __forceinline__ double uni(unsigned long long p) const { return L.pool[p & (POOL - 1)]; }
    // the exponential variate of word p (this lane's)
    __device__ __forceinline__ double expo(unsigned long long p) const {
        return L.epool[p & (POOL - 1)];
    }
    __device__ __forceinline__ void fill_pool(unsigned long long upto) {
        while (fill < upto) {
            const unsigned long long k = fill + (unsigned long long)lane;
            double u, e;
            if (a.rng_kind == 1) {
                u = k < n_words ? word_uniform(a.words[k]) : 0.5;
                e = k < n_words ? a.expo[k] : 1.0;
            } else {
                u = word_uniform(philox64(seed, a.stream_id, k));
                e = uniform_expo(u);
            }
            L.pool[k & (POOL - 1)] = u;
            L.epool[k & (POOL - 1)] = e;
            fill += WAVE;
        }
    }

    // ---- the queue ------------------------------------------------------------
    __device__ __forceinline__ void lower(int v, double t) { lds_min(L.lb + (v >> nvs), t); }

    // The whole near list back to its nodes (it has no room left).
    __device__ __forceinline__ void give_back() {
        sync_wave();
        for (int k = lane; k < nc; k += WAVE) lower(L.qv[k], L.qt[k]);
        nc = 0;
        far_t = tau_t;
        far_v = tau_v;
        sync_wave();
    }
    // Entries past the front's horizon, of the lanes in `m`, into the near
    // list or to their nodes.
    __device__ __forceinline__ void put(unsigned long long m, double t, int v) {
        if (!m) return;
        bool mine = (m >> lane) & 1ULL;
        unsigned long long h = __ballot(mine && !before(far_t, far_v, t, v));
        if (nc + (int)__popcll(h) > NEAR) {
            give_back();
            h = __ballot(mine && !before(far_t, far_v, t, v));
        }
        if ((h >> lane) & 1ULL) {
            const int k = nc + (int)__popcll(h & below(lane));
            L.qt[k] = t;
            L.qv[k] = v;
        } else if (mine) {
            lower(v, t);
        }
        nc += (int)__popcll(h);
    }

    // A voxel out of the near list: its last entry takes the place.
    __device__ __forceinline__ void drop_near(int v) {
        for (int c0 = 0; c0 < nc; c0 += WAVE) {
            const unsigned long long m = __ballot(c0 + lane < nc && L.qv[c0 + lane] == v);
            if (!m) continue;
            nc--;
            if (lane == 0) {
                const int k = c0 + (int)__builtin_ctzll(m);
                L.qt[k] = L.qt[nc];
                L.qv[k] = L.qv[nc];
            }
            sync_wave();
            break;
        }
    }

    // Scan up to GROUP listed nodes: entries past the second horizon up to
    // `to` join the near list, the node's bound becomes the minimum of the
    // rest.  Two (or more, for fewer nodes) lanes split a node.  A voxel past
    // the last one is skipped (the array is padded to a whole node).
    __device__ __forceinline__ void scan_nodes(const int *nodes, int m, const Lds::Scan &sc, double &drop) {
        int per = 2;
        while (per * 2 * m <= WAVE && per * 2 * 16 <= nv) per *= 2;
        const int slot = lane / per, sub = lane % per;
        const bool on = slot < m;
        const int node = on ? nodes[slot] : 0;
        if (on && sub == 0) L.lb[node] = INFINITY;
        sync_wave();
        if (on) {
            const int len = nv / per, b0 = node * nv + sub * len;
            double rest = INFINITY;
            for (int c0 = 0; c0 < len; c0 += 16) {
                double q[16];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const Pair w = *(const Pair *)(qtime + b0 + c0 + 2 * u);
                    q[2 * u] = w.a;
                    q[2 * u + 1] = w.b;
                }
                // most nodes bring one voxel or two: the rest goes into the
                // minimum without a branch
                unsigned in = 0;
#pragma unroll
                for (int u = 0; u < 16; u++) {
                    const int v = b0 + c0 + u;
                    const bool mine = (v < n) & before(sc.far_t, sc.far_v, q[u], v);
                    const bool hit = mine & (q[u] <= sc.to);
                    in |= hit ? 1u << u : 0u;
                    const double r = (mine & !hit) ? q[u] : INFINITY;
                    rest = r < rest ? r : rest;
                }
                while (in) {
                    const int u = __builtin_ctz(in);
                    in &= in - 1;
                    const double t = qtime[b0 + c0 + u];
                    const int k = atomicAdd(&L.scan->count, 1);
                    if (k < NEAR) {
                        L.qt[k] = t;
                        L.qv[k] = b0 + c0 + u;
                    } else {
                        drop = fmin(drop, t);
                        rest = fmin(rest, t);
                    }
                }
            }
            if (rest < INFINITY) lds_min(L.lb + node, rest);
        }
        sync_wave();
    }

    // Wavefront w's share of a scan: every nw-th 64 nodes whose bound lies
    // under it.
    __device__ __forceinline__ void scan_share(int w, int nw) {
        const Lds::Scan sc = *L.scan;
        int *const nodes = L.nodes + w * GROUP;
        double drop = INFINITY;
        int m = 0;
        for (int c = w * WAVE; c < nn; c += nw * WAVE) {
            const bool hit = c + lane < nn && L.lb[c + lane] <= sc.to;
            unsigned long long h = __ballot(hit);
            while (h) {
                // as many of these nodes as the list has room for
                const int room = GROUP - m, rank = (int)__popcll(h & below(lane));
                const bool mine = ((h >> lane) & 1ULL) && rank < room;
                if (mine) nodes[m + rank] = c + lane;
                const unsigned long long took = __ballot(mine);
                m += (int)__popcll(took);
                h &= ~took;
                if (m == GROUP) {
                    sync_wave();
                    scan_nodes(nodes, m, sc, drop);
                    m = 0;
                }
            }
        }
        if (m) {
            sync_wave();
            scan_nodes(nodes, m, sc, drop);
        }
        if (drop < INFINITY) lds_min(&L.scan->drop, drop);
    }
    // The other wavefronts: their shares of every scan, until the loop ends.
    __device__ __forceinline__ void help(int w) {
        for (;;) {
            __syncthreads();
            if (L.scan->stop) return;
            scan_share(w, waves);
            __syncthreads();
        }
    }

    // Every entry past the second horizon up to `to` into the near list; the
    // least time that found no room in it.
    __device__ __forceinline__ double collect(double to) {
        if (lane == 0) *L.scan = Lds::Scan{to, far_t, INFINITY, far_v, nc, 0, {}};
        // one wavefront's worth of nodes is not worth the barriers
        const bool team = waves > 1 && nn > WAVE;
        sync_wave();
        if (team) __syncthreads();
        scan_share(0, team ? waves : 1);
        if (team) __syncthreads();
        sync_wave();
        nc = min(__builtin_amdgcn_readfirstlane(L.scan->count), NEAR);
        return L.scan->drop;
    }

    // The least bound over the nodes.
    __device__ __forceinline__ double least_bound() const {
        double m = INFINITY;
        for (int c = lane; c < nn; c += WAVE) m = fmin(m, L.lb[c]);
        return wave_min(m);
    }

    // The earliest entry past both horizons alone (times that more voxels
    // than the near list holds share exactly: a horizon in time cannot
    // separate them).  The front and the near list are empty.
    __device__ __forceinline__ void take_one() {
        double t = INFINITY;
        int v = INT_MAX;
        for (int i = lane; i < n; i += WAVE) {
            const double q = qtime[i];
            if (before(far_t, far_v, q, i) && before(q, i, t, v)) { t = q; v = i; }
        }
        const double m = wave_min(t);
        if (!(m < INFINITY)) return;
        int c = t == m ? v : INT_MAX;
        for (int o = WAVE / 2; o > 0; o >>= 1) c = min(c, __shfl_xor(c, o, WAVE));
        if (lane == 0) { ft = m; fv = c; }
        cnt = 1;
        tau_t = far_t = m;
        tau_v = far_v = c;
    }

    // Move the second horizon on until the near list holds something, unless
    // every other voxel's time is +inf.
    __device__ __forceinline__ void refill_near() {
        for (int it = 0; it < 100; it++) {
            const double least = least_bound();
            if (!(least < INFINITY)) {
                // no other voxel has a next event: everything new comes here
                far_t = INFINITY;
                far_v = INT_MAX;
                return;
            }
            const int had = nc;
            const double step = gap * (double)(near_fill - had);
            const double to = fmax(far_t, least) + step;
            const double drop = collect(to);
            far_t = to;
            far_v = INT_MAX;
            if (drop < INFINITY) {
                // too many: those from the first that found no room on go back
                far_t = drop;
                far_v = -1;
                gap *= 0.1;
                int kept = 0;
                for (int c = 0; c < nc; c += WAVE) {
                    const int k = c + lane;
                    const double t = k < nc ? L.qt[k] : INFINITY;
                    const int v = k < nc ? L.qv[k] : 0;
                    const bool keep = k < nc && t < drop;
                    if (k < nc && !keep) lower(v, t);
                    const unsigned long long h = __ballot(keep);
                    sync_wave();
                    if (keep) {
                        const int w = kept + (int)__popcll(h & below(lane));
                        L.qt[w] = t;
                        L.qv[w] = v;
                    }
                    kept += (int)__popcll(h);
                }
                nc = kept;
            } else {
                const int g = nc - had;
                gap *= g > 0 ? fmin(fmax(step / ((double)g * gap), 0.1), 4.0) : 4.0;
            }
            sync_wave();
            if (nc > 0 || cnt > 0) return;
        }
        take_one();
    }

    // The near list's earliest into the front.
    __device__ __forceinline__ void refill() {
        if (nc < NEAR_LOW && far_t < INFINITY) refill_near();
        if (nc == 0) {
            if (cnt == 0 || before(tau_t, tau_v, far_t, far_v)) { tau_t = far_t; tau_v = far_v; }
            return;
        }
        const int room = WAVE - cnt;
        const double step = gap * (double)(FRONT_FILL - cnt);
        double from = tau_t, to;
        bool all;                              // up to the second horizon
        int g, kept;
        for (;;) {
            if (!(from > -INFINITY)) {
                // the first refill, or nothing within a step of an empty front
                from = INFINITY;
                for (int k = lane; k < nc; k += WAVE) from = fmin(from, L.qt[k]);
                from = wave_min(from);
            }
            to = from + step;
            all = !(to < far_t);
            // no more of them than one pass can rank (entries of one time
            // cannot be told apart that way: those take the longer path)
            for (int it = 0; it < 4; it++) {
                int m = 0;
                for (int c = 0; c < nc; c += WAVE)
                    m += (int)__popcll(__ballot((c + lane < nc) & (all | (L.qt[min(c + lane, NEAR - 1)] <= to))));
                if (m <= WAVE) break;
                to = from + (to - from) * (0.9 * WAVE) / (double)m;
                all = !(to < far_t);
            }
            // the entries up to `to` move out of the list
            g = kept = 0;
            for (int c = 0; c < nc; c += WAVE) {
                const int k = c + lane;
                const bool in = k < nc;
                const double t = in ? L.qt[k] : INFINITY;
                const int v = in ? L.qv[k] : 0;
                const bool take = in & (all | (t <= to));
                const unsigned long long h = __ballot(take), s = __ballot(in & !take);
                sync_wave();
                if (take) {
                    const int w = g + (int)__popcll(h & below(lane));
                    L.ht[w] = t;
                    L.hv[w] = v;
                } else if (in) {
                    const int w = kept + (int)__popcll(s & below(lane));
                    L.qt[w] = t;
                    L.qv[w] = v;
                }
                g += (int)__popcll(h);
                kept += (int)__popcll(s);
            }
            if (g > 0 || cnt > 0) break;
            from = -INFINITY;
        }
        nc = kept;
        sync_wave();
        if (g == 0) {
            tau_t = to;
            tau_v = INT_MAX;
            gap *= 2.0;
            return;
        }
        if (!all) gap = 0.5 * (gap + (to - from) / (double)g);
        // their ranks by (time, voxel); the earliest join the front behind its
        // last entry, the others go back
        int joined;
        double nt = INFINITY;
        int nvx = INT_MAX;
        if (g <= WAVE) {
            const double t = lane < g ? L.ht[lane] : INFINITY;
            const int v = lane < g ? L.hv[lane] : INT_MAX;
            int rank = 0;
            for (int i0 = 0; i0 < g; i0 += 4)
#pragma unroll
                for (int u = 0; u < 4; u++) rank += rl_d(t, i0 + u) < t ? 1 : 0;
            // by time alone two entries of one time share a rank
            if (lane < g) L.nodes[rank] = lane;
            sync_wave();
            if (__ballot(lane < g && L.nodes[rank] != lane)) {
                rank = 0;
                for (int i = 0; i < g; i++) rank += before(rl_d(t, i), rl_i(v, i), t, v) ? 1 : 0;
            }
            joined = min(g, room);
            if (lane < g) {
                if (rank < joined) {
                    L.ht[rank] = t;
                    L.hv[rank] = v;
                } else {
                    // (the list held it before: there is room)
                    L.qt[nc + rank - joined] = t;
                    L.qv[nc + rank - joined] = v;
                }
            }
            nc += g - joined;
            sync_wave();
            if (lane >= cnt && lane < cnt + joined) { nt = L.ht[lane - cnt]; nvx = L.hv[lane - cnt]; }
        } else {
            joined = room;
            for (int s0 = 0; s0 < g; s0 += WAVE) {
                const int k = s0 + lane;
                const double t = k < g ? L.ht[k] : INFINITY;
                const int v = k < g ? L.hv[k] : INT_MAX;
                int rank = 0;
                for (int i = 0; i < g; i++) rank += before(L.ht[i], L.hv[i], t, v) ? 1 : 0;
                const unsigned long long back = __ballot(k < g && rank >= room);
                for (unsigned long long w = __ballot(k < g && rank < room); w; w &= w - 1) {
                    const int l = (int)__builtin_ctzll(w);
                    if (lane == cnt + rl_i(rank, l)) { nt = rl_d(t, l); nvx = rl_i(v, l); }
                }
                if ((back >> lane) & 1ULL) {
                    const int w = nc + (int)__popcll(back & below(lane));
                    L.qt[w] = t;
                    L.qv[w] = v;
                }
                nc += (int)__popcll(back);
            }
        }
        if (lane >= cnt && lane < cnt + joined) { ft = nt; fv = nvx; }
        cnt += joined;
        if (joined < g) {
            tau_t = rl_d(ft, cnt - 1);
            tau_v = rl_i(fv, cnt - 1);
        } else if (all) {
            tau_t = far_t;
            tau_v = far_v;
        } else {
            tau_t = to;
            tau_v = INT_MAX;
        }
        sync_wave();
    }

    // ---- one event alone --------------------------------------------------
    // Into the sorted front, or past its horizon.
    __device__ __forceinline__ void insert(double t, int v) {
        if (before(tau_t, tau_v, t, v)) {
            put(1ULL, t, v);
            return;
        }
        const int at = (int)__popcll(__ballot(lane < cnt && before(ft, fv, t, v)));
        const double last_t = rl_d(ft, WAVE - 1);
        const int last_v = rl_i(fv, WAVE - 1);
        const double up_t = shift_up(t, ft);
        const int up_v = dpp_i<0x138, 0xF>(v, fv);
        if (lane >= at) {
            ft = lane == at ? t : up_t;
            fv = lane == at ? v : up_v;
        }
        if (cnt < WAVE) {
            cnt++;
            return;
        }
        // no lane for the last of them: the horizon moves back
        tau_t = rl_d(ft, WAVE - 1);
        tau_v = rl_i(fv, WAVE - 1);
        if (at < WAVE) put(1ULL, last_t, last_v);
        else put(1ULL, t, v);
    }
    // Out of the sorted front: the entry of lane `at`.
    __device__ __forceinline__ void remove(int at) {
        const double dn_t = dpp_d<0x130, 0xF>(INFINITY, ft);     // lane l gets lane l+1's
        const int dn_v = dpp_i<0x130, 0xF>(INT_MAX, fv);
        if (lane >= at) {
            ft = dn_t;
            fv = dn_v;
        }
        cnt--;
    }
    // What bounds it is the chain of two round trips and of the additions that
    // keep their order (about 7,000 cycles an event; a round with nothing to
    // share takes 17,000 with 2 species and reactions, 77,000 with 16).  The
    // evaluations are one lane each, the source's and the destination's side by
    // side, and the front is repaired in registers.
    // The front's first entry alone, one lane per species and per reaction of
    // its voxel (the upper half-wave: of a hop's destination), by the operations
    // of a round.  False, with nothing stored: an event off the common path.
    __device__ __forceinline__ bool event_alone(QueueState &q, int &stale) {
        static_assert(MS <= 32 && MR <= 32, "a half-wave each");
        if (pos + 4 > n_words) return false;
        const int l = lane & 31;
        const bool up = lane >= 32, sp = l < S, rc = l < R;
        const int sv = rl_i(fv, 0);
        const double t = rl_d(ft, 0);
        uint32_t x = sp ? xx[(size_t)sv * S + l] : 0u;
        const double D = sp ? a.Ddiag[(size_t)sv * S + l] : 0.0;
        double r = rc ? rrate[(size_t)sv * R + l] : 0.0;
        double sr = srrate[sv], sd = sdrate[sv];
        const double vol = a.vol[sv];
        const int tsv = a.type[sv], dg = __builtin_amdgcn_readfirstlane(a.deg[sv]);
        const EdgeRec *const row = a.erow + (size_t)sv * W;
        EdgeRec er = row[min(lane, W - 1)];
        fill_pool(pos + 4);
        sync_wave();

        // ---- reaction or hop, and which
        const double rand1 = uni(pos), totrate = sr + sd;
        const bool react = __ballot(rand1 <= sr / totrate) != 0;
        const bool textbook = a.textbook != 0;
        const double rv = react ? (textbook ? rand1 * totrate : rand1 * sr)
                                : (textbook ? rand1 * totrate - sr : rand1 * sd);
        const int m = react ? R : S;
        const double part = react ? r : D * x;
        int which = 0;
        double cum = rl_d(part, 0);
        while (which < m && rv > cum) {
            which++;
            cum += rl_d(part, which & 31);
        }
        which = __builtin_amdgcn_readfirstlane(which);
        if (which >= m) return false;

        // ---- the hop's destination
        int dv = sv, tds = tsv;
        double srd = 0.0, sdd = 0.0, Ddd = 0.0, qtd = INFINITY;
        const double Dw = rl_d(D, which & 31);
        if (!react) {
            const double rand2 = uni(pos + 1) * Dw;
            int jd = -1;
            double cum2 = 0.0;
            for (int k0 = 0; k0 < dg && jd < 0; k0 += WAVE) {
                if (k0 > 0) er = row[min(k0 + lane, W - 1)];
                const double w = er.D * L.Dmat[which * T + (T > 1 && k0 + lane < dg ? er.type - 1 : 0)];
                for (int k = 0; k < WAVE && k0 + k < dg; k++) {
                    cum2 += rl_d(w, k);
                    if (cum2 > rand2) {
                        jd = rl_i(er.j, k);
                        break;
                    }
                }
            }
            jd = __builtin_amdgcn_readfirstlane(jd);
            if (jd < 0 || jd == sv) return false;
            dv = jd;
            if (up) {
                x = sp ? xx[(size_t)dv * S + l] : 0u;
                r = rc ? rrate[(size_t)dv * R + l] : 0.0;
            }
            srd = srrate[dv];
            sdd = sdrate[dv];
            Ddd = a.Ddiag[(size_t)dv * S + which];
            qtd = qtime[dv];
            tds = a.type[dv];
        }

        // ---- the event
        const bool side = !up || !react;                     // lanes with a voxel of the event
        const unsigned dep = (unsigned)__builtin_amdgcn_readfirstlane((int)L.dep[react ? S + which : which]);
        const int d = react && sp && !up ? L.dN[which * MS + l] : 0;
        unsigned long long changed = 0;
        if (react) {
            changed = __ballot(d != 0);
            x += (uint32_t)d;
            for (unsigned long long h = changed; h; h &= h - 1) {
                const int s = (int)__builtin_ctzll(h);
                sd += rl_d(D, s) * rl_i(d, s);
            }
        } else if (l == which) {
            x += up ? 1u : ~0u;
        }
        const bool mine = rc && side && ((dep >> l) & 1u);
        if (dep) {
            const Rxn *const re = L.rx + (rc ? l : 0);
            const int kind = re->kind, at = lane & 32;
            const int xa = __shfl((int)x, at + (re->a & 31), WAVE), xb = __shfl((int)x, at + (re->b & 31), WAVE);
            double p;
            if (kind == 0) {
                p = re->k * vol;
            } else {
                p = re->k * xa;
                if (kind != 1) p = (p * (kind == 2 ? xb : xa - 1)) / vol;
            }
            if constexpr (VM) {
                if (L.vmx) {
                    if (sp) L.vmx[l * WAVE + at] = x;
                    sync_wave();
                    // each lane its own program: a round, which runs them one after
                    // the other, takes 120,000 cycles with 16 of them, an event
                    // this way 24,000
                    if (mine && kind == 4)
                        p = vm_run<uint32_t, WAVE>(L.vcode, re->a, L.vk, L.vmx + at, vol, t,
                                                   a.data_fn ? a.data_fn + (size_t)(up ? dv : sv) * a.n_df : nullptr);
                }
            }
            if (re->mask && !((re->mask >> (up ? tds : tsv)) & 1ULL)) p = 0.0;
            const double diff = p - r;
            double rd = 0.0, rdd = 0.0;
            for (unsigned h = dep; h; h &= h - 1) {
                const int j = __builtin_ctz(h);
                rd += rl_d(diff, j);
                rdd += rl_d(diff, 32 + j);
            }
            if (mine) r = p;
            sr += rd;
            if (!react) srd += rdd;
        }
        if (!react) {
            sd -= Dw;
            sdd += Ddd;
        }

        // ---- the new firing times
        unsigned long long pn = pos + (react ? 1 : 2);
        double ntv = INFINITY, ntd = INFINITY;
        int da = 0;
        if (const double tot = sr + sd; __ballot(tot <= 0.0)) da--;
        else ntv = expo(pn++) / tot + t;
        if (!react) {
            if (const double tot = srd + sdd; __ballot(tot <= 0.0)) {
                if (__ballot(qtd != INFINITY)) da--;
            } else {
                ntd = expo(pn++) / tot + t;
                if (__ballot(qtd == INFINITY)) da++;
            }
        }

        // ---- store
        const int at = up ? dv : sv;
        if (side) {
            if (sp && (react || l == which)) xx[(size_t)at * S + l] = x;
            if (mine) rrate[(size_t)at * R + l] = r;
            if (l == 0) {
                srrate[at] = up ? srd : sr;
                sdrate[at] = up ? sdd : sd;
                qtime[at] = up ? ntd : ntv;
            }
        }
        if (a.snap_tot && ((changed >> lane) & 1ULL)) atomicAdd(L.tot + l, (unsigned)d);
        if (a.trace && lane == 0 && q.events_traced < a.trace_cap) {
            ssasdpd_event ev;
            ev.t = t; ev.voxel = sv; ev.kind = react ? 0 : 1; ev.which = which; ev.dest = react ? -1 : dv;
            a.trace[q.events_traced] = ev;
        }
        pos = pn;
        q.rxnCount++;
        q.events_traced++;
        if (react) q.reactions++;
        else q.diffusions++;
        q.active = (unsigned long long)((long long)q.active + da);

        // ---- the queue
        qtd = rl_d(qtd, 0);
        ntv = rl_d(ntv, 0);
        ntd = rl_d(ntd, 0);
        remove(0);
        if (!react) {
            stale = dv;
            if (qtd < INFINITY) {
                if (!before(tau_t, tau_v, qtd, dv)) {
                    const unsigned long long h = __ballot(lane < cnt && fv == dv);
                    if (h) remove((int)__builtin_ctzll(h));
                } else if (!before(far_t, far_v, qtd, dv)) {
                    drop_near(dv);
                }
            }
        }
        if (ntv < INFINITY) insert(ntv, sv);
        if (ntd < INFINITY) insert(ntd, dv);
        return true;
    }
};

}  // namespace

// The event loop of one trajectory on one wavefront.  b: its index in a
// batch that shares one argument block (strides bs_*), else 0.
// VM: kind-4 reactions (custom propensities) through the expression VM.
// ALONE: where rounds keep too few events, they go one by one.
template <int MS, int MR, bool VM, bool ALONE>
__device__ __forceinline__ void ssa_run(const RdmeArgs &a, const size_t b) {
    extern __shared__ __align__(16) unsigned char smem[];
    QueueState *const qs_ = a.qs + b;
    QueueState q = *qs_;
    if (q.initialized != 1 || q.err) return;
    Loop<MS, MR, VM> lp(a);
    lp.lane = threadIdx.x & (WAVE - 1);
    lp.waves = blockDim.x / WAVE;
    const int tid = threadIdx.x, nthr = blockDim.x;
    lp.xx = a.xx + b * a.bs_xx;
    lp.rrate = a.rrate + b * a.bs_rr;
    lp.srrate = a.srrate + b * a.bs_n;
    lp.sdrate = a.sdrate + b * a.bs_n;
    lp.qtime = a.qtime + b * a.bs_n;
    double *const tmin = a.tmin + b * a.bs_tree;
    lp.seed = a.seeds ? a.seeds[b] : a.seed;
    lp.n = a.n; lp.S = a.S; lp.R = a.R; lp.T = a.T; lp.W = a.W;
    lp.nn = a.tree_nodes;
    lp.nv = WAVE * a.pl;
    lp.nvs = 31 - __builtin_clz(lp.nv);
    const int lane = lp.lane, S = a.S, R = a.R, T = a.T, W = a.W;
    Lds &L = lp.L;
    {
        auto al = [](size_t x) { return (x + 15) & ~(size_t)15; };
        size_t o = 0;
        auto take = [&](size_t bytes) { void *p = smem + o; o += al(bytes); return p; };
        L.lb = (double *)take(sizeof(double) * lp.nn);
        L.pool = (double *)take(sizeof(double) * POOL);
        L.epool = (double *)take(sizeof(double) * POOL);
        L.qt = (double *)take(sizeof(double) * NEAR);
        L.qv = (int *)take(sizeof(int) * NEAR);
        L.nodes = (int *)take(sizeof(int) * WAVES * GROUP);
        L.scan = (Lds::Scan *)take(sizeof(Lds::Scan));
        L.claim = (unsigned *)take(sizeof(unsigned) * 2 * CLAIMS);
        static_assert(sizeof(unsigned) * 2 * CLAIMS >= (sizeof(double) + sizeof(int)) * NEAR, "shared room");
        L.ht = (double *)L.claim;
        L.hv = (int *)(L.ht + NEAR);
        L.rx = (Rxn *)take(sizeof(Rxn) * R);
        L.Dmat = (double *)take(sizeof(double) * S * T);
        L.dN = (int *)take(sizeof(int) * R * MS);
        L.dep = (unsigned *)take(sizeof(unsigned) * (S + R));
        L.tot = (unsigned *)take(sizeof(unsigned) * S);
        L.vmx = nullptr;
        if (VM && a.vm_ncode > 0) {
            L.vmx = (uint32_t *)take(sizeof(uint32_t) * WAVE * S);
            L.vcode = (uint32_t *)take(sizeof(uint32_t) * a.vm_ncode);
            L.vk = (double *)take(sizeof(double) * a.vm_nk);
            for (int i = tid; i < a.vm_ncode; i += nthr) L.vcode[i] = a.vm_code[i];
            for (int i = tid; i < a.vm_nk; i += nthr) L.vk[i] = a.vm_k[i];
        }
        for (int i = tid; i < lp.nn; i += nthr) L.lb[i] = tmin[i];
        for (int i = tid; i < R; i += nthr) L.rx[i] = a.rx[i];
        for (int i = tid; i < S * T; i += nthr) L.Dmat[i] = a.Dmat[i];
        for (int i = tid; i < R * MS; i += nthr) L.dN[i] = 0;
        if (tid < S) L.tot[tid] = 0;
        if (tid < S + R) {
            unsigned d = 0;
            for (int k = a.jcG[tid]; k < a.jcG[tid + 1]; k++) d |= 1u << a.irG[k];
            L.dep[tid] = d;
        }
        __syncthreads();
        if (tid < R)
            for (int k = a.jcN[tid]; k < a.jcN[tid + 1]; k++) L.dN[tid * MS + a.irN[k]] = a.prN[k];
    }
    // species totals (persistent mode's snapshots)
    if (a.snap_tot) {
        uint32_t part[MS];
#pragma unroll
        for (int s = 0; s < MS; s++) part[s] = 0;
        for (int i = tid; i < a.n; i += nthr)
#pragma unroll
            for (int s = 0; s < MS; s++)
                if (s < S) part[s] += lp.xx[(size_t)i * S + s];
#pragma unroll
        for (int s = 0; s < MS; s++)
            if (s < S) atomicAdd(L.tot + s, part[s]);
    }
    __syncthreads();
    if (tid >= WAVE) {
        lp.help(tid / WAVE);
        return;
    }

    lp.n_words = a.rng_kind == 1 ? a.n_words : ~0ULL;
    lp.pos = q.rng_pos;
    lp.fill = q.rng_pos & ~63ULL;
    lp.ft = INFINITY;
    lp.fv = INT_MAX;
    lp.cnt = lp.nc = 0;
    lp.tau_t = lp.far_t = -INFINITY;
    lp.tau_v = lp.far_v = -1;
    lp.near_fill = (int)fmin(fmax((double)q.active * 0.25, 64.0), (double)NEAR_FILL);
    if constexpr (Loop<MS, MR, VM>::HELD) {
#pragma unroll
        for (int j = 0; j < MR; j++) {
            lp.ri[j] = 0;
            lp.rk[j] = 0.0;
            lp.rm[j] = 0;
            if (j < R) {
                const Rxn re = a.rx[j];
                lp.ri[j] = __builtin_amdgcn_readfirstlane(re.kind | re.a << 8 | re.b << 16);
                lp.rk[j] = rl_d(re.k, 0);
                lp.rm[j] = (uint64_t)(uint32_t)rl_i((int)(uint32_t)re.mask, 0) |
                           (uint64_t)(uint32_t)rl_i((int)(uint32_t)(re.mask >> 32), 0) << 32;
            }
        }
    }
    // one bin of the window holds 16 events on average (setBinNumberAndBounds)
    lp.gap = q.nbins > 0 ? (q.U - q.L) / (16.0 * (double)q.nbins) : a.dt;
    if (!(lp.gap > 0.0) || !(lp.gap < INFINITY)) lp.gap = a.dt;
    lp.guess_empty = 1.0;
    const int widest = VM ? WAVE / 2 : WAVE;
    int width = widest;   // lanes a round tries: about twice what the last ones kept
    // kept: 16 times what the last rounds kept, on average; below lone_at the
    // next events go alone, 32 << lone of them, then a round to see.  lone_at: 16
    // times a round's cost over an event's alone (2 at 2 species and reactions, 4
    // at 8, 12 at 16: 10 x 10 voxels with 8 of each 54.8 ms in rounds, 54.5 so)
    const int lone_at = VM ? 16 + 4 * R : MR <= 8 ? 24 + 11 * (S + R) / 4 : 6 * (S + R);
    int kept = lone_at - 1, lone = 0;
    const bool textbook = a.textbook != 0;
    const double inf = INFINITY;
    int err = 0;
    int ks = 0;
    const size_t nsS = (size_t)a.n * S;
    uint32_t *const snap_xx = a.snap_xx ? a.snap_xx + b * a.bs_snap : nullptr;
    uint32_t *const snap_tot = a.snap_tot ? a.snap_tot + b * a.n_snap * S : nullptr;

    const unsigned step_end = a.step_end > a.step ? a.step_end : a.step + 1;
    for (unsigned stp = a.step; stp < step_end; stp++) {
        while (ks < a.n_snap && a.snap_step[ks] <= stp)
            snapshot_counts(lp.xx, snap_xx, snap_tot, nsS, S, ks++, L.tot, lane);
        // one step of simulate_rdme (simulate_rdme.cpp:53-68): events while the
        // last one fired at or before the step's end; the destination carried
        // between diffusion events restarts each step
        const double t0 = a.step_end > a.step ? (double)stp * a.dt : a.t0;
        double tt = t0;
        const double end_time = t0 + a.dt;
        int stale = -1;                       // the last hop's destination
        unsigned long long guard = 0;
        bool more = false;
        do {
        // events alone, as long as the front holds the next ones
        if (ALONE && kept < lone_at) {
            int left = 32 << lone;
            for (; left > 0 && tt <= end_time && guard < a.max_events && lp.cnt > 0 &&
                   !(lp.cnt < FRONT_LOW && lp.tau_t < inf); left--) {
                const double first = rl_d(lp.ft, 0);
                if (!(first <= q.U) || !lp.event_alone(q, stale)) break;
                guard++;
                tt = first;
                sync_wave();
            }
        }
        more = false;
        while (tt <= end_time) {
            if (guard >= a.max_events) { err = SSASDPD_ERR_CAPACITY; break; }
            // ---- selectReaction: the earliest voxel inside the window [L, U]
            if (lp.cnt < FRONT_LOW && lp.tau_t < inf) lp.refill();
            const double first = lp.cnt > 0 ? rl_d(lp.ft, 0) : inf;
            if (!(lp.cnt > 0 && first <= q.U)) {
                if (!rebuild(q)) break;
                if (!(lp.cnt > 0 && first <= q.U)) break;   // window moved but still empty: empty queue this call
            }
            // the round's lanes: entries inside the window, the first one past
            // the step's end included
            int K = (int)__popcll(__ballot(lane < lp.cnt && lp.ft <= q.U));
            K = min(K, first_lane(__ballot(lane < lp.cnt && lp.ft > end_time)) + 1);
            K = min(K, width);
            if (a.max_events - guard < (unsigned long long)K) K = (int)(a.max_events - guard);
            const bool on = lane < K;
            const double t = on ? lp.ft : first;
            const int sv = on ? lp.fv : rl_i(lp.fv, 0);

            // ---- round trip 1: the voxels' states
            Voxel<MS, MR> vx;
            double Dd[MS];
#pragma unroll
            for (int s = 0; s < MS; s++) {
                vx.x[s] = 0;
                Dd[s] = 0.0;
                if (s < S) {
                    vx.x[s] = lp.xx[(size_t)sv * S + s];
                    Dd[s] = a.Ddiag[(size_t)sv * S + s];
                }
            }
#pragma unroll
            for (int j = 0; j < MR; j++) vx.r[j] = j < R ? lp.rrate[(size_t)sv * R + j] : 0.0;
            vx.sr = lp.srrate[sv];
            vx.sd = lp.sdrate[sv];
            const double vol = a.vol[sv];
            const int tsv = a.type[sv];
            const int dg = a.deg[sv];
            const double *const df = a.data_fn ? a.data_fn + (size_t)sv * a.n_df : nullptr;
            // most events are hops: the row's first entries come along
            const EdgeRec *const row = a.erow + (size_t)sv * W;
            EdgeRec er[ROW];
#pragma unroll
            for (int u = 0; u < ROW; u++) er[u] = row[min(u, W - 1)];
            // and where rows are longer, the next ones
            EdgeRec en[ROW];
            if (a.row_w > ROW)
#pragma unroll
                for (int u = 0; u < ROW; u++) en[u] = row[min(ROW + u, W - 1)];
            lp.fill_pool(lp.pos + 4ULL * WAVE);
            sync_wave();

            // ---- which outcomes leave the voxel without a next event (no
            // exponential is drawn then): only where the diffusion rate left
            // over is nothing next to the present one
            unsigned emS = 0, emR = 0;
            for (int q1 = 0; q1 < S + R; q1++) {
                // outcome q1: species q1 leaves, or reaction q1 - S fires
                const int r = q1 - S;
                const bool can = on && (r < 0 ? pick(vx.x, q1) > 0 : pick(vx.r, r) > 0.0);
                if (!__ballot(can)) continue;
                Voxel<MS, MR> w = vx;
                double sdn = vx.sd;
#pragma unroll
                for (int s = 0; s < MS; s++) {
                    const int d = r < 0 ? (s == q1 ? -1 : 0) : L.dN[r * MS + s];
                    w.x[s] += (uint32_t)d;
                    sdn += Dd[s] * d;
                }
                const bool amb = can && !(sdn > 1e-9 * vx.sd);
                if (!__ballot(amb)) continue;
                bool empty;
                if constexpr (VM) {
                    empty = lp.guess_empty != 0.0;
                } else {
                    const double srn = vx.sr + lp.update(w, L.dep[q1], vol, tsv, t, df, amb);
                    empty = srn + sdn <= 0.0;
                }
                const unsigned bit = amb && empty ? 1u : 0u;
                if (r < 0) emS |= bit << q1;
                else emR |= bit << r;
            }

            // ---- the draws: each lane's place in the stream and its choice
            const double totrate = vx.sr + vx.sd;
            const double share = vx.sr / totrate;
            double cr[MR], cs[MS];           // running sums of the selections
#pragma unroll
            for (int j = 0; j < MR; j++) cr[j] = j == 0 ? vx.r[0] : cr[j > 0 ? j - 1 : 0] + vx.r[j];
#pragma unroll
            for (int s = 0; s < MS; s++)
                cs[s] = s == 0 ? Dd[0] * vx.x[0] : cs[s > 0 ? s - 1 : 0] + Dd[s] * vx.x[s];
            // most lanes draw a number that hangs on reaction or hop alone
            unsigned canS = 0, canR = 0;
#pragma unroll
            for (int s = 0; s < MS; s++) canS |= vx.x[s] > 0 && Dd[s] > 0.0 ? 1u << s : 0u;
#pragma unroll
            for (int j = 0; j < MR; j++) canR |= vx.r[j] > 0.0 ? 1u << j : 0u;
            const bool plain = !__ballot(on && ((emS && (canS & ~emS)) || (emR && (canR & ~emR))));
            const int cR = emR ? 1 : 2, cS = emS ? 3 : 4;
            int c = on ? (share > 0.5 ? cR : cS) : 0, ex = 0, which = 0;
            bool react = false, over = false, act = false, hop = false;
            bool noop = false;       // the event changes nothing and leaves the queue as it is
            int forced = -1;         // lane 0's choice, when the first selection ran past the last entry
            int selfx = -1;          // the place in the stream at which this lane hops into its own voxel
            int lerr = 0, spec = 0, jd = -1, held = 0;
            double rand1 = 0.0;
            unsigned long long p0 = 0, cut = 0;
            for (int redo = 0;; redo++) {
                // the first entry whose running sum the value does not pass
                auto choose = [&]() {
                    const double rv = react ? (textbook ? rand1 * totrate : rand1 * vx.sr)
                                            : (textbook ? rand1 * totrate - vx.sr : rand1 * vx.sd);
                    int wr = R, ws = S;
#pragma unroll
                    for (int j = MR - 1; j >= 0; j--) wr = ((j < R) & !(rv > cr[j])) ? j : wr;
#pragma unroll
                    for (int s = MS - 1; s >= 0; s--) ws = ((s < S) & !(rv > cs[s])) ? s : ws;
                    which = react ? wr : ws;
                };
                for (int it = 0; it <= WAVE; it++) {
                    ex = scan_add(c) - c;
                    rand1 = lp.uni(lp.pos + ex);
                    react = rand1 <= share;
                    int cn = react ? cR : cS;
                    if (!plain) {
                        choose();
                        const int gone = (int)(((react ? emR : emS) >> which) & 1u);
                        cn = react ? 2 - gone : 4 - gone;
                    }
                    if (!react && selfx == ex) cn = 4;
                    cn = on ? cn : 0;
                    if (!__ballot(cn != c)) break;
                    c = cn;
                }
                choose();
                p0 = lp.pos + (unsigned long long)ex;

                // ---- lane 0's selections that ran past the last entry
                // (simulate_rdme.cpp:262-294, 322-349); other lanes wait for
                // their turn as lane 0.  cum: what the selection's sum ended at
                over = on && (react ? which >= R : which >= S);
                if (forced >= 0) { which = forced; over = false; }
                double cum = react ? (R > 0 ? pick(cr, R - 1) : 0.0) : pick(cs, S - 1);
                if (p0 >= lp.n_words) {
                    over = on;
                    if (lane == 0) lerr = SSASDPD_ERR_REPLAY_EXHAUSTED;
                } else {
                    if (redo == 0 && lane == 0 && over && react) {
                        if (cum != vx.sr) {
                            lp.stage(vx.x);
                            double rd = 0.0;
                            for (int j = 0; j < R; j++) {
                                const double p = lp.template prop<true>(j, vx.x, vol, tsv, t, df);
#pragma unroll
                                for (int u = 0; u < MR; u++)
                                    if (u == j) vx.r[u] = p;
                                rd += p;
                                lp.rrate[(size_t)sv * R + j] = p;
                            }
                            vx.sr = rd;
                            lp.srrate[sv] = rd;
                        }
                        if (vx.sr == 0.0) noop = true;
                        else {
                            const double rv2 = rand1 * vx.sr;
                            which = 0;
                            cum = vx.r[0];
                            while (which < R && rv2 > cum) { which++; cum += which < R ? pick(vx.r, which) : 0.0; }
                            if (which >= R) lerr = SSASDPD_ERR_PROPENSITY_OVERFLOW;
                        }
                    } else if (redo == 0 && lane == 0 && over) {
                        if (cum != vx.sd) {
                            double rd = 0.0;
#pragma unroll
                            for (int s = 0; s < MS; s++)
                                if (s < S) rd += Dd[s] * vx.x[s];
                            vx.sd = rd;
                            lp.sdrate[sv] = rd;
                        }
                        if (vx.sd == 0.0) noop = true;
                        else {
                            const double rv2 = cum * rand1;
                            which = 0;
                            cum = Dd[0] * vx.x[0];
                            while (which < S && rv2 > cum) {
                                which++;
                                cum += which < S ? pick(Dd, which) * pick(vx.x, which) : 0.0;
                            }
                            if (which >= S) {
                                which--;
                                bool bad = false;
                                while (pick(vx.x, which) <= 0) {
                                    which--;
                                    if (which <= 0) { bad = true; break; }
                                }
                                if (bad) lerr = SSASDPD_ERR_DIFFUSION_OVERFLOW;
                            }
                        }
                    }
                    if (redo == 0 && lane == 0 && over && !noop) { forced = which; over = false; }
                }
                if (rl_i(lerr, 0)) break;
                // the lanes still in the round
                cut = __ballot(over) & ~1ULL;
                act = on && lane < first_lane(cut) && !noop;
                hop = act && !react;
                spec = hop ? which : 0;

                // ---- the hop's destination: the neighbour row in list order
                const double r2 = lp.uni(p0 + 1);
                double rand2 = r2 * pick(Dd, spec);
                jd = -1;
                if (hop && p0 + 1 >= lp.n_words) {
                    if (lane == 0) lerr = SSASDPD_ERR_REPLAY_EXHAUSTED;
                } else if (hop) {
                    const double D1 = L.Dmat[spec * T];
                    for (int pass = 0; pass < 2 && jd < 0; pass++) {
                        double cum2 = 0.0;
                        for (int k0 = 0; k0 < dg && jd < 0; k0 += ROW) {
                            if (held != k0) {
                                if (held == k0 - ROW) {
#pragma unroll
                                    for (int u = 0; u < ROW; u++) er[u] = en[u];
                                } else {
#pragma unroll
                                    for (int u = 0; u < ROW; u++) er[u] = row[min(k0 + u, dg - 1)];
                                }
                                held = k0;
                                if (k0 + ROW < dg)
#pragma unroll
                                    for (int u = 0; u < ROW; u++) en[u] = row[min(k0 + ROW + u, dg - 1)];
                            }
#pragma unroll
                            for (int u = 0; u < ROW; u++) {
                                const double D = T > 1 ? L.Dmat[spec * T + (k0 + u < dg ? er[u].type - 1 : 0)] : D1;
                                const bool in = (k0 + u < dg) & (jd < 0);
                                const double nc2 = cum2 + er[u].D * D;
                                cum2 = in ? nc2 : cum2;
                                jd = (in & (nc2 > rand2)) ? er[u].j : jd;
                            }
                        }
                        if (jd >= 0 || lane != 0) break;
                        if (stale >= 0) { jd = stale; break; }   // simulate_rdme.cpp:368
                        rand2 = r2 * cum2;
                    }
                    if (jd < 0 && lane == 0) lerr = SSASDPD_ERR_DIFFUSION_OVERFLOW;
                }
                if (rl_i(lerr, 0)) break;
                // a hop into the own voxel does not empty it: the places after
                // such a lane that was expected to are wrong
                const bool again = hop && jd == sv && ((emS >> spec) & 1u) && selfx != ex;
                if (!__ballot(again) || redo == 3) break;
                if (again) selfx = ex;
            }
            if (rl_i(lerr, 0)) { err = rl_i(lerr, 0); break; }
            const bool self = hop && jd == sv;
            cut |= __ballot(hop && jd < 0) & ~1ULL;
            act = act && lane < first_lane(cut);

            // ---- round trip 2: the destinations' states
            const bool mv = act && !react;
            const int dv = mv ? jd : sv;
            Voxel<MS, MR> vd;
            vd.sr = vd.sd = 0.0;
            double Ddd = 0.0, qtd = inf;
            int tds = tsv;
#pragma unroll
            for (int s = 0; s < MS; s++) vd.x[s] = 0;
#pragma unroll
            for (int j = 0; j < MR; j++) vd.r[j] = 0.0;
            if (mv) {
#pragma unroll
                for (int s = 0; s < MS; s++)
                    if (s < S) vd.x[s] = lp.xx[(size_t)dv * S + s];
#pragma unroll
                for (int j = 0; j < MR; j++)
                    if (j < R) vd.r[j] = lp.rrate[(size_t)dv * R + j];
                vd.sr = lp.srrate[dv];
                vd.sd = lp.sdrate[dv];
                Ddd = a.Ddiag[(size_t)dv * S + spec];
                qtd = lp.qtime[dv];
                tds = a.type[dv];
            }

            // ---- the event
            const unsigned dep = act ? L.dep[react ? S + which : spec] : 0u;
            int act_d = 0;                     // change of the active count
            double ntv = inf, ntd = inf;
            unsigned long long pn = p0 + (react ? 1 : 2);   // the next word
            if (act && react) {
                // stoichiometry column (CSC order: ascending species)
#pragma unroll
                for (int s = 0; s < MS; s++)
                    if (s < S) {
                        const int d = L.dN[which * MS + s];
                        if (d != 0) {
                            vx.x[s] += (uint32_t)d;
                            vx.sd += Dd[s] * d;
                        }
                    }
            } else if (mv && !self) {
#pragma unroll
                for (int s = 0; s < MS; s++)
                    if (s == spec) { vx.x[s] -= 1u; vd.x[s] += 1u; }
            }
            const bool there = mv && !self;
            if constexpr (VM) {
                // an evaluation costs 7,000 cycles whatever the lanes hold: the
                // upper half-wave takes the lower one's destinations (the
                // 144-voxel model 97 -> 62 ms)
                const int peer = lane & 31;
                const bool up = lane >= 32;
                uint32_t xc[MS];
#pragma unroll
                for (int s = 0; s < MS; s++) {
                    const uint32_t o = (uint32_t)__shfl((int)vd.x[s], peer, WAVE);
                    xc[s] = up ? o : vx.x[s];
                }
                const double vol_c = __shfl(vol, peer, WAVE), t_c = __shfl(t, peer, WAVE);
                const int tds_c = __shfl(tds, peer, WAVE), dv_c = __shfl(dv, peer, WAVE);
                const int at_c = up ? dv_c : sv, tp_c = up ? tds_c : tsv;
                const double *const df_c = a.data_fn ? a.data_fn + (size_t)at_c * a.n_df : nullptr;
                lp.stage(xc);
                double rd = 0.0, rdd = 0.0;
                for (int j = 0; j < R; j++) {
                    // (only the lower half has lanes with a column: a destination
                    // takes its source's)
                    const bool now = act && ((dep >> j) & 1u);
                    if (!__ballot(now)) continue;
                    const double p = lp.template prop<true>(j, xc, vol_c, tp_c, t_c, df_c);
                    const double pd = __shfl(p, (lane & 31) + 32, WAVE);
#pragma unroll
                    for (int u = 0; u < MR; u++)
                        if (u == j && now) {
                            rd += p - vx.r[u];
                            vx.r[u] = p;
                            if (there) {
                                rdd += pd - vd.r[u];
                                vd.r[u] = pd;
                            }
                        }
                }
                if (act) vx.sr += rd;
                if (there) vd.sr += rdd;
            } else if (R > 0) {
                const double rd = lp.update(vx, dep, vol, tsv, t, df, act);
                if (act) vx.sr += rd;
                if (__ballot(there)) {
                    const double rdd = lp.update(vd, dep, vol, tds, t, nullptr, there);
                    if (there) vd.sr += rdd;
                }
            }
            if (mv) vx.sd -= pick(Dd, spec);
            if (mv && !self) vd.sd += Ddd;
            if (self) {
                // source and destination are one voxel, updated in turn
                // (simulate_rdme.cpp:402-445): the counts are what they were,
                // the second pass over the rates changes nothing
                vx.sd += pick(Dd, spec);
                vd = vx;
            }
            // ---- the new firing times (NRMConstant_v5::update,
            // NRMConstant_v5.cpp:89-132)
            if (act) {
                const double tot = vx.sr + vx.sd;
                if (tot <= 0.0) act_d--;       // the voxel's own time was finite
                else ntv = lp.expo(pn++) / tot + t;
                if (mv) {
                    const double dtot = vd.sr + vd.sd;
                    const double dold = self ? ntv : qtd;
                    if (dtot <= 0.0) {
                        if (dold != inf) act_d--;
                    } else {
                        ntd = lp.expo(pn++) / dtot + t;
                        if (dold == inf) act_d++;
                    }
                }
            }
            if (lane == 0 && act && pn > lp.n_words) lerr = SSASDPD_ERR_REPLAY_EXHAUSTED;
            if (rl_i(lerr, 0)) { err = rl_i(lerr, 0); break; }
            const int used = noop ? 1 : (int)(pn - p0);
            if (self) ntv = ntd;               // the voxel's one entry

            // ---- how many lanes stand: the first whose voxels an earlier
            // lane touched, or that comes after an earlier lane's new time,
            // or whose place in the stream was wrong
            unsigned long long bad = ~__ballot(act) & ~1ULL;
            bad |= __ballot(on && pn > lp.n_words) & ~1ULL;
            {
                const unsigned hs = (unsigned)sv * 2654435761u, hd = (unsigned)dv * 2654435761u;
                const unsigned s1 = hs >> 21, s2 = CLAIMS + ((hs >> 5) & (CLAIMS - 1));
                const unsigned d1 = hd >> 21, d2 = CLAIMS + ((hd >> 5) & (CLAIMS - 1));
                if (act) {
                    L.claim[s1] = ~0u;
                    L.claim[s2] = ~0u;
                    L.claim[d1] = ~0u;
                    L.claim[d2] = ~0u;
                }
                sync_wave();
                if (act) {
                    atomicMin(L.claim + s1, (unsigned)lane);
                    atomicMin(L.claim + s2, (unsigned)lane);
                    if (mv) {
                        atomicMin(L.claim + d1, (unsigned)lane);
                        atomicMin(L.claim + d2, (unsigned)lane);
                    }
                }
                sync_wave();
                bool touched = false;
                if (act) {
                    touched = L.claim[s1] < (unsigned)lane && L.claim[s2] < (unsigned)lane;
                    if (mv) touched = touched || (L.claim[d1] < (unsigned)lane && L.claim[d2] < (unsigned)lane);
                }
                bad |= __ballot(touched);
                sync_wave();
            }
            const double soonest = shift_up(inf, scan_min(act ? fmin(ntv, mv ? ntd : inf) : inf));
            bad |= __ballot(act && soonest <= t);
            const unsigned long long off = __ballot(act && used != c);   // later lanes' places are wrong
            int P = min(K, min(first_lane(bad), first_lane(off) + 1));
            if (rl_i(noop ? 1 : 0, 0)) P = 1;
            if (VM) {
                const int o = first_lane(off);
                if (o < WAVE) lp.guess_empty = rl_i(used, o) < rl_i(c, o) ? 1.0 : 0.0;
            }
            const bool done = act && lane < P;
            width = P == K ? min(2 * width, widest) : max(8, min(widest, (width + 3 * P + 8) / 2));

            if (ALONE && (P < K || K == 1 || 16 * K >= lone_at)) {
                kept += (16 * P - kept) / 8;
                lone = kept < lone_at ? min(lone + 1, 5) : 0;
            }

            // ---- store
            const unsigned long long m_done = __ballot(done), m_hop = __ballot(done && mv);
            if (done) {
                if (react) {
#pragma unroll
                    for (int s = 0; s < MS; s++)
                        if (s < S) lp.xx[(size_t)sv * S + s] = vx.x[s];
                } else {
                    if (!self) lp.xx[(size_t)sv * S + spec] = pick(vx.x, spec);
                    lp.xx[(size_t)dv * S + spec] = pick(vd.x, spec);
                }
#pragma unroll
                for (int j = 0; j < MR; j++)
                    if ((dep >> j) & 1u) {
                        lp.rrate[(size_t)sv * R + j] = vx.r[j];
                        if (mv) lp.rrate[(size_t)dv * R + j] = vd.r[j];
                    }
                lp.srrate[sv] = vx.sr;
                lp.sdrate[sv] = vx.sd;
                lp.qtime[sv] = ntv;
                if (mv) {
                    lp.srrate[dv] = vd.sr;
                    lp.sdrate[dv] = vd.sd;
                    lp.qtime[dv] = ntd;
                }
                if (a.snap_tot && react)
                    for (int s = 0; s < S; s++) {
                        const int d = L.dN[which * MS + s];
                        if (d != 0) atomicAdd(L.tot + s, (unsigned)d);
                    }
                if (a.trace) {
                    const unsigned long long ix = q.events_traced + (unsigned long long)lane;
                    if (ix < a.trace_cap) {
                        ssasdpd_event ev;
                        ev.t = t; ev.voxel = sv; ev.kind = react ? 0 : 1; ev.which = which; ev.dest = react ? -1 : dv;
                        a.trace[ix] = ev;
                    }
                }
            }
            lp.pos += (unsigned long long)(rl_i(ex, P - 1) + rl_i(used, P - 1));
            q.rxnCount += (unsigned long long)P;
            guard += (unsigned long long)P;
            tt = rl_d(t, P - 1);
            if (m_done) {
                q.events_traced += __popcll(m_done);
                q.diffusions += __popcll(m_hop);
                q.reactions += __popcll(m_done & ~m_hop);
                const int da = rl_i(scan_add(done ? act_d : 0), WAVE - 1);
                q.active = (unsigned long long)((long long)q.active + da);
                if (m_hop) stale = rl_i(dv, last_lane(m_hop));
                // ---- the queue: without the events done and the destinations
                // whose time changed, then the new times
                unsigned long long gone = below(P);
                const bool moved = done && mv && !self && qtd < inf;
                const bool inF = moved && !before(lp.tau_t, lp.tau_v, qtd, dv);
                for (unsigned long long h = __ballot(inF); h; h &= h - 1)
                    gone |= __ballot(lane < lp.cnt && lp.fv == rl_i(dv, (int)__builtin_ctzll(h)));
                for (unsigned long long h = __ballot(moved && !inF && !before(lp.far_t, lp.far_v, qtd, dv)); h;
                     h &= h - 1)
                    lp.drop_near(rl_i(dv, (int)__builtin_ctzll(h)));
                const bool newS = done && ntv < inf, newD = done && mv && !self && ntd < inf;
                const bool inS = newS && !before(lp.tau_t, lp.tau_v, ntv, sv);
                const bool inD = newD && !before(lp.tau_t, lp.tau_v, ntd, dv);
                lp.put(__ballot(newS && !inS), ntv, sv);
                lp.put(__ballot(newD && !inD), ntd, dv);
                // every entry's place among the others
                const unsigned long long stay = below(lp.cnt) & ~gone, mS = __ballot(inS), mD = __ballot(inD);
                const bool st = (stay >> lane) & 1ULL;
                int at = (int)__popcll(stay & below(lane)), atS = 0, atD = 0;
                for (int w = 0; w < 2; w++)
                    for (unsigned long long h = w ? mD : mS; h; h &= h - 1) {
                        const int l = (int)__builtin_ctzll(h);
                        const double tq = rl_d(w ? ntd : ntv, l);
                        const int vq = rl_i(w ? dv : sv, l);
                        const int less = (int)__popcll(__ballot(st & before(lp.ft, lp.fv, tq, vq)));
                        at += before(tq, vq, lp.ft, lp.fv) ? 1 : 0;
                        atS += before(tq, vq, ntv, sv) ? 1 : 0;
                        atD += before(tq, vq, ntd, dv) ? 1 : 0;
                        if (lane == l) {
                            if (w) atD += less;
                            else atS += less;
                        }
                    }
                if (st) { L.ht[at] = lp.ft; L.hv[at] = lp.fv; }
                if (inS) { L.ht[atS] = ntv; L.hv[atS] = sv; }
                if (inD) { L.ht[atD] = ntd; L.hv[atD] = dv; }
                const int total = (int)__popcll(stay) + (int)__popcll(mS) + (int)__popcll(mD);
                sync_wave();
                lp.cnt = min(total, WAVE);
                lp.ft = lane < lp.cnt ? L.ht[lane] : inf;
                lp.fv = lane < lp.cnt ? L.hv[lane] : INT_MAX;
                if (total > WAVE) {
                    // the horizon moves back to the last that has a lane
                    lp.tau_t = rl_d(lp.ft, WAVE - 1);
                    lp.tau_v = rl_i(lp.fv, WAVE - 1);
                    for (int c0 = WAVE; c0 < total; c0 += WAVE) {
                        const bool mine = c0 + lane < total;
                        lp.put(__ballot(mine), mine ? L.ht[c0 + lane] : inf, mine ? L.hv[c0 + lane] : 0);
                    }
                }
            }
            sync_wave();
            if (ALONE && kept < lone_at) {
                more = true;
                break;
            }
        }
        } while (ALONE && more);
        if (err) { q.err_step = stp; break; }
    }
    if (!err)
        while (ks < a.n_snap) snapshot_counts(lp.xx, snap_xx, snap_tot, nsS, S, ks++, L.tot, lane);
    // the bounds back for the next launch, the front's entries folded in
    if (lane < lp.cnt) lp.lower(lp.fv, lp.ft);
    lp.give_back();
    if (lane == 0) L.scan->stop = 1;
    sync_wave();
    if (lp.waves > 1) __syncthreads();
    for (int i = lane; i < lp.nn; i += WAVE) tmin[i] = L.lb[i];
    q.rng_pos = lp.pos;
    if (err) q.err = err;
    if (lane == 0) *qs_ = q;
}

template <int MS, int MR, bool VM, bool ALONE>
__global__ void __launch_bounds__(WAVE * WAVES) k_ssa(RdmeArgs a) {
    ssa_run<MS, MR, VM, ALONE>(a, blockIdx.x);
}

// Ensembles of different models: workgroup g runs the trajectory described
// by args[g] (its own domain, chemistry, queue and stream).
template <int MS, int MR, bool VM, bool ALONE>
__global__ void __launch_bounds__(WAVE * WAVES) k_ssa_multi(const RdmeArgs *__restrict__ args) {
    ssa_run<MS, MR, VM, ALONE>(args[blockIdx.x], 0);
}

// The per-lane tables are sized for 2, 4, 8 or 16 species and reactions (8 or
// 16 with custom propensities): the code of a round grows with them, and a
// round should stay in the instruction cache.
template <class F> static void by_size(bool vm, int m, F f) {
    if (vm) {
        if (m <= 8) f(std::integral_constant<int, 8>{}, std::true_type{});
        else f(std::integral_constant<int, 16>{}, std::true_type{});
    } else if (m <= 2) f(std::integral_constant<int, 2>{}, std::false_type{});
    else if (m <= 4) f(std::integral_constant<int, 4>{}, std::false_type{});
    else if (m <= 8) f(std::integral_constant<int, 8>{}, std::false_type{});
    else f(std::integral_constant<int, 16>{}, std::false_type{});
}

template <class K> static void allow_lds(K kernel, size_t lds) {
    if (lds > 65536)
        HIP_OK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
}

// Wavefronts per trajectory: they share the scans of the nodes (a 40^3
// lattice's trajectory 235 -> 173 ms with four instead of one, the 1M
// cylinder's event loop 93 -> 49 ms per 100 steps), as long as every
// trajectory still has a CU of its own; beyond that the extra wavefronts
// would only take the registers of other trajectories.
static int threads_for(int n_traj) { return n_traj <= 256 ? WAVE * WAVES : WAVE; }

// Whether a launch may take events alone: in domains of so few voxels that most
// rounds keep fewer than they cost, and where that few voxels have a next event.
// The lines (rounds / both ways, ms): up to 2 species and reactions, 16 voxels
// 87.5 / 82.1, 25 voxels 71.5 / 74.2; up to 4, 25 voxels 60.2 / 52.0, 36 voxels
// 57.1 / 57.8; up to 8, 64 voxels 76.1 / 60.8, 100 voxels 54.8 / 54.5, 144 voxels
// 26.7 / 27.8; 16, 256 voxels 80.5 / 70.3, 400 voxels 100.8 / 100.6.  20,000
// molecules in one of 3,600 voxels: 12.1 / 9.5.  Past them the kernel that only
// knows rounds is 2% faster.  Custom propensities: 6 of them, 4 voxels 3.5 / 2.7,
// 9 voxels 3.6 / 3.1 or, with exp and pow in them, 3.4 / 3.8; 8, 64 voxels 10.2 /
// 9.4, 144 voxels 19.7 / 17.0; 16, 16 voxels 16.4 / 5.3, 256 voxels 99 / 68, 576
// voxels 171 / 168.
bool nsm_alone(int n, int S, int R, bool vm, long long active) {
    const int m = S > R ? S : R;
    if (vm) return n <= (R <= 6 ? 4 : R <= 8 ? 150 : 300) || active <= 8;
    return n <= (m <= 2 ? 20 : m <= 4 ? 32 : m <= 8 ? 100 : 256) || active <= 8;
}

void rdme_take_step(hipStream_t s, const RdmeArgs &a, int n_traj) {
    by_size(a.vm_ncode > 0, a.S > a.R ? a.S : a.R, [&](auto m, auto vm) {
        constexpr int M = decltype(m)::value;
        constexpr bool V = decltype(vm)::value;
        auto launch = [&](auto kernel) {
            allow_lds(kernel, a.lds_bytes);
            hipLaunchKernelGGL(kernel, dim3(n_traj), dim3(threads_for(n_traj)), a.lds_bytes, s, a);
        };
        if (a.alone) launch(k_ssa<M, M, V, true>);
        else launch(k_ssa<M, M, V, false>);
    });
}

void rdme_take_step_multi(hipStream_t s, const RdmeArgs *d_args, int n_models, int max_sr, size_t lds, bool any_prog,
                          bool alone) {
    by_size(any_prog, max_sr, [&](auto m, auto vm) {
        constexpr int M = decltype(m)::value;
        constexpr bool V = decltype(vm)::value;
        auto launch = [&](auto kernel) {
            allow_lds(kernel, lds);
            hipLaunchKernelGGL(kernel, dim3(n_models), dim3(threads_for(n_models)), lds, s, d_args);
        };
        if (alone) launch(k_ssa_multi<M, M, V, true>);
        else launch(k_ssa_multi<M, M, V, false>);
    });
}

}  // namespace ssa
