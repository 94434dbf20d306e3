// SDPD substeps on gfx950: one thread per particle, neighbour lists read from
// the ELL layout (coalesced across threads at each list position).
//
//   sdpd_predict  take_step1     (ENG/src/simulate.cpp:56-109) + NaN check
//                                (ENG/src/particle.cpp:88-134)
//   sdpd_forces   pairwiseForce  (ENG/src/model.cpp:39-191)
//   sdpd_correct  take_step2 corrector + filterDensity (simulate.cpp:136-155,
//                                model.cpp:194-233)
//   sdpd_bvf      computeBoundaryVolumeFraction + applyBoundaryVolumeFraction
//                 + chem half step + boundary conditions (simulate.cpp:158-171,
//                 model.cpp:236-329)
//
// Neighbour rho inside the boundary volume fraction is read after every
// particle's density update of the same substep (snapshot order); the
// reference with one thread reads it in index order (model.cpp:285-293).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "engine.hpp"
#include "vm.hpp"

namespace ssa {

__device__ __forceinline__ void apply_bcs(const SdpdArgs &a, int i) {
    // generated applyBoundaryConditions (core/boundarycondition.py:121-167)
    for (int b = 0; b < a.nbc; b++) {
        const BcRule &r = a.bc[b];
        double x0 = a.x[i], x1 = a.x[(size_t)a.n + i], x2 = a.x[2 * (size_t)a.n + i];
        if (!((x0 >= r.lo[0]) && (x0 <= r.hi[0]) && (x1 >= r.lo[1]) && (x1 <= r.hi[1]) && (x2 >= r.lo[2]) &&
              (x2 <= r.hi[2])))
            continue;
        if (r.type >= 0 && a.type[i] != r.type) continue;
        switch (r.target) {
        case SSASDPD_BC_CHEM:
            if (r.species < a.Sc) a.C[(size_t)i * a.Sc + r.species] = r.value[0];
            break;
        case SSASDPD_BC_V:
            for (int k = 0; k < 3; k++) a.v[(size_t)k * a.n + i] = r.value[k];
            break;
        case SSASDPD_BC_NU: a.nu[i] = r.value[0]; break;
        case SSASDPD_BC_RHO: a.rho[i] = r.value[0]; break;
        }
    }
}

constexpr int MAXSC = 16;         // deterministic species the pair kernel sums

__device__ __forceinline__ bool bad(double x) { return isnan(x) || !isfinite(x); }

// Particle i's gather record from the arrays (eight 16-byte stores).
__device__ __forceinline__ void store_rec_to(const SdpdArgs &a, int i, double2 *p) {
    const size_t n = a.n;
    p[0] = make_double2(a.x[i], a.x[n + i]);
    p[1] = make_double2(a.x[2 * n + i], a.v[i]);
    p[2] = make_double2(a.v[n + i], a.v[2 * n + i]);
    p[3] = make_double2(a.vt[i], a.vt[n + i]);
    p[4] = make_double2(a.vt[2 * n + i], a.nu[i]);
    p[5] = make_double2(a.rho[i], a.mass[i]);
    ((int4 *)p)[6] = make_int4(a.type[i], a.solid[i], 0, 0);
    // what every pair with this particle as j forms from j alone, by the
    // same operations as the pair loop: P_j / rho_j^2 and m_j / rho_j
    const double rho = a.rho[i], P = a.P0 * (rho / a.rho0 - 1.0);
    p[7] = make_double2(P / (rho * rho), a.mass[i] / rho);
}
__device__ __forceinline__ void store_rec(const SdpdArgs &a, int i) { store_rec_to(a, i, (double2 *)(a.rec + i)); }

__device__ __forceinline__ double2 load_rho_mass(const PRec *r) { return *(const double2 *)&r->rho; }

__global__ void k_pack(SdpdArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    int i = chunk * blockDim.x + threadIdx.x;
    if (i < a.n) store_rec(a, i);
}

__device__ __forceinline__ void predict_one(const SdpdArgs &a, int i, double2 *rec_out) {
    const size_t n = a.n;
    bool nan = bad(a.rho[i]);
    for (int k = 0; k < 3; k++) nan = nan || bad(a.x[k * n + i]) || bad(a.v[k * n + i]);
    if (nan) {
        atomicCAS(&a.err->code, 0, (int)SSASDPD_ERR_NAN_STATE);
        atomicMin(&a.err->particle, i);
    }
    if (a.solid[i] == 0 && a.static_domain == 0) {
        for (int k = 0; k < 3; k++) {
            double v = a.v[k * n + i] + 0.5 * a.dt * a.F[k * n + i];
            double vt = v + 0.5 * a.dt * a.Fbp[k * n + i];
            a.v[k * n + i] = v;
            a.vt[k * n + i] = vt;
            a.x[k * n + i] = a.x[k * n + i] + a.dt * vt;
        }
        a.rho[i] = a.rho[i] + 0.5 * a.dt * a.Frho[i];
    }
    if (a.step > 0)
        for (int s = 0; s < a.Sc; s++) a.C[(size_t)i * a.Sc + s] += a.Q[(size_t)i * a.Sc + s] * a.dt * 0.5;
    apply_bcs(a, i);
    // F, Fbp, Frho and Q start anew here (simulate.cpp:92-105); k_forces, which
    // every step runs next, starts its sums from those values and stores all
    // that it sums, so only the others are stored here (a million moving
    // particles with 3 species: 80 of 560 MB, 125 -> 107 us)
    if (a.static_domain) {
        for (int k = 0; k < 3; k++) {
            a.F[k * n + i] = a.g[k];
            a.Fbp[k * n + i] = 0.0;
        }
        a.Frho[i] = 0.0;
    }
    for (int s = MAXSC; s < a.Sc; s++) a.Q[(size_t)i * a.Sc + s] = 0.0;
    a.old_rho[i] = a.rho[i];
    store_rec_to(a, i, rec_out);
}

// The gather records are staged in LDS and written as one contiguous range
// per block (a lane storing its own 128-byte record writes 16 bytes to each
// of 64 lines per instruction).
__global__ void __launch_bounds__(256) k_predict(SdpdArgs a) {
    __shared__ double2 srec[256 * 8];
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    const int base = chunk * 256;
    const int i = base + threadIdx.x;
    if (i < a.n) predict_one(a, i, srec + 8 * threadIdx.x);
    __syncthreads();
    const int nrec = min(256, a.n - base);
    double2 *dst = (double2 *)(a.rec + base);
    for (int q = threadIdx.x; q < nrec * 8; q += 256) dst[q] = srec[q];
}

// The model's tables are the same for all lanes and never written by a kernel:
// read through the constant address space they take scalar loads, also behind
// a kernel's stores.
__device__ __forceinline__ int tab_int(const int *p) { return *(const __attribute__((address_space(4))) int *)p; }
__device__ __forceinline__ Rxn tab_rxn(const Rxn *p) {
    Rxn r;
    constexpr int N = sizeof(Rxn) / 4;
    static_assert(sizeof(Rxn) % 4 == 0, "");
    int w[N];
#pragma unroll
    for (int k = 0; k < N; k++) w[k] = ((const __attribute__((address_space(4))) int *)p)[k];
    __builtin_memcpy(&r, w, sizeof r);
    return r;
}

// generated det<name> functions (solver.py:160-190), called with
// vol = mass/rho and t = current_step*dt (model.cpp:181-184); VM: kind-4
// rows through the expression VM (only k_chem instantiates it)
template <bool VM>
__device__ __forceinline__ double chem_rhs(const SdpdArgs &a, int i, int r) {
    const Rxn re = tab_rxn(a.rx + r);
    if (re.mask && !((re.mask >> a.type[i]) & 1ULL)) return 0.0;
    const double *c = a.C + (size_t)i * a.Sc;
    if constexpr (VM) {
        if (re.kind == 4)
            return vm_eval_f64(a.vm_code, re.b, a.vm_k, c, a.mass[i] / a.rho[i], (double)a.step * a.dt,
                               a.data_fn ? a.data_fn + (size_t)i * a.n_df : nullptr);
    }
    switch (re.kind) {
    case 0: return re.k;
    case 1: return re.k * c[re.a];
    case 2: return (re.k * c[re.a]) * c[re.b];
    default: return (re.k * c[re.a]) * c[re.a];
    }
}

// The particle this thread takes: the block's 256 particles in ascending order
// of their degree.  A wavefront walks its lists as far as the longest of them,
// 15 entries at 8.9 neighbours on average; with like degrees together the mean
// over a block's four wavefronts is 8 to 10.  (Which thread takes a particle
// decides nothing about its sums.)  Places past n count as degree 0.
__device__ __forceinline__ int by_degree(const SdpdArgs &a, int base) {
    constexpr int BINS = WAVE;
    __shared__ int bin[BINS], order[256];
    const int t = threadIdx.x;
    if (t < BINS) bin[t] = 0;
    __syncthreads();
    const int k = base + t < a.n ? min(a.deg[base + t], BINS - 1) : 0;
    const int at = atomicAdd(bin + k, 1);
    __syncthreads();
    if (t < BINS) {
        const int c = bin[t];
        int x = c;
        for (int o = 1; o < WAVE; o <<= 1) {
            const int y = __shfl_up(x, o, WAVE);
            if (t >= o) x += y;
        }
        bin[t] = x - c;
    }
    __syncthreads();
    order[bin[k] + at] = t;
    __syncthreads();
    return base + order[t];
}

// 16 bytes per lane from global memory straight to LDS, lane l's at dst + 16 l
// (no registers in between); dst is the same in every lane.
__device__ __forceinline__ void to_lds16(const void *src, void *dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t *)src,
                                     (__attribute__((address_space(3))) uint32_t *)dst, 16, 0, 0);
}

// pairwiseForce (model.cpp:39-191), list order.  Real = double is the
// reference's arithmetic operation for operation; Real = float evaluates the
// pair terms (kernel gradient, pressure, viscosity, background pressure,
// transport tensor, continuity) in FP32 from FP64-formed differences dx, dv
// and sums them into FP64 accumulators.  The species flux Q stays FP64.  For
// static domains only Q is observable, so the momentum part is left out.
// CHEM: the reaction fluxes are added here; otherwise k_chem adds them
// afterwards (models with custom deterministic rates), to the same Q in the
// same order.
// NSC: room for the sums of that many deterministic species (the fields of the
// first four are loaded an entry ahead).
//
// A lane sums its particle's list in order.  What bounds it is the FP64
// arithmetic of two wavefronts per SIMD (204 registers: 350 FP64 instructions
// an entry, 60% of the time at a million particles).  Three things kept it from
// that: the longest list of a wavefront (see by_degree); 40 divisions by 8
// different divisors (see Den); and the neighbours' records, one 128-byte line
// each and 7 loads apiece, whose 64 lines per wavefront pushed each other out
// of the 32 KB L1 between one load and the next (2.1 lines from L2 for each
// record) and made every entry wait for its own gather.  Now eight lanes fetch
// a record together, a line each time, straight to LDS, while the entry before
// it is computed; piece c of record r stands at place c ^ (r & 7) of it, so
// that 64 lanes reading one piece of their own records use all banks.
// Measured (cylinder, FP64, 3 species): 0.53 -> 0.32 ms at 1,000,000
// particles, 51 -> 37 us at 64,000.  Also tried, and slower: a lane per pair
// with the terms summed through LDS (0.49 to 0.64 ms: the sums and the search
// for a slot's particle cost more instructions than the idle lanes), and list
// entries loaded two ahead (0.33 ms).
template <typename Real, bool MOMENTUM, bool CHEM, int NSC>
__global__ void __launch_bounds__(256) k_forces(SdpdArgs a) {
    constexpr int NR = MOMENTUM ? 256 : 1;
    __shared__ __align__(16) char s_rec[NR * sizeof(PRec)];
    static_assert(__alignof__(s_rec) >= 16, "to_lds16 writes and double2 reads 16 bytes at a time");
    __shared__ int s_j[NR];
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    const int i = by_degree(a, chunk * 256);
    const bool mine = i < a.n;
    const size_t n = a.n, ii = mine ? i : 0;
    const double h = a.h;
    const Real hR = (Real)a.h, P0 = (Real)a.P0, rho0 = (Real)a.rho0, alpha = (Real)a.alpha;
    const double xi[3] = {a.x[ii], a.x[n + ii], a.x[2 * n + ii]};
    const double vi[3] = {a.v[ii], a.v[n + ii], a.v[2 * n + ii]};
    const double vti[3] = {a.vt[ii], a.vt[n + ii], a.vt[2 * n + ii]};
    const Real viR[3] = {(Real)vi[0], (Real)vi[1], (Real)vi[2]};
    const Real dvti[3] = {(Real)(vi[0] - vti[0]), (Real)(vi[1] - vti[1]), (Real)(vi[2] - vti[2])};
    const double rhoid = a.rho[ii], mid = a.mass[ii];
    const Real rhoi = (Real)rhoid, mi = (Real)mid, nui = (Real)a.nu[ii];
    const Real Pi = P0 * (rhoi / rho0 - (Real)1.0);
    // the sums start where the predictor resets them (F = g, Fbp, Frho and
    // Q = 0: simulate.cpp:92-105), not from the arrays, so a second launch
    // on the same lists (after a re-search) gives the same result
    double F[3] = {a.g[0], a.g[1], a.g[2]};
    double Fbp[3] = {0.0, 0.0, 0.0};
    double Frho = 0.0;
    constexpr bool SPECIES = NSC > 0;
    constexpr int NS = SPECIES ? NSC : 1;
    const int Sc = SPECIES ? min(a.Sc, NSC) : 0;
    constexpr int NE = NS < 4 ? NS : 4;      // species whose fields are loaded ahead
    double Q[NS], Ci[NE], Di[NE], Cj[NE];
    const int ti = a.type[ii];
    auto diffusion = [&](int s) {
        const long long kk = (long long)a.Sc * (ti - 1) + s;   // type-major, model.cpp:163
        return (kk < (long long)a.Sc * a.T) ? a.Dmat[kk] : 0.0;
    };
    for (int s = 0; s < NS; s++) Q[s] = 0.0;
#pragma unroll
    for (int s = 0; s < NE; s++) {
        Ci[s] = Di[s] = Cj[s] = 0.0;
        if (s < Sc) {
            Di[s] = diffusion(s);
            Ci[s] = a.C[ii * a.Sc + s];
        }
    }
    const int dg = mine ? a.deg[ii] : 0;
    const Den<Real> by_h(hR), by_hh(hR * hR);
    const Den<double> by_hd(h), by_hhd(h * h);
    const Real Pi_r = Pi / (rhoi * rhoi), inv_mi = (Real)1.0 / mi;

    int longest = dg;
    for (int o = 1; o < WAVE; o <<= 1) longest = max(longest, __shfl_xor(longest, o, WAVE));
    longest = __builtin_amdgcn_readfirstlane(longest);
    const int t = threadIdx.x & (WAVE - 1), wave = threadIdx.x & ~(WAVE - 1);
    char *const recs = s_rec + (MOMENTUM ? wave * (int)sizeof(PRec) : 0);
    int *const jrec = s_j + (MOMENTUM ? wave : 0);
    // entry k of the lane's list: the particle and its distance (places past
    // the end: the lane's own particle, which is skipped)
    int j1 = 0;
    double rd1 = 0.0;
    auto entry = [&](int k) {
        const size_t e = (size_t)k * n + ii;
        j1 = k < dg ? a.nidx[e] : (int)ii;
        rd1 = k < dg ? a.nr[e] : 0.0;
    };
    // the record of j1, without waiting for it
    double2 rm = make_double2(1.0, 1.0);
    const int piece = ((t & 7) ^ (t >> 3)) * 16;
    auto gather = [&]() {
        if constexpr (MOMENTUM) {
            jrec[(t & 7) * 8 + (t >> 3)] = j1;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            int jr[8];
#pragma unroll
            for (int u = 0; u < 8; u++) jr[u] = jrec[(t >> 3) * 8 + u];
#pragma unroll
            for (int u = 0; u < 8; u++) to_lds16((const char *)(a.rec + jr[u]) + piece, recs + u * 1024);
        } else {
            rm = load_rho_mass(a.rec + j1);
        }
#pragma unroll
        for (int s = 0; s < NE; s++)
            if (s < Sc) Cj[s] = a.C[(size_t)j1 * a.Sc + s];
    };
    if (longest > 0) {
        entry(0);
        gather();
    }
    Real dx[3] = {0, 0, 0}, dv[3] = {0, 0, 0};
    for (int k = 0; k < longest; k++) {
        const double rd = rd1;
        const int j = j1;
        double xj[3], vj[3], vtj[3], nujd, rhojd, mjd, dC[NE];
        double2 pmj = make_double2(0.0, 0.0);
        if constexpr (MOMENTUM) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            auto at = [&](int u) { return *(const double2 *)(recs + t * 128 + ((u ^ (t & 7)) * 16)); };
            const double2 a0 = at(0), a1 = at(1), a2 = at(2), a3 = at(3), a4 = at(4), a5 = at(5);
            pmj = at(7);
            xj[0] = a0.x; xj[1] = a0.y; xj[2] = a1.x;
            vj[0] = a1.y; vj[1] = a2.x; vj[2] = a2.y;
            vtj[0] = a3.x; vtj[1] = a3.y; vtj[2] = a4.x;
            nujd = a4.y; rhojd = a5.x; mjd = a5.y;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
            rhojd = rm.x;
            mjd = rm.y;
        }
#pragma unroll
        for (int s = 0; s < NE; s++) dC[s] = Ci[s] - Cj[s];
        if (k + 1 < longest) {
            entry(k + 1);
            gather();
        }
        const double Rd = by_hd.div(rd);
        if (Rd > 1.0) continue;
        if (rd == 0.0) continue;
        const Real r = (Real)rd;
        const Real R = by_h.div(r);
        const Real dWdr = alpha * by_hh.div((Real)-12 * r) * (((Real)1 - R) * ((Real)1 - R));
        const Real rhoj = (Real)rhojd, mj = (Real)mjd;
        const Den<Real> by_rh(r + (Real)0.001 * hR), by_rr(rhoi * rhoj);
        const Real inv_rh = by_rh.div((Real)1.0);
        if constexpr (MOMENTUM) {
            const Real nuj = (Real)nujd;
            Real dv_dx = 0;
            for (int d = 0; d < a.dim; d++) {
                dx[d] = (Real)(xi[d] - xj[d]);
                dv[d] = (Real)(vi[d] - vj[d]);
                dv_dx += dv[d] * dx[d];
            }
            const Real vjR[3] = {(Real)vj[0], (Real)vj[1], (Real)vj[2]};
            const Real dvtj[3] = {(Real)(vj[0] - vtj[0]), (Real)(vj[1] - vtj[1]), (Real)(vj[2] - vtj[2])};
            // P_j / rho_j^2 and m_j / rho_j from the record: the same
            // operations on the same values as here, done once per particle
            const Real Pj_r = (Real)pmj.x, mrj = (Real)pmj.y;
            Real pg = Pi_r + Pj_r;
            if (pg < 0) pg = -Pi_r + Pj_r;
            const Real fp = by_rh.div((Real)-1.0 * mj * pg * dWdr);
            const Real fv = by_rr.div(mj * Den<Real>(nui + nuj).div((Real)2.0 * (nui * nuj)) * inv_rh * dWdr);
            const Real mri = mi / rhoi;
            const Real vsum = mri * mri + mrj * mrj;
            const Real fbp = by_rh.div((Real)-10.0 * P0 * inv_mi * vsum * dWdr);
            Real ft[3];
            for (int p = 0; p < 3; p++) {
                Real acc = 0;
                Real Tp[3];
                for (int q = 0; q < 3; q++)
                    Tp[q] = (Real)0.5 * ((rhoi * viR[p] * (-dvti[q])) + (rhoj * vjR[p] * (-dvtj[q])));
                acc = Tp[0] * dx[0] + Tp[1] * dx[1] + Tp[2] * dx[2];
                ft[p] = by_rh.div(inv_mi * vsum * acc * dWdr);
            }
            for (int d = 0; d < a.dim; d++) {
                if (!a.skip_F) F[d] += (double)(fp * dx[d] + fv * dv[d] + ft[d]);
                Fbp[d] += (double)(fbp * dx[d]);
            }
            // model.cpp:143-146; its middle term (density diffusion) is
            // multiplied by 0.0 there: for finite states it adds a signed
            // zero, which leaves the sum (which starts at +0) unchanged, so
            // it is not formed
            Frho = Frho + (double)(rhoi * mrj * dv_dx * inv_rh * dWdr -
                                   mrj *
                                       (rhoi * (dvti[0] * dx[0] + dvti[1] * dx[1] + dvti[2] * dx[2]) +
                                        rhoj * (dvtj[0] * dx[0] + dvtj[1] * dx[1] + dvtj[2] * dx[2])) *
                                       inv_rh * dWdr);
        }
        if constexpr (SPECIES) {
            const double dWdrd = a.alpha * by_hhd.div(-12 * rd) * ((1 - Rd) * (1 - Rd));
            double inv_rhd, rsum;
            if constexpr (sizeof(Real) == 8) {
                inv_rhd = inv_rh;
                rsum = by_rr.div(rhoid + rhojd);
                if (rsum != rsum) rsum = (rhoid + rhojd) / (rhoid * rhojd);   // a density of 0
            } else {
                inv_rhd = Den<double>(rd + 0.001 * h).div(1.0);
                rsum = (rhoid + rhojd) / (rhoid * rhojd);
            }
            const double wfd = inv_rhd * dWdrd;
            const double dQc_base = Den<double>((rd * rd) + 0.01 * h * h)
                                        .div(2.0 * Den<double>(mid + mjd).div(mid * mjd) * rsum * (rd * rd) * wfd);
#pragma unroll
            for (int s = 0; s < NE; s++)
                if (s < Sc) Q[s] += Di[s] * dC[s] * dQc_base;
            for (int s = NE; s < Sc; s++)
                Q[s] += diffusion(s) * (a.C[ii * a.Sc + s] - a.C[(size_t)j * a.Sc + s]) * dQc_base;
        }
    }
    if (!mine) return;
    if constexpr (CHEM) {
        for (int r = 0; r < a.Rc; r++) {
            const double flux = chem_rhs<false>(a, i, r);
#pragma unroll
            for (int s = 0; s < NS; s++)
                if (s < Sc) {
                    const long long kk = (long long)a.Rc * r + s;             // model.cpp:186
                    const int nk = kk < (long long)a.Sc * a.Rc ? tab_int(a.Ndense + kk) : 0;
                    Q[s] += nk * flux;
                }
        }
    }
    if constexpr (MOMENTUM) {
        for (int d = 0; d < 3; d++) { a.F[d * n + i] = F[d]; a.Fbp[d * n + i] = Fbp[d]; }
        a.Frho[i] = Frho;
    }
#pragma unroll
    for (int s = 0; s < NS; s++)
        if (s < Sc) a.Q[(size_t)i * a.Sc + s] = Q[s];
}

__device__ __forceinline__ double cube(double x) { return x * x * x; }

__global__ void k_correct(SdpdArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    int i = chunk * blockDim.x + threadIdx.x;
    if (i >= a.n || a.static_domain) return;
    const size_t n = a.n;
    const bool filt = (a.step % 20) == 0;
    auto filter = [&]() {
        // filterDensity (model.cpp:194-233): no self term
        const double h = a.h;
        double num = 0.0, den = 0.0;
        const int dg = a.deg[i];
        for (int k = 0; k < dg; k++) {
            const size_t e = (size_t)k * n + i;
            const double r = a.nr[e], R = r / h;
            if (R > 1.0) continue;
            if (r == 0.0) continue;
            const double W = a.alpha * ((1 + 3 * R) * cube(1 - R));
            num += a.rec[a.nidx[e]].rho * W;     // old_rho of j (the record is written with it)
            den += W;
        }
        a.rho[i] = num / den;
    };
    if (a.solid[i] == 0) {
        for (int k = 0; k < 3; k++) a.v[k * n + i] = a.v[k * n + i] + 0.5 * a.dt * a.F[k * n + i];
        if (filt) filter();
        a.rho[i] = a.rho[i] + 0.5 * a.dt * a.Frho[i];
    } else if (a.solid[i] == 1) {
        if (filt) filter();
    }
}

__device__ __forceinline__ void bvf_one(const SdpdArgs &a, int i) {
    const size_t n = a.n;
    if (a.solid[i] == 0 && a.static_domain == 0) {
        const double h = a.h;
        double vos = 0.0, vtot = 0.0, nw[3] = {0.0, 0.0, 0.0}, dx[3] = {0.0, 0.0, 0.0};
        for (int d = 0; d < a.dim; d++) { a.normal[d * n + i] = 0.0; a.vt[d * n + i] = 0.0; }
        const double xi[3] = {a.x[i], a.x[n + i], a.x[2 * n + i]};
        const int dg = a.deg[i];
        if (a.no_solids) {
            // no solid neighbour: vos and nw stay 0, so phi = |0 / vtot| is 0
            // when some neighbour has W > 0 (0 < r < h, every (m/rho)^2 > 0)
            // and 0/0 = NaN otherwise; the normal is -0/0 = NaN and the
            // velocity is never reflected (phi >= 0.5 is false for both)
            bool pos = false;
            for (int k = 0; k < dg && !pos; k++) {
                const double r = a.nr[(size_t)k * n + i], R = r / h;
                pos = !(R > 1.0) && r != 0.0 && (1 + 3 * R) * cube(1 - R) > 0.0;
            }
            const double qnan = __longlong_as_double(0x7ff8000000000000LL);
            for (int d = 0; d < 3; d++) a.normal[d * n + i] = -qnan;
            a.bvf[i] = pos ? 0.0 : qnan;
            for (int s = 0; s < a.Sc; s++) a.C[(size_t)i * a.Sc + s] += a.Q[(size_t)i * a.Sc + s] * a.dt * 0.5;
            apply_bcs(a, i);
            return;
        }
        for (int k = 0; k < dg; k++) {
            const size_t e = (size_t)k * n + i;
            const int j = a.nidx[e];
            const double r = a.nr[e], R = r / h;
            if (R > 1.0) continue;
            if (r == 0.0) continue;
            const double W = a.alpha * ((1 + 3 * R) * cube(1 - R));
            const double dWdr = a.alpha * (-12 * r / (h * h)) * ((1 - R) * (1 - R));
            // x, mass and solid of j from its record (unchanged since the
            // predictor); rho[j] after the corrector from the array
            const PRec *pj = a.rec + j;
            const double2 x01 = *(const double2 *)&pj->x[0];
            const double xj[3] = {x01.x, x01.y, pj->x[2]};
            for (int d = 0; d < a.dim; d++) dx[d] = xi[d] - xj[d];
            const double mr = pj->mass / a.rho[j];
            const double mv = mr * mr;
            const bool sj = pj->solid != 0;
            if (sj) vos += mv * W;
            vtot += mv * W;
            if (sj)
                for (int d = 0; d < 3; d++) nw[d] += mv * dx[d] * dWdr / (r + 0.001 * h);
        }
        for (int d = 0; d < 3; d++) nw[d] = nw[d] / vtot;
        const double nn = sqrt(nw[0] * nw[0] + nw[1] * nw[1] + nw[2] * nw[2]);
        double nm[3];
        for (int d = 0; d < 3; d++) { nm[d] = -nw[d] / nn; a.normal[d * n + i] = nm[d]; }
        const double phi = fabs(vos / vtot);
        a.bvf[i] = phi;
        double v[3] = {a.v[i], a.v[n + i], a.v[2 * n + i]};
        const double vdn = v[0] * nm[0] + v[1] * nm[1] + v[2] * nm[2];
        if (phi >= 0.5)
            for (int d = 0; d < a.dim; d++) a.v[d * n + i] = -v[d] + 2.0 * fmax(0.0, vdn) * nm[d];
    }
    for (int s = 0; s < a.Sc; s++) a.C[(size_t)i * a.Sc + s] += a.Q[(size_t)i * a.Sc + s] * a.dt * 0.5;
    apply_bcs(a, i);
}
// The BVF, the corrector's species update and the BCs; then vol = mass/rho
// for the RDME of the step, from the final rho (the BCs may set it)
__global__ void k_bvf(SdpdArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    const int i = chunk * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    bvf_one(a, i);
    if (a.vol) a.vol[i] = a.mass[i] / a.rho[i];
}

static dim3 grid1(int n) { return xcd_grid((n + 255) / 256); }

void sdpd_predict(hipStream_t s, const SdpdArgs &a) { hipLaunchKernelGGL(k_predict, grid1(a.n), dim3(256), 0, s, a); }
// The reaction fluxes of models with custom deterministic rates
// (model.cpp:179-189), after k_forces has summed the pair fluxes into Q.
__global__ void __launch_bounds__(256) k_chem(SdpdArgs a) {
    const int chunk = xcd_chunk((a.n + 255) / 256);
    if (chunk < 0) return;
    const int i = chunk * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const int Sc = a.Sc;
    double *Q = a.Q + (size_t)i * Sc;
    for (int r = 0; r < a.Rc; r++) {
        const double flux = chem_rhs<true>(a, i, r);
        for (int s = 0; s < Sc; s++) {
            const long long kk = (long long)a.Rc * r + s;             // model.cpp:186
            const int nk = kk < (long long)a.Sc * a.Rc ? a.Ndense[kk] : 0;
            Q[s] += nk * flux;
        }
    }
}

template <bool CHEM, int NSC> static void forces_as(hipStream_t s, const SdpdArgs &a) {
    const dim3 g = grid1(a.n), b(256);
    if (a.static_domain) {
        if constexpr (NSC > 0) hipLaunchKernelGGL((k_forces<double, false, CHEM, NSC>), g, b, 0, s, a);
    } else if (a.fp32) {
        hipLaunchKernelGGL((k_forces<float, true, CHEM, NSC>), g, b, 0, s, a);
    } else {
        hipLaunchKernelGGL((k_forces<double, true, CHEM, NSC>), g, b, 0, s, a);
    }
}
void sdpd_forces(hipStream_t s, const SdpdArgs &a) {
    const bool vm = a.vm_code != nullptr && a.Rc > 0;
    if (a.Sc == 0) forces_as<false, 0>(s, a);
    else if (vm && a.Sc <= 4) forces_as<false, 4>(s, a);
    else if (vm) forces_as<false, MAXSC>(s, a);
    else if (a.Sc <= 4) forces_as<true, 4>(s, a);
    else forces_as<true, MAXSC>(s, a);
    if (vm && a.Sc > 0) hipLaunchKernelGGL(k_chem, grid1(a.n), dim3(256), 0, s, a);
}
void sdpd_correct(hipStream_t s, const SdpdArgs &a) {
    if (!a.static_domain) hipLaunchKernelGGL(k_correct, grid1(a.n), dim3(256), 0, s, a);
}
void sdpd_bvf(hipStream_t s, const SdpdArgs &a) { hipLaunchKernelGGL(k_bvf, grid1(a.n), dim3(256), 0, s, a); }
void sdpd_pack(hipStream_t s, const SdpdArgs &a) { hipLaunchKernelGGL(k_pack, grid1(a.n), dim3(256), 0, s, a); }


// Row permutation: gather dst[p][c] = src[map[p]][c], or scatter
// dst[map[p]][c] = src[p][c]; rows of `cols` elements of T.
template <class T>
__global__ void k_permute_rows(int n, int cols, const int *__restrict__ map, const T *__restrict__ src,
                               T *__restrict__ dst, int scatter) {
    const size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (e >= (size_t)n * cols) return;
    const int p = (int)(e / cols), c = (int)(e % cols);
    const size_t q = (size_t)map[p] * cols + c;
    if (scatter) dst[q] = src[e];
    else dst[e] = src[q];
}
void permute_rows(hipStream_t s, int n, int cols, int esz, const int *map, const void *src, void *dst, bool scatter) {
    if (n <= 0 || cols <= 0) return;
    const size_t m = (size_t)n * cols;
    const dim3 g((unsigned)((m + 255) / 256));
    if (esz == 8)
        hipLaunchKernelGGL(k_permute_rows<uint64_t>, g, dim3(256), 0, s, n, cols, map, (const uint64_t *)src,
                           (uint64_t *)dst, scatter ? 1 : 0);
    else
        hipLaunchKernelGGL(k_permute_rows<uint32_t>, g, dim3(256), 0, s, n, cols, map, (const uint32_t *)src,
                           (uint32_t *)dst, scatter ? 1 : 0);
}
}  // namespace ssa
