// sweep.h -- the schedule of the persistent workgroup-per-system kernels,
// shared by every storage mode.
//
// wg_drive runs one launch's worth of the reference's sweep loops on the
// system the workgroup owns: n plain sweeps, the whole schedule of an
// annealing temperature list, one segment of the parallel-tempering loop, or
// a chain of segments with the pairwise exchange after each.
// The per-site work comes from a "sweeper" object with the interface
//   int  n_sites()
//   void or_sweep(), det_sweep()               one coloured sweep
//   double metro(T, kind, sigma, ctr)          one Metropolis sweep, returns
//                                              the accepted count (all threads)
//   double metro_energy(T, kind, sigma, ctr, with_m, E, m)
//                              one Metropolis sweep, then the system's FP64
//                              energy E and, with_m, summed spin m, all in
//                              one workgroup reduction; returns the accepted
//                              count (all threads)
//   void magnet(double m[3])   FP64 summed spin, the same sums as metro_energy's
//   double *red                RED_BYTES of LDS scratch
//   bool leader()              this workgroup writes the system's shared
//                              results (false for all but one part of a
//                              system shared by several workgroups)
//   static constexpr bool LATE_EXCHANGE   resolve a chained exchange when its
//                              slot is next needed, not at once
// so each storage mode only provides its sweeps.
#pragma once
#include "device.h"
#include "kernels.h"

namespace csmc {

template <class R>
__device__ __forceinline__ const R *coef_of(const DevPools &P);
template <>
__device__ __forceinline__ const float *coef_of<float>(const DevPools &P) {
    return P.coefF;
}
template <>
__device__ __forceinline__ const double *coef_of<double>(const DevPools &P) {
    return P.coefD;
}

template <class R>
__device__ __forceinline__ spin4<double> to_d(const spin4<R> &s) {
    spin4<double> d;
    d.x = s.x;
    d.y = s.y;
    d.z = s.z;
    d.w = 0.0;
    return d;
}

// interaction field split by term kind (bilinear, cubic, quartic), FP64,
// for energies and gradients
template <bool GEN, bool SP = false, class NB, class LD>
__device__ __forceinline__ void field_parts(const LatView<double> &L, const NB &nb, int b, int i,
                                            LD &&ld, double F2[3], double F3[3], double F4[3]) {
    interaction_field<double, double, false>(L, nb, b, i, ld, F2);
    F3[0] = F3[1] = F3[2] = F4[0] = F4[1] = F4[2] = 0.0;
    if (!GEN) return;
    LatView<double> Lc = L;
    Lc.K2 = Lc.K2P = 0;
    Lc.K4 = 0;
    interaction_field<double, double, true, 0, 0, SP>(Lc, nb, b, i, ld, F3);
    LatView<double> Lq = L;
    Lq.K2 = Lq.K2P = 0;
    Lq.K3 = 0;
    interaction_field<double, double, true, 0, 0, SP>(Lq, nb, b, i, ld, F4);
}

// a value every lane holds, as a wave-uniform one: it then needs no vector
// register while it waits
__device__ __forceinline__ double uniform_d(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double combine_energy(const double p[5]) {
    // hamiltonian.jl:131
    return p[0] / 2 + p[1] / 3 + p[2] / 4 + p[3] + p[4];
}

// metropolis_adaptive! width update (metropolis.jl:129-131)
__device__ __forceinline__ double adapt_sigma(double sigma, double acc, double n) {
    double a = acc / n;
    double f = 0.5 / fmax(1.0 - a, 0.05);
    return fmin(fmax(sigma * f, 0.0), 100.0);
}

// one log-binning push (E or |M| with its square) into a slot's binner
__device__ __forceinline__ void bin_push(double *st, double v) {
    double c0 = v, c1 = v * v;
    for (int l = 0; l < BIN_LVLS; ++l) {
        double *q = st + l * 10;
        q[0] += 1.0;
        q[1] += c0;
        q[2] += c1;
        q[3] += c0 * c0;
        q[4] += c0 * c1;
        q[5] += c1 * c0;
        q[6] += c1 * c1;
        if (q[9] == 0.0) {
            q[7] = c0;
            q[8] = c1;
            q[9] = 1.0;
            return;
        }
        q[9] = 0.0;
        c0 = 0.5 * (q[7] + c0);
        c1 = 0.5 * (q[8] + c1);
    }
}

// Workgroup copy of n elements, get(i) -> put(i, v), with U independent
// loads in flight per thread (the index of each load is clamped to n - 1 so
// every load is unconditional; only the stores are guarded).
template <int U, class GET, class PUT>
__device__ __forceinline__ void wg_stage(int n, GET &&get, PUT &&put) {
    const int bd = (int)blockDim.x;
    for (int i0 = (int)threadIdx.x; i0 < n; i0 += U * bd) {
        decltype(get(0)) v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = get(min(i0 + u * bd, n - 1));
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * bd < n) put(i0 + u * bd, v[u]);
    }
}

// 64-bit words of (epoch << 32 | payload), each written and read as one
// relaxed device-scope atomic: a reader that sees the epoch it waits for sees
// that payload, with no fence or barrier between writer and reader.
__device__ __forceinline__ void ll_put(uint64_t *p, uint32_t v, uint32_t e) {
    __hip_atomic_store(p, ((uint64_t)e << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t ll_load(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the payload of word p once it carries epoch e (v: a first load of it); a
// wait that polls `limit` times, or sees another wait give up, sets *err and
// returns what it has, so every wave always reaches the end of the kernel
__device__ __forceinline__ uint32_t ll_wait(const uint64_t *p, uint64_t v, uint32_t e,
                                            uint32_t limit, uint32_t *err) {
    uint32_t n = 0;
    while ((uint32_t)(v >> 32) != e) {
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) break;
        if (++n > limit) {
            __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
        v = ll_load(p);
    }
    return (uint32_t)v;
}

__device__ __forceinline__ void ll_put_d(uint64_t *p, double v, uint32_t e) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    ll_put(p, (uint32_t)b, e);
    ll_put(p + 1, (uint32_t)(b >> 32), e);
}

__device__ __forceinline__ double ll_wait_d(const uint64_t *p, uint32_t e, uint32_t limit,
                                            uint32_t *err) {
    const uint64_t v0 = ll_load(p), v1 = ll_load(p + 1);
    const uint32_t lo = ll_wait(p, v0, e, limit, err), hi = ll_wait(p + 1, v1, e, limit, err);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The replica exchange (monte_carlo.jl:308-349) of a chained segment: the
// system in slot r publishes its energy and sigma for exchange xc = se / swap,
// waits for its partner slot's record (pairs (r, r+1) from 0 for an even xc,
// from 1 for an odd one) and decides its own pair: the same Philox draw and
// FP64 acceptance as the last-workgroup form, and both systems of a pair
// reach the same decision from the same two records.  Temperature labels
// move, spins stay.
// In two halves: exchange_publish right after the segment's last Metropolis
// sweep, exchange_resolve where the slot or its temperature is next needed
// (the next Metropolis sweep).  The overrelaxation sweeps between need
// neither, so the partner's record has arrived by then and nothing waits for
// it.  The partner slot's holder may by then have published two exchanges
// more; the ring of records holds them (PT_RECBUF).  Only the leader
// workgroup of a system publishes and counts.
__device__ __forceinline__ void exchange_publish(const WGArgs &a, int64_t se, int slot, double sigma, double E,
                                                 bool leader) {
    if (threadIdx.x == 0 && leader) {
        const PTDev &pt = a.pt;
        const uint32_t xc = (uint32_t)(se / pt.swap);
        uint64_t *rec = pt.rec + ((int64_t)pt_record_row(xc, pt.ring) * pt.R + slot) * 4;
        ll_put_d(rec, E, xc);
        ll_put_d(rec + 2, sigma, xc);
    }
}

// On return slot, sigma and T are those of the system's new slot.
// scratch: 3 doubles of LDS outside the reduction area.
__device__ __forceinline__ void exchange_resolve(const WGArgs &a, int64_t se, int &slot, double &sigma, double &T,
                                                 double E, double *scratch, bool leader) {
    if (threadIdx.x == 0) {
        const PTDev &pt = a.pt;
        const int R = pt.R, r = slot;
        const uint32_t xc = (uint32_t)(se / pt.swap), lim = a.spin_limit >> 4;
        uint64_t *rec = pt.rec + (int64_t)pt_record_row(xc, pt.ring) * R * 4;
        const int r0 = (xc % 2 == 0) ? 0 : 1;
        int lo = -1;
        if (r >= r0) lo = ((r - r0) % 2 == 0) ? r : r - 1;
        int ns = r;
        double nsig = sigma, nT = T;
        if (lo >= 0 && lo + 1 < R) {
            const int hi = lo + 1, p = (r == lo) ? hi : lo;
            const double Tp = pt.temps[p];
            const double Ep = ll_wait_d(rec + 4 * p, xc, lim, pt.err);
            const double sp = ll_wait_d(rec + 4 * p + 2, xc, lim, pt.err);
            const double E_lo = (r == lo) ? E : Ep, E_hi = (r == lo) ? Ep : E;
            const double T_lo = (r == lo) ? T : Tp, T_hi = (r == lo) ? Tp : T;
            uint4 rr = philox4x32_10(make_uint4((uint32_t)lo, 0xFFFFFFFFu, xc, TAG_EXCH), a.k0, a.k1);
            const double u = u01d(rr.x);
            const double dbeta = 1.0 / T_hi - 1.0 / T_lo;
            const double pacc = fmin(1.0, exp(dbeta * (E_hi - E_lo)));
            if (u < pacc) {
                ns = p;
                nsig = sp;
                nT = Tp;
                if (leader) __hip_atomic_fetch_add(pt.acc_exch + r, 1.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        scratch[0] = (double)ns;
        scratch[1] = nsig;
        scratch[2] = nT;
    }
    __syncthreads();
    slot = __builtin_amdgcn_readfirstlane((int)scratch[0]);
    sigma = uniform_d(scratch[1]);
    T = uniform_d(scratch[2]);
    __syncthreads();
}

template <int MODE, class SW>
__device__ __forceinline__ void wg_drive(const WGArgs &a, int sys, SW &sw) {
    uint32_t mctr = a.mcount[sys];
    auto metro_sweep = [&](double T, int kind, double &sigma) __attribute__((always_inline)) {
        double acc = sw.metro(T, kind, sigma, mctr);
        ++mctr;
        if (kind == CSMC_CONE_ADAPTIVE) sigma = adapt_sigma(sigma, acc, (double)sw.n_sites());
        return acc;
    };

    if constexpr (MODE == WG_SWEEPS || MODE >= WG_SWEEPS_OR) {
        const bool any = MODE == WG_SWEEPS;
        const double T = a.T_sys ? a.T_sys[sys] : 0.0;
        double sigma = a.sigma_sys ? a.sigma_sys[sys] : 60.0;
        double acc = 0.0;
        for (int s = 0; s < a.n_sweeps; ++s) {
            if (MODE == WG_SWEEPS_OR || (any && a.kind == CSMC_OVERRELAX)) sw.or_sweep();
            else if (MODE == WG_SWEEPS_DET || (any && a.kind == CSMC_DETERMINISTIC)) sw.det_sweep();
            else acc += metro_sweep(T, a.kind, sigma);
        }
        if (threadIdx.x == 0 && sw.leader()) {
            if (a.acc_sys) a.acc_sys[sys] = acc;
            if (a.T_keep) a.T_keep[sys] = T;
            if (a.sigma_sys) {
                a.sigma_out[sys] = sigma;
                if (a.sigma_keep) a.sigma_keep[sys] = sigma;
            }
        }
    } else if constexpr (MODE == WG_ANNEAL) {
        // simulated_annealing! (monte_carlo.jl:166-187), t = 1 .. t_th-1
        for (int k = 0; k < a.n_temps; ++k) {
            const double T = a.temps[k];
            double sigma = a.sigma0;
            double acc = 0.0;
            // a Metropolis sweep after every or_rate overrelaxation sweeps
            // (after none when or_rate == 0), the sweeps left over at the end
            for (int64_t t = 1; t < a.t_th;) {
                int64_t n = a.or_rate;
                const bool last = a.or_rate != 0 && a.t_th - t < n;
                if (last) n = a.t_th - t;
                for (int64_t q = 0; q < n; ++q) sw.or_sweep();
                if (!last) acc += metro_sweep(T, a.kind, sigma);
                t += a.or_rate != 0 ? n : 1;
            }
            if (threadIdx.x == 0 && sw.leader()) a.acc_T[(int64_t)sys * a.n_temps + k] = acc;
        }
    } else {
        // parallel_tempering! sweep loop (monte_carlo.jl:295-388).  State of
        // the system's current temperature slot, carried across segments.
        const PTDev &pt = a.pt;
        int slot = pt.slot_of_sys[sys];
        double T = pt.temps[slot];
        double sigma = pt.sigma[slot];
        double E = pt.E[sys];
        // probes go to the slot's series (binned later by launch_bin_fold);
        // every workgroup counts the same probe sweeps, so the index is shared
        int64_t probe_idx = a.probe_base;
        // accepted moves since the system took its slot; another system may
        // hold the slot later, with no ordering between the two but the
        // exchange records: added atomically
        double acc_local = 0.0;
        auto put_accepted = [&]() __attribute__((always_inline)) {
            if (threadIdx.x == 0 && sw.leader())
                __hip_atomic_fetch_add(pt.acc_local + slot, acc_local, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            acc_local = 0.0;
        };
        // an exchange published but not yet resolved (its sweep), and a probe
        // of that time whose slot the exchange decides: its index and |M|
        bool open_x = false, open_p = false;
        int64_t x_se = 0, p_idx = 0;
        double p_m = 0.0;
        auto put_probe = [&](int64_t idx, double absm) __attribute__((always_inline)) {
            if (threadIdx.x == 0 && sw.leader()) {
                double *q = pt.series + ((int64_t)slot * pt.series_cap + idx) * 2;
                q[0] = E;
                q[1] = absm;
            }
        };
        auto resolve = [&]() __attribute__((always_inline)) {
            if (MODE != WG_PT_CHAIN || !open_x) return;
            open_x = false;
            put_accepted();
            exchange_resolve(a, x_se, slot, sigma, T, E, sw.red + RED_XCHG, sw.leader());
            if (open_p) put_probe(p_idx, p_m);
            open_p = false;
        };
        // m: summed spin of the system's current state when m_now (the
        // exchange moves temperature labels, not spins, so it stays valid
        // across an exchange)
        double m[3] = {0, 0, 0};
        bool m_now = false;
        // Segments, each from the post-exchange part of sweep sb (bmid) to the
        // pre-exchange part of sweep se (emid).  WG_PT: one; WG_PT_CHAIN:
        // nseg that end with an exchange, decided pair by pair from the
        // partners' published records, then the tail, if any.
        const int nseg = MODE == WG_PT_CHAIN ? a.nseg + (a.chain_tail >= 0 ? 1 : 0) : 1;
        int64_t sb = a.seg_begin;
        bool bmid = a.begin_mid;
        // swp % dosweep and swp % probe as running remainders (a 64-bit
        // remainder is a long instruction sequence)
        int64_t r_do = sb % pt.dosweep, r_pr = sb % pt.probe;
        for (int g = 0; g < nseg; ++g) {
            const bool exch = MODE == WG_PT_CHAIN && g < a.nseg;
            const int64_t se = MODE != WG_PT_CHAIN ? a.seg_end
                               : exch              ? a.chain_e0 + (int64_t)g * a.chain_P
                                                   : a.chain_tail;
            const bool emid = MODE != WG_PT_CHAIN ? a.end_mid : exch;
            for (int64_t swp = sb; swp <= se;) {
                // k sweeps of overrelaxation alone, then sweep swp + k, which
                // may have a Metropolis sweep, a probe or the segment's end
                int64_t k = r_do ? pt.dosweep - r_do : 0;
                if (k > se - swp) k = se - swp;
                if (pt.measure) {
                    const int64_t kp = r_pr ? pt.probe - r_pr : 0;
                    k = k < kp ? k : kp;
                }
                const bool head = !(swp == sb && bmid && k == 0);
                int n_or = pt.or_rate != 0 ? (int)k + 1 : 0;
                if (n_or && swp == sb && bmid) --n_or;  // its overrelaxation is done
                for (int q = 0; q < n_or; ++q) sw.or_sweep();
                if (n_or) m_now = false;
                swp += k;
                r_do += k;
                if (r_do == pt.dosweep) r_do = 0;
                if (pt.measure) {
                    r_pr += k;
                    if (r_pr == pt.probe) r_pr = 0;
                }
                const bool metro = head && r_do == 0;
                const bool probe_at = pt.measure && swp >= pt.t_th && r_pr == 0;
                const bool probe_here = probe_at && !(swp == se && emid);
                if (SW::LATE_EXCHANGE && (metro || (probe_here && open_p))) resolve();
                if (metro) {
                    // the Metropolis sweep and total_energy
                    // (monte_carlo.jl:303-305); the energy pass also sums
                    // the spins when this sweep has a probe
                    const double acc = sw.metro_energy(T, pt.alg, sigma, mctr, probe_at, E, m);
                    ++mctr;
                    if (pt.alg == CSMC_CONE_ADAPTIVE) sigma = adapt_sigma(sigma, acc, (double)sw.n_sites());
                    acc_local += acc;
                    m_now = probe_at;
                }
                if (probe_here) {
                    if (!m_now) {
                        sw.magnet(m);
                        m_now = true;
                    }
                    const double absm = sqrt(m[0] * m[0] + m[1] * m[1] + m[2] * m[2]);
                    if (open_x) {  // no probe waits for its slot yet
                        open_p = true;
                        p_idx = probe_idx;
                        p_m = absm;
                    } else {
                        put_probe(probe_idx, absm);
                    }
                    ++probe_idx;
                }
                ++swp;
                if (++r_do == pt.dosweep) r_do = 0;
                if (pt.measure && ++r_pr == pt.probe) r_pr = 0;
            }
            if (exch) {
                exchange_publish(a, se, slot, sigma, E, sw.leader());
                open_x = true;
                x_se = se;
                if (!SW::LATE_EXCHANGE) resolve();
                // the next segment starts at the exchange's sweep, a multiple
                // of dosweep
                sb = se;
                bmid = true;
                r_do = 0;
                if (pt.measure) r_pr = (r_pr ? r_pr : pt.probe) - 1;
            }
        }
        if (SW::LATE_EXCHANGE) resolve();
        put_accepted();
        if (threadIdx.x == 0 && sw.leader()) {
            pt.E[sys] = E;
            pt.sigma[slot] = sigma;
            if (MODE == WG_PT_CHAIN) {
                pt.slot_of_sys[sys] = slot;
                pt.sys_of_slot[slot] = sys;
            }
        }
    }
    if (threadIdx.x == 0 && sw.leader()) a.mcount[sys] = mctr;
}

// Replica exchange (monte_carlo.jl:308-349) at the end of a PT segment, done
// by the last workgroup of the grid to finish: a completion counter, no
// waiting, so every wave reaches the end of the kernel.  Pairs (r, r+1)
// start at 0 for an even exchange index, at 1 for an odd one; the decision
// is FP64 with the Philox exchange stream; temperature labels move, spins
// stay.  Call from every thread after the workgroup's last global store;
// flag is one int of workgroup scratch in LDS.  (No static __shared__
// variable here: it would offset the dynamic LDS block and cost an address
// add on every LDS access of the sweep.)
__device__ __forceinline__ void pt_exchange_last(const WGArgs &a, int *flag) {
    // Only thread 0 fences: it wrote this system's energy and counters
    // (wg_drive), and an agent-scope fence writes back the L2, so one per
    // workgroup instead of one per wave keeps the launch tail short.  The
    // workgroup barrier then carries thread 0's acquire to the other threads.
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();  // release this workgroup's results
        unsigned prev = atomicAdd(a.pt.done, 1u);
        *flag = (prev == gridDim.x - 1);
        if (*flag) __threadfence();  // acquire every other workgroup's results
    }
    __syncthreads();
    if (*flag) {
        // the pairs are disjoint: one thread per pair
        const PTDev &pt = a.pt;
        const uint32_t xc = (uint32_t)(a.seg_end / pt.swap);
        const int r0 = (xc % 2 == 0) ? 0 : 1;
        for (int r = r0 + 2 * (int)threadIdx.x; r + 1 < pt.R; r += 2 * (int)blockDim.x) {
            const int p = r + 1;
            const int sr = pt.sys_of_slot[r], sp = pt.sys_of_slot[p];
            uint4 rr =
                philox4x32_10(make_uint4((uint32_t)r, 0xFFFFFFFFu, xc, TAG_EXCH), a.k0, a.k1);
            double u = u01d(rr.x);
            double dbeta = 1.0 / pt.temps[p] - 1.0 / pt.temps[r];
            double pacc = fmin(1.0, exp(dbeta * (pt.E[sp] - pt.E[sr])));
            if (u < pacc) {
                pt.sys_of_slot[r] = sp;
                pt.sys_of_slot[p] = sr;
                pt.slot_of_sys[sp] = r;
                pt.slot_of_sys[sr] = p;
                pt.acc_exch[r] += 1.0;
                pt.acc_exch[p] += 1.0;
            }
        }
        // visible to the next launch at the kernel boundary
        if (threadIdx.x == 0) *pt.done = 0u;
    }
}

}  // namespace csmc
