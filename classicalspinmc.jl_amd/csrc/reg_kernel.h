// reg_kernel.h -- register-table storage mode of the persistent
// workgroup-per-system sweep kernel (FP32 state, bilinear-only lattices).
//
// One workgroup of REG_THREADS threads owns one system.  Its spins sit in
// LDS as float4 records (16 B per site, plus the zero pad site), and each
// thread keeps, in registers, the spins of the sites it updates, their LDS
// addresses and those of their K2C bilinear neighbours: thread t owns site
// first + t of every slot (a REG_THREADS-site piece of one run of one colour
// class).  A site update is then one 16-byte LDS read per neighbour and one
// 16-byte write, with no neighbour-table traffic and no address arithmetic in
// the sweep.  The schedule (wg_drive) and the per-site physics (device.h) are
// the ones every other storage mode uses.
//
// Bound (honeycomb L=64, four sites a thread and colour phase): VALU issue
// (28 instructions per update, 16 waves on 4 SIMDs: 0.8 us a phase) and the
// LDS (4 x 16 B per update: 0.85 us), overlapping, plus what a phase waits
// for: so the couplings stay in scalar registers where they fit (loading them
// took two dependent round trips at the start of every phase), the slots of a
// phase are known without a load, and the neighbours of the next slot are
// read while a slot is computed.  An overrelaxation sweep takes 2.0 us
// within tempering and 1.7 alone (3.2 with the own spin read from LDS and the
// loads in place).
//
// Plain sweeps are compiled per kind (WG_SWEEPS_OR ...): one kernel with all
// three held the tables of each and spilled.  Metropolis sweep of square L=80
// with DM couplings 7.3 us, 10.4 in one kernel; overrelaxation of triangular
// L=30 1.6, 3.2.
#pragma once
#include "reg.h"

namespace csmc {

// TWO != 0: the lattice has two colour classes of SPT / 2 full
// REG_THREADS-site slots each, so every thread has a site in every slot, no
// update needs an ownership mask and both colours' couplings stay in scalar
// registers; TWO = 1: it has neither onsite terms nor a field.  TWO = 0: any
// layout.
template <int K2C, int SPT, bool DIAG, int TWO>
struct SweeperR {
    static constexpr bool LATE_EXCHANGE = true;
    static constexpr int SPC = TWO ? SPT / 2 : 0;  // slots per colour
    // couplings and field of the sites of one colour
    struct Coef {
        BilCoef<float, K2C, DIAG> M;
        float h[3];
    };
    // the neighbours' spins of one slot's site
    struct Near {
        spin4<float> sj[K2C];
    };

    const LatView<float> &L;
    const LatView<double> &Ld;
    SpinsV4 X;
    double *red;
    uint32_t stream, k0, k1;
    uint32_t valid;             // bit q: this thread owns a site in slot q
    uint64_t cmask;             // byte c: the slots of colour c (at most 8 of each)
    uint32_t cbasis, sbasis;    // 4 bits each: the basis of colour c, of slot q
    uint32_t own[SPT];          // LDS address of the owned site (the zero pad site if none)
    uint32_t nb[SPT][K2C];      // LDS address of each bilinear neighbour (pad site if absent)
    uint32_t refs[(SPT + 1) / 2];  // reference site indices, two to a word
    spin4<float> s[SPT];        // the owned spins (as in LDS), w = 0
    Coef cf[TWO ? 2 : 1];       // TWO: both colours; else of basis cfb
    int cfb;

    // slots: int4 records {first site, run end, basis, colour}; colslot:
    // first slot of each colour [ncol + 1], then the basis shared by a
    // colour's slots [ncol]
    __device__ __forceinline__ SweeperR(const LatView<float> &L_, const LatView<double> &Ld_, uint32_t base, double *red_,
                        const int32_t *slots, const int32_t *colslot, int nslots, uint32_t stream_,
                        uint32_t k0_, uint32_t k1_)
        : L(L_), Ld(Ld_), X(), red(red_), stream(stream_), k0(k0_), k1(k1_), valid(0), cmask(0), cbasis(0),
          sbasis(0), cfb(-1) {
        for (int c = 0; c < L.ncol; ++c) {
            const int qb = ldc(colslot + c), qe = ldc(colslot + c + 1);
            cmask |= (uint64_t)((1u << qe) - (1u << qb)) << (8 * c);
            cbasis |= (uint32_t)ldc(colslot + L.ncol + 1 + c) << (4 * c);
        }
#pragma unroll
        for (int q = 0; q < (SPT + 1) / 2; ++q) refs[q] = 0;
        // every table load is unconditional (slot index and site clamped to
        // valid entries) so all of them are in flight together
#pragma unroll
        for (int q = 0; q < SPT; ++q) {
            const int qq = q < nslots ? q : nslots - 1;
            const int first = ldc(slots + 4 * qq), end = ldc(slots + 4 * qq + 1);
            const int i = first + (int)threadIdx.x;
            const bool ok = q < nslots && i < end;
            const int ic = ok ? i : first;
            valid |= ok ? (1u << q) : 0u;
            sbasis |= (uint32_t)ldc(slots + 4 * qq + 2) << (4 * q);
            own[q] = pin_address(base + 16u * (uint32_t)(ok ? i : L.N));
            refs[q / 2] |= (uint32_t)L.ref[ic] << (16 * (q & 1));
#pragma unroll
            for (int k = 0; k < K2C; ++k)
                nb[q][k] = pin_address(base + 16u * (uint32_t)L.nbr2[(int64_t)k * L.N + ic]);
        }
    }
    // after the spins are staged in LDS
    __device__ __forceinline__ void start() {
        static_for<SPT>([&](auto Q) __attribute__((always_inline)) { s[Q] = X.ld(own[Q]); });
        if constexpr (TWO) {
            load_coef(cf[0], basis_of_colour(0));
            load_coef(cf[1], basis_of_colour(1));
        }
    }

    __device__ __forceinline__ int n_sites() const { return L.N; }
    __device__ __forceinline__ bool leader() const { return true; }  // the only workgroup of its system
    __device__ __forceinline__ bool owns(int q) const { return (valid >> q) & 1u; }
    __device__ __forceinline__ int basis_of_colour(int c) const { return (int)(cbasis >> (4 * c)) & 15; }

    __device__ __forceinline__ void load_coef(Coef &c, int b) const {
        // through an opaque address: kept where it is written
        c.M.load(per_site_coef(L.c2), L.K2P, b);
        const float *h = per_site_coef(L.field) + b * 3;
#pragma unroll
        for (int a = 0; a < 3; ++a) c.h[a] = ldc(h + a);
    }

    template <int Q>
    __device__ __forceinline__ uint32_t ref() const {
        // opaque where it is used: the first Philox product of every slot
        // would otherwise be kept across the sweeps, in scratch memory
        return pin_address((Q & 1) ? refs[Q / 2] >> 16 : refs[Q / 2] & 0xffffu);
    }
    template <int Q>
    __device__ __forceinline__ Near near() const {
        Near v;
#pragma unroll
        for (int k = 0; k < K2C; ++k) v.sj[k] = X.ld(nb[Q][k]);
        return v;
    }
    template <int Q>
    __device__ __forceinline__ void put(float x, float y, float z) {
        s[Q].x = x;
        s[Q].y = y;
        s[Q].z = z;
        X.st(own[Q], spin4<float>{x, y, z, 0.0f});
        // distinct per slot: the optimiser must not merge the ends of two
        // slots' branches, which would index s at run time (scratch memory)
        asm volatile("; slot %0" ::"n"(Q));
    }

    // One coloured sweep: colour classes in turn, a workgroup barrier after
    // each.  Every colour class has a single basis (the host only picks this
    // mode then).  upd(Q, basis, neighbours, C) updates slot Q with the
    // colour's couplings C; the sites of a phase are independent, so the
    // neighbours of a slot are read before the one before it is updated (the
    // scheduling barriers keep it to one slot ahead: more would not fit the
    // registers of 1024 threads).
    template <class UPD>
    __device__ __forceinline__ void colour_sweep(UPD &&upd) {
        if constexpr (TWO) {
            static_for<2>([&](auto C) __attribute__((always_inline)) {
                const int b = basis_of_colour(C);
                Near v = near<C * SPC>();
                static_for<SPC>([&](auto I) __attribute__((always_inline)) {
                    constexpr int q = C * SPC + I;
                    Near w;
                    if constexpr (I + 1 < SPC) w = near<q + 1>();
                    __builtin_amdgcn_sched_barrier(0);
                    upd(std::integral_constant<int, q>{}, b, v, cf[C]);
                    if constexpr (I + 1 < SPC) v = w;
                });
                __syncthreads();
            });
        } else {
            for (int c = 0; c < L.ncol; ++c) {
                const int b = basis_of_colour(c);
                const uint32_t m = (uint32_t)(cmask >> (8 * c));
                // a lattice of one basis loads its couplings once
                if (b != cfb) load_coef(cf[0], b);
                cfb = b;
                // One slot at a time: with two slots' neighbours read ahead
                // every update stands in the code three times (as a pair or
                // alone), and with full matrices the pair holds 32 registers
                // more.  Square L=80 with DM couplings: overrelaxation 4.43
                // us against 5.91 by pairs, Metropolis 10.4 against 12.8;
                // honeycomb L=8: 1.21 against 1.27, 2.10 against 2.48 (all of
                // them in a kernel of all three kinds).
                static_for<SPT>([&](auto q) __attribute__((always_inline)) {
                    if ((m >> q) & 1u) {
                        const Near v = near<q>();
                        if (owns(q)) upd(q, b, v, cf[0]);
                    }
                });
                __syncthreads();
            }
        }
    }

    // get_local_field (local_field) with the colour's field at hand
    template <int q>
    __device__ __forceinline__ void full_field(int b, const Near &v, const Coef &C, float H[3]) const {
        C.M.field(v.sj, H);
        if constexpr (TWO != 1) {
            if (L.flags & LAT_ONSITE) {
                const float *O = L.onsite + b * 9;
                const float x = s[q].x, y = s[q].y, z = s[q].z;
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    H[a] = fmaf(2.0f, dot3(ldc(O + 3 * a), ldc(O + 3 * a + 1), ldc(O + 3 * a + 2), x, y, z), H[a]);
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) H[a] -= C.h[a];
        }
    }

    __device__ __forceinline__ void or_sweep() {
        colour_sweep([&](auto q, int b, const Near &v, const Coef &C) __attribute__((always_inline)) {
            float H[3];
            full_field<q>(b, v, C, H);
            // or_reflect, with the H == 0 case (no change) taken by a select
            // instead of a branch: the spin is stored back unchanged
            const bool zero =
                __uint_as_float(__float_as_uint(H[0]) | __float_as_uint(H[1]) | __float_as_uint(H[2])) == 0.0f;
            const float x = s[q].x, y = s[q].y, z = s[q].z;
            const float hh = dot3(H[0], H[1], H[2], H[0], H[1], H[2]);
            const float proj = Math<float>::div(2.0f * dot3(x, y, z, H[0], H[1], H[2]), hh);
            put<q>(zero ? x : -x + proj * H[0], zero ? y : -y + proj * H[1], zero ? z : -z + proj * H[2]);
        });
    }
    __device__ __forceinline__ void det_sweep() {
        colour_sweep([&](auto q, int b, const Near &v, const Coef &C) __attribute__((always_inline)) {
            spin4<float> n;
            float H[3];
            full_field<q>(b, v, C, H);
            if (det_align<float>(L, H, n)) put<q>(n.x, n.y, n.z);
        });
    }

    __device__ __forceinline__ double metro(double T, int kind, double sigma, uint32_t ctr) {
        double w[1] = {(double)metro_local(T, kind, sigma, ctr)};
        block_sum<1>(w, red);
        return w[0];
    }

    // one Metropolis sweep; returns this thread's accepted count
    __device__ __forceinline__ int metro_local(double T, int kind, double sigma, uint32_t ctr) {
        const float Tf = (float)T, invT = 1.0f / Tf, sg = (float)sigma;
        int acc = 0;
        // opaque here, so that the round keys are formed in this sweep
        // instead of being held across the overrelaxation sweeps
        uint32_t k0 = this->k0, k1 = this->k1;
        asm volatile("" : "+s"(k0), "+s"(k1));
        colour_sweep([&](auto q, int b, const Near &v, const Coef &C) __attribute__((always_inline)) {
            // Philox counter: the reference index of the site
            const uint4 r = philox4x32_10(make_uint4(ref<q>(), stream, ctr, TAG_METRO), k0, k1);
            const spin4<float> n = metro_propose<float>(L, s[q], r, kind, sg);
            float F[3];
            C.M.field(v.sj, F);
            const int a = metro_accept<float>(metro_dE<float>(L, b, s[q], n, F, C.h), r, Tf, invT);
            // metro_commit
            if (a) {
                put<q>(n.x, n.y, n.z);
            } else {
                const float x = s[q].x, y = s[q].y, z = s[q].z;
                const float inv = Math<float>::rsqrt_(dot3(x, y, z, x, y, z)) * L.S;
                put<q>(x * inv, y * inv, z * inv);
            }
            acc += a;
        });
        return acc;
    }

    // thread_energy with the terms added row by row, as k_wg adds them, which
    // these lattices ran before: their energies keep their bits.  One slot's
    // FP64 matrix at a time (all six would take 108 scalar registers).
    __device__ __forceinline__ void thread_energy_rows(double &e, double m[3]) {
        double p[5] = {0, 0, 0, 0, 0};
        m[0] = m[1] = m[2] = 0.0;
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            if (!owns(q)) return;
            const int b = __builtin_amdgcn_readfirstlane((int)(sbasis >> (4 * q)) & 15);
            const double *c2 = per_site_coef(Ld.c2) + (int64_t)b * Ld.K2P * 9, *h = per_site_coef(Ld.field) + b * 3;
            const Near v = near<q>();
            const double sx = s[q].x, sy = s[q].y, sz = s[q].z;
            double F[3] = {0, 0, 0};
#pragma unroll
            for (int k = 0; k < K2C; ++k)
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    F[a] += dot3(ldc(c2 + 9 * k + 3 * a), ldc(c2 + 9 * k + 3 * a + 1), ldc(c2 + 9 * k + 3 * a + 2),
                                 (double)v.sj[k].x, (double)v.sj[k].y, (double)v.sj[k].z);
            p[0] += dot3(sx, sy, sz, F[0], F[1], F[2]);
            p[3] -= dot3(sx, sy, sz, ldc(h), ldc(h + 1), ldc(h + 2));
            p[4] += onsite_energy<double, double>(Ld, b, sx, sy, sz);
            m[0] += sx;
            m[1] += sy;
            m[2] += sz;
        });
        e = combine_energy(p);
    }

    // this thread's FP64 energy (bilinear / 2 + Zeeman + onsite: the lattice
    // has no cubic or quartic terms) and summed spin
    __device__ __forceinline__ void thread_energy(double &e, double m[3]) {
        if constexpr (K2C == 6 && SPT == 6) return thread_energy_rows(e, m);
        double bil = 0.0, zee = 0.0, ons = 0.0;
        m[0] = m[1] = m[2] = 0.0;
        BilCoef<double, K2C, DIAG> M;
        double h[3] = {0.0, 0.0, 0.0};
        int bl = -1;  // the basis M and h are of
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            const int b = (int)(sbasis >> (4 * q)) & 15;
            // slots of one colour share a basis: its FP64 couplings are
            // loaded once, where they are used
            if (TWO ? q % (TWO ? SPC : 1) == 0 : b != bl) {
                M.load(per_site_coef(Ld.c2), Ld.K2P, b);
                const double *hp = per_site_coef(Ld.field) + b * 3;
                h[0] = ldc(hp);
                h[1] = ldc(hp + 1);
                h[2] = ldc(hp + 2);
                bl = b;
            }
            if (owns(q)) {
                const Near v = near<q>();
                const double sx = s[q].x, sy = s[q].y, sz = s[q].z;
                double F[3];
                M.field(v.sj, F);
                bil += sx * F[0] + sy * F[1] + sz * F[2];
                zee -= sx * h[0] + sy * h[1] + sz * h[2];
                ons += onsite_energy<double, double>(Ld, b, sx, sy, sz);
                m[0] += sx;
                m[1] += sy;
                m[2] += sz;
            }
        });
        e = bil / 2 + zee + ons;
    }

    __device__ __forceinline__ double metro_energy(double T, int kind, double sigma, uint32_t ctr, bool with_m,
                                   double &E, double m[3]) {
        const int acc = metro_local(T, kind, sigma, ctr);
        double e, mm[3];
        thread_energy(e, mm);
        if (with_m) {
            double v[5] = {(double)acc, e, mm[0], mm[1], mm[2]};
            block_sum<5>(v, red);
            E = v[1];
            m[0] = v[2];
            m[1] = v[3];
            m[2] = v[4];
            return v[0];
        }
        double v[2] = {(double)acc, e};
        block_sum<2>(v, red);
        E = v[1];
        return v[0];
    }

    // the summed spin over the same per-thread sites, in the same order, as
    // thread_energy, so both give the same FP64 sums
    __device__ __forceinline__ void magnet(double out[3]) {
        double m[3] = {0, 0, 0};
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            if (owns(q)) {
                m[0] += s[q].x;
                m[1] += s[q].y;
                m[2] += s[q].z;
            }
        });
        block_sum<3>(m, red);
        for (int k = 0; k < 3; ++k) out[k] = m[k];
    }
};

template <int K2C, int SPT, bool DIAG, int MODE, int TWO>
__global__ __launch_bounds__(REG_THREADS) void k_wg_reg(WGArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *red = reinterpret_cast<double *>(smem);  // reduction scratch

    const int sys = blockIdx.x;
    const SysDev sd = a.P.sys[sys];
    const LatDev ld = a.P.lats[sd.lat];
    const int4 *runs = a.P.runs + ld.run_off;
    const LatView<float> L = lat_view<float>(ld, a.P.i32, runs, a.P.coefF);
    const LatView<double> Ld = lat_view<double>(ld, a.P.i32, runs, a.P.coefD);
    const SpinsG<float> G = spins_at<float>(a.spins, sd.spin_off);
    const int N = L.N;

    const uint32_t base = lds_address(smem + RED_BYTES);
    SpinsV4 X;
    // stage the system and its zero pad site N into LDS
    wg_stage<8>(N + 1, [&](int i) { return G.ld(i); },
                [&](int i, const spin4<float> &v) { X.st(base + 16u * (uint32_t)i, v); });
    SweeperR<K2C, SPT, DIAG, TWO> sw(L, Ld, base, red,
                                reinterpret_cast<const int32_t *>(a.P.runs + ld.slot_off),
                                a.P.i32 + ld.colslot_off, ld.nslots, (uint32_t)sd.stream, a.k0,
                                a.k1);
    __syncthreads();
    sw.start();
    wg_drive<MODE>(a, sys, sw);
    // the exchange goes first so that its fence writes back only the small
    // PT state, not the spins stored below
    if (MODE == WG_PT && a.exchange) pt_exchange_last(a, reinterpret_cast<int *>(red + RED_FLAG));
    __syncthreads();
    for (int i = threadIdx.x; i < N; i += REG_THREADS) G.st(i, X.ld(base + 16u * (uint32_t)i));
}

template <int K2C, int SPT, bool DIAG, int MODE, int TWO>
static hipError_t launch_reg_t(int nsys, size_t lds_bytes, const WGArgs &a, hipStream_t st) {
    const size_t bytes = RED_BYTES + lds_bytes;
    const void *fn = (const void *)k_wg_reg<K2C, SPT, DIAG, MODE, TWO>;
    if (bytes > 65536) {
        hipError_t e = allow_large_lds(fn);
        if (e != hipSuccess) return e;
    }
    if constexpr (MODE == WG_PT_CHAIN) return launch_cooperative(fn, nsys, REG_THREADS, bytes, a, st);
    hipLaunchKernelGGL((k_wg_reg<K2C, SPT, DIAG, MODE, TWO>), dim3(nsys), dim3(REG_THREADS), bytes, st, a);
    return hipGetLastError();
}

template <int K2C, int SPT, bool DIAG, int TWO>
static hipError_t launch_reg_m(int nsys, size_t lds_bytes, const WGArgs &a, hipStream_t st) {
    if (a.mode == WG_PT) return launch_reg_t<K2C, SPT, DIAG, WG_PT, TWO>(nsys, lds_bytes, a, st);
    if (a.mode == WG_PT_CHAIN)
        return launch_reg_t<K2C, SPT, DIAG, WG_PT_CHAIN, TWO>(nsys, lds_bytes, a, st);
    if (a.mode == WG_ANNEAL) return launch_reg_t<K2C, SPT, DIAG, WG_ANNEAL, TWO>(nsys, lds_bytes, a, st);
    if (a.kind == CSMC_OVERRELAX) return launch_reg_t<K2C, SPT, DIAG, WG_SWEEPS_OR, TWO>(nsys, lds_bytes, a, st);
    if (a.kind == CSMC_DETERMINISTIC) return launch_reg_t<K2C, SPT, DIAG, WG_SWEEPS_DET, TWO>(nsys, lds_bytes, a, st);
    return launch_reg_t<K2C, SPT, DIAG, WG_SWEEPS_METRO, TWO>(nsys, lds_bytes, a, st);
}

template <int K2C, int SPT>
static hipError_t launch_reg_d(bool diag, int two_colour, int nsys, size_t lds_bytes,
                               const WGArgs &a, hipStream_t st) {
    // the fixed two-colour layout is compiled for diagonal couplings with 3
    // or 4 neighbours (honeycomb, square and their Kitaev / XXZ variants)
    if constexpr (K2C <= 4) {
        if (diag && two_colour == 1) return launch_reg_m<K2C, SPT, true, 1>(nsys, lds_bytes, a, st);
        if (diag && two_colour == 2) return launch_reg_m<K2C, SPT, true, 2>(nsys, lds_bytes, a, st);
    }
    return diag ? launch_reg_m<K2C, SPT, true, 0>(nsys, lds_bytes, a, st)
                : launch_reg_m<K2C, SPT, false, 0>(nsys, lds_bytes, a, st);
}

// one translation unit per K2C (kernels_reg<K2C>.hip) instantiates this
template <int K2C>
hipError_t launch_reg_s(int spt, bool diag, int two_colour, int nsys, size_t lds_bytes,
                               const WGArgs &a, hipStream_t st) {
    if (spt == 4) return launch_reg_d<K2C, 4>(diag, two_colour, nsys, lds_bytes, a, st);
    // 8 slots of 6 neighbours exceed the register budget of 1024 threads; 6 fit
    if constexpr (K2C == 6) {
        if (spt == 6) return launch_reg_d<K2C, 6>(diag, two_colour, nsys, lds_bytes, a, st);
    } else {
        if (spt == 8) return launch_reg_d<K2C, 8>(diag, two_colour, nsys, lds_bytes, a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace csmc
