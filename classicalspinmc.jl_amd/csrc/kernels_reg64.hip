// kernels_reg64.hip -- the FP64 form of the register-table sweep kernel
// (bilinear lattices of 3 or 4 neighbours without self references, spins and
// zero pad site as 24-byte records in LDS).
//
// As in reg_kernel.h, thread t owns site first + t of every slot (here a
// 512-site piece of one run) and holds its spins and the LDS addresses of its
// sites and of their neighbours.  512 threads leave 256 vector registers a
// lane, enough for 8 slots (4096 sites a system); 16 slots spilled about 200
// registers.  The updates, the order of the energy sums and the draws are
// those of k_wg, bit for bit: each matrix row is added to the field as
// fma(m2, z, fma(m0, x, m1 y)), of which a diagonal matrix leaves the rounded
// product m_rr s_r (its other terms are exact zeros).
//
// Bound: the latency of a phase -- one wave per SIMD or two, a chain of about
// 70 dependent FP64 operations -- so what a phase needs is in registers when
// it starts; k_wg reads each partner index from LDS and each matrix with
// scalar loads between the slots.  Annealing of square L=16 (2 slots): 1.01 us
// a sweep, 1.87 in k_wg; square L=64 (8 slots) 4.28, 6.84.  Tempering, period
// of 10 overrelaxation sweeps and one Metropolis sweep: honeycomb L=24 with
// full matrices 25.5 us, 36.6 in k_wg; honeycomb L=32 27.4, 44.0.  Plain
// sweeps, a kernel for each kind, square L=64: overrelaxation 3.3 us, 6.2 in
// k_wg, Metropolis 10.2, 13.7; square L=45 with full matrices 3.2, 4.5 and 7.4,
// 8.4 (with every kind in one kernel they spilled: 3.8, 13.9; 5.0).
//
// Diagonal couplings (9 or 12 doubles) stay between the phases of one basis;
// full matrices (27 or 36) are read at the start of a phase: held across
// phases they spilled 100 to 180 vector registers and ran 1.5 times slower
// than k_wg.  Slots run one at a time: two slots' neighbours in flight
// together spilled as well, and the longer code (each update is unrolled per
// slot) took 1.6 us where the single form takes 1.07 (square L=16).
#include "reg.h"

namespace csmc {

namespace {

constexpr int R64_THREADS = 512;

struct SpinsD3 {
    using lds_d = __attribute__((address_space(3))) double;
    __device__ __forceinline__ spin4<double> ld(uint32_t a) const {
        const lds_d *p = (const lds_d *)(size_t)a;
        return spin4<double>{p[0], p[1], p[2], 0.0};
    }
    __device__ __forceinline__ void st(uint32_t a, double x, double y, double z) const {
        lds_d *p = (lds_d *)(size_t)a;
        p[0] = x;
        p[1] = y;
        p[2] = z;
    }
};

}  // namespace

template <int K2C, int SPT, bool DIAG>
struct SweeperD {
    static constexpr bool LATE_EXCHANGE = true;
    static constexpr int W = DIAG ? 3 : 9;
    struct Near {
        spin4<double> sj[K2C];
    };

    const LatView<double> &L;
    SpinsD3 X;
    double *red;
    uint32_t stream, k0, k1;
    uint32_t valid;           // bit q: this thread owns a site in slot q
    uint32_t cmask;           // 8 bits per colour: its slots (at most 4 colours)
    uint32_t sbasis;          // 4 bits per slot: its basis (at most 16)
    uint32_t own[SPT];        // LDS address of the owned site (the zero pad site if none)
    uint32_t nb[SPT][K2C];    // LDS address of each neighbour (pad site if absent)
    uint32_t refs[(SPT + 1) / 2];
    spin4<double> s[SPT];     // the owned spins
    double m[K2C][W], h[3];   // couplings and field of basis cfb
    int cfb;

    __device__ __forceinline__ SweeperD(const LatView<double> &L_, uint32_t base, double *red_, uint32_t stream_,
                                        uint32_t k0_, uint32_t k1_)
        : L(L_), X(), red(red_), stream(stream_), k0(k0_), k1(k1_), valid(0), cmask(0), sbasis(0), cfb(-1) {
        // the slots: every run in pieces of R64_THREADS sites, in run order;
        // every table load is unconditional (clamped), so they overlap
        int r = ldc(L.colrun), c = 0;
        const int rend = ldc(L.colrun + L.ncol);
        const int32_t *p = reinterpret_cast<const int32_t *>(L.runs + r);
        int first = ldc(p), end = ldc(p + 1), b = ldc(p + 2), cend = ldc(L.colrun + 1);
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            const bool live = r < rend;
            const int i = first + (int)threadIdx.x;
            const bool ok = live && i < end;
            const int ic = ok ? i : 0;
            valid |= ok ? (1u << q) : 0u;
            if (live) {
                cmask |= 1u << (q + 8 * c);
                sbasis |= (uint32_t)b << (4 * q);
            }
            own[q] = pin_address(base + 24u * (uint32_t)(ok ? i : L.N));
            if (q % 2 == 0) refs[q / 2] = 0;
            refs[q / 2] |= (uint32_t)L.ref[ic] << (16 * (q & 1));
#pragma unroll
            for (int k = 0; k < K2C; ++k)
                nb[q][k] = pin_address(base + 24u * (uint32_t)L.nbr2[(int64_t)k * L.N + ic]);
            if (live) {
                first += R64_THREADS;
                if (first >= end && ++r < rend) {
                    const int32_t *x = reinterpret_cast<const int32_t *>(L.runs + r);
                    first = ldc(x);
                    end = ldc(x + 1);
                    b = ldc(x + 2);
                    while (r >= cend) {
                        ++c;
                        cend = ldc(L.colrun + c + 1);
                    }
                }
            }
        });
    }
    // after the spins are staged in LDS
    __device__ __forceinline__ void start() {
        static_for<SPT>([&](auto q) __attribute__((always_inline)) { s[q] = X.ld(own[q]); });
    }

    __device__ __forceinline__ int n_sites() const { return L.N; }
    __device__ __forceinline__ bool leader() const { return true; }  // the only workgroup of its system
    __device__ __forceinline__ bool owns(int q) const { return (valid >> q) & 1u; }
    __device__ __forceinline__ int basis(int q) const { return (int)(sbasis >> (4 * q)) & 15; }
    template <int Q>
    __device__ __forceinline__ uint32_t ref() const {
        // opaque: see reg_kernel.h
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
    __device__ __forceinline__ void put(double x, double y, double z) {
        s[Q].x = x;
        s[Q].y = y;
        s[Q].z = z;
        X.st(own[Q], x, y, z);
        // distinct per slot: see reg_kernel.h
        asm volatile("; slot %0" ::"n"(Q));
    }
    // the couplings of basis b, unless they are held already
    __device__ __forceinline__ void want(int b) {
        if (b == cfb) return;
        const double *c2 = per_site_coef(L.c2) + (int64_t)b * L.K2P * 9, *f = per_site_coef(L.field) + b * 3;
#pragma unroll
        for (int k = 0; k < K2C; ++k)
#pragma unroll
            for (int e = 0; e < W; ++e) m[k][e] = ldc(c2 + k * 9 + (DIAG ? 4 * e : e));
#pragma unroll
        for (int a = 0; a < 3; ++a) h[a] = ldc(f + a);
        cfb = b;
    }
    // the interaction field (interaction_field's bilinear slots, in its order)
    __device__ __forceinline__ void field(const Near &v, double F[3]) const {
        F[0] = F[1] = F[2] = 0.0;
#pragma unroll
        for (int k = 0; k < K2C; ++k) {
            const spin4<double> &q = v.sj[k];
            if constexpr (DIAG) {
#pragma clang fp contract(off)
                F[0] += m[k][0] * q.x;
                F[1] += m[k][1] * q.y;
                F[2] += m[k][2] * q.z;
            } else {
#pragma unroll
                for (int r = 0; r < 3; ++r) F[r] += dot3(m[k][3 * r], m[k][3 * r + 1], m[k][3 * r + 2], q.x, q.y, q.z);
            }
        }
    }
    // get_local_field (local_field) with the field at hand
    __device__ __forceinline__ void full_field(int b, const spin4<double> &o, const Near &v, double H[3]) const {
        field(v, H);
        if (L.flags & LAT_ONSITE) {
            const double *O = L.onsite + b * 9;
#pragma unroll
            for (int a = 0; a < 3; ++a)
                H[a] = fma(2.0, dot3(ldc(O + 3 * a), ldc(O + 3 * a + 1), ldc(O + 3 * a + 2), o.x, o.y, o.z), H[a]);
        }
        if (L.flags & LAT_FIELD)
#pragma unroll
            for (int a = 0; a < 3; ++a) H[a] -= h[a];
    }

    // one coloured sweep: colour classes in turn, a workgroup barrier after each
    template <class UPD>
    __device__ __forceinline__ void colour_sweep(UPD &&upd) {
        for (int c = 0; c < L.ncol; ++c) {
            const uint32_t mc = (cmask >> (8 * c)) & 0xffu;
            if constexpr (!DIAG) cfb = -1;
            static_for<SPT>([&](auto q) __attribute__((always_inline)) {
                if ((mc >> q) & 1u) {
                    want(basis(q));
                    const Near v = near<q>();
                    if (owns(q)) upd(q, v);
                }
            });
            __syncthreads();
        }
    }

    __device__ __forceinline__ void or_sweep() {
        colour_sweep([&](auto q, const Near &v) __attribute__((always_inline)) {
            const spin4<double> o = s[q];
            spin4<double> n;
            double H[3];
            full_field(cfb, o, v, H);
            if (or_reflect<double>(o, H, n)) put<q>(n.x, n.y, n.z);
        });
    }
    __device__ __forceinline__ void det_sweep() {
        colour_sweep([&](auto q, const Near &v) __attribute__((always_inline)) {
            const spin4<double> o = s[q];
            spin4<double> n;
            double H[3];
            full_field(cfb, o, v, H);
            if (det_align<double>(L, H, n)) put<q>(n.x, n.y, n.z);
        });
    }
    // one Metropolis sweep; returns this thread's accepted count
    __device__ __forceinline__ int metro_local(double T, int kind, double sigma, uint32_t ctr) {
        const double invT = 1.0 / T;
        int acc = 0;
        uint32_t k0 = this->k0, k1 = this->k1;
        asm volatile("" : "+s"(k0), "+s"(k1));  // see reg_kernel.h
        colour_sweep([&](auto q, const Near &v) __attribute__((always_inline)) {
            const spin4<double> o = s[q];
            const uint4 r = philox4x32_10(make_uint4(ref<q>(), stream, ctr, TAG_METRO), k0, k1);
            const spin4<double> n = metro_propose<double>(L, o, r, kind, sigma);
            double F[3];
            field(v, F);
            const int a = metro_accept<double>(metro_dE<double>(L, cfb, o, n, F, h), r, T, invT);
            if (a) put<q>(n.x, n.y, n.z);
            acc += a;
        });
        return acc;
    }
    __device__ __forceinline__ double metro(double T, int kind, double sigma, uint32_t ctr) {
        double w[1] = {(double)metro_local(T, kind, sigma, ctr)};
        block_sum<1>(w, red);
        return w[0];
    }
    // this thread's FP64 energy and summed spin, as thread_energy of k_wg
    __device__ __forceinline__ void thread_energy(double &e, double mm[3]) {
        double p[5] = {0, 0, 0, 0, 0};
        mm[0] = mm[1] = mm[2] = 0.0;
        if constexpr (!DIAG) cfb = -1;
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            if (__any(owns(q))) {
                want(basis(q));
                const Near v = near<q>();
                if (owns(q)) {
                    const spin4<double> o = s[q];
                    double F[3];
                    field(v, F);
                    p[0] += dot3(o.x, o.y, o.z, F[0], F[1], F[2]);
                    p[3] -= dot3(o.x, o.y, o.z, h[0], h[1], h[2]);
                    p[4] += onsite_energy<double, double>(L, cfb, o.x, o.y, o.z);
                    mm[0] += o.x;
                    mm[1] += o.y;
                    mm[2] += o.z;
                }
            }
        });
        e = combine_energy(p);
    }
    __device__ __forceinline__ double metro_energy(double T, int kind, double sigma, uint32_t ctr, bool with_m,
                                                   double &E, double mo[3]) {
        const int acc = metro_local(T, kind, sigma, ctr);
        double e, mm[3];
        thread_energy(e, mm);
        if (with_m) {
            double v[5] = {(double)acc, e, mm[0], mm[1], mm[2]};
            block_sum<5>(v, red);
            E = v[1];
            mo[0] = v[2];
            mo[1] = v[3];
            mo[2] = v[4];
            return v[0];
        }
        double v[2] = {(double)acc, e};
        block_sum<2>(v, red);
        E = v[1];
        return v[0];
    }
    __device__ __forceinline__ void magnet(double out[3]) {
        double mm[3] = {0, 0, 0};
        static_for<SPT>([&](auto q) __attribute__((always_inline)) {
            if (owns(q)) {
                const spin4<double> o = s[q];
                mm[0] += o.x;
                mm[1] += o.y;
                mm[2] += o.z;
            }
        });
        block_sum<3>(mm, red);
        for (int k = 0; k < 3; ++k) out[k] = mm[k];
    }
};

template <int K2C, int SPT, bool DIAG, int MODE>
__global__ __launch_bounds__(R64_THREADS) void k_wg_reg64(WGArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *red = reinterpret_cast<double *>(smem);  // reduction scratch
    const int sys = blockIdx.x;
    const SysDev sd = a.P.sys[sys];
    const LatDev ld = a.P.lats[sd.lat];
    const LatView<double> L = lat_view<double>(ld, a.P.i32, a.P.runs + ld.run_off, a.P.coefD);
    const SpinsG<double> G = spins_at<double>(a.spins, sd.spin_off);
    const uint32_t base = lds_address(smem + RED_BYTES);
    SpinsD3 X;
    wg_stage<8>(L.N + 1, [&](int i) { return G.ld(i); },
                [&](int i, const spin4<double> &v) { X.st(base + 24u * (uint32_t)i, v.x, v.y, v.z); });
    SweeperD<K2C, SPT, DIAG> sw(L, base, red, (uint32_t)sd.stream, a.k0, a.k1);
    __syncthreads();
    sw.start();
    wg_drive<MODE>(a, sys, sw);
    // the exchange goes first so that its fence writes back only the small
    // PT state, not the spins stored below
    if (MODE == WG_PT && a.exchange) pt_exchange_last(a, reinterpret_cast<int *>(red + RED_FLAG));
    __syncthreads();
    for (int i = threadIdx.x; i < L.N; i += blockDim.x) G.st(i, X.ld(base + 24u * (uint32_t)i));
}

template <int K2C, int SPT, bool DIAG, int MODE>
static hipError_t launch_t(int nt, int nsys, size_t bytes, const WGArgs &a, hipStream_t st) {
    const void *fn = (const void *)k_wg_reg64<K2C, SPT, DIAG, MODE>;
    if (bytes > 65536) {
        hipError_t e = allow_large_lds(fn);
        if (e != hipSuccess) return e;
    }
    const int threads = nt > 0 && nt < R64_THREADS ? nt : R64_THREADS;
    if constexpr (MODE == WG_PT_CHAIN) return launch_cooperative(fn, nsys, threads, bytes, a, st);
    hipLaunchKernelGGL((k_wg_reg64<K2C, SPT, DIAG, MODE>), dim3(nsys), dim3(threads), bytes, st, a);
    return hipGetLastError();
}

template <int K2C, int SPT, bool DIAG>
static hipError_t launch_m(int nt, int nsys, size_t bytes, const WGArgs &a, hipStream_t st) {
    if (a.mode == WG_PT) return launch_t<K2C, SPT, DIAG, WG_PT>(nt, nsys, bytes, a, st);
    if (a.mode == WG_PT_CHAIN) return launch_t<K2C, SPT, DIAG, WG_PT_CHAIN>(nt, nsys, bytes, a, st);
    if (a.mode == WG_ANNEAL) return launch_t<K2C, SPT, DIAG, WG_ANNEAL>(nt, nsys, bytes, a, st);
    if (a.kind == CSMC_OVERRELAX) return launch_t<K2C, SPT, DIAG, WG_SWEEPS_OR>(nt, nsys, bytes, a, st);
    if (a.kind == CSMC_DETERMINISTIC) return launch_t<K2C, SPT, DIAG, WG_SWEEPS_DET>(nt, nsys, bytes, a, st);
    return launch_t<K2C, SPT, DIAG, WG_SWEEPS_METRO>(nt, nsys, bytes, a, st);
}

template <int K2C, int SPT>
static hipError_t launch_d(bool diag, int nt, int nsys, size_t bytes, const WGArgs &a, hipStream_t st) {
    return diag ? launch_m<K2C, SPT, true>(nt, nsys, bytes, a, st) : launch_m<K2C, SPT, false>(nt, nsys, bytes, a, st);
}

template <int K2C>
static hipError_t launch_s(int nslots, bool diag, int nt, int nsys, size_t bytes, const WGArgs &a, hipStream_t st) {
    if (nslots <= 4) return launch_d<K2C, 4>(diag, nt, nsys, bytes, a, st);
    return launch_d<K2C, 8>(diag, nt, nsys, bytes, a, st);
}

int reg64_slots(int run_sites) { return (run_sites + R64_THREADS - 1) / R64_THREADS; }

hipError_t launch_wg_reg64(int k2c, int nslots, bool diag, int nt, int nsys, int max_sites, const WGArgs &a,
                           hipStream_t st) {
    const size_t bytes = RED_BYTES + 24 * (size_t)(max_sites + 1);
    if (nslots > REG64_MAX_SLOTS) return hipErrorInvalidValue;
    if (k2c == 3) return launch_s<3>(nslots, diag, nt, nsys, bytes, a, st);
    if (k2c == 4) return launch_s<4>(nslots, diag, nt, nsys, bytes, a, st);
    return hipErrorInvalidValue;
}

}  // namespace csmc
