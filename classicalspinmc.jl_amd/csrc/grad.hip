// grad.hip -- dE/dJ of every unit-cell term of every system (the adjoint of
// total_energy, hamiltonian.jl:70-132, with respect to the couplings).
//
// The gradient of a term is a sum over sites of products of spin components,
// so it is a reduction: each workgroup takes one work item of one system,
// keeps the item's sums in registers over all the sites it walks, and adds
// them over the workgroup once at the end, in a fixed order.  An item is
//   a group of TG bilinear terms (the site's own spin is read once for the
//   group),
//   one cubic term with its first index fixed, one quartic term with its
//   first two fixed (9 sums each, the partners read again per item),
//   or the field and onsite entries of the system.
// Bound: the gathers of the partners' spins through L2.  128 FP64 triangular
// J1-J2 systems of 9216 sites (12 terms): 72 us; adding every site's products
// into LDS with FP64 atomics, 9 per bond on the same few addresses, took
// 1.2 ms.  Groups of 3 terms keep 27 FP64 sums a thread within the registers
// of 512-thread workgroups.  Systems whose runs all fit fewer threads get only
// the waves that hold a site (each thread then has the same sites, and an idle
// wave would add zeros): 4096 systems of 16 sites 134 us a call with one wave
// an item, 271 with eight.
#include "sweep.h"

namespace csmc {

namespace {

constexpr int TG = 3;              // bilinear terms per item
constexpr int GRAD_THREADS = 512;  // most threads of a workgroup

// Gradient tables at grad_off: t2[nb*K2], r2[nb*K2], t3[nb*K3], r3[nb*K3],
// t4[nb*K4], r4[nb*K4] (term and role of each slot), fsrc[nb], osrc[nb],
// then the term offsets {field, onsite, bilinear, cubic, quartic}.
struct GradTab {
    const int32_t *t2, *r2, *t3, *r3, *t4, *r4, *fsrc, *osrc;
    int off_f, off_o, off_2, off_3, off_4, len;
    __device__ __forceinline__ GradTab(const LatDev &ld, const int32_t *i32) {
        const int nb = ld.nb;
        t2 = i32 + ld.grad_off;
        r2 = t2 + nb * ld.K2;
        t3 = r2 + nb * ld.K2;
        r3 = t3 + nb * ld.K3;
        t4 = r3 + nb * ld.K3;
        r4 = t4 + nb * ld.K4;
        fsrc = r4 + nb * ld.K4;
        osrc = fsrc + nb;
        const int32_t *o = osrc + nb;
        off_f = ldc(o);
        off_o = ldc(o + 1);
        off_2 = ldc(o + 2);
        off_3 = ldc(o + 3);
        off_4 = ldc(o + 4);
        len = ld.grad_len;
    }
    __device__ __forceinline__ int n2() const { return (off_3 - off_2) / 9; }
    __device__ __forceinline__ int n3() const { return (off_4 - off_3) / 27; }
    __device__ __forceinline__ int n4() const { return (len - off_4) / 81; }
};

// every site of basis b, in the order of the runs
template <class R, class F>
__device__ __forceinline__ void sites_of_basis(const LatView<R> &L, int b, F &&f) {
    for (int r = ldc(L.colrun); r < ldc(L.colrun + L.ncol); ++r) {
        const int32_t *run = reinterpret_cast<const int32_t *>(L.runs + r);
        if (ldc(run + 2) != b) continue;
        const int end = ldc(run + 1);
        for (int i = ldc(run) + (int)threadIdx.x; i < end; i += (int)blockDim.x) f(i);
    }
}

// lanes k of the mask: slot k0 + k (< K) of the basis row belongs to term t
__device__ __forceinline__ unsigned long long slots_of_term(const int32_t *row, int k0, int K, int t) {
    const int k = k0 + (int)(threadIdx.x & 63);
    return __ballot(k < K && row[k] == t);
}

struct V3 {
    double c[3];
};

}  // namespace

template <class R>
__global__ __launch_bounds__(GRAD_THREADS) void k_grad_couplings(DevPools P, const void *spins, double *dEdJ) {
    __shared__ double red[BLOCK_SUM_SCRATCH];
    const int sys = blockIdx.y;
    const SysDev sd = P.sys[sys];
    const LatDev ld = P.lats[sd.lat];
    const LatView<double> L = lat_view<double>(ld, P.i32, P.runs + ld.run_off, P.coefD);
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    const GradTab g(ld, P.i32);
    const int nb = L.nb, N = L.N, n2 = g.n2(), n3 = g.n3(), n4 = g.n4(), groups = (n2 + TG - 1) / TG;
    const int items = groups + 3 * n3 + 9 * n4 + 1;
    double *out = dEdJ + (int64_t)sys * g.len;
    // the spin of site j; zero where ok is false (an absent partner)
    auto sp = [&](int j, bool ok) {
        const spin4<R> s = S.ld(ok ? j : N);
        return V3{{ok ? (double)s.x : 0.0, ok ? (double)s.y : 0.0, ok ? (double)s.z : 0.0}};
    };
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        if (item < groups) {
            double acc[TG][9];
#pragma unroll
            for (int u = 0; u < TG; ++u)
#pragma unroll
                for (int e = 0; e < 9; ++e) acc[u][e] = 0.0;
            for (int b = 0; b < nb; ++b)
                for (int k0 = 0; k0 < L.K2; k0 += 64) {
                    unsigned long long m[TG];
#pragma unroll
                    for (int u = 0; u < TG; ++u) m[u] = slots_of_term(g.t2 + b * L.K2, k0, L.K2, item * TG + u);
                    // one slot of each term at a time
                    for (;;) {
                        unsigned long long any = 0;
#pragma unroll
                        for (int u = 0; u < TG; ++u) any |= m[u];
                        if (!any) break;
                        int k[TG], rev[TG];
#pragma unroll
                        for (int u = 0; u < TG; ++u) {
                            k[u] = m[u] ? k0 + __builtin_ctzll(m[u]) : -1;
                            m[u] &= m[u] - 1;
                            rev[u] = k[u] >= 0 ? ldc(g.r2 + b * L.K2 + k[u]) : 0;
                        }
                        sites_of_basis(L, b, [&](int i) __attribute__((always_inline)) {
                            int j[TG];
#pragma unroll
                            for (int u = 0; u < TG; ++u) j[u] = k[u] >= 0 ? L.nbr2[(int64_t)k[u] * N + i] : N;
                            const V3 s = sp(i, true);
#pragma unroll
                            for (int u = 0; u < TG; ++u) {
                                const bool ok = j[u] < N;
                                const V3 q = sp(j[u], ok);
#pragma unroll
                                for (int a = 0; a < 3; ++a) {
                                    const double x = rev[u] ? q.c[a] : (ok ? s.c[a] : 0.0);
#pragma unroll
                                    for (int c = 0; c < 3; ++c)
                                        acc[u][a * 3 + c] += x * (rev[u] ? (ok ? s.c[c] : 0.0) : q.c[c]);
                                }
                            }
                        });
                    }
                }
#pragma unroll
            for (int u = 0; u < TG; ++u) {
                block_sum<9>(acc[u], red);
                const int t = item * TG + u;
                if (threadIdx.x == 0 && t < n2)
                    for (int e = 0; e < 9; ++e) out[g.off_2 + t * 9 + e] = 0.5 * acc[u][e];
            }
        } else if (item < groups + 3 * n3 + 9 * n4) {
            // v0[p] v1[q] v2[r] (v3[t]) over the term's slots, v the spins in
            // the term's own index order (the slot's site sits at its role)
            const bool cub = item < groups + 3 * n3;
            const int w = cub ? item - groups : item - groups - 3 * n3;
            const int t = w / (cub ? 3 : 9), sl = w - t * (cub ? 3 : 9), p = sl % 3, q = sl / 3;
            const int K = cub ? L.K3 : L.K4;
            double acc[9];
#pragma unroll
            for (int e = 0; e < 9; ++e) acc[e] = 0.0;
            for (int b = 0; b < nb; ++b)
                for (int k0 = 0; k0 < K; k0 += 64) {
                    unsigned long long m = slots_of_term((cub ? g.t3 : g.t4) + b * K, k0, K, t);
                    for (; m; m &= m - 1) {
                        const int k = k0 + __builtin_ctzll(m);
                        const int role = ldc((cub ? g.r3 : g.r4) + b * K + k);
                        sites_of_basis(L, b, [&](int i) __attribute__((always_inline)) {
                            const int32_t *nb0 = cub ? L.nbr3 + (int64_t)k * 2 * N : L.nbr4 + (int64_t)k * 3 * N;
                            const int j1 = nb0[i], j2 = nb0[N + i], j3 = cub ? N : nb0[2 * (int64_t)N + i];
                            const bool ok = j1 < N;
                            V3 v[4] = {sp(i, ok), sp(j1, ok), sp(j2, ok), sp(j3, ok && !cub)};
                            const V3 own = v[0];
                            v[0] = role == 1 ? v[1] : role == 2 ? v[2] : role == 3 ? v[3] : own;
#pragma unroll
                            for (int x = 1; x < 4; ++x)
                                if (role == x) v[x] = own;
                            const double vp = p == 0 ? v[0].c[0] : p == 1 ? v[0].c[1] : v[0].c[2];
                            const double vq = q == 0 ? v[1].c[0] : q == 1 ? v[1].c[1] : v[1].c[2];
                            // cubic: (q, r) = (v1, v2) with p fixed; quartic:
                            // (r, t) = (v2, v3) with p and q fixed
#pragma unroll
                            for (int y = 0; y < 3; ++y) {
                                const double z = cub ? vp : vp * vq;
#pragma unroll
                                for (int x = 0; x < 3; ++x)
                                    acc[x + 3 * y] += z * ((cub ? v[1].c[x] : v[2].c[x]) * (cub ? v[2].c[y] : v[3].c[y]));
                            }
                        });
                    }
                }
            block_sum<9>(acc, red);
            if (threadIdx.x == 0) {
                double *o = cub ? out + g.off_3 + t * 27 + p : out + g.off_4 + t * 81 + p + 3 * q;
                for (int e = 0; e < 9; ++e) o[(cub ? 3 : 9) * e] = acc[e] / (cub ? 3.0 : 4.0);
            }
        } else {
            // -sum s per field entry and sum s s^T per onsite entry; several
            // bases may share an entry
            if (threadIdx.x == 0)
                for (int e = g.off_f; e < g.off_2; ++e) out[e] = 0.0;
            for (int b = 0; b < nb; ++b) {
                const int f = ldc(g.fsrc + b), o = ldc(g.osrc + b);
                if (f < 0 && o < 0) continue;
                double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // s (3), then xx xy xz yy yz zz
                sites_of_basis(L, b, [&](int i) __attribute__((always_inline)) {
                    const V3 s = sp(i, true);
                    v[0] += s.c[0];
                    v[1] += s.c[1];
                    v[2] += s.c[2];
                    v[3] += s.c[0] * s.c[0];
                    v[4] += s.c[0] * s.c[1];
                    v[5] += s.c[0] * s.c[2];
                    v[6] += s.c[1] * s.c[1];
                    v[7] += s.c[1] * s.c[2];
                    v[8] += s.c[2] * s.c[2];
                });
                block_sum<9>(v, red);
                if (threadIdx.x == 0) {
                    if (f >= 0)
                        for (int a = 0; a < 3; ++a) out[g.off_f + f * 3 + a] -= v[a];
                    if (o >= 0) {
                        const double m[9] = {v[3], v[4], v[5], v[4], v[6], v[7], v[5], v[7], v[8]};
                        for (int e = 0; e < 9; ++e) out[g.off_o + o * 9 + e] += m[e];
                    }
                }
            }
        }
    }
}

int grad_items(int n2, int n3, int n4) { return (n2 + TG - 1) / TG + 3 * n3 + 9 * n4 + 1; }

int grad_threads(int max_run) { return max_run < GRAD_THREADS ? (max_run + 63) / 64 * 64 : GRAD_THREADS; }

// grid: items on x, systems on y (65535 a launch at most: the rest in turn)
hipError_t launch_grad_couplings(int prec, const DevPools &P, const void *spins, int nsys, int grad_len, int items,
                                 int threads, double *dEdJ, hipStream_t st) {
    for (int s0 = 0; s0 < nsys; s0 += 65535) {
        DevPools Q = P;
        Q.sys = P.sys + s0;
        const dim3 grid(items, nsys - s0 < 65535 ? nsys - s0 : 65535);
        double *o = dEdJ + (int64_t)s0 * grad_len;
        if (prec == 32) hipLaunchKernelGGL((k_grad_couplings<float>), grid, dim3(threads), 0, st, Q, spins, o);
        else hipLaunchKernelGGL((k_grad_couplings<double>), grid, dim3(threads), 0, st, Q, spins, o);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace csmc
