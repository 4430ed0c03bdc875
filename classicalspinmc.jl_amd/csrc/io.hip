// io.hip -- spins and per-site evaluations between the device and the host
// (reference site order, double[N][3], lattice.jl:6,29-33), and small results.
//
// The host side of every transfer is page-locked memory that the kernels
// address directly, so a call is one launch and one wait: bound by that
// round trip (11 us) for small lattices, then by the bus (54 GB/s).  A copy
// engine's transfer to or from the caller's pageable array costs a second
// round trip and the runtime's own staging (64 B: 25 us; 221 KB: 30 against
// 20 us here); large uploads still go through the runtime's copy, see
// csmc_set_spins.  Threads take consecutive reference sites and pass their three
// components through LDS, so that the bus sees whole 16-byte accesses of
// consecutive lanes whatever the device order is.
#include "sweep.h"

namespace csmc {

namespace {
constexpr int IO_THREADS = 256;
}

// the 3 doubles of each of the block's sites from LDS to dst (16-byte
// aligned): doubles [0, 3 n) of the block
__device__ __forceinline__ void rows_out(const double *sh, double *dst, int n) {
    __syncthreads();
    const int n3 = 3 * n;
    for (int e = 2 * (int)threadIdx.x; e < n3; e += 2 * IO_THREADS) {
        if (e + 1 < n3)
            *reinterpret_cast<double2 *>(dst + e) = make_double2(sh[e], sh[e + 1]);
        else
            dst[e] = sh[e];
    }
}

// spins of the reference sites [r0, r0 + n) of one system to dst[n][3]
template <class R>
__global__ __launch_bounds__(IO_THREADS) void k_spins_out(DevPools P, const void *spins, int sys, int r0, int n,
                                                          double *dst) {
    __shared__ double sh[3 * IO_THREADS];
    const SysDev sd = P.sys[sys];
    const int b0 = blockIdx.x * IO_THREADS, m = min(IO_THREADS, n - b0), t = threadIdx.x;
    if (t < m) {
        const spin4<R> s = spins_at<R>(spins, sd.spin_off).ld(P.i32[P.lats[sd.lat].dev_off + r0 + b0 + t]);
        sh[3 * t] = s.x;
        sh[3 * t + 1] = s.y;
        sh[3 * t + 2] = s.z;
    }
    rows_out(sh, dst + 3 * (int64_t)b0, m);
}

// src[n][3] to the reference sites [r0, r0 + n) of one system
template <class R>
__global__ __launch_bounds__(IO_THREADS) void k_spins_in(DevPools P, void *spins, int sys, int r0, int n,
                                                         const double *src) {
    __shared__ double sh[3 * IO_THREADS];
    const SysDev sd = P.sys[sys];
    const int b0 = blockIdx.x * IO_THREADS, m = min(IO_THREADS, n - b0), t = threadIdx.x, n3 = 3 * m;
    const double *p = src + 3 * (int64_t)b0;
    for (int e = 2 * t; e < n3; e += 2 * IO_THREADS) {
        if (e + 1 < n3) {
            const double2 v = *reinterpret_cast<const double2 *>(p + e);
            sh[e] = v.x;
            sh[e + 1] = v.y;
        } else {
            sh[e] = p[e];
        }
    }
    __syncthreads();
    if (t < m)
        spins_at<R>(spins, sd.spin_off)
            .st(P.i32[P.lats[sd.lat].dev_off + r0 + b0 + t],
                spin4<R>{(R)sh[3 * t], (R)sh[3 * t + 1], (R)sh[3 * t + 2], R(0)});
}

// get_local_field (H[n][3]) and energy(lattice, point) (e[n]) of the
// reference sites [r0, r0 + n), either may be null
template <class R>
__global__ __launch_bounds__(IO_THREADS) void k_site_eval(DevPools P, const void *spins, int sys, int r0, int n,
                                                          double *H, double *e) {
    __shared__ double sh[3 * IO_THREADS];
    const SysDev sd = P.sys[sys];
    const LatDev ld = P.lats[sd.lat];
    const LatView<double> L = lat_view<double>(ld, P.i32, P.runs + ld.run_off, P.coefD);
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    const int b0 = blockIdx.x * IO_THREADS, m = min(IO_THREADS, n - b0), t = threadIdx.x;
    if (t < m) {
        const int i = P.i32[ld.dev_off + r0 + b0 + t];
        const int b = L.sub[i];
        const spin4<double> s = to_d<R>(S.ld(i));
        double F[3], Hl[3];
        interaction_field<double, double>(L, NbrG{L.nbr2, L.N}, b, i, [&](int j) { return to_d<R>(S.ld(j)); }, F);
        local_field<double, double>(L, b, s, F, Hl);
        for (int a = 0; a < 3; ++a) sh[3 * t + a] = Hl[a];
        if (e) {
            const double *h = L.field + b * 3;
            e[b0 + t] = onsite_energy<double, double>(L, b, s.x, s.y, s.z) + s.x * F[0] + s.y * F[1] + s.z * F[2] -
                        (s.x * h[0] + s.y * h[1] + s.z * h[2]);
        }
    }
    if (H) rows_out(sh, H + 3 * (int64_t)b0, m);
}

// up to EXPORT_MAX blocks of 4-byte words to page-locked memory
__global__ __launch_bounds__(IO_THREADS) void k_export(ExportArgs a) {
    for (int k = 0; k < a.n; ++k)
        for (int64_t i = (int64_t)blockIdx.x * IO_THREADS + threadIdx.x; i < a.words[k];
             i += (int64_t)gridDim.x * IO_THREADS)
            a.dst[k][i] = a.src[k][i];
}

hipError_t launch_spins_out(int prec, const DevPools &P, const void *spins, int sys, int r0, int n, double *dst,
                            hipStream_t st) {
    const dim3 grid((n + IO_THREADS - 1) / IO_THREADS);
    if (prec == 32)
        hipLaunchKernelGGL((k_spins_out<float>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, dst);
    else
        hipLaunchKernelGGL((k_spins_out<double>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, dst);
    return hipGetLastError();
}

hipError_t launch_spins_in(int prec, const DevPools &P, void *spins, int sys, int r0, int n, const double *src,
                           hipStream_t st) {
    const dim3 grid((n + IO_THREADS - 1) / IO_THREADS);
    if (prec == 32)
        hipLaunchKernelGGL((k_spins_in<float>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, src);
    else
        hipLaunchKernelGGL((k_spins_in<double>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, src);
    return hipGetLastError();
}

hipError_t launch_site_eval(int prec, const DevPools &P, const void *spins, int sys, int r0, int n, double *H,
                            double *e, hipStream_t st) {
    const dim3 grid((n + IO_THREADS - 1) / IO_THREADS);
    if (prec == 32)
        hipLaunchKernelGGL((k_site_eval<float>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, H, e);
    else
        hipLaunchKernelGGL((k_site_eval<double>), grid, dim3(IO_THREADS), 0, st, P, spins, sys, r0, n, H, e);
    return hipGetLastError();
}

hipError_t launch_export(const ExportArgs &a, hipStream_t st) {
    int64_t most = 1;
    for (int k = 0; k < a.n; ++k) most = most < a.words[k] ? a.words[k] : most;
    const int64_t blocks = (most + IO_THREADS - 1) / IO_THREADS;
    hipLaunchKernelGGL(k_export, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(IO_THREADS), 0, st, a);
    return hipGetLastError();
}

}  // namespace csmc
