// energy.hip -- total energy (hamiltonian.jl:70-132) and magnetisation
// (observables.jl:12-18) of every system of a batch, FP64.
//
// A reduction over the sites of each system: workgroup (c, sys) sums the
// c-th range of `chunk` sites, and with more than one range a second kernel
// adds the ranges' sums in range order, so the result does not depend on
// which workgroup ran first.  Bound: one read of the records plus the gathers
// of the partners through L2.  64 FP32 systems of 524,288 sites (403 MB):
// energy 166 us, magnetisation 68 us; one 1024-thread workgroup per system,
// which leaves 192 of the 256 CUs idle, took 996 and 253 us.
#include "sweep.h"

namespace csmc {

namespace {
constexpr int EN_THREADS = 256;
}

// f(b, i) for this thread's sites of the range [i0, i1): the runs it meets
// in turn, so the basis b is wave-uniform
template <class F>
__device__ __forceinline__ void range_sites(const LatView<double> &L, int i0, int i1, F &&f) {
    for (int r = ldc(L.colrun); r < ldc(L.colrun + L.ncol); ++r) {
        const int32_t *run = reinterpret_cast<const int32_t *>(L.runs + r);
        const int lo = max(ldc(run), i0), hi = min(ldc(run + 1), i1);
        if (lo >= hi) continue;
        const int b = ldc(run + 2);
        for (int i = lo + (int)threadIdx.x; i < hi; i += EN_THREADS) f(b, i);
    }
}

// the five energy parts of range blockIdx.x of system blockIdx.y: into
// E / parts when the system is one range, else into part[sys][range][5]
template <class R, bool GEN>
__global__ __launch_bounds__(EN_THREADS) void k_energy(DevPools P, const void *spins, int s0, int chunk, double *E,
                                                       double *parts, double *part) {
    __shared__ double red[BLOCK_SUM_SCRATCH];
    const int sys = s0 + (int)blockIdx.y;
    const SysDev sd = P.sys[sys];
    const LatDev ld = P.lats[sd.lat];
    const LatView<double> L = lat_view<double>(ld, P.i32, P.runs + ld.run_off, P.coefD);
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    double p[5] = {0, 0, 0, 0, 0};
    const int64_t first = (int64_t)blockIdx.x * chunk, last = first + chunk;
    if (first < L.N)
        range_sites(L, (int)first, (int)(last < L.N ? last : L.N), [&](int b, int i) __attribute__((always_inline)) {
            const double *h = L.field + b * 3;
            const spin4<double> s = to_d<R>(S.ld(i));
            double F2[3], F3[3], F4[3];
            field_parts<GEN>(L, NbrG{L.nbr2, L.N}, b, i, [&](int j) { return to_d<R>(S.ld(j)); }, F2, F3, F4);
            p[0] += s.x * F2[0] + s.y * F2[1] + s.z * F2[2];
            if (GEN) {
                p[1] += s.x * F3[0] + s.y * F3[1] + s.z * F3[2];
                p[2] += s.x * F4[0] + s.y * F4[1] + s.z * F4[2];
            }
            p[3] -= s.x * ldc(h) + s.y * ldc(h + 1) + s.z * ldc(h + 2);
            p[4] += onsite_energy<double, double>(L, b, s.x, s.y, s.z);
        });
    block_sum<5>(p, red);
    if (threadIdx.x != 0) return;
    if (gridDim.x == 1) {
        E[sys] = combine_energy(p);
        if (parts)
            for (int k = 0; k < 5; ++k) parts[sys * 5 + k] = p[k];
    } else {
        for (int k = 0; k < 5; ++k) part[((int64_t)sys * gridDim.x + blockIdx.x) * 5 + k] = p[k];
    }
}

template <class R>
__global__ __launch_bounds__(EN_THREADS) void k_magnet(DevPools P, const void *spins, int s0, int chunk, double *M,
                                                       double *part) {
    __shared__ double red[BLOCK_SUM_SCRATCH];
    const int sys = s0 + (int)blockIdx.y;
    const SysDev sd = P.sys[sys];
    const int N = P.lats[sd.lat].N;
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    double m[3] = {0, 0, 0};
    const int64_t first = (int64_t)blockIdx.x * chunk, last = first + chunk;
    for (int64_t i = first + threadIdx.x; i < (last < N ? last : N); i += EN_THREADS) {
        const spin4<R> s = S.ld(i);
        m[0] += s.x;
        m[1] += s.y;
        m[2] += s.z;
    }
    block_sum<3>(m, red);
    if (threadIdx.x != 0) return;
    double *o = gridDim.x == 1 ? M + sys * 3 : part + ((int64_t)sys * gridDim.x + blockIdx.x) * 3;
    for (int k = 0; k < 3; ++k) o[k] = m[k];
}

// the ranges' sums of each system, added in range order by the lanes of one
// wave (lane l takes ranges l, l + 64, ...) and then over the lanes
template <int NV>
__device__ __forceinline__ void sum_ranges(const double *part, int nc, double v[NV]) {
    for (int k = 0; k < NV; ++k) v[k] = 0.0;
    for (int c = threadIdx.x; c < nc; c += 64)
        for (int k = 0; k < NV; ++k) v[k] += part[(int64_t)c * NV + k];
    for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
}

__global__ __launch_bounds__(64) void k_energy_sum(const double *part, int nc, double *E, double *parts) {
    const int sys = blockIdx.x;
    double p[5];
    sum_ranges<5>(part + (int64_t)sys * nc * 5, nc, p);
    if (threadIdx.x != 0) return;
    E[sys] = combine_energy(p);
    if (parts)
        for (int k = 0; k < 5; ++k) parts[sys * 5 + k] = p[k];
}

__global__ __launch_bounds__(64) void k_magnet_sum(const double *part, int nc, double *M) {
    const int sys = blockIdx.x;
    double m[3];
    sum_ranges<3>(part + (int64_t)sys * nc * 3, nc, m);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) M[sys * 3 + k] = m[k];
}

// Sites per range: at least 1024 (four a thread), and no more ranges than
// give the device about 16 workgroups per CU over the whole batch.  The
// ranges' sums (at most 5 doubles per 1024 sites) then fit the batch's
// staging buffer behind the results.
static int range_sites_of(int nsys, int maxN) {
    const int64_t total = (int64_t)nsys * maxN;
    int64_t chunk = (total + 4095) / 4096;
    chunk = (chunk + 1023) / 1024 * 1024;
    return (int)(chunk < 1024 ? 1024 : chunk);
}

template <class R>
static void energy_r(bool gen, dim3 grid, const DevPools &P, const void *spins, int s0, int chunk, double *E,
                     double *parts, double *part, hipStream_t st) {
    if (gen) hipLaunchKernelGGL((k_energy<R, true>), grid, dim3(EN_THREADS), 0, st, P, spins, s0, chunk, E, parts, part);
    else hipLaunchKernelGGL((k_energy<R, false>), grid, dim3(EN_THREADS), 0, st, P, spins, s0, chunk, E, parts, part);
}

hipError_t launch_energy(int prec, bool gen, const DevPools &P, const void *spins, int nsys, int maxN, double *E,
                         double *parts, double *part, hipStream_t st) {
    const int chunk = range_sites_of(nsys, maxN), nc = (maxN + chunk - 1) / chunk;
    for (int s0 = 0; s0 < nsys; s0 += 65535) {
        const dim3 grid(nc, nsys - s0 < 65535 ? nsys - s0 : 65535);
        if (prec == 32) energy_r<float>(gen, grid, P, spins, s0, chunk, E, parts, part, st);
        else energy_r<double>(gen, grid, P, spins, s0, chunk, E, parts, part, st);
    }
    if (nc > 1) hipLaunchKernelGGL(k_energy_sum, dim3(nsys), dim3(64), 0, st, part, nc, E, parts);
    return hipGetLastError();
}

hipError_t launch_magnet(int prec, const DevPools &P, const void *spins, int nsys, int maxN, double *M, double *part,
                         hipStream_t st) {
    const int chunk = range_sites_of(nsys, maxN), nc = (maxN + chunk - 1) / chunk;
    for (int s0 = 0; s0 < nsys; s0 += 65535) {
        const dim3 grid(nc, nsys - s0 < 65535 ? nsys - s0 : 65535);
        if (prec == 32)
            hipLaunchKernelGGL((k_magnet<float>), grid, dim3(EN_THREADS), 0, st, P, spins, s0, chunk, M, part);
        else
            hipLaunchKernelGGL((k_magnet<double>), grid, dim3(EN_THREADS), 0, st, P, spins, s0, chunk, M, part);
    }
    if (nc > 1) hipLaunchKernelGGL(k_magnet_sum, dim3(nsys), dim3(64), 0, st, part, nc, M);
    return hipGetLastError();
}

// doubles of scratch the ranges' sums need
size_t energy_scratch(int nsys, int maxN) {
    const int chunk = range_sites_of(nsys, maxN), nc = (maxN + chunk - 1) / chunk;
    return nc > 1 ? (size_t)nsys * nc * 5 : 0;
}

}  // namespace csmc
