// energy.hip -- total energy (hamiltonian.jl:70-132) and magnetisation
// (observables.jl:12-18) of every system of a batch, FP64.
//
// A reduction over the sites of each system: the batch's systems are cut into
// ranges of `chunk` sites (EnergyPlan), one workgroup sums each range, and
// where a system has more than one a second kernel adds their sums in range
// order, so the result does not depend on which workgroup ran first.  Bound: one read of the records plus the gathers
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

// the system and first site of range r; the first range of a system and its
// number of ranges
__device__ __forceinline__ void range_of(const EnergyPlan &pl, int r, int &sys, int &first) {
    if (pl.per) {
        sys = r / pl.per;
        first = (r - sys * pl.per) * pl.chunk;
    } else {
        sys = ldc(pl.range + 2 * r);
        first = ldc(pl.range + 2 * r + 1);
    }
}
__device__ __forceinline__ void ranges_of(const EnergyPlan &pl, int sys, int &r0, int &nr) {
    r0 = pl.per ? sys * pl.per : ldc(pl.off + sys);
    nr = pl.per ? pl.per : ldc(pl.off + sys + 1) - r0;
}

// the five energy parts of range blockIdx.x: into E / parts when it is the
// whole system, else into part[range][5]
template <class R, bool GEN>
__global__ __launch_bounds__(EN_THREADS) void k_energy(DevPools P, const void *spins, EnergyPlan pl, double *E,
                                                       double *parts, double *part) {
    __shared__ double red[BLOCK_SUM_SCRATCH];
    int sys, first;
    range_of(pl, (int)blockIdx.x, sys, first);
    const SysDev sd = P.sys[sys];
    const LatDev ld = P.lats[sd.lat];
    const LatView<double> L = lat_view<double>(ld, P.i32, P.runs + ld.run_off, P.coefD);
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    double p[5] = {0, 0, 0, 0, 0};
    range_sites(L, first, first + min(pl.chunk, L.N - first), [&](int b, int i) __attribute__((always_inline)) {
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
    if (L.N <= pl.chunk) {
        E[sys] = combine_energy(p);
        if (parts)
            for (int k = 0; k < 5; ++k) parts[sys * 5 + k] = p[k];
    } else {
        for (int k = 0; k < 5; ++k) part[(int64_t)blockIdx.x * 5 + k] = p[k];
    }
}

template <class R>
__global__ __launch_bounds__(EN_THREADS) void k_magnet(DevPools P, const void *spins, EnergyPlan pl, double *M,
                                                       double *part) {
    __shared__ double red[BLOCK_SUM_SCRATCH];
    int sys, first;
    range_of(pl, (int)blockIdx.x, sys, first);
    const SysDev sd = P.sys[sys];
    const int N = P.lats[sd.lat].N;
    const SpinsG<R> S = spins_at<R>(spins, sd.spin_off);
    double m[3] = {0, 0, 0};
    const int n = min(pl.chunk, N - first);
    for (int k = threadIdx.x; k < n; k += EN_THREADS) {
        const int i = first + k;
        const spin4<R> s = S.ld(i);
        m[0] += s.x;
        m[1] += s.y;
        m[2] += s.z;
    }
    block_sum<3>(m, red);
    if (threadIdx.x != 0) return;
    double *o = N <= pl.chunk ? M + (int64_t)sys * 3 : part + (int64_t)blockIdx.x * 3;
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

__global__ __launch_bounds__(64) void k_energy_sum(EnergyPlan pl, const double *part, double *E, double *parts) {
    const int sys = blockIdx.x;
    int r0, nr;
    ranges_of(pl, sys, r0, nr);
    if (nr == 1) return;  // k_energy wrote its result
    double p[5];
    sum_ranges<5>(part + (int64_t)r0 * 5, nr, p);
    if (threadIdx.x != 0) return;
    E[sys] = combine_energy(p);
    if (parts)
        for (int k = 0; k < 5; ++k) parts[(int64_t)sys * 5 + k] = p[k];
}

__global__ __launch_bounds__(64) void k_magnet_sum(EnergyPlan pl, const double *part, double *M) {
    const int sys = blockIdx.x;
    int r0, nr;
    ranges_of(pl, sys, r0, nr);
    if (nr == 1) return;
    double m[3];
    sum_ranges<3>(part + (int64_t)r0 * 3, nr, m);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) M[(int64_t)sys * 3 + k] = m[k];
}

// Sites per range: at least 1024 (four a thread), and no more ranges than
// give the device about 16 workgroups per CU over the sites of the whole
// batch, whatever their distribution: one square lattice of 262,144 FP64 sites
// beside 4095 of 64 takes 44 us (all of the large one in one workgroup
// if the batch counted as 4096 large ones: 734 us).
int energy_chunk(int64_t total_sites) {
    int64_t chunk = (total_sites + 4095) / 4096;
    chunk = (chunk + 1023) / 1024 * 1024;
    return (int)(chunk < 1024 ? 1024 : chunk);
}

hipError_t launch_energy(int prec, bool gen, const DevPools &P, const void *spins, int nsys, const EnergyPlan &pl,
                         double *E, double *parts, double *part, hipStream_t st) {
    const dim3 grid(pl.ranges), block(EN_THREADS);
    if (prec == 32) {
        if (gen) hipLaunchKernelGGL((k_energy<float, true>), grid, block, 0, st, P, spins, pl, E, parts, part);
        else hipLaunchKernelGGL((k_energy<float, false>), grid, block, 0, st, P, spins, pl, E, parts, part);
    } else {
        if (gen) hipLaunchKernelGGL((k_energy<double, true>), grid, block, 0, st, P, spins, pl, E, parts, part);
        else hipLaunchKernelGGL((k_energy<double, false>), grid, block, 0, st, P, spins, pl, E, parts, part);
    }
    if (pl.ranges > nsys) hipLaunchKernelGGL(k_energy_sum, dim3(nsys), dim3(64), 0, st, pl, part, E, parts);
    return hipGetLastError();
}

hipError_t launch_magnet(int prec, const DevPools &P, const void *spins, int nsys, const EnergyPlan &pl, double *M,
                         double *part, hipStream_t st) {
    const dim3 grid(pl.ranges), block(EN_THREADS);
    if (prec == 32) hipLaunchKernelGGL((k_magnet<float>), grid, block, 0, st, P, spins, pl, M, part);
    else hipLaunchKernelGGL((k_magnet<double>), grid, block, 0, st, P, spins, pl, M, part);
    if (pl.ranges > nsys) hipLaunchKernelGGL(k_magnet_sum, dim3(nsys), dim3(64), 0, st, pl, part, M);
    return hipGetLastError();
}

}  // namespace csmc
