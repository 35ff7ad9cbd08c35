// Diagnostics in FP64: probe (probe_global.F90:41-77), control-volume stress drag (flux_X.F90,
// flux_Y.F90), momentum-exchange drag (no reference counterpart), global means (diagno.F90) and the
// velocity / vorticity fields of the binary VTK writers (vtk_*.binary.F90).
//
// Populations are converted to double on load whatever the storage.  The control-volume drag
// computes one stress per face site on the GPU with the reference's expression order and returns
// them in the reference's loop order, so the host sums them exactly as flux_X/flux_Y do.  The
// momentum-exchange force and the global means are wavefront-reduced on the GPU in a fixed order
// (deterministic run to run).
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "eup_internal.h"
#include "eup_transfer.h"

// Device scratch of eup_drag_cv_noalloc: the per-site stresses of the two faces of one axis,
// at most kNoAllocFace sites per face (16 MiB per GPU, held for the life of the process).  Host
// code never passes this name to a kernel or a copy: it is a host-side stand-in; the device
// address comes from hipGetSymbolAddress, once per device (noalloc_scratch).
static constexpr int64_t kNoAllocFace = int64_t(1) << 20;
static __device__ __align__(256) double scratch[2 * kNoAllocFace];

namespace eup {

namespace {

constexpr int kRedBlocks = 2048;
constexpr int kTicketBlocks = 256; // largest grid whose last block adds the partial sums
constexpr int64_t kResultBytes = 4096; // of pinned memory for a few results

// population q of interior site (i, j, k) (1-based) as double
struct ParityAcc {
    const double *p[19]; // population q at its offset base
    int l, m, n, pitch;
    __device__ __forceinline__ double operator()(int q, int i, int j, int k) const
    {
        return p[q][(int64_t)i + (int64_t)pitch * ((int64_t)j + (int64_t)(m + 2) * k)];
    }
};

template <typename S> struct PhysAcc {
    using value_type = S;
    const S *base;
    PopIndex ix;
    DevRef ref;
    int l, m, n;
    __device__ __forceinline__ double operator()(int q, int i, int j, int k) const
    {
        return Store<S>::load64(base[ix(q, i - 1, j - 1, k - 1)], ref.r[q], q);
    }
};

template <typename Acc>
__global__ void k_site19(Acc acc, int i, int j, int k, double *out)
{
    const int q = threadIdx.x;
    if (q < 19) out[q] = acc(q, i, j, k);
}

// flux_X.F90:173-242 / flux_Y.F90:168-242 for one site; axis 0 -> sigma_xx, 1 -> sigma_xy
__device__ double site_sigma(const double *x, double omega, int axis)
{
    const double P1 = 1.0 / 18.0, P2 = 1.0 / 36.0, RF = 3.0, QF = 1.5;
    double rho = +x[0] + x[1] + x[2] + x[3] + x[4] + x[5] + x[6] + x[7] + x[8] + x[9] + x[10]
                 + x[11] + x[12] + x[13] + x[14] + x[15] + x[16] + x[17] + x[18];
    double rhoinv = 1.0 / rho;
    double xj = +(x[0] + x[1] + x[2] + x[3] + x[4] - x[9] - x[10] - x[11] - x[12] - x[13]) * rhoinv;
    double yj = +(x[2] + x[6] + x[7] + x[8] + x[11] - x[0] - x[9] - x[15] - x[16] - x[17]) * rhoinv;
    double zj = +(x[3] + x[5] + x[6] + x[12] + x[17] - x[1] - x[8] - x[10] - x[14] - x[15]) * rhoinv;
    double cvsq = xj * xj + yj * yj + zj * zj;
    double fe[18];
    fe[0] = rho * P2 * (1.0 + RF * (xj - yj) + QF * (3.0 * (xj - yj) * (xj - yj) - cvsq));
    fe[1] = rho * P2 * (1.0 + RF * (xj - zj) + QF * (3.0 * (xj - zj) * (xj - zj) - cvsq));
    fe[2] = rho * P2 * (1.0 + RF * (xj + yj) + QF * (3.0 * (xj + yj) * (xj + yj) - cvsq));
    fe[3] = rho * P2 * (1.0 + RF * (xj + zj) + QF * (3.0 * (xj + zj) * (xj + zj) - cvsq));
    fe[4] = rho * P1 * (1.0 + RF * (xj) + QF * (3.0 * (xj) * (xj)-cvsq));
    fe[5] = rho * P1 * (1.0 + RF * (zj) + QF * (3.0 * (zj) * (zj)-cvsq));
    fe[6] = rho * P2 * (1.0 + RF * (yj + zj) + QF * (3.0 * (yj + zj) * (yj + zj) - cvsq));
    fe[7] = rho * P1 * (1.0 + RF * (yj) + QF * (3.0 * (yj) * (yj)-cvsq));
    fe[8] = rho * P2 * (1.0 + RF * (yj - zj) + QF * (3.0 * (yj - zj) * (yj - zj) - cvsq));
    fe[9] = rho * P2 * (1.0 + RF * (-xj - yj) + QF * (3.0 * (xj + yj) * (xj + yj) - cvsq));
    fe[10] = rho * P2 * (1.0 + RF * (-xj - zj) + QF * (3.0 * (xj + zj) * (xj + zj) - cvsq));
    fe[11] = rho * P2 * (1.0 + RF * (-xj + yj) + QF * (3.0 * (xj - yj) * (xj - yj) - cvsq));
    fe[12] = rho * P2 * (1.0 + RF * (-xj + zj) + QF * (3.0 * (xj - zj) * (xj - zj) - cvsq));
    fe[13] = rho * P1 * (1.0 + RF * (-xj) + QF * (3.0 * (xj) * (xj)-cvsq));
    fe[14] = rho * P1 * (1.0 + RF * (-zj) + QF * (3.0 * (zj) * (zj)-cvsq));
    fe[15] = rho * P2 * (1.0 + RF * (-yj - zj) + QF * (3.0 * (yj + zj) * (yj + zj) - cvsq));
    fe[16] = rho * P1 * (1.0 + RF * (-yj) + QF * (3.0 * (yj) * (yj)-cvsq));
    fe[17] = rho * P2 * (1.0 + RF * (-yj + zj) + QF * (3.0 * (yj - zj) * (yj - zj) - cvsq));
    const double cxd[18] = {1, 1, 1, 1, 1, 0, 0, 0, 0, -1, -1, -1, -1, -1, 0, 0, 0, 0};
    const double cyd[18] = {-1, 0, 1, 0, 0, 0, 1, 1, 1, -1, 0, 1, 0, 0, 0, -1, -1, -1};
    const double c = (1 - 0.5 * omega);
    double sg;
    if (axis == 0) {
        sg = -rho / RF;
        for (int q = 0; q < 18; ++q) sg = sg - c * cxd[q] * cxd[q] * (x[q] - fe[q]);
    } else {
        sg = 0.0;
        for (int q = 0; q < 18; ++q) sg = sg - c * cxd[q] * cyd[q] * (x[q] - fe[q]);
    }
    return sg;
}

// face sites of one drag face in the reference's loop order (k outer, then j or i)
template <typename Acc>
__global__ void k_sigma(Acc acc, int axis, int plane, int lo, int hi, int k1, int k2, double omega,
                        double *out)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nin = hi - lo + 1;
    const int64_t total = (int64_t)nin * (k2 - k1 + 1);
    if (t >= total) return;
    const int u = lo + (int)(t % nin);
    const int k = k1 + (int)(t / nin);
    const int i = axis == 0 ? plane : u;
    const int j = axis == 0 ? u : plane;
    double x[19];
#pragma unroll
    for (int q = 0; q < 19; ++q) x[q] = acc(q, i, j, k);
    out[t] = site_sigma(x, omega, axis);
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// block partial sums of NV values; lane 0 of the block writes partial[blockIdx.x * NV + v]
template <int NV>
__device__ __forceinline__ void block_reduce(double (&v)[NV], double *partial)
{
    __shared__ double sh[NV][kBlock / 64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        double s = wave_sum(v[c]);
        if (lane == 0) sh[c][w] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            double s = 0.0;
            for (int ww = 0; ww < kBlock / 64; ++ww) s += sh[c][ww];
            partial[(int64_t)blockIdx.x * NV + c] = s;
        }
    }
}

// The blocks' partial sums and, with a ticket (0 between launches), by the block that ends last their
// sum, into pinned host memory: thread b of that block adds the partials b, b + 256, ..., so the
// order does not depend on which block it is, and is that of k_final.  One launch instead of two
// and no copy of the result: a step, its drag and a probe on 48 x 24 x 16 take 54.6 us instead of 78.4.  Every ticket is a release to
// the other XCDs, and 2048 of them cost more than the second launch: kTicketBlocks.
template <int NV>
__device__ __forceinline__ void grid_reduce(double (&v)[NV], double *partial, uint32_t *ticket, double *out)
{
    __shared__ bool last;
    block_reduce<NV>(v, partial);
    if (!ticket) return;
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
    for (int c = 0; c < NV; ++c) v[c] = 0.0;
    for (uint32_t b = threadIdx.x; b < gridDim.x; b += kBlock)
#pragma unroll
        for (int c = 0; c < NV; ++c) v[c] += partial[(int64_t)b * NV + c];
    block_reduce<NV>(v, out - (int64_t)blockIdx.x * NV);
    if (threadIdx.x == 0) *ticket = 0;
}

template <int NV>
__global__ __launch_bounds__(kBlock) void k_final(const double *partial, int nblocks, double *out)
{
    double v[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) v[c] = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += kBlock)
#pragma unroll
        for (int c = 0; c < NV; ++c) v[c] += partial[(int64_t)b * NV + c];
    block_reduce<NV>(v, out);
}

// momentum exchange over all interior sites (parity layout), neighbour test on the solid flags
template <typename Acc>
__global__ __launch_bounds__(kBlock) void k_mem_sites(Acc acc, const uint8_t *solid, int xopen,
                                                      double *partial)
{
    const int l = acc.l, m = acc.m, n = acc.n;
    const int64_t N = (int64_t)l * m * n;
    double v[3] = {0.0, 0.0, 0.0};
    const int cxs[18] = {1, 1, 1, 1, 1, 0, 0, 0, 0, -1, -1, -1, -1, -1, 0, 0, 0, 0};
    const int cys[18] = {-1, 0, 1, 0, 0, 0, 1, 1, 1, -1, 0, 1, 0, 0, 0, -1, -1, -1};
    const int czs[18] = {0, -1, 0, 1, 0, 1, 1, 0, -1, 0, -1, 0, 1, 0, -1, -1, 0, 1};
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < N; s += (int64_t)gridDim.x * blockDim.x) {
        if (solid[s]) continue;
        const int i = (int)(s % l);
        const int64_t r = s / l;
        const int j = (int)(r % m), k = (int)(r / m);
        for (int p = 0; p < 18; ++p) {
            int ti = i + cxs[p], tj = (j + cys[p] + m) % m, tk = (k + czs[p] + n) % n;
            if (ti < 0 || ti >= l) {
                if (xopen) continue;
                ti = (ti + l) % l;
            }
            if (!solid[(int64_t)ti + (int64_t)l * ((int64_t)tj + (int64_t)m * tk)]) continue;
            const double f2 = 2.0 * acc(p, i + 1, j + 1, k + 1);
            v[0] += cxs[p] * f2;
            v[1] += cys[p] * f2;
            v[2] += czs[p] * f2;
        }
    }
    block_reduce<3>(v, partial);
}

// momentum exchange over the mixed tiles only (physics layout): bit opp(p) of the link mask of a
// fluid site says that x + c_p is solid
template <typename S>
__global__ __launch_bounds__(kBlock) void k_mem_tiles(PhysAcc<S> acc, const int32_t *mixed_list,
                                                      int64_t nmixed, const uint32_t *link, int tpr,
                                                      double *partial, uint32_t *ticket, double *out)
{
    const int cxs[18] = {1, 1, 1, 1, 1, 0, 0, 0, 0, -1, -1, -1, -1, -1, 0, 0, 0, 0};
    const int cys[18] = {-1, 0, 1, 0, 0, 0, 1, 1, 1, -1, 0, 1, 0, 0, 0, -1, -1, -1};
    const int czs[18] = {0, -1, 0, 1, 0, 1, 1, 0, -1, 0, -1, 0, 1, 0, -1, -1, 0, 1};
    const int opp[18] = {11, 12, 9, 10, 13, 14, 15, 16, 17, 2, 3, 0, 1, 4, 5, 6, 7, 8};
    double v[3] = {0.0, 0.0, 0.0};
    const int lane = threadIdx.x & 63;
    const int64_t wpb = kBlock / 64;
    for (int64_t c = (int64_t)blockIdx.x * wpb + (threadIdx.x >> 6); c < nmixed; c += (int64_t)gridDim.x * wpb) {
        const uint32_t lm = link[c * kTile + lane];
        if (lm == 0 || (lm & 0x80000000u)) continue;
        const int64_t t = mixed_list[c];
        const int64_t row = t / tpr;
        const int i = (int)(t - row * tpr) * kTile + lane;
        if (i >= acc.l) continue;
        const int j = (int)(row % acc.m), k = (int)(row / acc.m);
        // all 18 loads at once (one behind a branch each waited for the one before: 170 x 77 x 51 with 3 %
        // scattered solid sites, FP32, 25.5 us, now 12.1); a site without
        // the link reads its population 0 and adds a zero, which changes no sum
        S x[18];
#pragma unroll
        for (int p = 0; p < 18; ++p) x[p] = acc.base[acc.ix((lm >> opp[p]) & 1u ? p : 0, i, j, k)];
#pragma unroll
        for (int p = 0; p < 18; ++p) {
            const double f2 = (lm >> opp[p]) & 1u ? 2.0 * Store<S>::load64(x[p], acc.ref.r[p], p) : 0.0;
            v[0] += cxs[p] * f2;
            v[1] += cys[p] * f2;
            v[2] += czs[p] * f2;
        }
    }
    grid_reduce<3>(v, partial, ticket, out);
}

// velocity of one site as the reference's binary VTK writers compute it (vtk_xy.binary.F90:93-115):
// momenta and density summed in FP64 in the written order, each rounded to float, divided in
// float (IEEE division; the translation unit is built without contraction)
template <typename Acc>
__device__ __forceinline__ void vtk_site(const Acc &acc, int i, int j, int k, float *o)
{
    double x[19];
#pragma unroll
    for (int q = 0; q < 19; ++q) x[q] = acc(q, i, j, k);
    const float u = (float)(x[0] + x[1] + x[2] + x[3] + x[4] - x[9] - x[10] - x[11] - x[12] - x[13]);
    const float w = (float)(x[2] + x[6] + x[7] + x[8] + x[11] - x[0] - x[9] - x[15] - x[16] - x[17]);
    const float v = (float)(x[3] + x[5] + x[6] + x[12] + x[17] - x[1] - x[8] - x[10] - x[14] - x[15]);
    const float den = (float)(x[0] + x[1] + x[2] + x[3] + x[4] + x[5] + x[6] + x[7] + x[8] + x[9]
                              + x[10] + x[11] + x[12] + x[13] + x[14] + x[15] + x[16] + x[17] + x[18]);
    o[0] = u / den;
    o[1] = w / den;
    o[2] = v / den;
}

// `count` velocities from site t0 on of a plane in the writers' loop order, into pinned host memory:
// plane 0 = yz at x = index (k, j), 1 = xz at y = index (k, i), 2 = xy at z = index (j, i), 3 = the
// lattice (k, j, i).  The block's 3 x 256 floats go through LDS, so that what crosses the bus is whole
// lines.
template <typename Acc>
__global__ __launch_bounds__(kBlock) void k_vtk_velocity(Acc acc, int plane, int index, int64_t t0, int64_t count,
                                                         float *out)
{
    __shared__ __align__(16) float sh[3 * kBlock];
    const int64_t b0 = (int64_t)blockIdx.x * kBlock;
    const int nb = (int)(count - b0 < kBlock ? count - b0 : kBlock);
    if ((int)threadIdx.x < nb) {
        const int64_t t = t0 + b0 + threadIdx.x;
        const uint32_t w = plane == 0 ? acc.m : acc.l; // the fastest coordinate's extent
        const uint64_t r = (uint64_t)t / w;
        const int u = 1 + (int)((uint64_t)t - r * w);
        int i = u, j = index, k = index;
        if (plane == 0) {
            i = index; j = u; k = 1 + (int)r;
        } else if (plane == 1) {
            k = 1 + (int)r;
        } else if (plane == 2) {
            j = 1 + (int)r;
        } else {
            const uint64_t z = r / (uint32_t)acc.m;
            j = 1 + (int)(r - z * (uint32_t)acc.m);
            k = 1 + (int)z;
        }
        vtk_site(acc, i, j, k, sh + 3 * threadIdx.x);
    }
    __syncthreads();
    float *o = out + 3 * b0;
    if (nb == kBlock) {
        if (threadIdx.x < 3 * kBlock / 4)
            reinterpret_cast<float4 *>(o)[threadIdx.x] = reinterpret_cast<const float4 *>(sh)[threadIdx.x];
    } else {
        for (int e = threadIdx.x; e < 3 * nb; e += kBlock) o[e] = sh[e];
    }
}

// vorticity of the xy plane z = k0 as vtk_om.binary.F90:88-131 computes it (i = 2..l-1 fastest,
// j = 2..m-1): densities rounded to float; in each momentum only the last population is divided
// by the density, as the writer's expression reads; the difference is formed in float
template <typename Acc>
__global__ void k_vtk_vorticity(Acc acc, int k0, int64_t t0, int64_t count, float *out)
{
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, t = t0 + o;
    const int l = acc.l;
    if (o >= count) return;
    const int i = 2 + (int)(t % (l - 2)), j = 2 + (int)(t / (l - 2));
    const int di[4] = {0, 0, -1, 1}, dj[4] = {1, -1, 0, 0}; // up, down, left, right
    float mom[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        double x[19];
#pragma unroll
        for (int q = 0; q < 19; ++q) x[q] = acc(q, i + di[s], j + dj[s], k0);
        const float d = (float)(x[0] + x[1] + x[2] + x[3] + x[4] + x[5] + x[6] + x[7] + x[8] + x[9]
                                + x[10] + x[11] + x[12] + x[13] + x[14] + x[15] + x[16] + x[17] + x[18]);
        if (s < 2)
            mom[s] = (float)(x[0] + x[1] + x[2] + x[3] + x[4] - x[9] - x[10] - x[11] - x[12] - x[13] / (double)d);
        else
            mom[s] = (float)(x[2] + x[6] + x[7] + x[8] + x[11] - x[0] - x[9] - x[15] - x[16] - x[17] / (double)d);
    }
    out[o] = 0.5f * (mom[0] - mom[1]) - 0.5f * (mom[3] - mom[2]);
}

// Site numbers in 32 bits (divided twice per site; in 64 bits 192 x 768 x 768, e3m12, took 1.63 ms, now
// 1.47): a lattice has less than 2^31 sites, and the last stride past them fits as well.
template <typename Acc>
__global__ __launch_bounds__(kBlock) void k_diagno(Acc acc, const uint8_t *solid, double *partial)
{
    const uint32_t l = (uint32_t)acc.l, m = (uint32_t)acc.m;
    const uint32_t N = l * m * (uint32_t)acc.n;
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < N; s += gridDim.x * kBlock) {
        double rho, xj, yj, zj;
        if (solid[s]) {
            rho = 1.0; xj = 0.0; yj = 0.0; zj = 0.0;
        } else {
            const uint32_t r = s / l, z = r / m;
            const int i = 1 + (int)(s - r * l), j = 1 + (int)(r - z * m), k = 1 + (int)z;
            double x[19];
#pragma unroll
            for (int q = 0; q < 19; ++q) x[q] = acc(q, i, j, k);
            rho = +x[0] + x[1] + x[2] + x[3] + x[4] + x[5] + x[6] + x[7] + x[8] + x[9] + x[10]
                  + x[11] + x[12] + x[13] + x[14] + x[15] + x[16] + x[17] + x[18];
            const double rhoinv = 1.0 / rho;
            xj = +(x[0] + x[1] + x[2] + x[3] + x[4] - x[9] - x[10] - x[11] - x[12] - x[13]) * rhoinv;
            yj = +(x[2] + x[6] + x[7] + x[8] + x[11] - x[0] - x[9] - x[15] - x[16] - x[17]) * rhoinv;
            zj = +(x[3] + x[5] + x[6] + x[12] + x[17] - x[1] - x[8] - x[10] - x[14] - x[15]) * rhoinv;
        }
        v[0] += rho;
        v[1] += xj;
        v[2] += yj;
        v[3] += zj;
        v[4] += xj * xj + yj * yj + zj * zj;
    }
    block_reduce<5>(v, partial);
}

ParityAcc parity_acc(Handle *h)
{
    ParityAcc a;
    const double *base = static_cast<const double *>(h->buf[h->cur]);
    for (int q = 0; q < 19; ++q) a.p[q] = base + (int64_t)q * h->stride + h->poff;
    a.l = h->g.l;
    a.m = h->g.m;
    a.n = h->g.n;
    a.pitch = h->ppitch;
    return a;
}

template <typename S> PhysAcc<S> phys_acc(Handle *h)
{
    PhysAcc<S> a;
    a.base = static_cast<const S *>(h->buf[h->cur]);
    a.ix = pop_index(h);
    a.ref = dev_ref(h);
    a.l = h->g.l;
    a.m = h->g.m;
    a.n = h->g.n;
    return a;
}

// run f(acc) with the accessor of the handle's layout
template <typename F> int with_acc(Handle *h, F &&f)
{
    if (h->cfg.mode == EUP_MODE_PARITY) return f(parity_acc(h));
    switch (h->cfg.storage) {
    case EUP_STORE_F64: return f(phys_acc<double>(h));
    case EUP_STORE_F32: return f(phys_acc<float>(h));
    case EUP_STORE_F16: return f(phys_acc<_Float16>(h));
    case EUP_STORE_BF16: return f(phys_acc<bf16_t>(h));
    case EUP_STORE_E3M12: return f(phys_acc<e3m12_t>(h));
    }
    return fail(h, EUP_EINVAL, "unknown storage");
}

int ensure_diag(Handle *h, int64_t len)
{
    if (h->diag_len >= len) return 0;
    hipFree(h->diag);
    h->diag = nullptr;
    h->diag_len = 0;
    if (hip_check(h, hipMalloc((void **)&h->diag, sizeof(double) * len), "hipMalloc diag")) return EUP_EHIP;
    h->diag_len = len;
    return 0;
}

} // namespace

int diag_site(Handle *h, int i, int j, int k, double out[19])
{
    if (pinned_ready(h, kResultBytes)) return EUP_EHIP;
    double *res = reinterpret_cast<double *>(h->pinned);
    int rc = with_acc(h, [&](auto acc) {
        hipLaunchKernelGGL((k_site19<decltype(acc)>), dim3(1), dim3(64), 0, h->stream, acc, i, j, k, res);
        return hip_check(h, hipGetLastError(), "site gather") ? EUP_EHIP : 0;
    });
    if (rc) return rc;
    if (hip_check(h, hipStreamSynchronize(h->stream), "sync")) return EUP_EHIP;
    memcpy(out, res, sizeof(double) * 19);
    return 0;
}

// index clipping of flux_X.F90:76-172 / flux_Y.F90:76-165 for a single task (offsets 0)
static bool clip_faces(const Geometry &g, const int32_t box[6], int axis, int *f1, int *f2,
                       double *n1, double *n2, int *lo, int *hi, int *k1, int *k2)
{
    const int L = axis == 0 ? g.l : g.m, M = axis == 0 ? g.m : g.l, n = g.n;
    const int s = axis == 0 ? box[0] : box[2], e = axis == 0 ? box[1] : box[3];
    const int os = axis == 0 ? box[2] : box[0], oe = axis == 0 ? box[3] : box[1];
    *n1 = 1.0;
    *n2 = 1.0;
    *f1 = *f2 = 0;
    if (s > 0 && e <= L) { *f1 = s; *f2 = e; }
    if (s > 0 && e > L) { *f1 = s; *f2 = L; *n2 = 0.0; }
    if (s <= 0 && e <= L) { *f1 = 1; *n1 = 0.0; *f2 = e; }
    if (s < 0 && e > L) return false;
    if (s > L || e < 0) return false;
    *lo = *hi = 0;
    if (os > 0 && oe <= M) { *lo = os; *hi = oe; }
    if (os > 0 && oe > M) { *lo = os; *hi = M; }
    if (os <= 0 && oe <= M) { *lo = 1; *hi = oe; }
    if (os < 0 && oe > M) { *lo = 1; *hi = M; }
    if (os > M || oe < 0) return false;
    *k1 = *k2 = 0;
    const int ks = box[4], ke = box[5];
    if (ks > 0 && ke <= n) { *k1 = ks; *k2 = ke; }
    if (ks > 0 && ke > n) { *k1 = ks; *k2 = n; }
    if (ks <= 0 && ke <= n) { *k1 = 1; *k2 = ke; }
    if (ks < 0 && ke > n) { *k1 = 1; *k2 = n; }
    if (ks > n || ke < 0) return false;
    return true;
}

// fixed != nullptr: the per-site stresses go to that device array (room for 2 * fixed_cap values),
// and are summed on the host through a stack buffer, so nothing is allocated
static int drag_axis(Handle *h, const int32_t box[6], int axis, double *res, double *fixed = nullptr,
                     int64_t fixed_cap = 0)
{
    *res = 0.0;
    int f[2], lo, hi, k1, k2;
    double n1, n2;
    if (!clip_faces(h->g, box, axis, &f[0], &f[1], &n1, &n2, &lo, &hi, &k1, &k2)) return 0;
    const int lim_in = axis == 0 ? h->g.m : h->g.l;
    const int lim_f = axis == 0 ? h->g.l : h->g.m;
    // a box ending at 0 puts its second face on plane 0: the ghost plane of the reference's arrays,
    // which only parity mode holds; the other layouts have no plane 0
    const int fmin = h->cfg.mode == EUP_MODE_PARITY ? 0 : 1;
    if (lo < 1 || hi > lim_in || k1 < 1 || k2 > h->g.n || f[0] < 1 || f[1] < fmin || f[1] > lim_f)
        return fail(h, EUP_ERANGE, "drag box outside the lattice after clipping");
    const int64_t per = (int64_t)(hi - lo + 1) * (k2 - k1 + 1);
    if (per <= 0) return 0;
    int rc = 0;
    double *buf = fixed;
    if (fixed) {
        if (per > fixed_cap)
            return fail(h, EUP_EINVAL, "eup_drag_cv_noalloc: a face of " + std::to_string(per) +
                                           " sites exceeds the no-allocation scratch (at most " +
                                           std::to_string(fixed_cap) + " sites per face)");
    } else {
        rc = ensure_diag(h, 2 * per);
        if (rc) return rc;
        buf = h->diag;
    }
    for (int ii = 0; ii < 2; ++ii) {
        rc = with_acc(h, [&](auto acc) {
            hipLaunchKernelGGL((k_sigma<decltype(acc)>), dim3((unsigned)((per + 255) / 256)), dim3(256), 0,
                               h->stream, acc, axis, f[ii], lo, hi, k1, k2, h->cfg.omega, buf + ii * per);
            return hip_check(h, hipGetLastError(), "sigma") ? EUP_EHIP : 0;
        });
        if (rc) return rc;
    }
    if (fixed) {
        // the same left-to-right sums as below, fed through a fixed host buffer
        double part[4096];
        double fl[2] = {0.0, 0.0};
        for (int ii = 0; ii < 2; ++ii)
            for (int64_t off = 0; off < per; off += 4096) {
                const int64_t cnt = per - off < 4096 ? per - off : 4096;
                if (hip_check(h, hipMemcpyAsync(part, buf + ii * per + off, sizeof(double) * cnt,
                                                hipMemcpyDeviceToHost, h->stream), "copy sigma") ||
                    hip_check(h, hipStreamSynchronize(h->stream), "sync"))
                    return EUP_EHIP;
                for (int64_t t = 0; t < cnt; ++t) fl[ii] = fl[ii] + part[t];
            }
        *res = axis == 0 ? -fl[0] * n1 + fl[1] * n2 : +fl[0] * n1 + fl[1] * n2;
        return 0;
    }
    std::vector<double> sg(2 * per);
    if (hip_check(h, hipMemcpyAsync(sg.data(), h->diag, sizeof(double) * 2 * per, hipMemcpyDeviceToHost,
                                    h->stream), "copy sigma") ||
        hip_check(h, hipStreamSynchronize(h->stream), "sync"))
        return EUP_EHIP;
    double fl[2] = {0.0, 0.0};
    for (int ii = 0; ii < 2; ++ii)
        for (int64_t t = 0; t < per; ++t) fl[ii] = fl[ii] + sg[ii * per + t];
    *res = axis == 0 ? -fl[0] * n1 + fl[1] * n2 : +fl[0] * n1 + fl[1] * n2;
    return 0;
}

int diag_drag_cv(Handle *h, const int32_t box[6], double *fx, double *fy)
{
    int rc = drag_axis(h, box, 0, fx);
    if (rc) return rc;
    return drag_axis(h, box, 1, fy);
}

// Device address of the no-allocation scratch on the handle's device (current when called):
// looked up once per device and kept.
static int noalloc_scratch(Handle *h, double **out)
{
    static std::mutex mu;
    static double *ptr[64] = {};
    const int dev = h->cfg.device;
    if (dev < 0 || dev >= 64) return fail(h, EUP_EINVAL, "eup_drag_cv_noalloc: device ordinal above 63");
    std::lock_guard<std::mutex> lock(mu);
    if (!ptr[dev]) {
        void *p = nullptr;
        if (hip_check(h, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)"))
            return EUP_EHIP;
        ptr[dev] = static_cast<double *>(p);
    }
    *out = ptr[dev];
    return 0;
}

int diag_drag_cv_noalloc(Handle *h, const int32_t box[6], double *fx, double *fy)
{
    double *s = nullptr;
    int rc = noalloc_scratch(h, &s);
    if (rc) return rc;
    rc = drag_axis(h, box, 0, fx, s, kNoAllocFace);
    if (rc) return rc;
    return drag_axis(h, box, 1, fy, s, kNoAllocFace);
}

// the scratch of a reduction to nv values: partial sums, ticket and result
static int reduce_ready(Handle *h, int nv)
{
    if (ensure_diag(h, nv * kRedBlocks) || pinned_ready(h, kResultBytes)) return EUP_EHIP;
    if (h->ticket) return 0;
    if (hip_check(h, hipMalloc((void **)&h->ticket, sizeof(uint32_t)), "hipMalloc ticket") ||
        hip_check(h, hipMemsetAsync(h->ticket, 0, sizeof(uint32_t), h->stream), "clear ticket"))
        return EUP_EHIP;
    return 0;
}

int diag_drag_mem(Handle *h, double F[3])
{
    const int xopen = h->cfg.front != EUP_FACE_PERIODIC;
    if (h->cfg.mode != EUP_MODE_PARITY && h->tiles_mixed == 0) {
        F[0] = F[1] = F[2] = 0.0;
        return 0;
    }
    int rc = reduce_ready(h, 3);
    if (rc) return rc;
    double *res = reinterpret_cast<double *>(h->pinned);
    // physics: no more blocks than tiles to give them (the partials left out were zeros)
    int blocks = kRedBlocks;
    if (h->cfg.mode != EUP_MODE_PARITY)
        blocks = (int)std::min<int64_t>(blocks, (h->tiles_mixed + kBlock / 64 - 1) / (kBlock / 64));
    uint32_t *ticket = blocks <= kTicketBlocks ? h->ticket : nullptr;
    rc = with_acc(h, [&](auto acc) -> int {
        using A = decltype(acc);
        if constexpr (std::is_same_v<A, ParityAcc>) {
            hipLaunchKernelGGL((k_mem_sites<A>), dim3(blocks), dim3(kBlock), 0, h->stream, acc, h->solid, xopen,
                               h->diag);
        } else {
            using S = typename A::value_type;
            hipLaunchKernelGGL((k_mem_tiles<S>), dim3(blocks), dim3(kBlock), 0, h->stream, acc, h->mixed_list,
                               h->tiles_mixed, h->link_mask, h->g.tiles_per_row, h->diag, ticket, res);
        }
        return 0;
    });
    if (rc) return rc;
    if (!ticket) hipLaunchKernelGGL((k_final<3>), dim3(1), dim3(kBlock), 0, h->stream, h->diag, blocks, res);
    if (hip_check(h, hipGetLastError(), "mem drag") || hip_check(h, hipStreamSynchronize(h->stream), "sync"))
        return EUP_EHIP;
    for (int c = 0; c < 3; ++c) F[c] = res[c];
    return 0;
}

int diag_vtk_velocity(Handle *h, int plane, int index, float *out)
{
    const Geometry &g = h->g;
    const int64_t count = plane == 0   ? (int64_t)g.m * g.n
                          : plane == 1 ? (int64_t)g.l * g.n
                          : plane == 2 ? (int64_t)g.l * g.m
                                       : g.sites;
    return with_acc(h, [&](auto acc) {
        return transfer<false>(h, (char *)out, 12 * count, 12 * kBlock, [=](int64_t at, int64_t len, char *pinned) {
            hipLaunchKernelGGL((k_vtk_velocity<decltype(acc)>), dim3((unsigned)((len / 12 + kBlock - 1) / kBlock)),
                               dim3(kBlock), 0, h->stream, acc, plane, index, at / 12, len / 12, (float *)pinned);
        });
    });
}

int diag_vtk_vorticity(Handle *h, int k0, float *out)
{
    const int64_t count = (int64_t)(h->g.l - 2) * (h->g.m - 2);
    return with_acc(h, [&](auto acc) {
        return transfer<false>(h, (char *)out, 4 * count, 4, [=](int64_t at, int64_t len, char *pinned) {
            hipLaunchKernelGGL((k_vtk_vorticity<decltype(acc)>), dim3((unsigned)((len / 4 + 255) / 256)), dim3(256), 0,
                               h->stream, acc, k0, at / 4, len / 4, (float *)pinned);
        });
    });
}

int diag_diagno(Handle *h, double out[5])
{
    int rc = reduce_ready(h, 5);
    if (rc) return rc;
    double *tot = reinterpret_cast<double *>(h->pinned);
    rc = with_acc(h, [&](auto acc) {
        using A = decltype(acc);
        hipLaunchKernelGGL((k_diagno<A>), dim3(kRedBlocks), dim3(kBlock), 0, h->stream, acc, h->solid, h->diag);
        return 0;
    });
    if (rc) return rc;
    hipLaunchKernelGGL((k_final<5>), dim3(1), dim3(kBlock), 0, h->stream, h->diag, kRedBlocks, tot);
    if (hip_check(h, hipGetLastError(), "diagno") || hip_check(h, hipStreamSynchronize(h->stream), "sync"))
        return EUP_EHIP;
    const double rdv = 1. / ((double)h->g.l * (double)h->g.m * (double)h->g.n);
    for (int c = 0; c < 5; ++c) out[c] = tot[c] * rdv;
    return 0;
}

} // namespace eup
