// Grey-lattice mode: partial bounce-back on a solid-fraction field s in [0, 1], the drag
// objective averaged over a step window, and its discrete adjoint with checkpoint-recompute.
// (No reference counterpart; the binary-mask limit is the physics step's bounce-back.)
//
// Link model: the link between x and its source y = x - c_q has the fraction
//   sigma = 1 - (1 - s(x))(1 - s(y))          (s = 0 on the inlet / outlet ghosts)
// and the pulled population is f_q(x) = (1 - sigma) src_q + sigma a_qbar(x), with src_q = a_q(y),
// the inlet equilibrium or the outlet equilibrium of bcond.bc.F90.  sigma is symmetric in the
// link, so every link conserves mass; s in {0, 1} gives the halfway bounce-back exactly.
// Force on the grey body: F = sum over interior links (x, q) of sigma c_q (a_q(y) - a_qbar(x)).
// Objective: J = (1 / ((t1 - t0 + 1) norm)) sum_{t = t0..t1} F_x(a^t).
//
// Adjoint: lam^t = (d a^{t+1} / d a^t)^T lam^{t+1} + [t >= t0] w dF_x/da(a^t), and
// dJ/ds accumulates (d a^{t+1} / ds)^T lam^{t+1} + [t >= t0] w dF_x/ds(a^t).  Per step two kernels:
// k_adj_collide recomputes the pulled populations f(x) of a^t and applies the transposed BGK
// Jacobian to lam^{t+1}, and adds the gradient terms of the links the site pulls through;
// k_adj_stream gathers the transposed pull (all gathers, no atomics):
//   lam_p(z) = (1 - sigma_l) lin_p(z + c_p) + sigma_l lin_pbar(z)   (sigma_l of link z -- z + c_p)
// plus the outlet-equilibrium transpose on the last x column and the objective terms, and adds the
// gradient terms of the links of which the site is the source (FP64 accumulation).
// Inside a segment k_adj_fused runs the stream half of step t and the collide half of step t - 1 in
// one pass, so lam^t is never stored.
// States are checkpointed every K steps; each segment but the last, whose states the forward sweep
// leaves in place, is recomputed forward before its backward sweep, so memory is (t1/K + K) states
// instead of t1.
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "eup_internal.h"

namespace eup {

namespace {

// direction table (0-based population index; bgk3d.F90:31-49), folded into the fully unrolled
// loops below
constexpr int kCX[19] = {1, 1, 1, 1, 1, 0, 0, 0, 0, -1, -1, -1, -1, -1, 0, 0, 0, 0, 0};
constexpr int kCY[19] = {-1, 0, 1, 0, 0, 0, 1, 1, 1, -1, 0, 1, 0, 0, 0, -1, -1, -1, 0};
constexpr int kCZ[19] = {0, -1, 0, 1, 0, 1, 1, 0, -1, 0, -1, 0, 1, 0, -1, -1, 0, 1, 0};
constexpr int kOPP[19] = {11, 12, 9, 10, 13, 14, 15, 16, 17, 2, 3, 0, 1, 4, 5, 6, 7, 8, 18};

// A state: 19 SoA arrays of l*m*n sites, population q at A + q * stride, then the outlet ghost plane
// of the state (5 x m x n: the equilibria that bcond.bc.F90:138-164 gives for its x = l column), which
// the kernel that writes the state writes too.  (Evaluated by each reader instead, an x = l site
// loaded 19 populations for each of its five outlet links, and every wavefront with such a site
// waited for it.)
template <typename R> struct GArgs {
    const R *A; // the state read
    R *B;       // the state written, or null
    int64_t stride;
    const R *s;
    const uint8_t *zero; // per 64 consecutive sites: s = 0 there and at all their neighbours
    double *partial;     // three force sums per block
    R inl[5];
    R omega;
    int l, m, n;
    int xopen;
    UDiv dl, dm;
};

// addresses: element e of an array; 32-bit byte offsets (one scalar base per array, one lane offset)
// where the array is smaller than 4 GiB, 64-bit ones otherwise
template <bool BIG, typename R> __device__ __forceinline__ R ldg(const R *p, uint32_t e)
{
    if constexpr (BIG) return p[(uint64_t)e];
    else return *reinterpret_cast<const R *>(reinterpret_cast<const char *>(p) + (uint64_t)(e * (uint32_t)sizeof(R)));
}

template <bool BIG, typename R> __device__ __forceinline__ void stg(R *p, uint32_t e, R v)
{
    if constexpr (BIG) p[(uint64_t)e] = v;
    else *reinterpret_cast<R *>(reinterpret_cast<char *>(p) + (uint64_t)(e * (uint32_t)sizeof(R))) = v;
}

// one thread per site: its index, coordinates and the index steps to its neighbours (d = -1, 0, +1 at
// [d + 1]), wrapped in y and z (and x when periodic; with open x a step past the end stays on the site
// and the caller takes the ghost instead)
struct Site {
    uint32_t x;
    int i, j, k;
    uint32_t dx[3], dy[3], dz[3];
    bool first, last; // open x: the first and the last column
    bool valid;
    __device__ __forceinline__ uint32_t at(int cx, int cy, int cz) const { return x + dx[cx + 1] + dy[cy + 1] + dz[cz + 1]; }
    // open x: the neighbour at +c_x is the inlet or outlet ghost
    __device__ __forceinline__ bool ghost(int cx) const { return cx == 1 ? last : (cx == -1 && first); }
};

template <typename R> __device__ __forceinline__ Site site_of(const GArgs<R> &a)
{
    Site p;
    const uint32_t l = (uint32_t)a.l, m = (uint32_t)a.m, n = (uint32_t)a.n, N = l * m * n;
    p.x = blockIdx.x * blockDim.x + threadIdx.x;
    p.valid = p.x < N;
    const uint32_t x = p.valid ? p.x : N - 1, row = a.dl.div(x), k = a.dm.div(row);
    p.x = x;
    p.i = (int)(x - row * l);
    p.j = (int)(row - k * m);
    p.k = (int)k;
    p.first = a.xopen && p.i == 0;
    p.last = a.xopen && p.i == a.l - 1;
    p.dx[0] = p.i > 0 ? 0u - 1u : (a.xopen ? 0u : l - 1);
    p.dx[2] = p.i < a.l - 1 ? 1u : (a.xopen ? 0u : 0u - (l - 1));
    p.dy[0] = p.j > 0 ? 0u - l : (m - 1) * l;
    p.dy[2] = p.j < a.m - 1 ? l : 0u - (m - 1) * l;
    const uint32_t lm = l * m;
    p.dz[0] = p.k > 0 ? 0u - lm : (n - 1) * lm;
    p.dz[2] = p.k < a.n - 1 ? lm : 0u - (n - 1) * lm;
    p.dx[1] = p.dy[1] = p.dz[1] = 0u;
    return p;
}

template <typename R> __device__ __forceinline__ R wq(int q)
{
    return q == 18 ? R(1) / R(3) : ((kCX[q] * kCX[q] + kCY[q] * kCY[q] + kCZ[q] * kCZ[q]) == 1 ? R(1) / R(18) : R(1) / R(36));
}

// whether the wavefront's sites are free fluid with free neighbours (s = 0: every link sigma is zero)
template <typename R> __device__ __forceinline__ bool chunk_zero(const GArgs<R> &a, const Site &p)
{
    return a.zero[__builtin_amdgcn_readfirstlane(p.x >> 6)] != 0;
}

// outlet ghost values that the last column pulls as populations 9..13: entry (j - c_y, k - c_z)
template <typename R> __device__ __forceinline__ void outlet_pulls(const GArgs<R> &a, const Site &p, R *src)
{
    const R *out = a.A + 19 * a.stride;
    const uint32_t mn = (uint32_t)a.m * (uint32_t)a.n;
    const uint32_t jm = p.j > 0 ? p.j - 1 : a.m - 1, jp = p.j < a.m - 1 ? p.j + 1 : 0;
    const uint32_t km = p.k > 0 ? p.k - 1 : a.n - 1, kp = p.k < a.n - 1 ? p.k + 1 : 0;
#pragma unroll
    for (int q = 9; q < 14; ++q) {
        const uint32_t jj = kCY[q] == 0 ? (uint32_t)p.j : (kCY[q] > 0 ? jm : jp);
        const uint32_t kk = kCZ[q] == 0 ? (uint32_t)p.k : (kCZ[q] > 0 ? km : kp);
        src[q] = out[(uint32_t)(q - 9) * mn + jj + (uint32_t)a.m * kk];
    }
}

// source values src[0..17] that site p pulls (population 18 stays): interior sources, the inlet
// equilibrium, the outlet ghost plane
template <bool BIG, typename R> __device__ __forceinline__ void sources(const GArgs<R> &a, const Site &p, R *src)
{
#pragma unroll
    for (int q = 0; q < 18; ++q) src[q] = ldg<BIG>(a.A + q * a.stride, p.at(-kCX[q], -kCY[q], -kCZ[q]));
    if (p.first) {
#pragma unroll
        for (int q = 0; q < 5; ++q) src[q] = a.inl[q];
    }
    if (p.last) outlet_pulls(a, p, src);
}

// solid fraction of the source of population q (0 on the ghosts)
template <bool BIG, typename R> __device__ __forceinline__ R source_s(const GArgs<R> &a, const Site &p, int q)
{
    const R v = ldg<BIG>(a.s, p.at(-kCX[q], -kCY[q], -kCZ[q]));
    return p.ghost(-kCX[q]) ? R(0) : v;
}

__device__ __forceinline__ double wsum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// partial[3 * block ..] += the block's sums of the first NF components of v (one block is always the
// same sites, so the sums over sites and steps have a fixed order)
template <int NF> __device__ __forceinline__ void add_partial(const double *v, double *partial)
{
    __shared__ double sh[NF][4];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int c = 0; c < NF; ++c) {
        const double t = wsum(v[c]);
        if (lane == 0) sh[c][w] = t;
    }
    __syncthreads();
    if (threadIdx.x < NF)
        partial[blockIdx.x * 3 + threadIdx.x] += sh[threadIdx.x][0] + sh[threadIdx.x][1] + sh[threadIdx.x][2] + sh[threadIdx.x][3];
}

// One step of the grey lattice and the force of the state read, its first NF components (both pull the
// same links).  Without STEP only the force.  Memory-bound: 19 reads and 19 writes per site, and 18 + 18
// more reads, of own populations and solid fractions, that mostly hit the caches and that wavefronts
// of free fluid skip.  128 x 64 x 64 FP32: 18.1 us (23.3 with 64-bit index arithmetic, every outlet
// value evaluated where it is read and no chunk flags), 21.8 with the force (it took 17.6 + 4.6 us on
// its own); FP64 70 x 45 x 36 10.9 us (15.4).
template <typename R, bool BIG, bool STEP, int NF> __global__ __launch_bounds__(256) void k_grey(GArgs<R> a)
{
    const Site p = site_of(a);
    const bool zero = chunk_zero(a, p);
    double v[3] = {0.0, 0.0, 0.0};
    if (STEP || !zero) {
        R f[19];
        sources<BIG>(a, p, f);
        f[18] = ldg<BIG>(a.A + 18 * a.stride, p.x);
        if (!zero) {
            const R sx = ldg<BIG>(a.s, p.x);
            R own[18];
#pragma unroll
            for (int q = 0; q < 18; ++q) own[q] = ldg<BIG>(a.A + kOPP[q] * a.stride, p.x);
#pragma unroll
            for (int q = 0; q < 18; ++q) {
                const R sg = R(1) - (R(1) - sx) * (R(1) - source_s<BIG>(a, p, q));
                if (NF > 1 || (NF == 1 && kCX[q])) {
                    const double d = p.valid && !p.ghost(-kCX[q]) ? (double)sg * ((double)f[q] - (double)own[q]) : 0.0;
                    if (kCX[q]) v[0] += kCX[q] * d;
                    if (NF > 1 && kCY[q]) v[1] += kCY[q] * d;
                    if (NF > 1 && kCZ[q]) v[2] += kCZ[q] * d;
                }
                f[q] = (R(1) - sg) * f[q] + sg * own[q];
            }
        }
        if constexpr (STEP) {
            collide<R>(f, f, a.omega, R(0));
            if (p.valid) {
#pragma unroll
                for (int q = 0; q < 19; ++q) stg<BIG>(a.B + q * a.stride, p.x, f[q]);
                if (p.last) {
                    R o[5];
                    outlet_eq<R>(f, o);
                    const uint32_t mn = (uint32_t)a.m * (uint32_t)a.n;
#pragma unroll
                    for (uint32_t u = 0; u < 5; ++u) a.B[19 * a.stride + u * mn + p.j + (uint32_t)a.m * (uint32_t)p.k] = o[u];
                }
            }
        }
    }
    if constexpr (NF > 0) {
        if (__syncthreads_or(!zero)) add_partial<NF>(v, a.partial);
    }
}

// outlet ghost plane of a state that the host set
template <typename R> __global__ __launch_bounds__(256) void k_grey_outlet(R *A, int64_t stride, int l, int m, int n)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x, mn = (uint32_t)m * (uint32_t)n;
    if (r >= mn) return;
    R y[19], o[5];
#pragma unroll
    for (int q = 0; q < 19; ++q) y[q] = A[q * stride + (int64_t)r * l + l - 1];
    outlet_eq<R>(y, o);
#pragma unroll
    for (uint32_t u = 0; u < 5; ++u) A[19 * stride + u * mn + r] = o[u];
}

// the sums of the blocks' partial forces (single block, fixed order)
__global__ __launch_bounds__(1024) void k_force_sum(const double *partial, int nb, double *out)
{
    __shared__ double sh[3][1024];
    double v[3] = {0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nb; b += blockDim.x)
        for (int c = 0; c < 3; ++c) v[c] += partial[b * 3 + c];
    for (int c = 0; c < 3; ++c) sh[c][threadIdx.x] = v[c];
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st)
            for (int c = 0; c < 3; ++c) sh[c][threadIdx.x] += sh[c][threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x < 3) out[threadIdx.x] = sh[threadIdx.x][0];
}

// Transposed BGK Jacobian at density rho and momentum j applied to lam[19], in place:
//   out_p = (1 - omega) lam_p + omega (A + B . c_p),
//   A = sum_q lam_q w_q (1 + 1.5 u^2 - 4.5 (c_q.u)^2),
//   B = sum_q lam_q w_q (3 c_q + 9 (c_q.u) c_q - 3 u).
// Only the terms with c != 0 are formed (a product with a constant 0 is not dropped by the compiler).
template <typename R> __device__ __forceinline__ void collide_adj(R rho, R jx, R jy, R jz, R omega, R *lam)
{
    const R inv = R(1) / rho, ux = jx * inv, uy = jy * inv, uz = jz * inv, usq = ux * ux + uy * uy + uz * uz;
    R S = 0, Q = 0, Bx = 0, By = 0, Bz = 0;
#pragma unroll
    for (int q = 0; q < 19; ++q) {
        const R lw = lam[q] * wq<R>(q);
        S += lw;
        if (q == 18) continue;
        R cu = R(0);
        if (kCX[q]) cu = kCX[q] > 0 ? ux : -ux;
        if (kCY[q]) cu = kCY[q] > 0 ? cu + uy : cu - uy;
        if (kCZ[q]) cu = kCZ[q] > 0 ? cu + uz : cu - uz;
        Q += lw * (cu * cu);
        const R g = lw * (R(3) + R(9) * cu);
        if (kCX[q]) Bx = kCX[q] > 0 ? Bx + g : Bx - g;
        if (kCY[q]) By = kCY[q] > 0 ? By + g : By - g;
        if (kCZ[q]) Bz = kCZ[q] > 0 ? Bz + g : Bz - g;
    }
    const R A = S * (R(1) + R(1.5) * usq) - R(4.5) * Q, S3 = R(3) * S;
    Bx -= S3 * ux;
    By -= S3 * uy;
    Bz -= S3 * uz;
    const R o1 = R(1) - omega;
#pragma unroll
    for (int p = 0; p < 19; ++p) {
        R e = A;
        if (kCX[p]) e = kCX[p] > 0 ? e + Bx : e - Bx;
        if (kCY[p]) e = kCY[p] > 0 ? e + By : e - By;
        if (kCZ[p]) e = kCZ[p] > 0 ? e + Bz : e - Bz;
        lam[p] = o1 * lam[p] + omega * e;
    }
}

template <typename R> struct AdjArgs {
    GArgs<R> g;
    const R *lam_in; // lam^{t+1} (the state layout of g)
    R *lin;          // J_C^T lam^{t+1} at every site
    R *lam_out;      // lam^t
    double *gs;
    double wobj;     // objective weight at time t (0 outside the window)
};

// lin(x) = J_C(f(x))^T lam^{t+1}(x) from lam[19] = lam^{t+1}(x) (overwritten), stored to a.lin;
// g gets the gradient terms of the links that x pulls through (x as the pulling site:
// d f_q(x) / d s(x) on every link, plus the objective's force term).  Of f only the moments are
// kept; the source values and the site's own populations wait in registers for the gradient.
template <bool BIG, bool ZERO, typename R>
__device__ __forceinline__ void adj_collide_site(const AdjArgs<R> &a, const Site &p, R *lam, double &g)
{
    const double w = a.wobj;
    R src[18], own[18], sy[18];
    sources<BIG>(a.g, p, src);
#pragma unroll
    for (int q = 0; q < 18; ++q) own[q] = ldg<BIG>(a.g.A + kOPP[q] * a.g.stride, p.x);
    R rho = 0, jx = 0, jy = 0, jz = 0;
    R sx = R(0);
    if constexpr (!ZERO) sx = ldg<BIG>(a.g.s, p.x);
#pragma unroll
    for (int q = 0; q < 18; ++q) {
        R f = src[q];
        sy[q] = R(0);
        if constexpr (!ZERO) {
            sy[q] = source_s<BIG>(a.g, p, q);
            const R sg = R(1) - (R(1) - sx) * (R(1) - sy[q]);
            f = (R(1) - sg) * f + sg * own[q];
        }
        rho += f;
        if (kCX[q]) jx = kCX[q] > 0 ? jx + f : jx - f;
        if (kCY[q]) jy = kCY[q] > 0 ? jy + f : jy - f;
        if (kCZ[q]) jz = kCZ[q] > 0 ? jz + f : jz - f;
    }
    rho += ldg<BIG>(a.g.A + 18 * a.g.stride, p.x);
    collide_adj<R>(rho, jx, jy, jz, a.g.omega, lam);
    if (p.valid) {
#pragma unroll
        for (int q = 0; q < 19; ++q) stg<BIG>(a.lin + q * a.g.stride, p.x, lam[q]);
    }
#pragma unroll
    for (int q = 0; q < 18; ++q) {
        // (L - w c_x) (abar - src) (1 - s(y)); the objective's term on interior links only
        double L = (double)lam[q];
        if (kCX[q] && w != 0.0 && !p.ghost(-kCX[q])) L -= w * kCX[q];
        double d = L * ((double)own[q] - (double)src[q]);
        if constexpr (!ZERO) d *= 1.0 - (double)sy[q];
        g += d;
    }
}

// lam^t(z) into lam[19]: the transposed pull gathered from a.lin at the sites z + c_p that pull
// from z, the outlet-equilibrium transpose on the last x column and the objective's force term;
// g gets the gradient terms of the links of which z is the source
template <bool BIG, bool ZERO, typename R>
__device__ __forceinline__ void adj_stream_site(const AdjArgs<R> &a, const Site &z, R *lam, double &g)
{
    const int64_t st = a.g.stride;
    const double w = a.wobj;
    R sz = R(0);
    if constexpr (!ZERO) sz = ldg<BIG>(a.g.s, z.x);
#pragma unroll
    for (int p = 0; p < 18; ++p) {
        const int pb = kOPP[p];
        const uint32_t zp = z.at(kCX[p], kCY[p], kCZ[p]); // the site pulling p from z
        const bool gh = z.ghost(kCX[p]);
        const double Lp = (double)ldg<BIG>(a.lin + p * st, zp);
        const double d = (double)ldg<BIG>(a.g.A + pb * st, zp) - (double)ldg<BIG>(a.g.A + p * st, z.x);
        double lp = Lp, e = Lp;
        if (kCX[p] && w != 0.0) e -= w * kCX[p];
        e *= d;
        if constexpr (!ZERO) {
            const double s2 = (double)ldg<BIG>(a.g.s, zp), own = (double)ldg<BIG>(a.lin + pb * st, z.x);
            const double sl = 1.0 - (1.0 - (double)sz) * (1.0 - s2);
            lp = (1.0 - sl) * Lp + sl * own;
            if (kCX[p] && w != 0.0) lp += 2.0 * w * sl * kCX[p];
            lp = gh ? (double)sz * own : lp; // ghost link: sigma = s(z)
            e *= 1.0 - s2;
        } else {
            lp = gh ? 0.0 : lp;
        }
        g += gh ? 0.0 : e;
        lam[p] = (R)lp;
    }
    lam[18] = ldg<BIG>(a.lin + 18 * st, z.x);
    // Outlet equilibrium transpose: z on the last x column feeds the ghost values read by the sites
    // x = (l-1, j + cy, k + cz) for q = 10..14 (0-based 9..13).  With Lw_q = w_q (1 - s(x)) lin_q(x):
    //   lam_p += sum_q Lw_q (3 c_q.c_p + 9 (c_q.J) (c_q.c_p) - 3 J.c_p) = c_p . V
    if (z.last) {
        double J[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int p = 0; p < 18; ++p) {
            const double yp = (double)ldg<BIG>(a.g.A + p * st, z.x);
            if (kCX[p]) J[0] += kCX[p] * yp;
            if (kCY[p]) J[1] += kCY[p] * yp;
            if (kCZ[p]) J[2] += kCZ[p] * yp;
        }
        double V[3] = {0.0, 0.0, 0.0}, sum = 0.0;
#pragma unroll
        for (int q = 9; q < 14; ++q) {
            const uint32_t x = z.at(0, kCY[q], kCZ[q]);
            const double sg = (double)ldg<BIG>(a.g.s, x); // sigma of the ghost link
            const double Lw = (1.0 - sg) * (double)ldg<BIG>(a.lin + q * st, x) * wq<double>(q);
            const double t = Lw * (3.0 + 9.0 * (kCX[q] * J[0] + kCY[q] * J[1] + kCZ[q] * J[2]));
            sum += Lw;
            if (kCX[q]) V[0] += kCX[q] * t;
            if (kCY[q]) V[1] += kCY[q] * t;
            if (kCZ[q]) V[2] += kCZ[q] * t;
        }
        for (int c = 0; c < 3; ++c) V[c] -= 3.0 * sum * J[c];
#pragma unroll
        for (int p = 0; p < 18; ++p)
            lam[p] = (R)((double)lam[p] + (kCX[p] * V[0] + kCY[p] * V[1] + kCZ[p] * V[2]));
    }
}

// the collide half of an adjoint step on its own: lin = J_C^T lam_in, and the gradient terms of
// the links that x pulls through
template <typename R, bool BIG> __global__ __launch_bounds__(256) void k_adj_collide(AdjArgs<R> a)
{
    const Site p = site_of(a.g);
    R lam[19];
#pragma unroll
    for (int q = 0; q < 19; ++q) lam[q] = ldg<BIG>(a.lam_in + q * a.g.stride, p.x);
    double g = 0.0;
    if (chunk_zero(a.g, p)) adj_collide_site<BIG, true>(a, p, lam, g);
    else adj_collide_site<BIG, false>(a, p, lam, g);
    if (p.valid) a.gs[p.x] += g;
}

// the stream half of an adjoint step on its own: lam_out = P^T lin (+ objective terms)
template <typename R, bool BIG> __global__ __launch_bounds__(256) void k_adj_stream(AdjArgs<R> a)
{
    const Site z = site_of(a.g);
    R lam[19];
    double g = 0.0;
    if (chunk_zero(a.g, z)) adj_stream_site<BIG, true>(a, z, lam, g);
    else adj_stream_site<BIG, false>(a, z, lam, g);
    if (!z.valid) return;
#pragma unroll
    for (int p = 0; p < 19; ++p) stg<BIG>(a.lam_out + p * a.g.stride, z.x, lam[p]);
    a.gs[z.x] += g;
}

// the stream half of step t (sa: state a^t, lin^t in sa.lin) and the collide half of step t - 1
// (ca: state a^{t-1}, lin^{t-1} into ca.lin) in one pass: lam^t stays in registers, so the
// adjoint field is read and written once per step instead of twice.  The gradient sum of each
// site takes the two halves' terms in the same order as the split kernels, so the result is
// bit-identical to running k_adj_stream(t) and k_adj_collide(t - 1).  Bound by latency at two (FP32, 251
// registers) and one (FP64) wavefronts per SIMD with every load of a half in flight: held to three
// wavefronts, or with the loads in groups of 6, it spills or waits more (FP32 45 us; about 85 us at
// three).
template <typename R, bool BIG> __global__ __launch_bounds__(256) void k_adj_fused(AdjArgs<R> sa, AdjArgs<R> ca)
{
    const Site z = site_of(sa.g);
    R lam[19];
    double g1 = 0.0, g2 = 0.0;
    if (chunk_zero(sa.g, z)) {
        adj_stream_site<BIG, true>(sa, z, lam, g1);
        adj_collide_site<BIG, true>(ca, z, lam, g2);
    } else {
        adj_stream_site<BIG, false>(sa, z, lam, g1);
        adj_collide_site<BIG, false>(ca, z, lam, g2);
    }
    if (!z.valid) return;
    double v = sa.gs[z.x];
    v += g1;
    v += g2;
    sa.gs[z.x] = v;
}

// objective seed at t1: lam = w dF/da, gs += w dF/ds
template <typename R, bool BIG> __global__ __launch_bounds__(256) void k_force_adj_seed(AdjArgs<R> a)
{
    const Site z = site_of(a.g);
    if (!z.valid) return;
    const int64_t st = a.g.stride;
    const double w = a.wobj;
    const double sz = (double)ldg<BIG>(a.g.s, z.x);
    double g = 0.0;
#pragma unroll
    for (int q = 0; q < 18; ++q) { // z as x: pair (z, q) with interior source y = z - c_q
        if (!kCX[q] || z.ghost(-kCX[q])) continue;
        const uint32_t y = z.at(-kCX[q], -kCY[q], -kCZ[q]);
        const double d = (double)ldg<BIG>(a.g.A + q * st, y) - (double)ldg<BIG>(a.g.A + kOPP[q] * st, z.x);
        g += w * kCX[q] * d * (1.0 - (double)ldg<BIG>(a.g.s, y));
    }
#pragma unroll
    for (int p = 0; p < 18; ++p) {
        double lam = 0.0;
        if (kCX[p] && !z.ghost(kCX[p])) {
            const uint32_t zp = z.at(kCX[p], kCY[p], kCZ[p]);
            const double s2 = (double)ldg<BIG>(a.g.s, zp);
            const double sl = 1.0 - (1.0 - sz) * (1.0 - s2);
            lam = 2.0 * w * sl * kCX[p];
            const double d = (double)ldg<BIG>(a.g.A + p * st, z.x) - (double)ldg<BIG>(a.g.A + kOPP[p] * st, zp);
            g += w * kCX[p] * d * (1.0 - s2);
        }
        stg<BIG>(a.lam_out + p * st, z.x, (R)lam);
    }
    stg<BIG>(a.lam_out + 18 * st, z.x, R(0));
    a.gs[z.x] += g;
}

// The solid fraction as the kernels hold it, and the chunks of 64 sites without any in or next to them.
// One launch, the neighbours read from the caller's field: in a second one, over the field just
// stored, setting a field in device memory took 19 to 20 us (70 x 45 x 36, 128 x 64 x 64 FP32) instead of 13 to 14.5.
template <typename R, typename T>
__global__ __launch_bounds__(256) void k_grey_field(GArgs<R> a, const T *__restrict__ src, R *__restrict__ s, uint8_t *zero)
{
    const Site p = site_of(a);
    const R v = (R)src[p.x];
    bool any = v != R(0);
#pragma unroll
    for (int q = 0; q < 18; ++q) any |= (R)src[p.at(kCX[q], kCY[q], kCZ[q])] != R(0);
    const uint64_t b = __ballot(any);
    if (!p.valid) return;
    s[p.x] = v;
    if ((threadIdx.x & 63) == 0) zero[p.x >> 6] = b == 0;
}

__global__ void k_to_f32(const double *src, float *dst, int64_t N)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x < N) dst[x] = (float)src[x];
}

__global__ void k_fill0(double *p, int64_t N)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x < N) p[x] = 0.0;
}

unsigned blocks_of(int64_t n) { return (unsigned)((n + 255) / 256); }

template <typename R> GArgs<R> gargs(Handle *h, const void *from, void *to)
{
    GArgs<R> a;
    a.A = static_cast<const R *>(from);
    a.B = static_cast<R *>(to);
    a.stride = h->stride;
    a.s = static_cast<const R *>(h->grey);
    a.zero = h->grey_zero;
    a.partial = h->diag;
    R inl[5];
    inlet_eq<R>((R)h->cfg.u_inflow, inl);
    for (int u = 0; u < 5; ++u) a.inl[u] = inl[u];
    a.omega = (R)h->cfg.omega;
    a.l = h->g.l;
    a.m = h->g.m;
    a.n = h->g.n;
    a.xopen = h->cfg.front != EUP_FACE_PERIODIC;
    a.dl = UDiv::make((uint32_t)a.l);
    a.dm = UDiv::make((uint32_t)a.m);
    return a;
}

// f(std::bool_constant<BIG>): arrays of 4 GiB and more take 64-bit offsets (EUP_GREY_64BIT=1: all)
template <typename R, typename F> void by_size(Handle *h, F &&f)
{
    const char *e = getenv("EUP_GREY_64BIT");
    if (!(e && atoi(e) != 0) && (uint64_t)h->g.sites * sizeof(R) < (1ull << 32)) f(std::false_type{});
    else f(std::true_type{});
}

// one step (to != null), the first nf force components of `from` added to the blocks' partial sums,
// or both (the objective needs F_x alone)
template <typename R> void launch_grey(Handle *h, const void *from, void *to, int nf)
{
    const GArgs<R> a = gargs<R>(h, from, to);
    const dim3 grid(blocks_of(h->g.sites)), block(256);
    by_size<R>(h, [&](auto big) {
        constexpr bool B = decltype(big)::value;
        if (to && nf) hipLaunchKernelGGL((k_grey<R, B, true, 1>), grid, block, 0, h->stream, a);
        else if (to) hipLaunchKernelGGL((k_grey<R, B, true, 0>), grid, block, 0, h->stream, a);
        else if (nf == 1) hipLaunchKernelGGL((k_grey<R, B, false, 1>), grid, block, 0, h->stream, a);
        else hipLaunchKernelGGL((k_grey<R, B, false, 3>), grid, block, 0, h->stream, a);
    });
}

// the outlet plane of the handle's current state, after the host set populations
template <typename R> void refresh_outlet(Handle *h)
{
    if (h->outlet_dirty && h->cfg.front != EUP_FACE_PERIODIC)
        hipLaunchKernelGGL((k_grey_outlet<R>), dim3(blocks_of((int64_t)h->g.m * h->g.n)), dim3(256), 0, h->stream,
                           static_cast<R *>(h->buf[h->cur]), h->stride, h->g.l, h->g.m, h->g.n);
    h->outlet_dirty = false;
}

template <typename R> int grey_step_t(Handle *h)
{
    refresh_outlet<R>(h);
    launch_grey<R>(h, h->buf[h->cur], h->buf[h->cur ^ 1], 0);
    if (hip_check(h, hipGetLastError(), "grey step")) return EUP_EHIP;
    h->cur ^= 1;
    return 0;
}

// the blocks' partial force sums, cleared, and pinned memory for their total
int force_scratch(Handle *h)
{
    const int64_t np = 3 * (int64_t)blocks_of(h->g.sites);
    if (pinned_ready(h, 3 * sizeof(double))) return EUP_EHIP;
    if (h->diag_len < np) {
        hipFree(h->diag);
        h->diag = nullptr;
        h->diag_len = 0;
        if (hip_check(h, hipMalloc((void **)&h->diag, sizeof(double) * np), "hipMalloc")) return EUP_EHIP;
        h->diag_len = np;
    }
    hipLaunchKernelGGL(k_fill0, dim3(blocks_of(np)), dim3(256), 0, h->stream, h->diag, np);
    return hip_check(h, hipGetLastError(), "force scratch") ? EUP_EHIP : 0;
}

int force_result(Handle *h, double F[3])
{
    double *const sum = reinterpret_cast<double *>(h->pinned);
    hipLaunchKernelGGL(k_force_sum, dim3(1), dim3(1024), 0, h->stream, h->diag, (int)blocks_of(h->g.sites), sum);
    if (hip_check(h, hipGetLastError(), "grey force") || hip_check(h, hipStreamSynchronize(h->stream), "sync"))
        return EUP_EHIP;
    for (int c = 0; c < 3; ++c) F[c] = sum[c];
    return 0;
}

template <typename R> int grey_force_t(Handle *h, double F[3])
{
    if (int rc = force_scratch(h)) return rc;
    refresh_outlet<R>(h);
    launch_grey<R>(h, h->buf[h->cur], nullptr, 3);
    return force_result(h, F);
}

// A handle keeps its objective's device memory for the next call if it is at most this much
// (allocating and freeing on each call: 128 x 64 x 64 FP32, 100 steps, 8.60 against 8.03 ms).
constexpr size_t kKeepBytes = size_t(2) << 30;

template <typename R>
int objective_t(Handle *h, int t0, int t1, int K, double norm, double *J, void *grad_dev, int gdtype,
                double *grad_host)
{
    const int64_t N = h->g.sites;
    const size_t S = (grey_state_bytes(h) + 255) / 256 * 256; // one state with its outlet plane
    const bool want_grad = grad_dev || grad_host;
    if (int rc = force_scratch(h)) return rc;
    // Checkpoints: the states K, 2 K, ... up to t1 - 1, written by the forward sweep in place (state 0
    // is the handle's own).  A segment's other states, at most min(K, t1) - 1; the forward sweep leaves
    // those of the last segment there.  Two states for the rest of the forward sweep, the last one t1.
    const int ncheck = want_grad ? (t1 - 1) / K : 0, nseg = want_grad ? (K < t1 ? K : t1) - 1 : 0;
    const size_t gbytes = want_grad ? (sizeof(double) * (size_t)N + 255) / 256 * 256 : 0;
    const size_t need = S * (size_t)(ncheck + nseg + 2 + (want_grad ? 3 : 0)) + gbytes;
    if (h->work_len < need) {
        hipFree(h->work);
        h->work = nullptr;
        h->work_len = 0;
        if (hipMalloc(&h->work, need) != hipSuccess) {
            (void)hipGetLastError();
            h->work = nullptr;
            return fail(h, EUP_EHIP, "eup_grey_objective: out of device memory for checkpoints and the adjoint");
        }
        h->work_len = need;
    }
    struct Give { // back after the call, unless small
        Handle *h;
        ~Give()
        {
            if (h->work_len <= kKeepBytes) return;
            hipStreamSynchronize(h->stream);
            hipFree(h->work);
            h->work = nullptr;
            h->work_len = 0;
        }
    } give{h};
    char *mem = static_cast<char *>(h->work);
    auto take = [&](size_t states) {
        char *p = mem;
        mem += S * states;
        return p;
    };
    char *const ck = take((size_t)ncheck), *const seg = take((size_t)nseg);
    void *const work[2] = {take(1), take(1)};
    refresh_outlet<R>(h);
    const int tlast = want_grad ? ncheck * K : t1; // first state of the last segment
    auto check = [&](int c) -> void * { return c == 0 ? h->buf[h->cur] : ck + S * (size_t)(c - 1); };
    auto segment = [&](int t, int tb) -> void * { return t == tb ? check(tb / K) : seg + S * (size_t)(t - tb - 1); };
    // where the forward sweep keeps state t
    auto state = [&](int t) -> void * {
        if (t == 0) return check(0);
        if (want_grad && t < t1 && t % K == 0) return check(t / K);
        if (want_grad && t > tlast && t < t1) return segment(t, tlast);
        return work[t & 1];
    };
    for (int t = 0; t < t1; ++t) launch_grey<R>(h, state(t), state(t + 1), t >= t0 ? 1 : 0);
    launch_grey<R>(h, state(t1), nullptr, 1);
    double F[3];
    if (int rc = force_result(h, F)) return rc;
    const double wobj = 1.0 / ((double)(t1 - t0 + 1) * norm);
    *J = F[0] * wobj;
    if (!want_grad) return 0;
    void *const lam = take(1);                    // lam^t between the halves of a step
    void *const linb[2] = {take(1), take(1)};     // lin^t, lin^{t-1}
    double *const gs = reinterpret_cast<double *>(mem);
    const dim3 grid(blocks_of(N)), block(256);
    hipLaunchKernelGGL(k_fill0, grid, block, 0, h->stream, gs, N);
    auto adj = [&](const void *st, const void *lam_in, void *lin, void *lam_out, double w) {
        AdjArgs<R> q;
        q.g = gargs<R>(h, st, nullptr);
        q.lam_in = static_cast<const R *>(lam_in);
        q.lin = static_cast<R *>(lin);
        q.lam_out = static_cast<R *>(lam_out);
        q.gs = gs;
        q.wobj = w;
        return q;
    };
    // Per segment: the collide half of its last step, then the stream half of step t fused with the
    // collide half of step t - 1 (both states are in the segment), then the stream half of its first
    // step.  Fused, 128 x 64 x 64 (MI355X): FP32 45 us against 30 + 28 us apart, FP64 70 x 45 x 36 24.6
    // against 15.2 + 13.1 us.  EUP_ADJ_FUSED=0 / 1 forces the halves apart or together; both give the
    // same results bit for bit.
    bool fuse = true;
    if (const char *e = getenv("EUP_ADJ_FUSED")) fuse = atoi(e) != 0;
    by_size<R>(h, [&](auto big) {
        constexpr bool B = decltype(big)::value;
        hipLaunchKernelGGL((k_force_adj_seed<R, B>), grid, block, 0, h->stream, adj(state(t1), nullptr, nullptr, lam, wobj));
        for (int cc = ncheck; cc >= 0; --cc) {
            const int tb = cc * K, te = (cc + 1) * K < t1 ? (cc + 1) * K : t1;
            if (cc < ncheck) // the last segment's states are those of the forward sweep
                for (int t = tb + 1; t < te; ++t) launch_grey<R>(h, segment(t - 1, tb), segment(t, tb), 0);
            auto at = [&](int t) { return static_cast<const void *>(segment(t, tb)); };
            auto wt = [&](int t) { return t >= t0 ? wobj : 0.0; };
            int b = 0; // linb[b] holds lin^t
            hipLaunchKernelGGL((k_adj_collide<R, B>), grid, block, 0, h->stream,
                               adj(at(te - 1), lam, linb[b], nullptr, wt(te - 1)));
            for (int t = te - 1; t > tb; --t) {
                if (fuse) {
                    hipLaunchKernelGGL((k_adj_fused<R, B>), grid, block, 0, h->stream,
                                       adj(at(t), nullptr, linb[b], nullptr, wt(t)),
                                       adj(at(t - 1), nullptr, linb[b ^ 1], nullptr, wt(t - 1)));
                    b ^= 1;
                } else {
                    hipLaunchKernelGGL((k_adj_stream<R, B>), grid, block, 0, h->stream,
                                       adj(at(t), nullptr, linb[b], lam, wt(t)));
                    hipLaunchKernelGGL((k_adj_collide<R, B>), grid, block, 0, h->stream,
                                       adj(at(t - 1), lam, linb[b], nullptr, wt(t - 1)));
                }
            }
            hipLaunchKernelGGL((k_adj_stream<R, B>), grid, block, 0, h->stream,
                               adj(at(tb), nullptr, linb[b], lam, wt(tb)));
        }
    });
    if (grad_dev && gdtype == EUP_STORE_F32)
        hipLaunchKernelGGL(k_to_f32, grid, block, 0, h->stream, gs, static_cast<float *>(grad_dev), N);
    if (hip_check(h, hipGetLastError(), "adjoint sweep")) return EUP_EHIP;
    if ((grad_host || gdtype == EUP_STORE_F64) &&
        hip_check(h, hipMemcpyAsync(grad_host ? (void *)grad_host : grad_dev, gs, sizeof(double) * N,
                                    grad_host ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice, h->stream), "copy grad"))
        return EUP_EHIP;
    return hip_check(h, hipStreamSynchronize(h->stream), "sync") ? EUP_EHIP : 0;
}

template <typename F> int rdispatch(Handle *h, F &&f)
{
    if (h->cfg.storage == EUP_STORE_F64) return f((double *)nullptr);
    return f((float *)nullptr);
}

} // namespace

int grey_step(Handle *h)
{
    return rdispatch(h, [&](auto *p) { return grey_step_t<std::remove_pointer_t<decltype(p)>>(h); });
}

int grey_set_field(Handle *h, const void *s, int dtype, bool on_device)
{
    const int64_t N = h->g.sites;
    const size_t rb = h->cfg.storage == EUP_STORE_F64 ? 8 : 4;
    if (!h->grey && hip_check(h, hipMalloc(&h->grey, rb * N), "hipMalloc grey")) return EUP_EHIP;
    if (!h->grey_zero && hip_check(h, hipMalloc((void **)&h->grey_zero, (N + 63) / 64), "hipMalloc grey")) return EUP_EHIP;
    const void *src = s;
    void *tmp = nullptr;
    if (!on_device) {
        if (hip_check(h, hipMalloc(&tmp, sizeof(double) * N), "hipMalloc") ||
            hip_check(h, hipMemcpy(tmp, s, sizeof(double) * N, hipMemcpyHostToDevice), "copy grey")) {
            hipFree(tmp);
            return EUP_EHIP;
        }
        src = tmp;
        dtype = EUP_STORE_F64;
    }
    int rc = rdispatch(h, [&](auto *p) {
        using R = std::remove_pointer_t<decltype(p)>;
        const GArgs<R> a = gargs<R>(h, nullptr, nullptr);
        R *const field = static_cast<R *>(h->grey);
        if (dtype == EUP_STORE_F64)
            hipLaunchKernelGGL((k_grey_field<R, double>), dim3(blocks_of(N)), dim3(256), 0, h->stream, a,
                               static_cast<const double *>(src), field, h->grey_zero);
        else
            hipLaunchKernelGGL((k_grey_field<R, float>), dim3(blocks_of(N)), dim3(256), 0, h->stream, a,
                               static_cast<const float *>(src), field, h->grey_zero);
        return hip_check(h, hipGetLastError(), "grey field") ? EUP_EHIP : 0;
    });
    if (!rc && hip_check(h, hipStreamSynchronize(h->stream), "sync")) rc = EUP_EHIP;
    hipFree(tmp);
    return rc;
}

int grey_force(Handle *h, double F[3])
{
    return rdispatch(h, [&](auto *p) { return grey_force_t<std::remove_pointer_t<decltype(p)>>(h, F); });
}

int grey_objective(Handle *h, int t0, int t1, int K, double norm, double *J, void *grad_dev, int gdtype,
                   double *grad_host)
{
    return rdispatch(h, [&](auto *p) {
        return objective_t<std::remove_pointer_t<decltype(p)>>(h, t0, t1, K, norm, J, grad_dev, gdtype,
                                                               grad_host);
    });
}

} // namespace eup
