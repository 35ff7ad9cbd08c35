// Two physics steps in one launch, FP64 and FP32 storage (included by eup_physics.hip, which defines
// XArgs and the helpers used here).
//
// The single-step kernel is bound by HBM: it reads and writes every population once per step.  Here
// a workgroup marches through z over a column of the lattice and carries the state between the two
// steps on the chip, so that memory is read and written once per two steps:
//   * a window of WX x WY sites (one thread each) runs the first step on plane kz; its inner
//     TX x TY sites (WX = TX + 2, WY = TY + 2) run the second step on plane kz - 1, whose pulls
//     reach one site beyond them;
//   * LDS holds the first step's results of the window: for the 16 populations that move in x or y
//     the planes that a second step still pulls from (two planes, three of those with c_z = +1),
//     also the sources of its bounce-back; populations 5, 14 and 18, which stay in their column,
//     are kept in registers;
//   * the pulls of plane kz + 1 are issued before plane kz is computed, one between every few
//     arithmetic instructions (all at once they filled the address queue while the VALU idled), with
//     the link masks and tile codes of the planes after it already at hand;
//   * wavefronts hold whole window rows, aligned to the tiles, so that the 19 stores of a row write
//     whole lines (a row split between wavefronts wrote 1.23 x the bytes); the two halo columns are
//     one more wavefront;
//   * planes are accessed through buffer resources, whose bounds check takes the place of branches
//     (raw_load_at).
// A column is cut into chunks of zc planes (PairMap), each with two planes of run-up.  The arithmetic
// per site is the single-step kernel's, so the state after a pair is the state after two single
// steps, bit for bit.
//
// Open x: the window's column x = l stands for the outlet ghost.  Its threads run the first step of
// the site x = l - 1 once more and put the outlet equilibrium of the result in place of the
// populations that the second step pulls from there.
//
// Bound: memory, short of a copy's 6.2 TB/s.  Sponge 512 x 256 x 256 FP32: 0.57 to 0.61 ms per step
// between boxes against 0.82 to 0.83 in single steps, for 2.95 GB (5.1 TB/s at 0.58 ms); FP64 1.27 ms
// against 1.66, 6.21 GB (4.9 TB/s).  Without obstacles 0.569 ms with open and 0.52 to 0.53 with periodic
// x (FP32); the latter took 0.150 without the kernel's loads and stores, 0.226 without the loads, 0.346
// without the stores, 0.520 without the collisions.  It read 3.4 GB and wrote 2.55 GB per two steps,
// 5.7 TB/s: the extra reads are the halo (15 / 13 rows, 34 / 32 planes and the lines that cut the columns).
// What keeps it below the copy rate: one workgroup per CU (its LDS), whose wavefronts meet at two barriers
// per plane.  The 2-byte storages stay with single steps: a form of this kernel for FP16 took 0.424
// against 0.418 ms with open x and 0.470 against 0.427 on the sponge, though 0.374 against 0.418 with
// periodic x.  What bounds that form is not known: neither its arithmetic (about 0.23 ms with the
// conversions) nor its bytes (0.26) come to as much.
#pragma once

template <typename S> struct PairShape; // inner sites of a window
// FP32: 16 wavefronts of at most 128 registers, 143 KB of LDS.  Others in the same builds: 32 x 28
// 697 against 612 us (sponge), 64 x 9 754 / 649 (sponge), 64 x 5, two workgroups per CU, 568 / 538
// (no obstacles).
template <> struct PairShape<float> { static constexpr int tx = 64, ty = 13; };
// FP64: 8 wavefronts of at most 256 registers, 138 KB of LDS.  64 x 5: 1.29 against 1.24 ms (no
// obstacles); 32 x 14 (9 wavefronts, 168 registers, spills) 1.62 / 1.30 (sponge).
template <> struct PairShape<double> { static constexpr int tx = 32, ty = 12; };

// storages that take two steps per launch
template <typename S> constexpr bool kPairs = std::is_same_v<S, float> || std::is_same_v<S, double>;

// LDS values per window site: the last two planes of the 4 populations with c_z = -1 and of the 8
// with c_z = 0 that move in x or y, the last three of the 4 with c_z = +1
constexpr int kPairSlots = 2 * 4 + 2 * 8 + 3 * 4;

// slot of such a population among those with its c_z
__device__ constexpr int pair_slot(int q)
{
    constexpr int slot[18] = {0, 0, 1, 0, 2, -1, 1, 3, 1, 4, 2, 5, 2, 6, -1, 3, 7, 3};
    return slot[q];
}

// threads: the window's rows and one wavefront for its two halo columns (32 rows at most)
template <typename S> constexpr int pair_threads()
{
    static_assert(PairShape<S>::tx * (PairShape<S>::ty + 2) % 64 == 0 && PairShape<S>::ty + 2 <= 32,
                  "whole wavefronts of window rows");
    return PairShape<S>::tx * (PairShape<S>::ty + 2) + 64;
}

// (with a margin before and after the slots for reads next to any site of the window)
template <typename S> constexpr size_t pair_lds_bytes()
{
    constexpr int wx = PairShape<S>::tx + 2, wy = PairShape<S>::ty + 2;
    return sizeof(S) * (kPairSlots * wx * wy + 2 * (wx + 1));
}

struct PairMap {
    uint32_t nx, ny;  // window columns in x and y
    uint32_t zc;      // planes per chunk
    uint32_t blocks;  // columns x chunks
    UDiv dnx, dny;
    uint32_t plane;   // bytes of one plane of tiles (below 2^31)
    int mixed;        // mixed tiles
};

// Consecutive workgroups (x fastest, then y, then z) that one XCD takes from each group of 8 of
// these (hardware block b runs on XCD b % 8): windows that share halo lines run on one XCD, at the same
// time.  512 x 256 x 256 FP32: 579 us per step with 32, 580 with 16, 588 with 64, 610 with 1, 590
// with one contiguous range per XCD.
constexpr uint32_t kPairGroup = 32;

// v, opaque to the optimiser: keeps what is computed from it (addresses) out of the registers that
// the plane loop holds throughout, or a loaded value from being loaded later
template <typename T> __device__ __forceinline__ T here(T v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// The kernel's arguments, read again where they are used: for what only a few workgroups need (the
// outlet planes), which would otherwise hold scalar registers throughout.
template <typename S> using LateArgs = const __attribute__((address_space(4))) XArgs<S>;
template <typename S> __device__ __forceinline__ LateArgs<S> *late_args()
{
    auto *p = __builtin_amdgcn_kernarg_segment_ptr(); // XArgs is the kernel's first argument
    asm volatile("" : "+s"(p));
    return (LateArgs<S> *)p;
}

// the workgroup's LDS accesses in order; global loads and stores stay in flight
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Buffer resources: an access whose offset lies outside reads zero or writes nothing, so lanes and
// planes without work need no branch around their accesses.  (Past a branch the compiler cannot count
// the accesses that a skipped path does not issue, and waits for all of them.)
using Rsrc = __amdgpu_buffer_rsrc_t;
constexpr uint32_t kOutside = 0x80000000u; // beyond every resource here

__device__ __forceinline__ Rsrc rsrc_of(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}

template <typename S> __device__ __forceinline__ S rsrc_load(Rsrc r, uint32_t off, int base)
{
    if constexpr (sizeof(S) == 4) return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, base, 0));
    else return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, base, 0));
}

// population Q of a plane's sites at byte offset off (the instruction's own offset has 12 bits)
template <typename S, int Q> __device__ __forceinline__ S raw_load_at(Rsrc r, uint32_t off)
{
    constexpr int b = Q * kTile * (int)sizeof(S);
    return rsrc_load<S>(r, off + (b & 4095), b & ~4095);
}

template <typename S, bool NT, int Q> __device__ __forceinline__ void raw_store_at(Rsrc r, uint32_t off, S v)
{
    constexpr int b = Q * kTile * (int)sizeof(S), lo = b & 4095, hi = b & ~4095;
    constexpr int aux = NT ? 2 : 0; // non-temporal
    if constexpr (sizeof(S) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)(off + lo), hi, aux);
    } else {
        typedef uint32_t u2 __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)(off + lo), hi, aux);
    }
}

// byte offsets, within a plane, of a window site's sources: xo[c_x + 1] those of its own row, plus
// ym (c_y = +1, the row y - 1) or yp (c_y = -1)
struct PairCol {
    uint32_t xo[3], ym, yp;
};

template <typename S, int... Qs>
__device__ __forceinline__ void pair_pull(QSeq<Qs...>, const Rsrc (&pl)[3], const PairCol &w, S *p)
{
    ((p[Qs] = raw_load_at<S, Qs>(pl[1 - Dir<Qs>::cz], w.xo[Dir<Qs>::cx + 1] +
                                                          (Dir<Qs>::cy == 0 ? 0u : (Dir<Qs>::cy > 0 ? w.ym : w.yp)))),
     ...);
}

// bounce-back in the first step: the site's own opposite population over the one pulled from a
// solid source
template <typename S, int Q> __device__ __forceinline__ void pair_own(Rsrc own, uint32_t off, uint32_t lm, S *p)
{
    if ((lm >> Q) & 1u) p[Q] = raw_load_at<S, Dir<Q>::opp>(own, off);
}

template <typename S, int... Qs>
__device__ __forceinline__ void pair_own_all(QSeq<Qs...>, Rsrc own, uint32_t off, uint32_t lm, S *p)
{
    (pair_own<S, Qs>(own, off, lm, p), ...);
}

// byte offsets of the rows y, y - 1, y + 1 in a plane of outlet ghost values
struct PairRow {
    int o, m, p;
};

// outlet ghost values that a site x = l - 1 of the row pulls: population 9 + v from the plane's entry
// (y - c_y, k - c_z)
template <typename S>
__device__ __forceinline__ void pair_outlet_pulls(const PairRow &row, int k, int km, int kp, S *p)
{
    LateArgs<S> &a = *late_args<S>();
    const int m = a.m, mn = a.m * a.n;
    const Rsrc o = rsrc_of(a.out_cur, 5u * (uint32_t)mn * (uint32_t)sizeof(S));
    auto at = [&](int v, int off, int z) { return rsrc_load<S>(o, (uint32_t)off, (v * mn + m * z) * (int)sizeof(S)); };
    p[9] = at(0, row.p, k);
    p[10] = at(1, row.o, kp);
    p[11] = at(2, row.m, k);
    p[12] = at(3, row.o, km);
    p[13] = at(4, row.o, k);
}

template <typename S> __device__ __forceinline__ void pair_collide(S *x, const XArgs<S> &a)
{
    if constexpr (kOnStored<S>) collide_dev<false>(x, a.bgk);
    else collide<S>(x, x, a.omega, a.fgrad);
}

// where a plane's first-step results are in LDS (of(i): the entries of window site i)
template <typename S, int WX, int SW> struct PairPlane {
    S *m, *z, *p; // c_z = -1, 0, +1
    __device__ __forceinline__ PairPlane of(int i) const { return {m + i, z + i, p + i}; }
    template <int Q> __device__ __forceinline__ S &at() const
    {
        constexpr int cz = Dir<Q>::cz;
        return (cz < 0 ? m : (cz == 0 ? z : p))[pair_slot(Q) * SW];
    }
    template <int Q> __device__ __forceinline__ void put(const S *x) const
    {
        if constexpr (Q != 5 && Q != 14) at<Q>() = x[Q];
    }
    // what the site pulls as population Q, if this is the plane it comes from
    template <int Q> __device__ __forceinline__ S source() const { return (&at<Q>())[-Dir<Q>::cy * WX - Dir<Q>::cx]; }
};

template <typename P, typename S, int... Qs>
__device__ __forceinline__ void pair_put(QSeq<Qs...>, const P &w, const S *x)
{
    (w.template put<Qs>(x), ...);
}

// second step, plane k: population Q from plane k - c_z (pl: planes k - 1, k, k + 1)
template <typename P, typename S, int Q> __device__ __forceinline__ void pair_take(const P (&pl)[3], S *x)
{
    if constexpr (Q != 5 && Q != 14) x[Q] = pl[1 - Dir<Q>::cz].template source<Q>();
}

template <typename P, typename S, int... Qs>
__device__ __forceinline__ void pair_take_all(QSeq<Qs...>, const P (&pl)[3], S *x)
{
    (pair_take<P, S, Qs>(pl, x), ...);
}

// Bounce-back in the second step: the site's own opposite populations of the first step, then a
// per-lane choice (o5, o14: populations 5 and 14, which are not in LDS).  A few at a time, and read
// before the choice: one by one inside a branch each, they cost the sponge 7 %, all 18 at once too
// many registers.
template <int Q, typename P, typename S> __device__ __forceinline__ S pair_own_of(const P &own, S o5, S o14)
{
    constexpr int op = Dir<Q>::opp;
    if constexpr (op == 5) return o5;
    else if constexpr (op == 14) return o14;
    else return own.template at<op>();
}

template <typename P, typename S, int... Qs>
__device__ __forceinline__ void pair_bounce(QSeq<Qs...>, uint32_t lm, const P &own, S o5, S o14, S *x)
{
    S b[18];
    ((b[Qs] = pair_own_of<Qs>(own, o5, o14)), ...);
    ((b[Qs] = here(b[Qs])), ...);
    ((x[Qs] = ((lm >> Qs) & 1u) ? b[Qs] : x[Qs]), ...);
}

template <typename S, bool NT, int... Qs>
__device__ __forceinline__ void pair_store(QSeq<Qs...>, Rsrc r, uint32_t off, const S *x)
{
    (raw_store_at<S, NT, Qs>(r, off, x[Qs]), ...);
}

template <typename S, bool XOPEN, bool NT>
__global__ __launch_bounds__((pair_threads<S>())) void k_pair(XArgs<S> a, PairMap pm)
{
    extern __shared__ __align__(16) char pair_lds[];
    constexpr int TX = PairShape<S>::tx, TY = PairShape<S>::ty;
    constexpr int WX = TX + 2, WY = TY + 2, SW = WX * WY;
    using Plane = PairPlane<S, WX, SW>;
    S *const lds = reinterpret_cast<S *>(pair_lds);

    uint32_t lb = blockIdx.x;
    {
        const uint32_t r8 = lb >> 3, g = r8 / kPairGroup, g0 = g * 8u * kPairGroup;
        if (g0 + 8u * kPairGroup <= gridDim.x) lb = g0 + (lb & 7u) * kPairGroup + (r8 - g * kPairGroup);
    }
    const uint32_t cr = pm.dnx.div(lb), bx = lb - cr * pm.nx, bz = pm.dny.div(cr), by = cr - bz * pm.ny;
    const int l = a.l, m = a.m, n = a.n;
    const int X0 = (int)bx * TX, Y0 = (int)by * TY, k0 = (int)(bz * pm.zc);
    const int planes = min((int)pm.zc, n - k0) + 2; // first-step planes k0 - 1 .. k0 + zc
    const int klast = k0 + planes - 2;              // the last of them (<= n)

    // the thread's window site; x = l (open) is the outlet ghost, run as the site l - 1
    constexpr int kMain = TX * WY;
    const int t = (int)threadIdx.x, h = t - kMain;
    const int wy = t < kMain ? t / TX : (h & 31), wx = t < kMain ? 1 + t % TX : (h < 32 ? 0 : TX + 1);
    int x = X0 + wx - 1, y = Y0 + wy - 1;
    bool active = wy < WY && x <= l && y <= m;
    bool ghost = false;
    if constexpr (XOPEN) {
        active = active && x >= 0;
        ghost = active && x == l;
        if (ghost) x = l - 1;
    } else {
        x = x < 0 ? l - 1 : (x >= l ? x - l : x);
    }
    y = y < 0 ? m - 1 : (y >= m ? y - m : y);
    const bool inner = active && wx >= 1 && wx <= TX && wy >= 1 && wy <= TY && X0 + wx - 1 < l && Y0 + wy - 1 < m;
    if (!active) { // any valid site
        x = 0;
        y = 0;
    }
    const int site = WX + 1 + min(wy, WY - 1) * WX + wx; // LDS index (lanes past the window: any)
    const bool at0 = XOPEN && x == 0, at1 = XOPEN && x == l - 1;

    const uint32_t tpr = (uint32_t)a.tpr, tpm = tpr * (uint32_t)m;
    PairCol w;
    {
        auto tile_at = [&](int xs, int ys) {
            return (((uint32_t)(xs >> 6) + tpr * (uint32_t)ys) * (uint32_t)kTileElems + (uint32_t)(xs & 63)) *
                   (uint32_t)sizeof(S);
        };
        int xm = x - 1, xp = x + 1;
        if constexpr (XOPEN) { // replaced by inlet and outlet values
            xm = max(xm, 0);
            xp = min(xp, l - 1);
        } else {
            xm = xm < 0 ? l - 1 : xm;
            xp = xp >= l ? 0 : xp;
        }
        w.xo[0] = tile_at(xp, y);
        w.xo[1] = tile_at(x, y);
        w.xo[2] = tile_at(xm, y);
        w.ym = tile_at(x, y == 0 ? m - 1 : y - 1) - w.xo[1];
        w.yp = tile_at(x, y == m - 1 ? 0 : y + 1) - w.xo[1];
    }
    const PairRow row{y * (int)sizeof(S), (y == 0 ? m - 1 : y - 1) * (int)sizeof(S),
                      (y == m - 1 ? 0 : y + 1) * (int)sizeof(S)};
    const uint32_t tile0 = (uint32_t)(x >> 6) + tpr * (uint32_t)y;
    const int lane = x & 63;
    const char *A = reinterpret_cast<const char *>(a.A);
    char *B = reinterpret_cast<char *>(a.B);

    auto wrap = [&](int k) { return k < 0 ? k + n : (k >= n ? k - n : k); }; // -2 <= k <= n + 1
    auto code_of = [&](int k) -> int32_t { return a.tile_code[tile0 + tpm * (uint32_t)wrap(min(k, klast))]; };
    // (after the mixed tiles' masks the table holds those of a fluid and of a solid tile)
    auto link_of = [&](int32_t code) -> uint32_t {
        const int e = code >= 0 ? code : pm.mixed + (code == kTileSolid ? 1 : 0);
        return a.link[(size_t)(uint32_t)e * kTile + (size_t)(uint32_t)lane];
    };
    auto plane_of = [&](const char *p, int k, uint32_t bytes) { return rsrc_of(p + (uint64_t)wrap(k) * pm.plane, bytes); };

    S P[19]; // pulls of plane kz
    // the pulls of plane k (nothing past the last one) ...
    auto load = [&](int k) {
        const uint32_t bytes = k <= klast ? pm.plane : 0u;
        k = min(k, klast);
        const Rsrc pl[3] = {plane_of(A, k - 1, bytes), plane_of(A, k, bytes), plane_of(A, k + 1, bytes)};
        const PairCol c{{w.xo[0], w.xo[1], w.xo[2]}, here(w.ym), here(w.yp)};
        pair_pull<S>(Q19{}, pl, c, P);
    };
    // ... and what replaces some of them: bounce-back and outlet ghost values
    auto load_other = [&](int k, uint32_t lm) {
        const uint32_t bytes = k <= klast ? pm.plane : 0u;
        k = min(k, klast);
        if (__ballot((lm & 0x7FFFFFFFu) != 0)) pair_own_all<S>(Q18{}, plane_of(A, k, bytes), w.xo[1], lm, P);
        if constexpr (XOPEN) {
            if (at1) pair_outlet_pulls<S>(row, wrap(k), wrap(k - 1), wrap(k + 1), P);
        }
    };

    // link masks of planes kz - 1, kz and kz + 1, and the tile code of plane kz + 2
    uint32_t lm_prev = 0x80000000u, lm, lm1;
    int32_t code2;
    {
        const int32_t c0 = code_of(k0 - 1), c1 = code_of(k0);
        code2 = code_of(k0 + 1);
        lm = link_of(c0);
        lm1 = link_of(c1);
    }
    load(k0 - 1);
    load_other(k0 - 1, lm);
    S o5 = S(0), o14 = S(0), o18 = S(0); // first-step results 5, 14 and 18 of plane kz - 1
    S oo5 = S(0);                        // and 5 of plane kz - 2
    S *const ldm = lds, *const ldz = lds + 8 * SW;
    S *p0 = lds + 24 * SW, *p1 = p0 + 4 * SW, *p2 = p1 + 4 * SW; // c_z = +1: planes kz, kz - 1, kz - 2

    for (int it = 0; it < planes; ++it) {
        const int kz = k0 - 1 + it, par = it & 1;
        const bool solid = (lm & 0x80000000u) != 0;
        // first step, plane kz (values of solid sites and of lanes past the window: not used)
        S x1[19];
#pragma unroll
        for (int q = 0; q < 19; ++q) x1[q] = P[q];
        if constexpr (XOPEN) {
            if (at0) {
#pragma unroll
                for (int q = 0; q < 5; ++q) x1[q] = a.inl[q];
            }
        }
        // the link mask and tile code of the planes after, then the pulls (loads return in order:
        // what the next plane waits for first goes first)
        const uint32_t lm2 = link_of(code2);
        code2 = code_of(kz + 3);
        load(kz + 1);
        pair_collide<S>(x1, a);
#pragma unroll
        for (int q = 0; q < 19; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x0020, 1, 0); // one load,
            __builtin_amdgcn_sched_group_barrier(0x0002, 9, 0); // nine VALU instructions
        }
        load_other(kz + 1, lm1);
        if constexpr (XOPEN) {
            if (ghost) {
                S o[5];
                if (solid) {
                    // a frozen site's outlet values never change
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        const S *p = late_args<S>()->out_cur + ((size_t)v * m * n + (size_t)m * wrap(kz));
                        o[v] = here(*at<S>(reinterpret_cast<const char *>(p), 0, (uint32_t)row.o));
                    }
                } else {
                    outlet_eq<S>(x1, o);
                }
#pragma unroll
                for (int v = 0; v < 5; ++v) x1[9 + v] = o[v];
            }
        }
        // into LDS, over planes kz - 2 (c_z <= 0) and kz - 3, which the second step of the previous
        // plane was the last to read
        const Plane cur{ldm + par * (4 * SW), ldz + par * (8 * SW), p0};
        const Plane prv{ldm + (par ^ 1) * (4 * SW), ldz + (par ^ 1) * (8 * SW), p1};
        lds_barrier();
        if (wy < WY) pair_put(Q18{}, cur.of(site), x1);
        lds_barrier();
        // second step, plane kz - 1
        S x2[19];
        const Plane own = prv.of(site);
        const Plane pl[3] = {Plane{ldm, ldz, p2}.of(site), own, cur.of(site)};
        pair_take_all(Q18{}, pl, x2);
        x2[5] = oo5;
        x2[14] = x1[14];
        x2[18] = o18;
        if (__ballot((lm_prev & 0x7FFFFFFFu) != 0)) {
            pair_bounce(QSeq<0, 1, 2, 3, 4, 5>{}, lm_prev, own, o5, o14, x2);
            pair_bounce(QSeq<6, 7, 8, 9, 10, 11>{}, lm_prev, own, o5, o14, x2);
            pair_bounce(QSeq<12, 13, 14, 15, 16, 17>{}, lm_prev, own, o5, o14, x2);
        }
        if constexpr (XOPEN) {
            if (at0) {
#pragma unroll
                for (int q = 0; q < 5; ++q) x2[q] = a.inl[q];
            }
        }
        pair_collide<S>(x2, a);
        const int ko = max(kz - 1, 0); // kz - 1, 0 <= ko < n, where a lane stores
        const bool out = it >= 2 && inner && !(lm_prev & 0x80000000u);
        pair_store<S, NT>(Q19{}, plane_of(B, ko, pm.plane), out ? w.xo[1] : kOutside, x2);
        if constexpr (XOPEN) {
            if (out && at1) {
                S o[5];
                outlet_eq<S>(x2, o);
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    S *p = late_args<S>()->out_next + ((size_t)v * m * n + (size_t)m * ko);
                    *reinterpret_cast<S *>(reinterpret_cast<char *>(p) + (uint32_t)row.o) = o[v];
                }
            }
        }
        oo5 = o5;
        o5 = x1[5];
        o14 = x1[14];
        o18 = x1[18];
        S *const pn = p2;
        p2 = p1;
        p1 = p0;
        p0 = pn;
        lm_prev = lm;
        lm = lm1;
        lm1 = lm2;
    }
}
