// gfx950 kernels of the FargoCPT hydro step.
//
// Every kernel restates one loop nest of the reference (file:line given above
// it) with the same expression order; the library is compiled with
// -ffp-contract=off so that add/mul/div/sqrt round exactly like the
// reference's host build.  Threads map x -> azimuthal index j (contiguous in
// HBM, so a wavefront reads 64 consecutive values) and y -> ring index i.
//
// Storage: every kernel is instantiated twice.  SPLIT = false keeps each field
// in FP64.  SPLIT = true keeps each 2-D field as an FP32 deviation from an FP64
// per-ring background (value = bg[ring] + (double)deviation), which halves the
// HBM traffic; the arithmetic is FP64 in both instantiations and the FP64
// instantiation performs exactly the operations of the reference.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "fcpt_device.hpp"
#include "fcpt_kernels.hpp"

namespace fcpt {

#define IX(i, j) ((size_t)(i) * (size_t)ns + (size_t)(j))

__device__ __forceinline__ double std_min(double a, double b) { return (b < a) ? b : a; }
__device__ __forceinline__ double std_max(double a, double b) { return (a < b) ? b : a; }
__device__ __forceinline__ double van_leer_lim(double a, double b)
{
    // TransportEuler.cpp:306-312, evaluated without a branch (the quotient of
    // a rejected pair is discarded)
    const double r = 2.0 * a * b / (a + b);
    return (a * b > 0.0) ? r : 0.0;
}
// Split storage rounds every stored value to an FP32 deviation, so its
// kernels may form quantities that only scale a correction term in FP32 and
// replace divisions by a reciprocal; the FP64 instantiations keep the
// reference's IEEE operations.  van Leer limiter: FP32 in split storage (the
// slope multiplies the second-order term of the interface value), its
// quotient through the hardware reciprocal (1 ulp; an FP32 division without
// fast-math is the IEEE sequence of about ten instructions).
template <bool SPLIT>
__device__ __forceinline__ double vl_lim(double a, double b)
{
    if constexpr (SPLIT) {
        const float fa = (float)a, fb = (float)b;
        const float r = 2.0f * fa * fb * __builtin_amdgcn_rcpf(fa + fb);
        return (fa * fb > 0.0f) ? (double)r : 0.0;
    } else {
        return van_leer_lim(a, b);
    }
}

// Quotients n / d that share one denominator d.  The compiler's IEEE FP64
// division on gfx950 is v_div_scale (range scaling of d and n), v_rcp, two
// Newton steps on the reciprocal, the quotient, one FMA correction
// (v_div_fmas) and v_div_fixup (zeros, infinities, NaNs, out-of-range
// results).  For |d| in [2^-250, 2^250) and |n| in [2^-400, 2^250) neither
// the scaling nor the fix-up changes anything, so the same reciprocal and
// correction steps written out give the same bits, and the reciprocal part
// (five instructions) is formed once per denominator: a quotient then costs
// three.  Other operands (zero aside, which returns the signed zero n * r)
// take the division itself.
struct SharedDen {
    double d, r;
    bool ok;
};
__device__ __forceinline__ SharedDen shared_den(double d)
{
    const double r0 = __builtin_amdgcn_rcp(d);
    const double e0 = fma(-d, r0, 1.0);
    const double r1 = fma(r0, e0, r0);
    const double e1 = fma(-d, r1, 1.0);
    const double r2 = fma(r1, e1, r1);
    const unsigned ed = (unsigned)((unsigned long long)__double_as_longlong(d) >> 52) & 0x7ffu;
    return SharedDen{d, r2, ed - 773u < 500u};
}
__device__ __forceinline__ double shared_div(double n, const SharedDen &D)
{
    const double q0 = n * D.r;
    const double rem = fma(-D.d, q0, n);
    double q = fma(rem, D.r, q0);
    const unsigned en = (unsigned)((unsigned long long)__double_as_longlong(n) >> 52) & 0x7ffu;
    if (n == 0.0) q = q0;
    else if (!D.ok || en - 623u >= 650u) q = n / D.d;
    return q;
}

// n / D.d by the shared reciprocal, for |n| below 2^900 and D.d in
// [2^-100, 2^100); below 2^-900 the quotient may be off by a unit of its last place
__device__ __forceinline__ double quot_fast(double n, const SharedDen &D)
{
    const double q0 = n * D.r;
    return fma(fma(-D.d, q0, n), D.r, q0);
}

// A denominator with its refined reciprocal, shared by several quotients: in
// FP64 storage shared_den's, so that in range (ok) the quotient is the IEEE one
// at three instructions; in split storage recip<true>'s, a product.  ok says
// that the denominator lies in [2^-100, 2^100) and the numerators the caller
// forms are within [2^-400, 2^250) or zero (quot_range); others divide.
__device__ __forceinline__ bool quot_range(double x)
{
    const unsigned e = (unsigned)((unsigned long long)__double_as_longlong(x) >> 52) & 0x7ffu;
    return e - 923u < 200u;
}
struct Den {
    double d, r;
    bool ok;
};
template <bool SPLIT>
__device__ __forceinline__ double quot_by(double n, const Den &D)
{
    if constexpr (SPLIT) {
        return n * D.r;
    } else {
        const double q0 = n * D.r;
        double q = fma(fma(-D.d, q0, n), D.r, q0);
        if (!D.ok) {
            __builtin_amdgcn_s_sleep(0);  // a branch: the division is not formed and selected
            q = n / D.d;
        }
        return q;
    }
}

// IEEE FP64 square root.  The compiler's sqrt on gfx950 scales x by 2^256
// below 2^-767, refines v_rsq by one Goldschmidt step and two Newton
// corrections, scales back, and passes zeros and +inf through a class test.
// For x in [2^-767, inf) the scalings are by 2^0 and the class test passes
// the refined value, so the refinement written out gives the same bits;
// other operands take sqrt itself.
__device__ __forceinline__ double sqrt_ieee(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    double e = fma(-g, g, x);
    g = fma(e, h, g);
    e = fma(-g, g, x);
    g = fma(e, h, g);
    if (!(x >= 0x1p-767 && x < __builtin_inf())) {
        __builtin_amdgcn_s_sleep(0);  // a branch: not both roots formed and selected
        g = sqrt(x);
    }
    return g;
}

// FP64 reciprocal: one IEEE division, or in split storage the hardware
// reciprocal refined by two Newton steps (error a few ulp)
template <bool SPLIT>
__device__ __forceinline__ double recip(double x)
{
    if constexpr (SPLIT) {
        double y = __builtin_amdgcn_rcp(x);
        y = y * (2.0 - x * y);
        return y * (2.0 - x * y);
    } else {
        return 1.0 / x;
    }
}

// 1 / sqrt(x): IEEE square root and division, or in split storage the
// hardware reciprocal square root refined by two Newton steps
template <bool SPLIT>
__device__ __forceinline__ double inv_sqrt(double x)
{
    if constexpr (SPLIT) {
        double y = __builtin_amdgcn_rsq(x);
        y = y * (1.5 - 0.5 * x * y * y);
        return y * (1.5 - 0.5 * x * y * y);
    } else {
        return 1.0 / sqrt(x);
    }
}

// n / d: the IEEE quotient, or in split storage the product of n with the
// refined reciprocal of d
template <bool SPLIT>
__device__ __forceinline__ double quot(double n, double d)
{
    if constexpr (SPLIT) return n * recip<true>(d);
    else return n / d;
}

__device__ __forceinline__ double omega_kepler(const KParams &P, double r)
{
    return sqrt(P.G * P.mstar / (r * r * r));  // Theo.cpp:246-249
}


// dt and time of the running kick (no kernel that reads them writes them, so they
// are scalar loads that stores do not repeat)
__device__ __forceinline__ double kick_dt(const KParams &P)
{
    const double dt = *(const __attribute__((address_space(4))) double *)&P.s->dt;
    return P.kick ? dt / 2 : dt;
}
__device__ __forceinline__ double kick_time(const KParams &P)
{
    const double t = *(const __attribute__((address_space(4))) double *)&P.s->time;
    return P.kick == 2 ? t + kick_dt(P) : t;
}

// Per-ring arrays (metric, backgrounds, ring means, shifts) are never written
// by the kernel that reads them.  Reading them through the constant address
// space says so: with a wave-uniform index they become scalar loads, which
// use their own counter and do not wait behind the wavefront's vector loads.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *cst(const T *p)
{
    return (const __attribute__((address_space(4))) T *)p;
}

// Split storage rounds each deviation to FP32 either to nearest or
// stochastically: up or down with probabilities proportional to the distances
// to the two neighbouring FP32 values (the rounding is unbiased, so the
// per-step roundings of a slowly changing value do not add up in one
// direction: an increment below half an FP32 unit of the deviation survives
// on average instead of being lost every step).  The uniform variate of a
// store is one multiply-xorshift round (Wellons' hash prospector, public
// domain) of the cell index, the deviation's high word (sign, exponent and
// leading mantissa bits: independent of the dropped bits, and different for
// the several values one field of one cell takes in a step) and a key drawn
// per field and step (sr_key, Wellons' lowbias32): a value always rounds the
// same way at its cell within one kernel (a thread can form what another
// thread stores) and differently from step to step.
__device__ __forceinline__ unsigned sr_hash(unsigned x)
{
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}
// one multiply-xorshift round (the first half of lowbias32)
__device__ __forceinline__ unsigned sr_bits(unsigned x)
{
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    return x;
}
__device__ __forceinline__ float round_dev(double d, unsigned key, unsigned c)
{
    if (!key) return (float)d;
    // add a 29-bit variate below the FP32 unit of the FP64 deviation and drop
    // those 29 bits: rounded away from zero with probability (dropped
    // bits) / 2^29.  Exact for |d| in [2^-126, 2^128) (the sign bit is never
    // reached); smaller deviations are rounded once more by the conversion,
    // infinities stay infinite.
    const unsigned long long b0 = (unsigned long long)__double_as_longlong(d);
    const unsigned u = sr_bits(c ^ key ^ (unsigned)(b0 >> 32)) >> 3;
    const unsigned long long b = b0 + (unsigned long long)u;
    return (float)__longlong_as_double((long long)(b & ~0x1fffffffull));
}
__device__ __forceinline__ unsigned sr_key(int id, unsigned step)
{
    return sr_hash(step * 0x85ebca77u + (unsigned)id * 0xc2b2ae3du) | 1u;
}

// field accessor: an FP64 array, or FP32 deviations from an FP64 ring background.
// An element's address is its row's (scalar where the ring is) plus a 32-bit
// byte offset along the ring, which the load and store instructions add
// themselves: no 64-bit address per lane (a row is at most 2 MiB).
template <bool SPLIT>
struct Fld {
    using T = typename std::conditional<SPLIT, float, double>::type;
    T *p;
    const double *bg;
    int ns;
    unsigned key;  // split storage: 0 rounds to nearest, else the stochastic rounding's key
    __device__ __forceinline__ T &at(int i, int j) const
    {
        char *row = reinterpret_cast<char *>(p) + (size_t)i * (size_t)ns * sizeof(T);
        return *reinterpret_cast<T *>(row + (unsigned)j * (unsigned)sizeof(T));
    }
    // the rounding's cell number (its low 32 bits)
    __device__ __forceinline__ unsigned cell(int i, int j) const { return (unsigned)i * (unsigned)ns + (unsigned)j; }
    __device__ __forceinline__ double operator()(int i, int j) const
    {
        if constexpr (SPLIT) return cst(bg)[i] + (double)at(i, j);
        else return at(i, j);
    }
    __device__ __forceinline__ void set(int i, int j, double v) const
    {
        if constexpr (SPLIT) at(i, j) = round_dev(v - cst(bg)[i], key, cell(i, j));
        else at(i, j) = v;
    }
    // the stored value alone, and its decoding: lets a kernel issue a load
    // early and pay for it where the value is used
    __device__ __forceinline__ T raw(int i, int j) const { return at(i, j); }
    __device__ __forceinline__ void set_raw(int i, int j, T x) const { at(i, j) = x; }
    // store v at (i, j) and return it as a later load of it returns it
    __device__ __forceinline__ double set_get(int i, int j, double v) const
    {
        if constexpr (SPLIT) {
            const double b = cst(bg)[i];
            const float x = round_dev(v - b, key, cell(i, j));
            at(i, j) = x;
            return b + (double)x;
        } else {
            at(i, j) = v;
            return v;
        }
    }
    // v as a later load of the value stored at (i, j) returns it
    __device__ __forceinline__ double stored(int i, int j, double v) const
    {
        if constexpr (SPLIT) return cst(bg)[i] + (double)round_dev(v - cst(bg)[i], key, cell(i, j));
        else return v;
    }
    // the stored form of v at (i, j)
    __device__ __forceinline__ T enc(int i, int j, double v) const
    {
        if constexpr (SPLIT) return round_dev(v - cst(bg)[i], key, cell(i, j));
        else return v;
    }
    __device__ __forceinline__ double dec(int i, T x) const
    {
        if constexpr (SPLIT) return cst(bg)[i] + (double)x;
        else return x;
    }
};

// value t of ring i in KParams::ring_tab (formed once by k_ring_tables with
// the expressions of its users: the same bits)
__device__ __forceinline__ double ring_tab(const KParams &P, int t, int i)
{
    return cst(P.ring_tab)[i * kRingTabs + t];
}
// the same for a ring walk, whose wavefront holds the rows of its rings in LDS
// from row0 on: a scalar load per value and ring misses the scalar cache once
// per ring and stalls the walk at every use
struct KWalk : KParams {
    const double *rows;
    int row0;
    double dt;  // of the running kick
};
__device__ __forceinline__ double kick_dt(const KWalk &P) { return P.dt; }
__device__ __forceinline__ double kick_time(const KWalk &P)
{
    const double t = *(const __attribute__((address_space(4))) double *)&P.s->time;
    return P.kick == 2 ? t + P.dt : t;
}
__device__ __forceinline__ double ring_tab(const KWalk &P, int t, int i)
{
    return P.rows[(i - P.row0) * kRingTabs + t];
}

// the rounding key of split-storage stores of field (or buffer) `id` in the
// current step; 0 (to nearest) in FP64 storage, with stochastic rounding off,
// and (split_rounding 1) for the fields derived afresh from the state every
// step, whose roundings do not accumulate: stochastic rounding then applies
// to the evolved fields Sigma, v_r, v_phi, E and the transported momenta
constexpr int kBufMom = 64;
__device__ __forceinline__ bool carries_state(int id)
{
    return id == FCPT_SIGMA || id == FCPT_VRAD || id == FCPT_VAZI || id == FCPT_ENERGY || id >= kBufMom;
}
template <bool SPLIT>
__device__ __forceinline__ unsigned store_key(const KParams &P, int id)
{
    if constexpr (SPLIT) {
        const int mode = P.split_rounding;
        return (mode == 2 || (mode == 1 && carries_state(id))) ? sr_key(id, *cst(P.step_at)) : 0u;
    } else {
        return 0u;
    }
}
template <bool SPLIT>
__device__ __forceinline__ Fld<SPLIT> fld(const KParams &P, int f)
{
    return Fld<SPLIT>{static_cast<typename Fld<SPLIT>::T *>(P.f[f]), P.bg[f], P.ns, store_key<SPLIT>(P, f)};
}
// a derived field as the end of the last step (or the caller) rounded it
template <bool SPLIT>
__device__ __forceinline__ Fld<SPLIT> fld_derived(const KParams &P, int f)
{
    Fld<SPLIT> x = fld<SPLIT>(P, f);
    if constexpr (SPLIT)
        if (P.split_rounding == 2) x.key = sr_key(f, *cst(&P.s->count_derived));
    return x;
}
// a work buffer; id names it for the rounding key (the momenta: kBufMom + q)
template <bool SPLIT>
__device__ __forceinline__ Fld<SPLIT> buf(const KParams &P, void *p, const double *bg, int id = -1)
{
    return Fld<SPLIT>{static_cast<typename Fld<SPLIT>::T *>(p), bg, P.ns, id >= 0 ? store_key<SPLIT>(P, id) : 0u};
}

#define FLD(name, id) const Fld<SPLIT> name = fld<SPLIT>(P, id)

// The transported momenta, read by the end of the step: FP64 in both storage
// modes (in split storage their FP32 rounding, once per step, was the largest
// part of the error near the planets, and the sweeps are bound by their
// instructions, which the stochastic rounding of four stores per cell adds to)
__device__ __forceinline__ Fld<false> mom_out(const KParams &P, int q)
{
    return Fld<false>{static_cast<double *>(P.mom[q]), nullptr, P.ns, 0u};
}

// The gas potential is stored in FP64 in both storage modes: its radial and
// azimuthal differences drive the source terms, and near a body the
// potential's deviation from any ring profile is large, so an FP32 deviation
// would round the gradient there by about 2^-24 |dev| / |difference|.
__device__ __forceinline__ Fld<false> phi_fld(const KParams &P)
{
    return Fld<false>{static_cast<double *>(P.f[FCPT_POTENTIAL]), nullptr, P.ns, 0u};
}

// Neighbour values within a wavefront: the value of lane - 1 and of lane + 1,
// moved by the DPP wavefront shifts (wave_shr:1, wave_shl:1) on both 32-bit
// halves; the edge lanes, which have no source lane, receive 0 (bound_ctrl,
// so no old value has to be set first) and their results are discarded
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)(b & 0xffffffffll), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double from_left(double x) { return dpp_move<0x138>(x); }
__device__ __forceinline__ double from_right(double x) { return dpp_move<0x130>(x); }

// Kernels read every input before their first store: the compiler must
// assume that a store may alias any later load, so a load written after a
// store waits for it and the memory latency is paid once per such phase.

// Cell kernels run 64 x 4 blocks: one wavefront is one 64-sector piece of
// one ring, so the ring index is the same in every lane.  Reading it through
// readfirstlane tells the compiler so, and the per-ring metric values and
// backgrounds become scalar loads.
__device__ __forceinline__ int wave_ring(int r0, int by)
{
    return __builtin_amdgcn_readfirstlane(r0 + by * (int)blockDim.y + (int)threadIdx.y);
}

// XCD-aware block order.  The dispatcher hands workgroup b of a launch to XCD
// b mod 8 (each XCD has its own L2), so blocks adjacent in the grid, which
// share stencil halos (sector halo lanes, cache lines at segment edges, the
// rings a walk reloads), would run on different XCDs and fetch the shared
// lines once per XCD.  xcd_block gives each XCD a contiguous run of the grid
// instead: the workgroups XCD x receives (b = x, x + 8, ...) take the x-th
// run of linear indices in order, so neighbours share an L2 and run close in
// time.  A bijection of [0, gx gy); the block's work is unchanged.
struct BlockXY {
    int x, y;
};
__device__ __forceinline__ BlockXY xcd_block()
{
    constexpr unsigned kXcds = 8;
    const unsigned gx = gridDim.x, G = gridDim.x * gridDim.y;
    const unsigned b = blockIdx.y * gx + blockIdx.x;
    const unsigned xcd = b % kXcds, idx = b / kXcds, q = G / kXcds, r = G % kXcds;
    const unsigned L = xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
    return BlockXY{(int)(L % gx), (int)(L / gx)};
}

// 2-D launch over rows [r0, r1) x all sectors; (bx, by) is the block's place
// in the disk's own grid
#define CELL_LOOP_HEAD(r0, r1)                                   \
    const int ns = P.ns;                                         \
    const int j = bx * (int)blockDim.x + (int)threadIdx.x;       \
    const int i = wave_ring(r0, by);                             \
    if (j >= ns || i >= (r1)) return;

// Every kernel body takes the disk's parameters and its block coordinates
// (bx, by) in that disk's grid, and comes in up to two launch forms: k_NAME runs
// one disk on its own grid; kb_NAME, of the batched step's stages, many disks in
// one launch, each
// block reading (disk, by << 16 | bx) from a per-stage work table and the
// disk's parameters from a device array (constant address space: scalar
// loads).
__device__ __forceinline__ BatchEntry batch_entry(const BatchEntry *map)
{
    const auto *m = cst(map) + blockIdx.x;
    return BatchEntry{m->disk, m->yx};
}
__device__ __forceinline__ KParams batch_disk(const KParams *Ps, unsigned d)
{
    // a copy through the constant address space, word by word: the fields a
    // kernel uses become scalar loads at its start, as kernel arguments do
    static_assert(sizeof(KParams) % 8 == 0, "KParams is copied in 8-byte words");
    KParams P;
    const auto src = cst(reinterpret_cast<const unsigned long long *>(Ps + d));
    unsigned long long *dst = reinterpret_cast<unsigned long long *>(&P);
#pragma unroll
    for (unsigned k = 0; k < sizeof(KParams) / 8; ++k) dst[k] = src[k];
    return P;
}

#define FCPT_ONE0(name, BOUNDS)                                                                   \
    template <bool SPLIT>                                                                         \
    __global__ void __launch_bounds__(BOUNDS) k_##name(KParams P)                                 \
    {                                                                                             \
        b_##name<SPLIT>(P, (int)blockIdx.x, (int)blockIdx.y);                                     \
    }

#define FCPT_PAIR0(name, BOUNDS)                                                                  \
    FCPT_ONE0(name, BOUNDS)                                                                       \
    template <bool SPLIT>                                                                         \
    __global__ void __launch_bounds__(BOUNDS) kb_##name(const KParams *Ps, const BatchEntry *map)  \
    {                                                                                             \
        const BatchEntry e = batch_entry(map);                                                \
        b_##name<SPLIT>(batch_disk(Ps, e.disk), (int)(e.yx & 0xffffu), (int)(e.yx >> 16));        \
    }

#define FCPT_ONE1(name, BOUNDS, T1, a1)                                                           \
    template <bool SPLIT>                                                                         \
    __global__ void __launch_bounds__(BOUNDS) k_##name(KParams P, T1 a1)                          \
    {                                                                                             \
        b_##name<SPLIT>(P, (int)blockIdx.x, (int)blockIdx.y, a1);                                 \
    }

#define FCPT_PAIR1(name, BOUNDS, T1, a1)                                                          \
    FCPT_ONE1(name, BOUNDS, T1, a1)                                                               \
    template <bool SPLIT>                                                                         \
    __global__ void __launch_bounds__(BOUNDS)                                                     \
        kb_##name(const KParams *Ps, const BatchEntry *map, T1 a1)                                \
    {                                                                                             \
        const BatchEntry e = batch_entry(map);                                                \
        b_##name<SPLIT>(batch_disk(Ps, e.disk), (int)(e.yx & 0xffffu), (int)(e.yx >> 16), a1);    \
    }

// ---------------------------------------------------------------------------
// ring sums (cfl.cpp:196-205, TransportEuler.cpp:174-190): one block per ring,
// pairwise tree order
// 256 threads' values, the first 256 of the block, summed in pairwise tree order
// (t + 128, t + 64, ..., t + 1): every wavefront adds the four wavefronts'
// values and then its lanes' (the two lanes of a pair form the same sum), so
// the tree takes one barrier and every thread has the result.  With a barrier
// per level the step took 0.4 to 0.8 us longer (128x384: 28.3 -> 27.6).
__device__ __forceinline__ double wave_tree(double v)
{
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) v = v + __shfl_xor(v, s, 64);
    return v;
}
__device__ __forceinline__ double block_sum(double v, double *sh)
{
    const int t = (int)(threadIdx.y * blockDim.x + threadIdx.x), l = t & 63;
    if (t < 256) sh[t] = v;
    __syncthreads();
    return wave_tree((sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192]));
}

// The ring sum and the sum of the magnitudes of its terms in one tree: the
// sum's additions are exactly those of block_sum.
__device__ __forceinline__ double2 block_sum_abs(double v, double a, double2 *sh)
{
    const int t = (int)threadIdx.x, l = t & 63;
    sh[t] = double2{v, a};
    __syncthreads();
    const double2 p = sh[l], q = sh[l + 64], r = sh[l + 128], u = sh[l + 192];
    return double2{wave_tree((p.x + r.x) + (q.x + u.x)), wave_tree((p.y + r.y) + (q.y + u.y))};
}

// mode 0: CFL ring mean
// mode 1: transport ring mean + FARGO shift (TransportEuler.cpp:215-220) +
//         uniform residual (:207-236)
// The reference sums a ring left to right (TransportEuler.cpp:178-183); the
// block's tree sums the same terms in another order.  Any two summation
// orders of n terms differ by at most 2 gamma_(n-1) sum |term| (gamma_k =
// k u / (1 - k u), u = 2^-53), and the shift floor(Ntilde + 0.5) is a
// monotone function of the sum (a division by ns and products with positive
// ring constants, each rounded monotonically).  So when both ends of the
// interval sum -/+ that bound give the same shift, the left-to-right sum
// gives it too; otherwise thread 0 forms the left-to-right sum itself
// (seq_sum: the ring's terms in order) and the ring's mean, shift and
// residual come from it, as in the reference.
// What a ring's FARGO shift needs besides its sum, loaded (and 1 / dt formed)
// while the ring's values are under way
struct MeanConst {
    double dt, invdt, inv_rmed, rmed;
};
__device__ __forceinline__ MeanConst mean_const(const KParams &P, int i)
{
    const double dt = P.s->dt;
    return MeanConst{dt, 1.0 / dt, cst(P.InvRmed)[i], cst(P.Rmed)[i]};
}
// the first wavefront's lanes 0, 1 and 2 form the shift of the sum and of its
// interval's ends at once
template <typename SeqSum>
__device__ __forceinline__ void ring_mean_store(const KParams &P, int i, double sum, double asum, int mode,
                                                const MeanConst &c, SeqSum seq_sum)
{
    const int t = (int)threadIdx.x;
    if (t >= 64) return;
    const double nsd = (double)P.ns;
    if (mode == 1) {
        const double bound = asum * (2.02 * nsd * 0x1p-53) + fabs(sum) * 0x1p-50;
        double vm = (t == 1 ? sum - bound : t == 2 ? sum + bound : sum) / nsd;
        double Ntilde = vm * c.inv_rmed * c.dt * P.invdphi;
        double Nround = floor(Ntilde + 0.5);
        const double lo = __shfl(Nround, 1, 64), hi = __shfl(Nround, 2, 64);
        if (t != 0) return;
        if (!(lo == hi)) {
            vm = seq_sum() / nsd;
            Ntilde = vm * c.inv_rmed * c.dt * P.invdphi;
            Nround = floor(Ntilde + 0.5);
        }
        P.vmean[i] = vm;
        P.nshift[i] = (int)Nround;
        P.vuni[i] = (Ntilde - Nround) * c.rmed * c.invdt * P.dphi;
    } else if (t == 0) {
        P.vmean[i] = sum / nsd;
    }
}

// One thread's share of a ring sum: the sectors t, t + STRIDE, t + 2 STRIDE,
// ... below ns, added in that order.  Eight sectors' loads are issued before
// their additions (a loop of one load and one addition keeps one load in
// flight per thread and waits for each): the same additions in the same
// order, so the same bits.
template <int STRIDE, class Load, class Add>
__device__ __forceinline__ void strided_row(int ns, int t, Load &&load, Add &&add)
{
    constexpr int U = 8;
    int j = t;
    for (; j + STRIDE * (U - 1) < ns; j += STRIDE * U) {
        double x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = load(j + STRIDE * u);
#pragma unroll
        for (int u = 0; u < U; ++u) add(x[u]);
    }
    for (; j < ns; j += STRIDE) add(load(j));
}

template <bool SPLIT>
__device__ __forceinline__ void b_ring_mean(const KParams &P, int bx, int by, int mode)
{
    __shared__ double2 sh[256];
    const int ns = P.ns;
    const int i = bx;
    FLD(v, FCPT_VAZI);
    const MeanConst c = mode == 1 ? mean_const(P, i) : MeanConst{};
    double acc = 0.0, aacc = 0.0;
    strided_row<256>(ns, (int)threadIdx.x, [&](int j) { return v(i, j); }, [&](double x) {
        acc += x;
        aacc += fabs(x);
    });
    const double2 r = block_sum_abs(acc, aacc, sh);
    ring_mean_store(P, i, r.x, r.y, mode, c, [&]() {
        double seq = 0.0;
        for (int j = 0; j < ns; ++j) seq += v(i, j);
        return seq;
    });
}
FCPT_ONE1(ring_mean, 256, int, mode)

// The fold of the CFL limits (cfl.cpp:210-376): the rings' smallest
// (b_cfl_ring's slots) and the shear limits between the rings' means.
// mode 0: condition_cfl only; 1: sim::CalculateTimeStep (simulation.cpp:100-118);
// 2: CalculateTimeStep + the monitor clip of sim::run (simulation.cpp:526-542).
// One block of 256 threads (thread index t) folds them in a fixed pairwise
// order: deterministic and free of atomics.
__device__ __forceinline__ double cfl_shear(const KParams &P, int k)
{
    // the limit of the shear between rings k and k + 1 (cfl.cpp:223-233)
    const double *vm = P.vmean;
    const double denom = fabs(vm[k] * P.InvRmed[k] - vm[k + 1] * P.InvRmed[k + 1]) + 1.0e-100;
    return P.cfl * P.dphi / denom;
}

// the monitor clip of sim::run (simulation.cpp:526-542)
__device__ __forceinline__ double monitor_clip(const KParams &P, double rv, int n_monitor, double time)
{
    const double time_next_monitor = (n_monitor + 1) * P.monitor_timestep;
    const double time_left_till_write = time_next_monitor - time;
    const bool overshoot = rv > time_left_till_write;
    const double dt_stretch_factor = 0.05;
    const bool almost_there = time_left_till_write < rv * (1 + dt_stretch_factor);
    return (overshoot || almost_there) ? time_left_till_write : rv;
}

__device__ __forceinline__ void b_cfl_fold(const KParams &P, int mode, int t)
{
    __shared__ double sh[256];
    double m = __longlong_as_double(0x7FF0000000000000ll);
    for (int k = t; k < P.nr; k += 256) m = std_min(m, P.ring_min[k]);
    for (int k = t; k < P.nr - 1; k += 256) m = std_min(m, cfl_shear(P, k));
    sh[t] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) sh[t] = std_min(sh[t], sh[t + w]);
        __syncthreads();
    }
    if (t != 0) return;
    DevScalars *s = P.s;
    const double cfl_dt = sh[0];
    s->cfl_dt = cfl_dt;
    s->step_count += 1u;
    s->count_next = s->step_count + 1u;
    if (!(cfl_dt > 0.0) || !isfinite(cfl_dt)) s->error_flags |= 1;
    if (mode >= 1) {
        const double rv = std_min(P.cfl_max_var * s->last_dt, cfl_dt);
        s->last_dt = rv;
        s->last_prev = rv;
        s->cfl_dt = rv;
        if (mode == 2) s->dt = monitor_clip(P, rv, s->n_monitor, s->time);
    }
}

// The fold (mode 2) by one wavefront of the kick walk: every wavefront forms
// the same dt from the ring minima and means, and the one with `writes` stores
// the clock; none reads what that one writes (last_prev and count_next are
// the last_dt and the next step_count that the last step left).  The shear limits take
// one division: the smallest quotient is that of the largest shear.
constexpr int kFoldRings = 512;  // most rings: eight per lane
struct FoldLoads {
    double lim[kFoldRings / 64], vm[kFoldRings / 64], rm[kFoldRings / 64];
};
__device__ __forceinline__ void cfl_fold_load(const KParams &P, int lane, FoldLoads &x)
{
#pragma unroll
    for (int q = 0; q < kFoldRings / 64; ++q) {
        if (64 * q >= P.nr) continue;  // uniform
        const int c = lane + 64 * q < P.nr ? lane + 64 * q : P.nr - 1;
        x.lim[q] = P.ring_min[c];
        x.vm[q] = P.vmean[c];
        x.rm[q] = P.InvRmed[c];
    }
}
__device__ __forceinline__ double cfl_fold_wave(const KParams &P, int lane, bool writes, const FoldLoads &x)
{
    double m = __longlong_as_double(0x7FF0000000000000ll), shear = 1.0e-100, next = 0.0;
#pragma unroll
    for (int q = kFoldRings / 64 - 1; q >= 0; --q) {
        if (64 * q >= P.nr) continue;
        m = std_min(m, x.lim[q]);
        // the ring outside is the next lane's; the last lane's the next round's first
        const double om = x.vm[q] * x.rm[q], right = from_right(om);
        const double out = lane == 63 ? next : right;
        if (lane + 64 * q < P.nr - 1) shear = std_max(shear, fabs(om - out) + 1.0e-100);
        next = __shfl(om, 0, 64);
    }
    for (int off = 32; off > 0; off >>= 1) {
        m = std_min(m, __shfl_xor(m, off, 64));
        shear = std_max(shear, __shfl_xor(shear, off, 64));
    }
    const double cfl_dt = std_min(m, P.cfl * P.dphi / shear);
    const double rv = std_min(P.cfl_max_var * *cst(&P.s->last_prev), cfl_dt);
    const double dt = monitor_clip(P, rv, *cst(&P.s->n_monitor), *cst(&P.s->time));
    if (writes && lane == 0) {
        DevScalars *s = P.s;
        if (!(cfl_dt > 0.0) || !isfinite(cfl_dt)) s->error_flags |= 1;
        s->step_count = s->count_next;
        s->last_dt = rv;
        s->cfl_dt = rv;
        s->dt = dt;
    }
    return dt;
}

// adiabatic sound speed, scale height and viscosity of one cell
// (compute_sound_speed, compute_scale_height, compute_viscosity)
template <bool SPLIT>
__device__ __forceinline__ Den make_den(double d, bool in_range)
{
    if constexpr (SPLIT) {
        return Den{d, recip<true>(d), true};
    } else {
        const SharedDen s = shared_den(d);
        return Den{d, s.r, in_range && quot_range(d)};
    }
}
struct AdiDerived {
    double cs, h, nu;
};
template <bool SPLIT>
__device__ __forceinline__ AdiDerived adi_derived(const KParams &P, int i, double e, double sig)
{
    AdiDerived d;
    const double g = P.gamma;
    const double inv_omega_kepler = ring_tab(P, TAB_INV_OMEGA_K, i);  // 1 / Omega_K(Rmed)
    if constexpr (SPLIT) {  // products with reciprocals (the 1 / sqrt(gamma) is launch-wide)
        d.cs = sqrt(g * (g - 1.0) * e * recip<true>(sig));
        d.h = d.cs * inv_sqrt<true>(g) * inv_omega_kepler;
    } else {
        d.cs = sqrt_ieee(g * (g - 1.0) * e / sig);
        d.h = d.cs / (sqrt(g)) * inv_omega_kepler;
    }
    const double alpha = P.alpha;
    d.nu = alpha * d.h * d.cs;
    return d;
}

// the same (FP64 storage) with the quotients by Sigma and sqrt(gamma) through
// their reciprocals where `fine` says that E, Sigma and the constants are in range
template <bool SPLIT, class PP>
__device__ __forceinline__ AdiDerived adi_derived_in(const PP &P, int i, double e, double sig, bool fine)
{
    if constexpr (SPLIT) {
        return adi_derived<true>(P, i, e, sig);
    } else {
        AdiDerived d;
        d.cs = sqrt_ieee(quot_by<false>(ring_tab(P, TAB_G_GM1, i) * e, Den{sig, shared_den(sig).r, fine}));
        const Den sg{ring_tab(P, TAB_SQRT_GAMMA, i), ring_tab(P, TAB_SQRT_GAMMA_RCP, i), fine};
        d.h = quot_by<false>(d.cs, sg) * ring_tab(P, TAB_INV_OMEGA_K, i);
        const double alpha = P.alpha;
        d.nu = alpha * d.h * d.cs;
        return d;
    }
}

// split storage: c_s and nu as a step that stores them reads them back
template <bool SPLIT>
__device__ __forceinline__ AdiDerived adi_derived_stored(const KParams &P, int i, int j, double e, double sig)
{
    AdiDerived a = adi_derived<SPLIT>(P, i, e, sig);
    if (SPLIT && (P.split_emul & SPLIT_EMUL_DERIVED)) {
        a.cs = fld_derived<SPLIT>(P, FCPT_SOUNDSPEED).stored(i, j, a.cs);
        a.nu = fld_derived<SPLIT>(P, FCPT_VISCOSITY).stored(i, j, a.nu);
    }
    return a;
}

// The CFL limit of cell (i, j) is CFL / sqrt(sum) (cfl.cpp:235-376), sum the
// squares of six inverse times added in their order; vm_i is the ring's mean
// v_phi, and h receives the scale height where the derived fields are formed
// here.  Division and root round monotonically, so the smallest limit is that
// of the largest sum: the kernels take the largest sums and form one limit
// (cfl_limit).  FAST divides by the ring's cell sizes and by E through refined
// reciprocals, which gives the same bits for finite numerators below 2^400 and
// sizes and E in [2^-100, 2^100); the caller forms a sum that is not below
// 2^400 again without it.
struct CflRing {
    double inv_cell2;  // split storage
    SharedDen dr, daz, cell, cell2;
    bool fast;
};
// the ring's cell sizes and their reciprocals: in FP64 storage from
// KParams::cfl_tab through scalar loads, in split storage (no fall-back, two
// reciprocals) formed here, where as many scalars would spill
template <bool SPLIT>
__device__ __forceinline__ CflRing cfl_ring(const KParams &P, int i)
{
    CflRing R{};
    if constexpr (SPLIT) {
        const double dr = cst(P.Rsup)[i] - cst(P.Rinf)[i], daz = cst(P.Rmed)[i] * P.dphi;
        R.dr.r = cst(P.InvDiffRsup)[i];
        R.daz.r = recip<true>(daz);
        R.cell.r = recip<true>(std_min(dr, daz));
        R.inv_cell2 = R.cell.r * R.cell.r;
    } else {
        const auto t = cst(P.cfl_tab) + 8 * i;
        R.dr = SharedDen{t[0], t[1], true};
        R.daz = SharedDen{t[2], t[3], true};
        R.cell = SharedDen{t[4], t[5], true};
        R.cell2 = SharedDen{t[6], t[7], true};
        R.fast = quot_range(R.dr.d) && quot_range(R.daz.d) && quot_range(R.cell2.d);
    }
    return R;
}
template <bool SPLIT>
struct CflCell {
    double vr0, vr1, va0, va1, e, qp, qm, cs, nu, h;
};
template <bool SPLIT>
__device__ __forceinline__ CflCell<SPLIT> cfl_load(const KParams &P, int i, int j)
{
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const double vr0 = vr(i, j), vr1 = vr(i + 1, j);
    const double va0 = vaz(i, j), va1 = vaz(i, j == P.ns - 1 ? 0 : j + 1);
    // one block of loads: a value decoded in a block of its own waits there
    double e = 0.0, qp = 0.0, qm = 0.0, cs, nu, h = 0.0;
    if (!P.adiabatic) {  // ring profiles
        cs = cst(P.iso_cs)[i];
        nu = cst(P.iso_nu)[i];
    } else if (P.lazy_derived) {
        e = fld<SPLIT>(P, FCPT_ENERGY)(i, j);
        const double sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
        qp = fld<SPLIT>(P, FCPT_QPLUS)(i, j);
        qm = fld<SPLIT>(P, FCPT_QMINUS)(i, j);
        // as recalculate_derived forms them from the same E and Sigma
        const AdiDerived a = adi_derived_stored<SPLIT>(P, i, j, e, sig);
        cs = a.cs;
        nu = a.nu;
        h = a.h;
    } else {
        e = fld<SPLIT>(P, FCPT_ENERGY)(i, j);
        qp = fld<SPLIT>(P, FCPT_QPLUS)(i, j);
        qm = fld<SPLIT>(P, FCPT_QMINUS)(i, j);
        cs = fld<SPLIT>(P, FCPT_SOUNDSPEED)(i, j);
        nu = fld<SPLIT>(P, FCPT_VISCOSITY)(i, j);
    }
    return CflCell<SPLIT>{vr0, vr1, va0, va1, e, qp, qm, cs, nu, h};
}
template <bool SPLIT, bool FAST>
__device__ __forceinline__ double cfl_sum(const KParams &P, int i, double vm_i, const CflRing &R, const CflCell<SPLIT> &c)
{
    auto by = [](double n, const SharedDen &D) { return FAST ? quot_fast(n, D) : n / D.d; };
    const double fac2 = P.artvisc_factor * P.artvisc_factor;
    const double v_residual = c.va0 - vm_i;
    const double csv = c.cs, nuv = c.nu;
    const double invdt1 = SPLIT ? csv * R.cell.r : by(csv, R.cell);
    const double invdt2 = SPLIT ? c.vr0 * R.dr.r : by(c.vr0, R.dr);
    const double invdt3 = SPLIT ? v_residual * R.daz.r : by(v_residual, R.daz);
    // the LeapFrog scheme applies the source terms twice with dt / 2 and
    // relaxes their limits (cfl.cpp:254-261); the Euler factor 1.0 is exact
    const double lf = P.integrator == FCPT_INTEGRATOR_LEAPFROG ? 0.6 : 1.0;
    double invdt4;
    if (P.artvisc == FCPT_ARTVISC_SN) {
        double dvRadial = c.vr1 - c.vr0;
        double dvAzimuthal = c.va1 - c.va0;
        if (dvRadial > 0.0) dvRadial = 0.0;
        else dvRadial = -dvRadial;
        if (dvAzimuthal > 0.0) dvAzimuthal = 0.0;
        else dvAzimuthal = -dvAzimuthal;
        if constexpr (SPLIT)
            invdt4 = 4.0 * fac2 * std_max(dvRadial * R.dr.r, dvAzimuthal * R.daz.r) * lf;
        else
            invdt4 = 4.0 * fac2 * std_max(by(dvRadial, R.dr), by(dvAzimuthal, R.daz)) * lf;
    } else {
        const double eps_rr = (c.vr1 - c.vr0) * cst(P.InvDiffRsup)[i];
        const double eps_pp = cst(P.InvRmed)[i] * ((c.va1 - c.va0) * P.invdphi + 0.5 * (c.vr1 + c.vr0));
        const double mdiv_V = -std_min(eps_rr + eps_pp, 0.0);
        invdt4 = 4.0 * fac2 * mdiv_V * lf;
    }
    const double invdt5 = SPLIT ? 4.0 * nuv * R.inv_cell2 * lf : by(4.0 * nuv, R.cell2) * lf;
    double invdt6 = 0.0;
    if (P.adiabatic) {
        const double inv_limit = 1.0 / P.heating_cooling_cfl_limit;
        double q;
        if constexpr (SPLIT) q = (c.qp - c.qm) * recip<true>(c.e);
        else if constexpr (FAST) q = quot_fast(c.qp - c.qm, shared_den(c.e));
        else q = (c.qp - c.qm) / c.e;
        invdt6 = inv_limit * fabs(q) * lf;
    }
    return invdt1 * invdt1 + invdt2 * invdt2 + invdt3 * invdt3 + invdt4 * invdt4 + invdt5 * invdt5 + invdt6 * invdt6;
}
template <bool SPLIT>
__device__ __forceinline__ double cfl_cell_sum(const KParams &P, int i, double vm_i, const CflRing &R,
                                               const CflCell<SPLIT> &c)
{
    double sum = cfl_sum<SPLIT, true>(P, i, vm_i, R, c);
    if constexpr (!SPLIT) {
        if (!(R.fast && sum < 0x1p400 && (!P.adiabatic || quot_range(c.e)))) {
            __builtin_amdgcn_s_sleep(0);  // a branch: not both sums formed and selected
            sum = cfl_sum<SPLIT, false>(P, i, vm_i, R, c);
        }
    }
    return sum;
}
template <bool SPLIT>
__device__ __forceinline__ double cfl_limit(const KParams &P, double sum)
{
    return SPLIT ? P.cfl * inv_sqrt<true>(sum) : P.cfl / sqrt(sum);
}

__global__ void __launch_bounds__(256) k_cfl_fold(KParams P, int mode) { b_cfl_fold(P, mode, (int)threadIdx.x); }
__global__ void __launch_bounds__(256) kb_cfl_fold(const KParams *Ps, const BatchEntry *map, int mode)
{
    b_cfl_fold(batch_disk(Ps, batch_entry(map).disk), mode, (int)threadIdx.x);
}
__global__ void k_set_dt(KParams P, double dt) { P.s->dt = dt; }
__global__ void k_set_clock(KParams P, double time) { P.s->time = time; }

__global__ void k_set_time(KParams P, double time, double last_dt, int n_monitor)
{
    P.s->time = time;
    P.s->last_dt = last_dt;
    P.s->last_prev = last_dt;
    P.s->n_monitor = n_monitor;
}

__global__ void k_set_params(KParams P, fcpt_step_params sp, BodySmoothing sm)
{
    DevScalars *s = P.s;
    s->n_planets = sp.n_planets;
    for (int k = 0; k < sp.n_planets; ++k) {
        s->planet[k].x = sp.planet[k].x;
        s->planet[k].y = sp.planet[k].y;
        s->planet[k].mass = sp.planet[k].mass;
        s->planet[k].r_cubic = sp.planet[k].r_cubic;
        s->planet[k].smooth = sm.s[k];
    }
    s->indirect_x = sp.indirect_x;
    s->indirect_y = sp.indirect_y;
    s->has_mid = 0;
}

// the bodies of a LeapFrog step's second kick
__global__ void k_set_mid_params(KParams P, fcpt_step_params sp, BodySmoothing sm)
{
    DevScalars *s = P.s;
    s->n_planets_mid = sp.n_planets;
    for (int k = 0; k < sp.n_planets; ++k) {
        s->planet_mid[k].x = sp.planet[k].x;
        s->planet_mid[k].y = sp.planet[k].y;
        s->planet_mid[k].mass = sp.planet[k].mass;
        s->planet_mid[k].r_cubic = sp.planet[k].r_cubic;
        s->planet_mid[k].smooth = sm.s[k];
    }
    s->indirect_mid_x = sp.indirect_x;
    s->indirect_mid_y = sp.indirect_y;
    s->has_mid = 1;
}

// step_LeapFrog's clock (simulation.cpp:278-281, 378, 441): phase 0 before
// the first kick (dt / 2 at the start time), 1 before the drift (dt), 2 before
// the second kick (dt / 2 at the midstep time, the midstep bodies), 3 before
// the final boundaries (dt at the start time: they advance the time to
// start + dt, the reference's end_time)
__global__ void k_leapfrog_phase(KParams P, int phase)
{
    DevScalars *s = P.s;
    if (phase == 0) {
        s->dt_step = s->dt;
        s->t_step = s->time;
        s->dt = s->dt_step / 2;
    } else if (phase == 1) {
        s->dt = s->dt_step;
    } else if (phase == 2) {
        s->dt = s->dt_step / 2;
        s->time = s->t_step + s->dt;
        if (s->has_mid) {
            s->n_planets_first = s->n_planets;
            s->indirect_first_x = s->indirect_x;
            s->indirect_first_y = s->indirect_y;
            for (int k = 0; k < kMaxPlanets; ++k) s->planet_first[k] = s->planet[k];
            s->n_planets = s->n_planets_mid;
            s->indirect_x = s->indirect_mid_x;
            s->indirect_y = s->indirect_mid_y;
            for (int k = 0; k < kMaxPlanets; ++k) s->planet[k] = s->planet_mid[k];
        }
    } else {
        s->dt = s->dt_step;
        s->time = s->t_step;
        if (s->has_mid) {
            s->n_planets = s->n_planets_first;
            s->indirect_x = s->indirect_first_x;
            s->indirect_y = s->indirect_first_y;
            for (int k = 0; k < kMaxPlanets; ++k) s->planet[k] = s->planet_first[k];
        }
    }
}

// ---------------------------------------------------------------------------
// x^4 and x^3 of the Klahr-Kley factor by compensated powering (Graillat, Langlois and Louvet,
// "Algorithms for accurate, validated and fast polynomial evaluation",
// Japan J. Indust. Appl. Math. 26, 2009): the square is carried as the
// unevaluated sum p + e (e from an FMA), and the last product's rounding error
// is added back before the one final rounding, so the result is within 0.5 +
// 2^-49 ulp of the exact power: the correctly rounded value but for inputs
// within 2^-49 ulp of a rounding boundary, as the C library's pow (within
// 0.52 ulp) returns it.  An overflowing power returns the rounded product.
__device__ __forceinline__ double pow4_comp(double x)
{
    const double p = x * x, e = fma(x, x, -p);
    const double q = p * p, eq = fma(p, p, -q);
    const double r = q + (eq + 2.0 * p * e);
    return isfinite(q) ? r : q;
}
__device__ __forceinline__ double pow3_comp(double x)
{
    const double p = x * x, e = fma(x, x, -p);
    const double q = p * x, eq = fma(p, x, -q);
    const double r = q + (eq + e * x);
    return isfinite(q) ? r : q;
}

// one body's term at (x, y) with smoothing length `smooth`
template <bool SPLIT>
__device__ __forceinline__ double potential_body(const KParams &P, double x, double y, double smooth,
                                                 double px, double py, double mass, double r_sm)
{
    const double dx = x - px;
    const double dy = y - py;
    const double dist_2 = dx * dx + dy * dy;
    const double d2 = dist_2 + smooth * smooth;
    // split storage: one reciprocal square root instead of sqrt and division
    const double inv_d = SPLIT ? inv_sqrt<true>(d2) : 0.0;
    const double d_smoothed = SPLIT ? d2 * inv_d : sqrt_ieee(d2);
    double smooth_factor_klahr = 1.0;
    if (r_sm > 0.0 && d_smoothed < r_sm) {
        const double q = d_smoothed / r_sm;
        smooth_factor_klahr = (pow4_comp(q) - 2.0 * pow3_comp(q) + 2.0 * d_smoothed / r_sm);
    }
    if constexpr (SPLIT) return -P.G * mass * inv_d * smooth_factor_klahr;
    else return shared_div(-P.G * mass, shared_den(d_smoothed)) * smooth_factor_klahr;
}

// CalculateNbodyPotential, Pframeforce.cpp:44-85 (+ compute_smoothing,
// Force.cpp:145-159: a body's fixed smoothing length, or ThicknessSmoothing *
// H of the cell), for kPotCells cells of ring i, sectors j0 + 64 c (those
// below ns), with the bodies' loop outside the cells': every cell still adds the bodies
// in order and then the indirect term, and a body's parameters are loaded
// once per kPotCells cells.  The potential is stored in FP64 in both storage
// modes.
constexpr int kPotCells = 4;
template <bool SPLIT>
__device__ __forceinline__ void potential_ring_cells(const KParams &P, int i, int j0)
{
    const DevScalars *s = P.s;
    const int ns = P.ns;
    double x[kPotCells], y[kPotCells], sm[kPotCells], acc[kPotCells];
#pragma unroll
    for (int c = 0; c < kPotCells; ++c) {
        const int j = min(j0 + 64 * c, ns - 1);  // past ns: formed, not stored
        x[c] = cst(P.Rmed)[i] * P.cosphi[j];
        y[c] = cst(P.Rmed)[i] * P.sinphi[j];
        const double H = P.adiabatic ? fld<SPLIT>(P, FCPT_SCALE_HEIGHT)(i, j) : cst(P.iso_h)[i];
        sm[c] = P.thickness_smoothing * H;
        acc[c] = 0.0;
    }
    // the bodies through scalar loads (this launch writes none of them)
    const bool mid = P.kick == 2 && *cst(&s->has_mid);
    const auto bodies = mid ? cst(s->planet_mid) : cst(s->planet);
    const int np = mid ? *cst(&s->n_planets_mid) : *cst(&s->n_planets);
    for (int k = 0; k < np; ++k) {
        const double px = bodies[k].x, py = bodies[k].y;
        const double mass = bodies[k].mass, r_sm = bodies[k].r_cubic;
        const double smk = bodies[k].smooth;
#pragma unroll
        for (int c = 0; c < kPotCells; ++c)
            acc[c] += potential_body<SPLIT>(P, x[c], y[c], smk >= 0.0 ? smk : sm[c], px, py, mass, r_sm);
    }
    const double ix = mid ? *cst(&s->indirect_mid_x) : *cst(&s->indirect_x);
    const double iy = mid ? *cst(&s->indirect_mid_y) : *cst(&s->indirect_y);
#pragma unroll
    for (int c = 0; c < kPotCells; ++c) {
        const int j = j0 + 64 * c;
        if (j >= ns) break;
        phi_fld(P).set(i, j, acc[c] + (-ix * x[c] - iy * y[c]));
    }
}

// the potential, blocks of 64 x kPotCells sectors by 4 rings
template <bool SPLIT>
__device__ __forceinline__ void b_potential(const KParams &P, int bx, int by)
{
    const int i = wave_ring(0, by);
    const int j0 = bx * 64 * kPotCells + (int)threadIdx.x;
    if (j0 >= P.ns || i >= P.nr) return;
    potential_ring_cells<SPLIT>(P, i, j0);
}
FCPT_PAIR0(potential, 256)

// The potential of a single disk in one launch (b_potential); fold_mode >= 0:
// one extra block row runs the CFL fold of the step's start
// (k_cfl_fold; the potential reads none of the scalars the fold
// writes, and dt is first read by the kernels after this one).
template <bool SPLIT>
__global__ void __launch_bounds__(256) k_potential_fold(KParams P, int fold_mode)
{
    // block row 0 is the fold (dispatched first, it ends under the others)
    const int bx = (int)blockIdx.x, by = (int)blockIdx.y - 1;
    if (by < 0) {
        if (bx == 0 && fold_mode >= 0)
            b_cfl_fold(P, fold_mode, (int)(threadIdx.y * blockDim.x + threadIdx.x));
        return;
    }
    b_potential<SPLIT>(P, bx, by);
}

// The CFL ring means and the cells' limits, one block per ring: the block forms
// the ring's mean v_phi exactly as k_ring_mean does (same per-thread sums, same
// tree) and stores it, then the limits of the ring's cells (rings 1 .. nr-2)
// with that mean, and puts the ring's smallest in its slot; the fold adds the
// shear limits between neighbouring rings' means (cfl.cpp:185-382).  The first
// 256 threads form the mean, all of them the cells: 512 where a disk is alone
// (256: 128x384 27.6 -> 28.6 us per step, 2048x6144 adiabatic 1112 -> 1133; 1024
// slower everywhere), 256 in a batch, whose rings fill the device anyway and
// leave fewer of them idle (16 disks of 128 to 512 rings: 437 -> 418 us).
// POT: also the potential of the ring's cells, for steps whose derived fields
// are formed where they are needed; the scale height of its smoothing comes with
// the sound speed of the limits, so no step stores it.
// 4096x12288 beta, FP64: 718 us where the two launches take 506 + 306, and the end
// of the step 796 us instead of 880 without the store of H; 73 B/cell at 5.1 TB/s,
// with instruction issue for 0.59 of its time.
template <bool SPLIT, bool POT, int THREADS>
__device__ __forceinline__ void b_cfl_ring(const KParams &P, int i)
{
    __shared__ double sh[256];
    __shared__ double wmax[THREADS / 64];
    const int ns = P.ns;
    const int t = (int)threadIdx.x;
    FLD(v, FCPT_VAZI);
    const Fld<SPLIT> Hf = fld_derived<SPLIT>(P, FCPT_SCALE_HEIGHT);
    double acc = 0.0;
    if (t < 256) strided_row<256>(ns, t, [&](int j) { return v(i, j); }, [&](double x) { acc += x; });
    const bool active = i >= 1 && i < P.nr - 1;
    // a disk alone waits for its first cells' loads during the sum; a batch has
    // other rings to run and keeps the registers
    constexpr bool AHEAD = THREADS == 512;
    CflCell<SPLIT> c;
    if constexpr (AHEAD) c = cfl_load<SPLIT>(P, active ? i : 1, t < ns ? t : 0);
    const CflRing R = cfl_ring<SPLIT>(P, i);
    const double r = cst(P.Rmed)[i];
    const DevScalars *s = P.s;
    const int np = POT ? *cst(&s->n_planets) : 0;
    const double ix = POT ? *cst(&s->indirect_x) : 0.0, iy = POT ? *cst(&s->indirect_y) : 0.0;
    const double vm = block_sum(acc, sh) / (double)ns;
    if (t == 0) P.vmean[i] = vm;
    double most = 0.0;
    // a loop for the active rings and one for the ghost rings: a test of the
    // ring in the loop keeps its scalar loads there
    auto cells = [&](auto act) {
        for (int j = t; j < ns; j += THREADS) {
            double H = P.adiabatic ? 0.0 : cst(P.iso_h)[i];
            if constexpr (decltype(act)::value) {
                if (!AHEAD || j != t) c = cfl_load<SPLIT>(P, i, j);
                // NaN never wins a comparison, exactly like the reference's "if (dt_cell < dt_core)"
                most = std_max(most, cfl_cell_sum<SPLIT>(P, i, vm, R, c));
                if (POT && P.adiabatic) H = Hf.stored(i, j, c.h);
            } else {
                if (P.adiabatic) H = Hf(i, j);  // the ghost rings' is stored
            }
            if constexpr (POT) {
                const double sm = P.thickness_smoothing * H;
                const double px = r * P.cosphi[j], py = r * P.sinphi[j];
                double a = 0.0;
                for (int k = 0; k < np; ++k) {
                    const auto b = cst(s->planet) + k;
                    const double smk = b->smooth;
                    a += potential_body<SPLIT>(P, px, py, smk >= 0.0 ? smk : sm, b->x, b->y, b->mass, b->r_cubic);
                }
                phi_fld(P).set(i, j, a + (-ix * px - iy * py));
            }
        }
    };
    if (active) cells(std::true_type{});
    else if (POT) cells(std::false_type{});
    for (int off = 32; off > 0; off >>= 1) most = std_max(most, __shfl_xor(most, off, 64));
    if ((t & 63) == 0) wmax[t >> 6] = most;
    __syncthreads();
    if (t == 0) {
        double m = wmax[0];
        for (int k = 1; k < THREADS / 64; ++k) m = std_max(m, wmax[k]);
        P.ring_min[i] = m > 0.0 ? cfl_limit<SPLIT>(P, m) : __longlong_as_double(0x7FF0000000000000ll);
    }
}
template <bool SPLIT, bool POT>
__global__ void __launch_bounds__(512) k_cfl_ring(KParams P)
{
    b_cfl_ring<SPLIT, POT, 512>(P, (int)blockIdx.x);
}
template <bool SPLIT, bool POT>
__global__ void __launch_bounds__(256) kb_cfl_ring(const KParams *Ps, const BatchEntry *map)
{
    const BatchEntry e = batch_entry(map);
    b_cfl_ring<SPLIT, POT, 256>(batch_disk(Ps, e.disk), (int)(e.yx & 0xffffu));
}

// ---------------------------------------------------------------------------
// momentum_update_radial, SourceEuler.cpp:325-372, for one cell: pressure and
// potential gradients between rings i - 1 and i, and the centrifugal term of
// the four v_phi around the interface (summed in that order)
// inv = 2 / (Sigma(i) + Sigma(i - 1))
template <class PP>
__device__ __forceinline__ double src_vr_by(const PP &P, int i, double dt, double v, double inv, double p0,
                                            double pm, double phi0, double phim, double va00, double va01,
                                            double va10, double va11)
{
    double gradp = inv;
    gradp *= (p0 - pm);
    gradp *= ring_tab(P, TAB_INV_DIFF_RMED, i);
    const double gradphi = (phi0 - phim) * ring_tab(P, TAB_INV_DIFF_RMED, i);
    const double vsum = va00 + va01 + va10 + va11;
    const double vt = 0.25 * vsum + ring_tab(P, TAB_RINF_OMEGA, i);
    const double vt2 = vt * vt;
    const double centrifugal_accel = vt2 * ring_tab(P, TAB_INV_RINF, i);
    return v + dt * (-gradp - gradphi + centrifugal_accel);
}
template <bool SPLIT = false>
__device__ __forceinline__ double src_vr_new(const KParams &P, int i, double dt, double v, double s0,
                                             double sm, double p0, double pm, double phi0, double phim,
                                             double va00, double va01, double va10, double va11)
{
    return src_vr_by(P, i, dt, v, quot<SPLIT>(2.0, s0 + sm), p0, pm, phi0, phim, va00, va01, va10, va11);
}

// momentum_update_azimuthal, SourceEuler.cpp:375-428, for one cell
// inv = 2 / (Sigma(j) + Sigma(j - 1))
template <class PP>
__device__ __forceinline__ double src_vphi_by(const PP &P, int i, double dt, double va, double inv, double p0,
                                              double pjp, double phi0, double phijp)
{
    const double invdxtheta = ring_tab(P, TAB_SRC_INVDXTHETA, i);  // 2 / (dphi (Rsup + Rinf))
    const double gradp = inv * (p0 - pjp) * invdxtheta;
    const double gradphi = (phi0 - phijp) * invdxtheta;
    return va + dt * (-gradp - gradphi);
}
template <bool SPLIT = false>
__device__ __forceinline__ double src_vphi_new(const KParams &P, int i, double dt, double va, double s0,
                                               double sjp, double p0, double pjp, double phi0,
                                               double phijp)
{
    return src_vphi_by(P, i, dt, va, quot<SPLIT>(2.0, s0 + sjp), p0, pjp, phi0, phijp);
}

// momentum_update_radial, SourceEuler.cpp:325-372
template <bool SPLIT>
__device__ __forceinline__ void b_src_vr(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(2, P.nr - 1)
    FLD(S, FCPT_SIGMA);
    FLD(Pr, FCPT_PRESSURE);
    const Fld<false> Phi = phi_fld(P);
    FLD(vaz, FCPT_VAZI);
    FLD(vr, FCPT_VRAD);
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    vr.set(i, j, src_vr_new<SPLIT>(P, i, dt, vr(i, j), S(i, j), S(i - 1, j), Pr(i, j), Pr(i - 1, j), Phi(i, j),
                            Phi(i - 1, j), vaz(i, j), vaz(i, jn), vaz(i - 1, j), vaz(i - 1, jn)));
}
FCPT_ONE0(src_vr, 256)

// momentum_update_azimuthal, SourceEuler.cpp:375-428
template <bool SPLIT>
__device__ __forceinline__ void b_src_vphi(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(1, P.nr - 1)
    FLD(S, FCPT_SIGMA);
    FLD(Pr, FCPT_PRESSURE);
    const Fld<false> Phi = phi_fld(P);
    FLD(vaz, FCPT_VAZI);
    const double dt = P.s->dt;
    const int jp = j == 0 ? ns - 1 : j - 1;
    vaz.set(i, j, src_vphi_new<SPLIT>(P, i, dt, vaz(i, j), S(i, j), S(i, jp), Pr(i, j), Pr(i, jp), Phi(i, j),
                               Phi(i, jp)));
}
FCPT_ONE0(src_vphi, 256)

// compression_heating, SourceEuler.cpp:459-493, for one cell (rings 0 .. nr-2)
// from v_r(i), v_r(i + 1), v_phi(j), v_phi(j + 1)
template <class PP>
__device__ __forceinline__ double src_energy_new(const PP &P, int i, double dt, double e, double vr0,
                                                 double vr1, double va0, double va1)
{
    const double DIV_V = (vr1 * ring_tab(P, TAB_RINF, i + 1) - vr0 * ring_tab(P, TAB_RINF, i)) * ring_tab(P, TAB_INV_DIFF_RSUP_RB, i) +
                         (va1 - va0) * P.invdphi * ring_tab(P, TAB_INV_RMED, i);
    return e * exp(-(P.gamma - 1.0) * dt * DIV_V);
}

template <bool SPLIT>
__device__ __forceinline__ void b_src_energy(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr - 1)
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(E, FCPT_ENERGY);
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    E.set(i, j, src_energy_new(P, i, dt, E(i, j), vr(i, j), vr(i + 1, j), vaz(i, j), vaz(i, jn)));
}
FCPT_PAIR0(src_energy, 256)

// the energy of temperature t, t sigma / mu R / (gamma - 1) (split storage:
// one product with the launch-wide R / (mu (gamma - 1)))
template <bool SPLIT = false>
__device__ __forceinline__ double energy_at(const KParams &P, double t, double sigma)
{
    if constexpr (SPLIT) return t * sigma * (P.Rgas * recip<true>(P.mu * (P.gamma - 1.0)));
    else return t * sigma / P.mu * P.Rgas / (P.gamma - 1.0);
}
template <bool SPLIT = false>
__device__ __forceinline__ double energy_floor(const KParams &P, double sigma)
{
    return energy_at<SPLIT>(P, P.t_min, sigma);
}
// assure_temperature_range for one cell, SourceEuler.cpp:136-202
// (FP64 storage: an e clear of both limits by more than the rounding of the
// limits' products is unchanged, so the limits' four divisions are formed
// only for the others)
template <bool SPLIT = false>
__device__ __forceinline__ double temperature_floor(const KParams &P, double e, double sigma)
{
    if constexpr (!SPLIT) {
        const double es = sigma * P.energy_per_t;
        const double lo = P.t_min * es, hi = P.t_max * es;
        if (lo >= 0x1p-900 && e > lo * (1.0 + 0x1p-40) && e < hi * (1.0 - 0x1p-40)) return e;
        __builtin_amdgcn_s_sleep(0);  // a branch: the divisions are not formed and selected
    }
    const double minimum_energy = energy_floor<SPLIT>(P, sigma);
    const double maximum_energy = energy_at<SPLIT>(P, P.t_max, sigma);
    if (!(e > minimum_energy)) e = minimum_energy;
    if (!(e < maximum_energy)) e = maximum_energy;
    return e;
}

// temperature_floor at a cell of ring i whose Sigma is in range (fine)
template <bool SPLIT, class PP>
__device__ __forceinline__ double temperature_floor_in(const PP &P, int i, double e, double sig, bool fine)
{
    if constexpr (!SPLIT) {
        if (fine && e > sig * ring_tab(P, TAB_E_LO, i) && e < sig * ring_tab(P, TAB_E_HI, i)) return e;
        __builtin_amdgcn_s_sleep(0);
    }
    return temperature_floor<SPLIT>(P, e, sig);
}

template <bool SPLIT>
__device__ __forceinline__ void b_temperature_floor(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(E, FCPT_ENERGY);
    FLD(S, FCPT_SIGMA);
    E.set(i, j, temperature_floor<SPLIT>(P, E(i, j), S(i, j)));
}
FCPT_PAIR0(temperature_floor, 256)

// ---------------------------------------------------------------------------
// compute_sound_speed / compute_scale_height / update_viscosity for one cell
// (SourceEuler.cpp:957-995, 1121-1154; viscosity.cpp:98-137), as a load of
// the inputs and a store of the results
// locally isothermal pressure Sigma c_s^2 (the value recalculate_derived
// stores, SourceEuler.cpp:225-249, with the ring profile of c_s)
__device__ __forceinline__ double iso_pressure(const KParams &P, int i, double sig)
{
    const double c_s = cst(P.iso_cs)[i];
    return sig * (c_s * c_s);
}

struct DerivedIn {
    double e, sig, cs, h;
};

template <bool SPLIT>
__device__ __forceinline__ DerivedIn derived_load(const KParams &P, int i, int j, bool with_pressure)
{
    DerivedIn d{0.0, 0.0, 0.0, 0.0};
    if (P.adiabatic) {
        d.e = fld<SPLIT>(P, FCPT_ENERGY)(i, j);
        d.sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
    } else {
        // locally isothermal: c_s and H are the ring profiles of k_iso_rings
        d.cs = cst(P.iso_cs)[i];
        d.h = cst(P.iso_h)[i];
        if (with_pressure) d.sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
    }
    return d;
}

template <bool SPLIT>
__device__ __forceinline__ void derived_store(const KParams &P, int i, int j, const DerivedIn &d,
                                             bool with_temperature, bool with_pressure,
                                             bool force_nu = false)
{
    double c_s, h;
    if (P.lazy_derived) {
        // the only derived field a step reads stored: H, by the potential where
        // that is a launch of its own (h_lazy 0) and in the ghost rings, whose
        // Sigma and E a boundary call of the caller's may change alone
        if (P.adiabatic && (!P.h_lazy || i == 0 || i == P.nr - 1))
            fld<SPLIT>(P, FCPT_SCALE_HEIGHT).set(i, j, adi_derived<SPLIT>(P, i, d.e, d.sig).h);
        return;
    }
    if (P.adiabatic) {
        const double e = d.e;
        const double sig = d.sig;
        if (with_temperature) {
            const double c_v_inv = P.mu / P.Rgas * (P.gamma - 1.0);
            fld<SPLIT>(P, FCPT_TEMPERATURE).set(i, j, c_v_inv * e / sig);
        }
        const AdiDerived a = adi_derived<SPLIT>(P, i, e, sig);
        c_s = a.cs;
        h = a.h;
        fld<SPLIT>(P, FCPT_SOUNDSPEED).set(i, j, c_s);
        fld<SPLIT>(P, FCPT_SCALE_HEIGHT).set(i, j, h);
        if (with_pressure) fld<SPLIT>(P, FCPT_PRESSURE).set(i, j, (P.gamma - 1.0) * e);
    } else {
        c_s = d.cs;
        h = d.h;
        if (with_pressure) fld<SPLIT>(P, FCPT_PRESSURE).set(i, j, d.sig * (c_s * c_s));
        // locally isothermal: nu = alpha H c_s is the ring profile iso_nu,
        // already in the field since the state was uploaded
        if (!force_nu) return;
    }
    const double alpha = P.alpha;
    fld<SPLIT>(P, FCPT_VISCOSITY).set(i, j, alpha * h * c_s);
}

// ---------------------------------------------------------------------------
// The tensor of the TW artificial viscosity at one cell from its velocities
// v_r(i), v_r(i + 1), v_phi(j), v_phi(j + 1) (artificial_viscosity.cpp:44-70)
struct TwQ {
    double qr, qp, eps_rr, eps_pp, div_V, l_sq;
};

template <class PP>
__device__ __forceinline__ TwQ tw_q_cell(const PP &P, int i, double vr0, double vr1, double va0,
                                         double va1, double sig)
{
    TwQ q;
    q.eps_rr = (vr1 - vr0) * ring_tab(P, TAB_INV_DIFF_RSUP, i);
    q.eps_pp = ring_tab(P, TAB_INV_RMED, i) * ((va1 - va0) * P.invdphi + 0.5 * (vr1 + vr0));
    q.div_V = std_min(q.eps_rr + q.eps_pp, 0.0);
    q.l_sq = ring_tab(P, TAB_TW_LSQ, i);
    q.qr = q.l_sq * sig * -q.div_V * (q.eps_rr - 1.0 / 3.0 * q.div_V);
    q.qp = q.l_sq * sig * -q.div_V * (q.eps_pp - 1.0 / 3.0 * q.div_V);
    return q;
}

// energy after the TW dissipation and the temperature floor
// (artificial_viscosity.cpp:72-86, then SetTemperatureFloorCeilValues, :19-21)
template <class PP>
__device__ __forceinline__ double tw_heat(const PP &P, int i, const TwQ &q, double sig, double dt, double e)
{
    if (i > 1 && i < P.nr - 1) {
        const double d = q.eps_rr - q.eps_pp;
        const double Qplus =
            -q.l_sq * q.div_V * sig * 1.0 / 3.0 * (q.eps_rr * q.eps_rr + q.eps_pp * q.eps_pp + d * d);
        e += Qplus * dt;
    }
    return e;
}
template <class PP>
__device__ __forceinline__ double tw_dissipation(const PP &P, int i, const TwQ &q, double sig,
                                                 double dt, double e)
{
    return temperature_floor(P, tw_heat(P, i, q, sig, dt, e), sig);
}

// update_with_artificial_viscosity_TW, artificial_viscosity.cpp:35-88
template <bool SPLIT>
__device__ __forceinline__ void b_tw_q(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    const bool diss = P.adiabatic && P.artvisc_dissipation;
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const double vr0 = vr(i, j), vr1 = vr(i + 1, j), va0 = vaz(i, j), va1 = vaz(i, jn);
    const double sig = S(i, j);
    const double e_in = diss ? E(i, j) : 0.0;
    const TwQ q = tw_q_cell(P, i, vr0, vr1, va0, va1, sig);
    fld<SPLIT>(P, FCPT_Q_R).set(i, j, q.qr);
    fld<SPLIT>(P, FCPT_Q_PHI).set(i, j, q.qp);
    if (diss) E.set(i, j, tw_dissipation(P, i, q, sig, dt, e_in));
}
FCPT_ONE0(tw_q, 256)

// the TW velocity updates of one cell from the tensors around it
// (artificial_viscosity.cpp:90-139)
// (inv = 2 dt / ((Rsup + Rinf) Sigma_avg))
template <class PP>
__device__ __forceinline__ double tw_vphi_by(const PP &P, double va, double inv, double qp0, double qpj)
{
    const double dVp = inv * (qp0 - qpj) * P.invdphi;
    return va + dVp;
}
template <bool SPLIT = false>
__device__ __forceinline__ double tw_vphi_new(const KParams &P, int i, double dt, double va, double s0,
                                              double sjp, double qp0, double qpj)
{
    const double sigma_phi_avg = 0.5 * (s0 + sjp);
    return tw_vphi_by(P, va, quot<SPLIT>(2.0 * dt, ring_tab(P, TAB_RSUP_RINF, i) * sigma_phi_avg), qp0, qpj);
}

// (c = f dt / Sigma_avg 2 / (Rmed(i)^2 - Rmed(i - 1)^2))
template <class PP>
__device__ __forceinline__ double tw_vr_by(const PP &P, int i, double v, double c, double qr0, double qrm,
                                           double qp0, double qpm)
{
    const double r0 = ring_tab(P, TAB_RMED, i), r1 = ring_tab(P, TAB_RMED, i - 1);
    const double dVr = c * ((qr0 * r0 - qrm * r1) - 0.5 * (qp0 + qpm) * ring_tab(P, TAB_RMED_DIFF, i));
    return v + dVr;
}
template <bool SPLIT = false>
__device__ __forceinline__ double tw_vr_new(const KParams &P, int i, double dt, double v, double s0,
                                            double sm, double qr0, double qrm, double qp0, double qpm)
{
    const double sigma_r_avg = 0.5 * (s0 + sm);
    const double c = quot<SPLIT>(quot<SPLIT>(P.radial_viscosity_factor * dt, sigma_r_avg) * 2.0,
                                 ring_tab(P, TAB_RMED_SQ_DIFF, i));
    return tw_vr_by(P, i, v, c, qr0, qrm, qp0, qpm);
}

template <bool SPLIT>
__device__ __forceinline__ void b_tw_vel(const KParams &P, int bx, int by, int with_viscosity)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(S, FCPT_SIGMA);
    FLD(Qr, FCPT_Q_R);
    FLD(Qp, FCPT_Q_PHI);
    FLD(vaz, FCPT_VAZI);
    FLD(vr, FCPT_VRAD);
    const double dt = P.s->dt;
    const bool inner = i >= 1 && i < P.nr - 1;
    const bool radial = i >= 2 && inner;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const int im = i >= 1 ? i - 1 : 0;
    // in the fused step, recalculate_viscosity (SourceEuler.cpp:205-223), which is
    // pointwise in Sigma and E and follows this kernel, is done here for every ring
    DerivedIn din{0.0, 0.0, 0.0, 0.0};
    const bool visc = with_viscosity && P.adiabatic;  // constant ring profile when isothermal
    if (visc) din = derived_load<SPLIT>(P, i, j, false);
    double s0 = 0.0, sjp = 0.0, sm = 0.0, qp0 = 0.0, qpj = 0.0, qpm = 0.0, qr0 = 0.0, qrm = 0.0;
    double va = 0.0, v = 0.0;
    if (inner) {
        s0 = S(i, j);
        sjp = S(i, jp);
        qp0 = Qp(i, j);
        qpj = Qp(i, jp);
        va = vaz(i, j);
    }
    if (radial) {
        sm = S(im, j);
        qr0 = Qr(i, j);
        qrm = Qr(im, j);
        qpm = Qp(im, j);
        v = vr(i, j);
    }
    if (visc) derived_store<SPLIT>(P, i, j, din, false, false);
    if (!inner) return;
    vaz.set(i, j, tw_vphi_new<SPLIT>(P, i, dt, va, s0, sjp, qp0, qpj));
    if (radial) vr.set(i, j, tw_vr_new<SPLIT>(P, i, dt, v, s0, sm, qr0, qrm, qp0, qpm));
}
FCPT_ONE1(tw_vel, 256, int, with_viscosity)

// The von Neumann-Richtmyer tensor at one cell (artificial_viscosity.cpp:160-185)
struct SnQ {
    double qr, qp, dv_r, dv_phi;
};

template <class PP>
__device__ __forceinline__ SnQ sn_q_cell(const PP &P, int i, double vr0, double vr1, double va0,
                                         double va1, double sig)
{
    SnQ q;
    const double fac2 = ring_tab(P, TAB_ARTVISC_SQ, i);
    q.dv_r = vr1 - vr0;
    q.qr = q.dv_r < 0.0 ? fac2 * sig * (q.dv_r * q.dv_r) : 0.0;
    q.dv_phi = va1 - va0;
    q.qp = q.dv_phi < 0.0 ? fac2 * sig * (q.dv_phi * q.dv_phi) : 0.0;
    return q;
}

// energy after the SN dissipation and the temperature floor
// (artificial_viscosity.cpp:187-205, then SetTemperatureFloorCeilValues)
template <class PP>
__device__ __forceinline__ double sn_heat(const PP &P, int i, const SnQ &q, double dt, double e)
{
    if (i >= 1 && i < P.nr - 1) {
        const double invdxtheta = ring_tab(P, TAB_INV_DXTHETA, i);  // 1 / (dphi Rmed)
        e = e - dt * q.qr * q.dv_r * ring_tab(P, TAB_INV_DIFF_RSUP, i) - dt * q.qp * q.dv_phi * invdxtheta;
    }
    return e;
}
template <class PP>
__device__ __forceinline__ double sn_dissipation(const PP &P, int i, const SnQ &q, double sig,
                                                 double dt, double e)
{
    return temperature_floor(P, sn_heat(P, i, q, dt, e), sig);
}

// update_with_artificial_viscosity_SN, artificial_viscosity.cpp:148-211
template <bool SPLIT>
__device__ __forceinline__ void b_sn_q(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    const bool diss = P.adiabatic && P.artvisc_dissipation;
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const double vr0 = vr(i, j), vr1 = vr(i + 1, j), va0 = vaz(i, j), va1 = vaz(i, jn);
    const double sig = S(i, j);
    const double e_in = diss ? E(i, j) : 0.0;
    const SnQ q = sn_q_cell(P, i, vr0, vr1, va0, va1, sig);
    fld<SPLIT>(P, FCPT_Q_R).set(i, j, q.qr);
    fld<SPLIT>(P, FCPT_Q_PHI).set(i, j, q.qp);
    if (diss) E.set(i, j, sn_dissipation(P, i, q, sig, dt, e_in));
}
FCPT_ONE0(sn_q, 256)

// the SN velocity updates of one cell (artificial_viscosity.cpp:214-248)
// (inv = 2 dt / (Sigma + its neighbour's))
template <class PP>
__device__ __forceinline__ double sn_vr_by(const PP &P, int i, double v, double inv, double qr0, double qrm)
{
    return v - inv * (qr0 - qrm) * ring_tab(P, TAB_INV_DIFF_RMED, i);
}
template <class PP>
__device__ __forceinline__ double sn_vphi_by(const PP &P, int i, double va, double inv, double qp0, double qpj)
{
    return va - inv * (qp0 - qpj) * ring_tab(P, TAB_INV_DXTHETA, i);  // 1 / (dphi Rmed)
}
template <bool SPLIT = false>
__device__ __forceinline__ double sn_vr_new(const KParams &P, int i, double dt, double v, double s0,
                                            double sm, double qr0, double qrm)
{
    return sn_vr_by(P, i, v, quot<SPLIT>(dt * 2.0, s0 + sm), qr0, qrm);
}

template <bool SPLIT = false>
__device__ __forceinline__ double sn_vphi_new(const KParams &P, int i, double dt, double va, double s0,
                                              double sjp, double qp0, double qpj)
{
    return sn_vphi_by(P, i, va, quot<SPLIT>(dt * 2.0, s0 + sjp), qp0, qpj);
}

template <bool SPLIT>
__device__ __forceinline__ void b_sn_vel(const KParams &P, int bx, int by, int with_viscosity)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(S, FCPT_SIGMA);
    FLD(Qr, FCPT_Q_R);
    FLD(Qp, FCPT_Q_PHI);
    FLD(vaz, FCPT_VAZI);
    FLD(vr, FCPT_VRAD);
    const double dt = P.s->dt;
    const bool inner = i >= 1 && i < P.nr - 1;
    const bool radial = i >= 2 && inner;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const int im = i >= 1 ? i - 1 : 0;
    // in the fused step, recalculate_viscosity (SourceEuler.cpp:205-223), which is
    // pointwise in Sigma and E and follows this kernel, is done here for every ring
    DerivedIn din{0.0, 0.0, 0.0, 0.0};
    const bool visc = with_viscosity && P.adiabatic;  // constant ring profile when isothermal
    if (visc) din = derived_load<SPLIT>(P, i, j, false);
    double s0 = 0.0, sjp = 0.0, sm = 0.0, qp0 = 0.0, qpj = 0.0, qr0 = 0.0, qrm = 0.0;
    double va = 0.0, v = 0.0;
    if (inner) {
        s0 = S(i, j);
        sjp = S(i, jp);
        qp0 = Qp(i, j);
        qpj = Qp(i, jp);
        va = vaz(i, j);
    }
    if (radial) {
        sm = S(im, j);
        qr0 = Qr(i, j);
        qrm = Qr(im, j);
        v = vr(i, j);
    }
    if (visc) derived_store<SPLIT>(P, i, j, din, false, false);
    if (!inner) return;
    if (radial) vr.set(i, j, sn_vr_new<SPLIT>(P, i, dt, v, s0, sm, qr0, qrm));
    vaz.set(i, j, sn_vphi_new<SPLIT>(P, i, dt, va, s0, sjp, qp0, qpj));
}
FCPT_ONE1(sn_vel, 256, int, with_viscosity)

// recalculate_viscosity, SourceEuler.cpp:205-223
template <bool SPLIT>
__device__ __forceinline__ void b_recalc_viscosity(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    derived_store<SPLIT>(P, i, j, derived_load<SPLIT>(P, i, j, false), false, false, true);
}
FCPT_PAIR0(recalc_viscosity, 256)

// recalculate_derived_disk_quantities, SourceEuler.cpp:225-249
template <bool SPLIT>
__device__ __forceinline__ void b_derived(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    if (i == 0 && j == 0) P.s->count_derived = *P.step_at;
    derived_store<SPLIT>(P, i, j, derived_load<SPLIT>(P, i, j, true), true, true);
}
FCPT_ONE0(derived, 256)


// compute_pressure (SourceEuler.cpp): (gamma - 1) E, or Sigma c_s^2 with the
// isothermal ring profile of c_s
template <bool SPLIT>
__device__ __forceinline__ void b_pressure(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    const double v = P.adiabatic ? (P.gamma - 1.0) * fld<SPLIT>(P, FCPT_ENERGY)(i, j)
                                 : iso_pressure(P, i, fld<SPLIT>(P, FCPT_SIGMA)(i, j));
    fld<SPLIT>(P, FCPT_PRESSURE).set(i, j, v);
}
FCPT_PAIR0(pressure, 256)

// locally isothermal sound speed and scale height from the initial setup
// (compute_sound_speed_normal / compute_scale_height_old, isothermal branches)
template <bool SPLIT>
__device__ __forceinline__ void b_iso_profile(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    const double r = ring_tab(P, TAB_RMED, i);
    const double vK = sqrt(P.G * P.mstar / r);
    const double h = P.aspect_ratio * pow(r, P.flaring);
    const double c_s = h * vK;
    fld<SPLIT>(P, FCPT_SOUNDSPEED).set(i, j, c_s);
    const double inv_omega_kepler = 1.0 / omega_kepler(P, r);
    fld<SPLIT>(P, FCPT_SCALE_HEIGHT).set(i, j, c_s * inv_omega_kepler);
    const double sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
    const double pr = sig * (c_s * c_s);
    fld<SPLIT>(P, FCPT_PRESSURE).set(i, j, pr);
    fld<SPLIT>(P, FCPT_TEMPERATURE).set(i, j, P.mu / P.Rgas * pr / sig);
}
FCPT_PAIR0(iso_profile, 256)

// KParams::ring_tab: the metric, and each ring-uniform product or quotient
// with the expression of the cell formula that reads it (the same bits)
__global__ void __launch_bounds__(256) k_ring_tables(KParams P, double *out)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i > P.nr) return;
    double *tab = out + (size_t)i * kRingTabs;
    tab[TAB_RINF] = P.Rinf[i];
    tab[TAB_INV_RINF] = P.InvRinf[i];
    tab[TAB_RMED] = P.Rmed[i];
    tab[TAB_INV_RMED] = P.InvRmed[i];
    tab[TAB_INV_DIFF_RMED] = P.InvDiffRmed[i];
    tab[TAB_INV_DIFF_RSUP] = P.InvDiffRsup[i];
    tab[TAB_INV_DIFF_RSUP_RB] = P.InvDiffRsupRb[i];
    tab[TAB_SRC_INVDXTHETA] = 2.0 / (P.dphi * (P.Rsup[i] + P.Rinf[i]));
    const double dxtheta = P.dphi * P.Rmed[i];
    tab[TAB_INV_DXTHETA] = 1.0 / dxtheta;
    tab[TAB_INV_OMEGA_K] = 1.0 / omega_kepler(P, P.Rmed[i]);
    tab[TAB_OMEGA_K] = omega_kepler(P, P.Rmed[i]);
    const double a0 = P.Rinf[i] * P.Rinf[i], a1 = P.Rsup[i] * P.Rsup[i];  // Rsup[i] is Rinf[i + 1]
    tab[TAB_VISC_AREA] = 2.0 / (a1 - a0);
    tab[TAB_RINF_SQ] = a0;
    tab[TAB_RINF_OMEGA] = P.Rinf[i] * P.omega_frame;
    // the length scale of the TW tensor (artificial_viscosity.cpp:52-62)
    const double Dr = P.Rsup[i] - P.Rinf[i], rDphi = P.Rmed[i] * P.dphi;
    const double dxm = (P.ns <= 16) ? std_min(Dr, rDphi) : std_max(Dr, rDphi);
    tab[TAB_TW_LSQ] = (P.artvisc_factor * P.artvisc_factor) * (dxm * dxm);
    tab[TAB_RSUP_RINF] = P.Rsup[i] + P.Rinf[i];
    const double r0 = P.Rmed[i], r1 = i > 0 ? P.Rmed[i - 1] : 0.0;
    const SharedDen sum = shared_den(r0 + r1);
    tab[TAB_RMED_SUM] = sum.d;
    tab[TAB_RMED_SUM_RCP] = P.split ? recip<true>(sum.d) : sum.r;
    const SharedDen sq = shared_den(r0 * r0 - r1 * r1);
    tab[TAB_RMED_SQ_DIFF] = sq.d;
    tab[TAB_RMED_SQ_DIFF_RCP] = P.split ? recip<true>(sq.d) : sq.r;
    tab[TAB_RMED_DIFF] = r0 - r1;
    // disk-wide constants, repeated per ring: the walks load them with the
    // ring's values instead of holding them in registers throughout
    tab[TAB_E_LO] = P.t_min * P.energy_per_t * (1.0 + 0x1p-40);
    tab[TAB_E_HI] = P.t_max * P.energy_per_t * (1.0 - 0x1p-40);
    const SharedDen sg = shared_den(sqrt(P.gamma)), cl = shared_den(P.c_light);
    tab[TAB_SQRT_GAMMA] = sg.d;
    tab[TAB_SQRT_GAMMA_RCP] = sg.r;
    tab[TAB_C_LIGHT] = cl.d;
    tab[TAB_C_LIGHT_RCP] = cl.r;
    tab[TAB_G_GM1] = P.gamma * (P.gamma - 1.0);
    tab[TAB_MU_GM1] = P.mu * (P.gamma - 1.0);
    tab[TAB_SIGMA_FLOOR10] = 10.0 * P.sigma0 * P.sigma_floor;
    tab[TAB_BETA_INV] = 1 / P.cooling_beta;
    tab[TAB_ARTVISC_SQ] = P.artvisc_factor * P.artvisc_factor;
    double *sw = P.sweep_tab + (size_t)i * kSweepTabs;
    sw[SW_RMED] = P.Rmed[i];
    sw[SW_INV_DIFF_RMED] = P.InvDiffRmed[i];
    sw[SW_RINF] = P.Rinf[i];
    sw[SW_INV_SURF] = P.InvSurf[i];
    sw[SW_WIDTH] = P.Rsup[i] - P.Rinf[i];
    sw[SW_DXTHETA] = dxtheta;
    const double dr = P.Rsup[i] - P.Rinf[i], daz = P.Rmed[i] * P.dphi, cell = std_min(dr, daz);
    const double size[4] = {dr, daz, cell, cell * cell};
    for (int q = 0; q < 4; ++q) {
        P.cfl_tab[8 * i + 2 * q] = size[q];
        P.cfl_tab[8 * i + 2 * q + 1] = shared_den(size[q]).r;
    }
    sw[SW_INV_DXTHETA] = 1.0 / dxtheta;
    for (int v = 0; v < 2; ++v) {
        double *t = P.damp_tab + 8 * i + 4 * v;
        const double r = v ? P.Rinf[i] : P.Rmed[i < P.nr ? i : P.nr - 1];
        const double lin = P.damping_inner_limit, lout = P.damping_outer_limit;
        if (i <= P.zone_in[v]) {
            const double a = (r - P.rmin * lin) / (P.rmin - P.rmin * lin);
            t[0] = a * a;
            t[1] = P.damping_time_factor * 2.0 * M_PI / omega_kepler(P, P.rmin);
        }
        if (i >= P.zone_out[v]) {
            const double a = (r - P.rmax * lout) / (P.rmax - P.rmax * lout);
            t[2] = a * a;
            t[3] = P.damping_time_factor * 2.0 * M_PI / omega_kepler(P, P.damping_time_radius_outer);
        }
    }
}

void launch_ring_tables(const KParams &P, hipStream_t st)
{
    hipLaunchKernelGGL(k_ring_tables, dim3((unsigned)((P.nr + 256) / 256)), dim3(256), 0, st, P, P.ring_tab);
}

// the locally isothermal ring profiles c_s, H and nu = alpha H c_s, with the
// expressions of the 2-D kernels above (k_iso_profile, derived_store)
__global__ void __launch_bounds__(256) k_iso_rings(KParams P)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= P.nr) return;
    const double r = ring_tab(P, TAB_RMED, i);
    const double vK = sqrt(P.G * P.mstar / r);
    const double h = P.aspect_ratio * pow(r, P.flaring);
    const double c_s = h * vK;
    const double inv_omega_kepler = 1.0 / omega_kepler(P, r);
    const double H = c_s * inv_omega_kepler;
    const double alpha = P.alpha;
    P.iso_cs[i] = c_s;
    P.iso_h[i] = H;
    P.iso_nu[i] = alpha * H * c_s;
}

// ---------------------------------------------------------------------------
// compute_viscous_stress_tensor, viscosity.cpp:139-254: the cell-centred
// divergence and diagonal components at (i, j) from v_r(i), v_r(i + 1),
// v_phi(j), v_phi(j + 1), nu and Sigma of the cell
struct StressDiag {
    double divv, trr, tpp;
};

template <class PP>
__device__ __forceinline__ StressDiag stress_diag(const PP &P, int i, double vr0, double vr1,
                                                  double va0, double va1, double n, double s)
{
    StressDiag d;
    d.divv = (vr1 * ring_tab(P, TAB_RINF, i + 1) - vr0 * ring_tab(P, TAB_RINF, i)) * ring_tab(P, TAB_INV_DIFF_RSUP_RB, i) +
             (va1 - va0) * P.invdphi * ring_tab(P, TAB_INV_RMED, i);
    const double drr = (vr1 - vr0) * ring_tab(P, TAB_INV_DIFF_RSUP, i);
    d.trr = 2.0 * n * s * (drr - 1.0 / 3.0 * d.divv);
    const double dpp = (va1 - va0) * P.invdphi * ring_tab(P, TAB_INV_RMED, i) + 0.5 * (vr1 + vr0) * ring_tab(P, TAB_INV_RMED, i);
    d.tpp = 2.0 * n * s * (dpp - 1.0 / 3.0 * d.divv);
    return d;
}

// the corner component tau_r_phi at (i >= 1, j) from v_phi(i), v_phi(i - 1),
// v_r(j), v_r(j - 1) and nu, Sigma of the four cells around the corner
template <class PP>
__device__ __forceinline__ double stress_rp(const PP &P, int i, double va0, double vam, double vr0,
                                            double vrp, double n, double nm, double njp, double nmp,
                                            double s, double sm, double sjp, double smp)
{
    const double dvazirdr = (va0 * ring_tab(P, TAB_INV_RMED, i) - vam * ring_tab(P, TAB_INV_RMED, i - 1)) * ring_tab(P, TAB_INV_DIFF_RMED, i);
    const double dvrdphi = (vr0 - vrp) * P.invdphi;
    const double drp = ring_tab(P, TAB_RINF, i) * dvazirdr + dvrdphi * ring_tab(P, TAB_INV_RINF, i);
    const double n4 = 0.25 * (n + nm + njp + nmp);
    const double s4 = 0.25 * (s + sm + sjp + smp);
    return n4 * s4 * drp;
}

template <bool SPLIT>
__device__ __forceinline__ void b_stress(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(nu, FCPT_VISCOSITY);
    FLD(S, FCPT_SIGMA);
    const int jn = j == ns - 1 ? 0 : j + 1;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const int im = i >= 1 ? i - 1 : 0;
    const double vr0 = vr(i, j), vr1 = vr(i + 1, j), va0 = vaz(i, j), va1 = vaz(i, jn);
    const bool iso = !P.adiabatic;  // nu is a ring profile
    const double n = iso ? cst(P.iso_nu)[i] : nu(i, j), s = S(i, j);
    const double vam = vaz(im, j), vrp = vr(i, jp);
    const double nm = iso ? cst(P.iso_nu)[im] : nu(im, j);
    const double njp = iso ? n : nu(i, jp), nmp = iso ? nm : nu(im, jp);
    const double sm = S(im, j), sjp = S(i, jp), smp = S(im, jp);
    const StressDiag d = stress_diag(P, i, vr0, vr1, va0, va1, n, s);
    fld<SPLIT>(P, FCPT_DIV_V).set(i, j, d.divv);
    fld<SPLIT>(P, FCPT_TAU_R_R).set(i, j, d.trr);
    fld<SPLIT>(P, FCPT_TAU_PHI_PHI).set(i, j, d.tpp);
    if (i >= 1)
        fld<SPLIT>(P, FCPT_TAU_R_PHI).set(i, j, stress_rp(P, i, va0, vam, vr0, vrp, n, nm, njp, nmp, s, sm, sjp, smp));
}
FCPT_ONE0(stress, 256)

// update_velocities_with_viscosity, viscosity.cpp:355-426, for one cell
// (inv = dt / Rmed / Sigma_avg)
template <class PP>
__device__ __forceinline__ double visc_vphi_by(const PP &P, int i, double va, double inv, double trp0,
                                               double trp1, double tpp0, double tppj)
{
    const double a1 = ring_tab(P, TAB_RINF_SQ, i + 1), a0 = ring_tab(P, TAB_RINF_SQ, i);
    const double dVp = inv * (ring_tab(P, TAB_VISC_AREA, i) * (a1 * trp1 - a0 * trp0) + (tpp0 - tppj) * P.invdphi);
    return va + dVp;
}
template <bool SPLIT = false>
__device__ __forceinline__ double visc_vphi_new(const KParams &P, int i, double dt, double va, double s0,
                                                double sjp, double trp0, double trp1, double tpp0,
                                                double tppj)
{
    const double sigma_avg = 0.5 * (s0 + sjp);
    return visc_vphi_by(P, i, va, quot<SPLIT>(dt * ring_tab(P, TAB_INV_RMED, i), sigma_avg), trp0, trp1, tpp0, tppj);
}

// (c = dt / Sigma_avg f 2 / (Rmed(i) + Rmed(i - 1)))
template <class PP>
__device__ __forceinline__ double visc_vr_by(const PP &P, int i, double v, double c, double trr0, double trrm,
                                             double trp0, double trpn, double tpp0, double tppm)
{
    const double dVr = c * ((ring_tab(P, TAB_RMED, i) * trr0 - ring_tab(P, TAB_RMED, i - 1) * trrm) *
                                ring_tab(P, TAB_INV_DIFF_RMED, i) +
                            (trpn - trp0) * P.invdphi - 0.5 * (tpp0 + tppm));
    return v + dVr;
}
template <bool SPLIT = false>
__device__ __forceinline__ double visc_vr_new(const KParams &P, int i, double dt, double v, double s0,
                                              double sm, double trr0, double trrm, double trp0,
                                              double trpn, double tpp0, double tppm)
{
    const double sigma_avg = 0.5 * (s0 + sm);
    const double c = quot<SPLIT>(quot<SPLIT>(dt, sigma_avg) * P.radial_viscosity_factor * 2.0,
                                 ring_tab(P, TAB_RMED_SUM, i));
    return visc_vr_by(P, i, v, c, trr0, trrm, trp0, trpn, tpp0, tppm);
}

template <bool SPLIT>
__device__ __forceinline__ void b_visc_update(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(1, P.nr - 1)
    FLD(S, FCPT_SIGMA);
    FLD(trr, FCPT_TAU_R_R);
    FLD(tpp, FCPT_TAU_PHI_PHI);
    FLD(trp, FCPT_TAU_R_PHI);
    FLD(vaz, FCPT_VAZI);
    FLD(vr, FCPT_VRAD);
    const double dt = P.s->dt;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const double s0 = S(i, j), sjp = S(i, jp), sm = S(i - 1, j);
    const double trp0 = trp(i, j), trp1 = trp(i + 1, j), trpn = trp(i, jn);
    const double tpp0 = tpp(i, j), tppj = tpp(i, jp), tppm = tpp(i - 1, j);
    const double trr0 = trr(i, j), trrm = trr(i - 1, j);
    const double va = vaz(i, j), v = vr(i, j);
    vaz.set(i, j, visc_vphi_new<SPLIT>(P, i, dt, va, s0, sjp, trp0, trp1, tpp0, tppj));
    if (i >= 2) vr.set(i, j, visc_vr_new<SPLIT>(P, i, dt, v, s0, sm, trr0, trrm, trp0, trpn, tpp0, tppm));
}
FCPT_ONE0(visc_update, 256)

// ---------------------------------------------------------------------------
// Fused kernels of the step.  Each reads the velocities of its view (P.f[VRAD],
// P.f[VAZI]) and writes the velocities of every row, updated or passed
// through, to the view's partner buffers P.valt: a cell's neighbours then
// always see the old values, exactly as between the separate kernels above,
// whose per-cell expressions they call, and whose intermediate tensors they
// recompute where a neighbour needs them instead of storing and reloading
// them.  The step alternates two views with swapped velocity pointers; the
// transport's velocity kernel writes the final velocities to the fields.
template <bool SPLIT>
__device__ __forceinline__ Fld<SPLIT> alt_vr(const KParams &P)
{
    return buf<SPLIT>(P, P.valt[0], P.bg[FCPT_VRAD], FCPT_VRAD);
}
template <bool SPLIT>
__device__ __forceinline__ Fld<SPLIT> alt_vaz(const KParams &P)
{
    return buf<SPLIT>(P, P.valt[1], P.bg[FCPT_VAZI], FCPT_VAZI);
}

// update_with_sourceterms' two momentum updates (SourceEuler.cpp:325-428) in
// one pass over rows 0 .. nr; v_r is updated on rings 2 .. nr-2, v_phi on
// 1 .. nr-2.  A locally isothermal disk's pressure is formed from Sigma.
template <bool SPLIT>
__device__ __forceinline__ void b_src_fused(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr + 1)
    const int nr = P.nr;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const Fld<SPLIT> vr_o = alt_vr<SPLIT>(P);
    const Fld<SPLIT> vaz_o = alt_vaz<SPLIT>(P);
    const bool upd_p = i >= 1 && i < nr - 1;
    const bool upd_r = i >= 2 && upd_p;
    if (!upd_p) {
        vr_o.set_raw(i, j, vr.raw(i, j));
        if (i < nr) vaz_o.set_raw(i, j, vaz.raw(i, j));
        return;
    }
    FLD(S, FCPT_SIGMA);
    FLD(Pr, FCPT_PRESSURE);
    const Fld<false> Phi = phi_fld(P);
    const bool iso = !P.adiabatic;
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const double s0 = S(i, j), sjp = S(i, jp);
    const double p0 = iso ? iso_pressure(P, i, s0) : Pr(i, j);
    const double pjp = iso ? iso_pressure(P, i, sjp) : Pr(i, jp);
    const double phi0 = Phi(i, j), phijp = Phi(i, jp);
    const double va0 = vaz(i, j);
    double v = 0.0, sm = 0.0, pm = 0.0, phim = 0.0, va1 = 0.0, vam0 = 0.0, vam1 = 0.0;
    if (upd_r) {
        v = vr(i, j);
        sm = S(i - 1, j);
        pm = iso ? iso_pressure(P, i - 1, sm) : Pr(i - 1, j);
        phim = Phi(i - 1, j);
        va1 = vaz(i, jn);
        vam0 = vaz(i - 1, j);
        vam1 = vaz(i - 1, jn);
    }
    const typename Fld<SPLIT>::T vr_raw = vr.raw(i, j);
    vaz_o.set(i, j, src_vphi_new<SPLIT>(P, i, dt, va0, s0, sjp, p0, pjp, phi0, phijp));
    if (upd_r) vr_o.set(i, j, src_vr_new<SPLIT>(P, i, dt, v, s0, sm, p0, pm, phi0, phim, va0, va1, vam0, vam1));
    else vr_o.set_raw(i, j, vr_raw);
}
FCPT_PAIR0(src_fused, 256)

// the TW or SN artificial viscosity (artificial_viscosity.cpp:35-248) in one
// pass: the tensor of the cell, of its azimuthal neighbour j - 1 and of its
// radial neighbour i - 1, the dissipation and temperature floor of E, the
// viscosity recalculation when asked, and the velocity updates
template <bool SPLIT>
__device__ __forceinline__ void b_av_fused(const KParams &P, int bx, int by, int with_viscosity)
{
    CELL_LOOP_HEAD(0, P.nr + 1)
    const int nr = P.nr;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const Fld<SPLIT> vr_o = alt_vr<SPLIT>(P);
    const Fld<SPLIT> vaz_o = alt_vaz<SPLIT>(P);
    if (i == nr) {
        vr_o.set_raw(i, j, vr.raw(i, j));
        return;
    }
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    const bool sn = P.artvisc == FCPT_ARTVISC_SN;
    const bool diss = P.adiabatic && P.artvisc_dissipation;
    const bool visc = with_viscosity && P.adiabatic;  // constant ring profile when isothermal
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const bool inner = i >= 1 && i < nr - 1;
    const bool radial = i >= 2 && inner;
    const int im = i >= 1 ? i - 1 : 0;
    // rows that are not updated are copied as stored (in split storage a
    // decode / encode round trip would round the deviation)
    const typename Fld<SPLIT>::T vr_raw = vr.raw(i, j), va_raw = vaz.raw(i, j);
    const double vr0 = vr.dec(i, vr_raw), vr1 = vr(i + 1, j), va0 = vaz.dec(i, va_raw), va1 = vaz(i, jn);
    const double sig = S(i, j);
    const double e_in = (diss || visc) ? E(i, j) : 0.0;
    double vrj0 = 0.0, vrj1 = 0.0, vaj0 = 0.0, sjp = 0.0;  // cell (i, j - 1)
    if (inner) {
        vrj0 = vr(i, jp);
        vrj1 = vr(i + 1, jp);
        vaj0 = vaz(i, jp);
        sjp = S(i, jp);
    }
    double vrm0 = 0.0, vam0 = 0.0, vam1 = 0.0, sm = 0.0;  // cell (i - 1, j)
    if (radial) {
        vrm0 = vr(im, j);
        vam0 = vaz(im, j);
        vam1 = vaz(im, jn);
        sm = S(im, j);
    }
    double qr0, qp0, qpj = 0.0, qrm = 0.0, qpm = 0.0, e = e_in;
    if (sn) {
        const SnQ q = sn_q_cell(P, i, vr0, vr1, va0, va1, sig);
        qr0 = q.qr;
        qp0 = q.qp;
        if (diss) e = sn_dissipation(P, i, q, sig, dt, e_in);
        if (inner) qpj = sn_q_cell(P, i, vrj0, vrj1, vaj0, va0, sjp).qp;
        if (radial) qrm = sn_q_cell(P, im, vrm0, vr0, vam0, vam1, sm).qr;
    } else {
        const TwQ q = tw_q_cell(P, i, vr0, vr1, va0, va1, sig);
        qr0 = q.qr;
        qp0 = q.qp;
        if (diss) e = tw_dissipation(P, i, q, sig, dt, e_in);
        if (inner) qpj = tw_q_cell(P, i, vrj0, vrj1, vaj0, va0, sjp).qp;
        if (radial) {
            const TwQ m = tw_q_cell(P, im, vrm0, vr0, vam0, vam1, sm);
            qrm = m.qr;
            qpm = m.qp;
        }
    }
    if (diss) e = E.set_get(i, j, e);
    if (visc) derived_store<SPLIT>(P, i, j, DerivedIn{e, sig, 0.0, 0.0}, false, false);
    if (inner)
        vaz_o.set(i, j, sn ? sn_vphi_new<SPLIT>(P, i, dt, va0, sig, sjp, qp0, qpj)
                           : tw_vphi_new<SPLIT>(P, i, dt, va0, sig, sjp, qp0, qpj));
    else
        vaz_o.set_raw(i, j, va_raw);
    if (radial)
        vr_o.set(i, j, sn ? sn_vr_new<SPLIT>(P, i, dt, vr0, sig, sm, qr0, qrm)
                          : tw_vr_new<SPLIT>(P, i, dt, vr0, sig, sm, qr0, qrm, qp0, qpm));
    else
        vr_o.set_raw(i, j, vr_raw);
}
FCPT_PAIR1(av_fused, 256, int, with_viscosity)

// compute_viscous_stress_tensor and update_velocities_with_viscosity
// (viscosity.cpp:139-426) in one pass: the stress components a cell's update
// needs -- tau_rr at (i, j), (i - 1, j); tau_pp at (i, j), (i, j - 1),
// (i - 1, j); tau_rp at (i, j), (i + 1, j), (i, j + 1) -- from the velocities,
// nu and Sigma around it.  The tensor and div v of the cell are stored when a
// later kernel of the step reads them (the viscous heating of SubStep3 in an
// adiabatic disk).
template <bool SPLIT>
__device__ __forceinline__ void b_visc_fused(const KParams &P, int bx, int by)
{
    const bool store_tensor = P.adiabatic && P.heating_viscous;
    CELL_LOOP_HEAD(0, P.nr + 1)
    const int nr = P.nr;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const Fld<SPLIT> vr_o = alt_vr<SPLIT>(P);
    const Fld<SPLIT> vaz_o = alt_vaz<SPLIT>(P);
    if (i == nr) {
        vr_o.set_raw(i, j, vr.raw(i, j));
        return;
    }
    FLD(nu, FCPT_VISCOSITY);
    FLD(S, FCPT_SIGMA);
    const bool iso = !P.adiabatic;  // nu is a ring profile
    const double dt = P.s->dt;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const int jp = j == 0 ? ns - 1 : j - 1;
    const int im = i >= 1 ? i - 1 : 0;
    const bool upd_p = i >= 1 && i < nr - 1;
    const bool upd_r = i >= 2 && upd_p;
    const int ip = upd_p ? i + 1 : i;
    // the cell and the corner (i, j); rows that are not updated are copied as stored
    const typename Fld<SPLIT>::T vr_raw = vr.raw(i, j), va_raw = vaz.raw(i, j);
    const double vr0 = vr.dec(i, vr_raw), vr1 = vr(i + 1, j), va0 = vaz.dec(i, va_raw), va1 = vaz(i, jn);
    const double n = iso ? cst(P.iso_nu)[i] : nu(i, j), s = S(i, j);
    const double vam = vaz(im, j), vrp = vr(i, jp);
    const double nm = iso ? cst(P.iso_nu)[im] : nu(im, j);
    const double njp = iso ? n : nu(i, jp), nmp = iso ? nm : nu(im, jp);
    const double sm = S(im, j), sjp = S(i, jp), smp = S(im, jp);
    // corner (i + 1, j) and cell (i, j - 1): the v_phi update
    double va_p = 0.0, vr1p = 0.0, np_ = 0.0, npj = 0.0, sp = 0.0, spj = 0.0, vaj = 0.0;
    if (upd_p) {
        va_p = vaz(ip, j);
        vr1p = vr(ip, jp);
        np_ = iso ? cst(P.iso_nu)[ip] : nu(ip, j);
        npj = iso ? np_ : nu(ip, jp);
        sp = S(ip, j);
        spj = S(ip, jp);
        vaj = vaz(i, jp);
    }
    // cell (i - 1, j) and corner (i, j + 1): the v_r update
    double vrm = 0.0, vam1 = 0.0, vrn = 0.0, nn = 0.0, nmn = 0.0, sn = 0.0, smn = 0.0;
    if (upd_r) {
        vrm = vr(im, j);
        vam1 = vaz(im, jn);
        vrn = vr(i, jn);
        nn = iso ? n : nu(i, jn);
        nmn = iso ? nm : nu(im, jn);
        sn = S(i, jn);
        smn = S(im, jn);
    }
    const StressDiag d = stress_diag(P, i, vr0, vr1, va0, va1, n, s);
    const double trp0 = i >= 1 ? stress_rp(P, i, va0, vam, vr0, vrp, n, nm, njp, nmp, s, sm, sjp, smp) : 0.0;
    if (store_tensor) {
        fld<SPLIT>(P, FCPT_DIV_V).set(i, j, d.divv);
        fld<SPLIT>(P, FCPT_TAU_R_R).set(i, j, d.trr);
        fld<SPLIT>(P, FCPT_TAU_PHI_PHI).set(i, j, d.tpp);
        if (i >= 1) fld<SPLIT>(P, FCPT_TAU_R_PHI).set(i, j, trp0);
    }
    if (upd_p) {
        const double trp1 = stress_rp(P, ip, va_p, va0, vr1, vr1p, np_, n, npj, njp, sp, s, spj, sjp);
        const double tppj = stress_diag(P, i, vrp, vr1p, vaj, va0, njp, sjp).tpp;
        vaz_o.set(i, j, visc_vphi_new<SPLIT>(P, i, dt, va0, s, sjp, trp0, trp1, d.tpp, tppj));
    } else {
        vaz_o.set_raw(i, j, va_raw);
    }
    if (upd_r) {
        const StressDiag dm = stress_diag(P, im, vrm, vr0, vam, vam1, nm, sm);
        const double trpn = stress_rp(P, i, va1, vam1, vrn, vr0, nn, nmn, n, nm, sn, smn, s, sm);
        vr_o.set(i, j, visc_vr_new<SPLIT>(P, i, dt, vr0, s, sm, d.trr, dm.trr, trp0, trpn, d.tpp, dm.tpp));
    } else {
        vr_o.set_raw(i, j, vr_raw);
    }
}
FCPT_PAIR0(visc_fused, 256)

// the velocities of view P copied as stored to its partner buffers (a LeapFrog
// step whose second kick ends on the swapped view hands them back this way)
template <bool SPLIT>
__device__ __forceinline__ void b_copy_velocities(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr + 1)
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    alt_vr<SPLIT>(P).set_raw(i, j, vr.raw(i, j));
    if (i < P.nr) alt_vaz<SPLIT>(P).set_raw(i, j, vaz.raw(i, j));
}
FCPT_PAIR0(copy_velocities, 256)

// ---------------------------------------------------------------------------
// Q- of the beta cooling (thermal_relaxation, SourceEuler.cpp:632-690) for
// one active cell
template <bool SPLIT, class PP>
__device__ __forceinline__ double cooling_beta_cell(const PP &P, int i, int j, double time, double e,
                                                    double sig)
{
    if (!P.cooling_beta_enabled) return 0.0;
    const double omega_k = ring_tab(P, TAB_OMEGA_K, i);  // Omega_K(Rmed)
    double beta_inv = ring_tab(P, TAB_BETA_INV, i);
    if (P.cooling_beta_ramp_up > 0.0) {
        const double x = 2 * time / P.cooling_beta_ramp_up;
        const double ramp_factor = 1 - exp(-(x * x));
        beta_inv = beta_inv * ramp_factor;
    }
    double delta_E = e;
    if (P.cooling_beta_ref == FCPT_BETA_REF_REFERENCE)
        delta_E -= fld<SPLIT>(P, FCPT_ENERGY0)(i, j) / fld<SPLIT>(P, FCPT_SIGMA0)(i, j) * sig;
    if (P.cooling_beta_ref == FCPT_BETA_REF_FLOOR)
        delta_E -= energy_floor<SPLIT>(P, sig);
    return 0.0 + delta_E * omega_k * beta_inv;
}

// Q+ of the viscous heating (viscous_heating, SourceEuler.cpp:496-536) from
// the cell's stress tensor; tau_r_phi is the mean of the cell's four corners
template <bool SPLIT = false>
__device__ __forceinline__ double viscous_heating_q(const KParams &P, double nu, double sig, double trr,
                                                    double tpp, double dv, double tau_r_phi, bool fine = false)
{
    double q = quot_by<SPLIT>(1.0, make_den<SPLIT>(2.0 * nu * sig, fine)) * (trr * trr + 2 * (tau_r_phi * tau_r_phi) + tpp * tpp);
    q += (2.0 / 9.0) * nu * sig * (dv * dv);
    q *= P.heating_viscous_factor;
    return 0.0 + q;
}

// Q- and Q+ for one active cell, the tensor read from its fields
template <bool SPLIT>
__device__ __forceinline__ void heating_cooling_cell(const KParams &P, int i, int j, double time,
                                                     double e, double sig, double &qplus,
                                                     double &qminus)
{
    const int ns = P.ns;
    qminus = cooling_beta_cell<SPLIT>(P, i, j, time, e, sig);
    qplus = 0.0;
    if (P.heating_viscous) {
        const double nu = fld<SPLIT>(P, FCPT_VISCOSITY)(i, j);
        if (nu != 0.0) {
            FLD(trp, FCPT_TAU_R_PHI);
            const int jn = j == ns - 1 ? 0 : j + 1;
            const double tau_r_phi = 0.25 * (trp(i, j) + trp(i + 1, j) + trp(i, jn) + trp(i + 1, jn));
            qplus = viscous_heating_q<SPLIT>(P, nu, sig, fld<SPLIT>(P, FCPT_TAU_R_R)(i, j),
                                      fld<SPLIT>(P, FCPT_TAU_PHI_PHI)(i, j), fld<SPLIT>(P, FCPT_DIV_V)(i, j),
                                      tau_r_phi);
        }
    }
}


// the radiative correction of SubStep3 (SourceEuler.cpp:920-924; its
// std::pow(., 4) and std::pow(., 3) by compensated powering)
template <bool SPLIT = false>
__device__ __forceinline__ double rad_alpha(const KParams &P, double h, double sig, double e)
{
    const double inv_pow4 = pow4_comp(quot<SPLIT>(P.mu * (P.gamma - 1.0), P.Rgas * sig));
    return 1.0 + 2.0 * h * 4.0 * P.sigma_sb / P.c_light * inv_pow4 * pow3_comp(e);
}
// the same at a cell of ring i whose Sigma, E and H are in range (fine)
template <bool SPLIT, class PP>
__device__ __forceinline__ double rad_alpha_in(const PP &P, int i, double h, double sig, double e, bool fine)
{
    if constexpr (SPLIT) {
        return rad_alpha<true>(P, h, sig, e);
    } else {
        const double d = P.Rgas * sig;
        const double inv_pow4 = pow4_comp(quot_by<false>(ring_tab(P, TAB_MU_GM1, i), Den{d, shared_den(d).r, fine}));
        const Den c{ring_tab(P, TAB_C_LIGHT, i), ring_tab(P, TAB_C_LIGHT_RCP, i), fine};
        return 1.0 + quot_by<false>(2.0 * h * 4.0 * P.sigma_sb, c) * inv_pow4 * pow3_comp(e);
    }
}

// SubStep3 (SourceEuler.cpp:859-954) at one cell from its Q+ and Q- before
// the radiative correction; writes T, Q+, Q- and (to Eo) E
template <bool SPLIT, class PP>
__device__ __forceinline__ void substep3_cell(const PP &P, const Fld<SPLIT> &Eo, int i, int j, double e,
                                              double sig, double h, double qplus, double qminus, bool fine = false)
{
    const double dt = kick_dt(P);
    if (!P.lazy_derived) {
        // compute_temperature (SourceEuler.cpp:1378-1408) before the update
        const double c_v_inv = P.mu / P.Rgas * (P.gamma - 1.0);
        fld<SPLIT>(P, FCPT_TEMPERATURE).set(i, j, c_v_inv * e / sig);
    }
    if (i >= 1 && i < P.nr - 1) {
        const double alpha = rad_alpha_in<SPLIT>(P, i, h, sig, e, fine);
        if constexpr (SPLIT) {
            const double ra = recip<true>(alpha);
            qplus *= ra;
            qminus *= ra;
        } else {  // the same bits through one reciprocal
            const SharedDen A = shared_den(alpha);
            qplus = shared_div(qplus, A);
            qminus = shared_div(qminus, A);
        }
        double energy_new = e + dt * (qplus - qminus);
        if (sig < ring_tab(P, TAB_SIGMA_FLOOR10, i)) {
            // TAU_EFF is never computed without surface cooling: it holds 0
            const double tau_eff = 0.0;
            const double e4 = qplus * tau_eff / (2.0 * P.sigma_sb);
            const double constant = (P.Rgas / P.mu * sig / (P.gamma - 1.0));
            energy_new = sqrt(sqrt(e4)) * constant;  // pow(e4, 1 / 4): 0 here, as tau_eff is 0
            qminus = qplus;
        }
        e = energy_new;
    } else {
        qplus = qminus = 0.0;
    }
    fld<SPLIT>(P, FCPT_QPLUS).set(i, j, qplus);
    fld<SPLIT>(P, FCPT_QMINUS).set(i, j, qminus);
    Eo.set(i, j, temperature_floor_in<SPLIT>(P, i, e, sig, fine));
}

template <bool SPLIT>
__device__ __forceinline__ void b_substep3(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    const double sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
    const double e = fld<SPLIT>(P, FCPT_ENERGY)(i, j);
    const double h = fld<SPLIT>(P, FCPT_SCALE_HEIGHT)(i, j);
    double qplus = 0.0, qminus = 0.0;
    if (i >= 1 && i < P.nr - 1) heating_cooling_cell<SPLIT>(P, i, j, P.s->time, e, sig, qplus, qminus);
    substep3_cell<SPLIT>(P, fld<SPLIT>(P, FCPT_ENERGY), i, j, e, sig, h, qplus, qminus);
}
FCPT_PAIR0(substep3, 256)

// compute_heating_cooling_for_CFL, SourceEuler.cpp:1410-1450 (after update_viscosity
// and the stress tensor)
template <bool SPLIT>
__device__ __forceinline__ void b_heatcool_cfl(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    double qplus = 0.0, qminus = 0.0;
    if (i >= 1 && i < P.nr - 1) {
        const double e = fld<SPLIT>(P, FCPT_ENERGY)(i, j);
        const double sig = fld<SPLIT>(P, FCPT_SIGMA)(i, j);
        heating_cooling_cell<SPLIT>(P, i, j, P.s->time, e, sig, qplus, qminus);
        const double alpha = rad_alpha<SPLIT>(P, fld<SPLIT>(P, FCPT_SCALE_HEIGHT)(i, j), sig, e);
        qplus /= alpha;
        qminus /= alpha;
    }
    fld<SPLIT>(P, FCPT_QPLUS).set(i, j, qplus);
    fld<SPLIT>(P, FCPT_QMINUS).set(i, j, qminus);
}
FCPT_PAIR0(heatcool_cfl, 256)

// The fused viscous pass as a radial walk.  A wavefront owns kViscSegW
// consecutive sectors and `tile` consecutive rings: lane k holds sector
// j0 - 1 + k (lanes 0 and 63 are the halo) and walks the rings outwards.
// Each ring is loaded once (v_r, v_phi, Sigma, nu of the lane's own sector;
// the ring after next is prefetched before the current ring's stores), the
// neighbouring sectors' values come from the adjacent lanes by DPP moves,
// and every stress component is formed once per cell: the diagonal of ring
// i, whose tau_phi_phi at sector j - 1 is the left lane's, and tau_rp of
// corner (i + 1, j), whose value at sector j + 1 is the right lane's; the
// diagonal of ring i - 1 and the corners of ring i carry over from the
// previous step.  Every value goes through the helpers b_visc_fused calls,
// with the same arguments, so the two are bit-identical.  With ENERGY the walk
// also runs SubStep3 on each cell it updates, its viscous heating formed from
// the tensor in registers (the corner mean takes tau_rp of corner (i + 1,
// j + 1) from the right lane), exactly as b_substep3 forms it from the stored
// tensor, which the walk then does not store.
constexpr int kViscSegW = 62;  // sectors written per wavefront

struct ViscRing {
    double vr, va, s, n;  // the lane's sector
    double vrL, sL, nL;   // sector j - 1
    double vaR;           // v_phi of sector j + 1
};

template <bool SPLIT, bool ENERGY>
__device__ __forceinline__ void b_visc_walk(const KParams &P, int bx, int by, int tile)
{
    const int ns = P.ns, nr = P.nr;
    const int k = (int)threadIdx.x;  // lane
    const int i0 = __builtin_amdgcn_readfirstlane((by * (int)blockDim.y + (int)threadIdx.y) * tile);
    if (i0 >= nr) return;
    const int i1 = i0 + tile < nr ? i0 + tile : nr;  // rings [i0, i1)
    const int j0 = bx * kViscSegW;
    const int Ls = ns - j0 < kViscSegW ? ns - j0 : kViscSegW;
    const int j = (j0 - 1 + k + ns) % ns;
    const bool wr = k >= 1 && k <= Ls;  // lanes that write
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(nu, FCPT_VISCOSITY);
    FLD(S, FCPT_SIGMA);
    const Fld<SPLIT> vr_o = alt_vr<SPLIT>(P);
    const Fld<SPLIT> vaz_o = alt_vaz<SPLIT>(P);
    const bool iso = !P.adiabatic;  // nu is a ring profile
    const bool store = !ENERGY && P.adiabatic && P.heating_viscous;
    const double dt = P.s->dt;
    // the lane's values of ring r (r < nr); ring nr holds only v_r
    struct Raw {
        double vr, va, s, n;
    };
    auto load = [&](int r) {
        Raw w;
        w.vr = vr(r, j);
        if (r < nr) {
            w.va = vaz(r, j);
            w.s = S(r, j);
            w.n = iso ? cst(P.iso_nu)[r] : nu(r, j);
        } else {
            w.va = w.s = w.n = 0.0;
        }
        return w;
    };
    auto ring = [&](const Raw &w) {
        ViscRing g;
        g.vr = w.vr;
        g.va = w.va;
        g.s = w.s;
        g.n = w.n;
        g.vrL = from_left(w.vr);
        g.sL = from_left(w.s);
        g.nL = iso ? w.n : from_left(w.n);
        g.vaR = from_right(w.va);
        return g;
    };
    // tau_rp at corner (r, j) from rings a = r - 1 and b = r
    auto corner = [&](int r, const ViscRing &a, const ViscRing &b) {
        return stress_rp(P, r, b.va, a.va, b.vr, b.vrL, b.n, a.n, b.nL, a.nL, b.s, a.s, b.sL, a.sL);
    };
    ViscRing A, B;  // rings i, i + 1
    StressDiag dprev{0.0, 0.0, 0.0};
    double trp_c = 0.0, s_prev = 0.0;  // tau_rp(i, j), Sigma(i - 1, j)
    if (i0 >= 1) {
        const ViscRing Z = ring(load(i0 - 1));
        A = ring(load(i0));
        dprev = stress_diag(P, i0 - 1, Z.vr, A.vr, Z.va, Z.vaR, Z.n, Z.s);
        trp_c = corner(i0, Z, A);
        s_prev = Z.s;
    } else {
        A = ring(load(i0));
    }
    B = ring(load(i0 + 1));
    for (int i = i0; i < i1; ++i) {
        const Raw Cn = load(i + 2 <= nr ? i + 2 : nr);  // prefetch, before this ring's stores
        const bool upd_p = i >= 1 && i < nr - 1;
        const bool upd_r = i >= 2 && upd_p;
        const StressDiag d = stress_diag(P, i, A.vr, B.vr, A.va, A.vaR, A.n, A.s);
        const double tppj = from_left(d.tpp);  // diagonal of (i, j - 1)
        const double trp_n = from_right(trp_c);  // corner (i, j + 1)
        const double trp1 = i + 1 <= nr - 1 ? corner(i + 1, A, B) : 0.0;
        const double trp1_n = ENERGY ? from_right(trp1) : 0.0;  // corner (i + 1, j + 1)
        if (wr) {
            if (store) {
                fld<SPLIT>(P, FCPT_DIV_V).set(i, j, d.divv);
                fld<SPLIT>(P, FCPT_TAU_R_R).set(i, j, d.trr);
                fld<SPLIT>(P, FCPT_TAU_PHI_PHI).set(i, j, d.tpp);
                if (i >= 1) fld<SPLIT>(P, FCPT_TAU_R_PHI).set(i, j, trp_c);
            }
            if (upd_p)
                vaz_o.set(i, j, visc_vphi_new<SPLIT>(P, i, dt, A.va, A.s, A.sL, trp_c, trp1, d.tpp, tppj));
            else
                vaz_o.set_raw(i, j, vaz.raw(i, j));
            if (upd_r)
                vr_o.set(i, j, visc_vr_new<SPLIT>(P, i, dt, A.vr, A.s, s_prev, d.trr, dprev.trr, trp_c, trp_n,
                                           d.tpp, dprev.tpp));
            else
                vr_o.set_raw(i, j, vr.raw(i, j));
            if constexpr (ENERGY) {
                FLD(E, FCPT_ENERGY);
                const double e = E(i, j);
                const double h = fld<SPLIT>(P, FCPT_SCALE_HEIGHT)(i, j);
                double qplus = 0.0, qminus = 0.0;
                if (upd_p) {
                    qminus = cooling_beta_cell<SPLIT>(P, i, j, P.s->time, e, A.s);
                    if (P.heating_viscous && A.n != 0.0)
                        qplus = viscous_heating_q<SPLIT>(P, A.n, A.s, d.trr, d.tpp, d.divv,
                                                  0.25 * (trp_c + trp1 + trp_n + trp1_n));
                }
                substep3_cell<SPLIT>(P, E, i, j, e, A.s, h, qplus, qminus);
            }
        }
        dprev = d;
        trp_c = trp1;
        s_prev = A.s;
        A = B;
        B = ring(Cn);
    }
    if (i1 == nr && wr) vr_o.set_raw(nr, j, vr.raw(nr, j));  // the outer v_r row, untouched
}
template <bool SPLIT, bool ENERGY>
__global__ void __launch_bounds__(256) k_visc_walk(KParams P, int tile)
{
    const BlockXY bb = xcd_block();
    b_visc_walk<SPLIT, ENERGY>(P, bb.x, bb.y, tile);
}
// batched form: each disk's tile is its resolved visc_tile
template <bool SPLIT, bool ENERGY>
__global__ void __launch_bounds__(256) kb_visc_walk(const KParams *Ps, const BatchEntry *map)
{
    const BatchEntry e = batch_entry(map);
    const KParams &P = batch_disk(Ps, e.disk);
    b_visc_walk<SPLIT, ENERGY>(P, (int)(e.yx & 0xffffu), (int)(e.yx >> 16), P.visc_tile);
}

// The whole kick of the fused step as one radial walk, after the potential
// pass: update_with_sourceterms, compression_heating (adiabatic), the TW or SN
// artificial viscosity with its dissipation and recalculate_viscosity, then
// the viscous stress, the velocity update and (adiabatic) SubStep3: the
// per-cell steps of b_src_fused, b_src_energy, b_av_fused, b_visc_fused and
// b_substep3 in that order.
//
// A wavefront owns kKvSegW consecutive sectors and `tile` consecutive rings:
// lane k holds sector j0 - 3 + k and walks the rings outwards.  Each ring is
// loaded once (v_r, v_phi, Sigma, the potential, and E of an adiabatic disk,
// whose pressure is (gamma - 1) E); neighbouring sectors' values come from the
// adjacent lanes by DPP moves, and every stage runs one ring behind the one it
// reads: the source-term velocities at ring m + 1, the artificial viscosity at
// m, the viscous update and SubStep3 at m - 1.  The stages spoil three lanes
// at the lower and two at the upper edge: the source terms read sectors j - 1
// and j + 1, the artificial viscosity the tensor of j - 1 and v_phi of j + 1,
// the viscous update tau_phi_phi of j - 1 and tau_r_phi of j + 1.  Results go
// to partner buffers (the velocities' valt, E's ealt), so no wavefront reads
// what another writes; rows that are not updated are copied as stored.
//
// Every value goes through the helpers of the separate kernels with the same
// arguments, so FP64 storage gives the same fields bit for bit.  Split storage
// rounds what the stages hand over (v_r, v_phi, E and nu between the
// artificial viscosity and the viscous update) as if it had been stored;
// KParams::split_emul adds the roundings of the forms that store more.
//
// What bounds it: its instructions, whose issue is 0.61 of its time at 4096 x
// 12288 adiabatic (0.74 in split storage), and beyond them the latency of its
// chain of stages, at the 3 wavefronts per SIMD (4 isothermal) that its registers
// allow.  Hence one pass for the whole kick (a walk for the sources and
// artificial viscosity and one for the rest moved 188 B/cell at 4096 x 12288
// adiabatic, 2161 us; this one 88 B/cell, 1190 us; 2048 x 6144 isothermal 256
// -> 170 us), the loads of ring m + 2 in flight during ring m, no load behind
// a store in the loop (rows that are only copied are copied after it: 240 us
// at 4096 x 12288), the ring's metric in LDS (KWalk), and quotients that share
// a denominator through one reciprocal.
// doubles of LDS per wavefront: the ring-table rows of its rings
__host__ __device__ inline int kv_lds_doubles(int tile) { return (tile + 5) * kRingTabs; }
extern __shared__ __align__(16) double kv_lds[];

constexpr int kKvSegW = 59;   // sectors written per wavefront
constexpr int kKvHalo = 3;    // sectors before them
template <bool SPLIT, bool ADI, bool SN, bool EMUL>
__device__ __forceinline__ void b_kv_walk(const KParams &K, int bx, int by, int tile, double *lds)
{
    const int ns = K.ns, nr = K.nr;
    const int k = (int)threadIdx.x;  // lane
    const int i0 = __builtin_amdgcn_readfirstlane((by * (int)blockDim.y + (int)threadIdx.y) * tile);
    if (i0 >= nr) return;
    const int i1 = i0 + tile < nr ? i0 + tile : nr;  // rings [i0, i1)
    const int j0 = bx * kKvSegW;
    const int Ls = ns - j0 < kKvSegW ? ns - j0 : kKvSegW;
    const int j = (j0 - kKvHalo + k + ns) % ns;
    const bool own = k >= kKvHalo && k < kKvHalo + Ls;  // lanes that write
    // this wavefront's rows of the ring table: rings i0 - 3 .. i1 + 1
    KWalk P{K, lds + (int)threadIdx.y * kv_lds_doubles(tile), i0 >= 3 ? i0 - 3 : 0, 0.0};
    if (K.fold_in_kick) P.step_at = &K.s->count_next;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    const Fld<SPLIT> vr_o = alt_vr<SPLIT>(P);
    const Fld<SPLIT> vaz_o = alt_vaz<SPLIT>(P);
    // one ring of the lane's sector as loaded
    struct Raw {
        typename Fld<SPLIT>::T vr, va, s, e;
        double phi;
    };
    auto load = [&](int r) {
        Raw w;
        const int c = r < nr ? r : nr - 1;  // ring nr holds only v_r
        w.vr = vr.raw(r, j);
        w.va = vaz.raw(c, j);
        w.s = S.raw(c, j);
        if constexpr (ADI) w.e = E.raw(c, j);
        w.phi = phi_fld(P)(c, j);
        return w;
    };
    // The walk's start issues every load before it waits for one: the window's
    // rings, the rows of the ring table and the fold's ring minima (with a wait
    // per round of them a 1024x3072 step took 301.7 us, now 299.4).
    const int m0 = i0 >= 1 ? i0 - 1 : 0;  // the first ring of the artificial viscosity
    const Raw x2 = load(m0 >= 2 ? m0 - 2 : 0), x1 = load(m0 >= 1 ? m0 - 1 : 0), x0 = load(m0);
    Raw X = load(m0 + 1);  // ring m + 1, in flight
    FoldLoads fold;
    if (K.fold_in_kick) cfl_fold_load(K, k, fold);
    {
        constexpr int U = 6;
        const int last = i1 + 1 <= nr ? i1 + 1 : nr, n = (last - P.row0 + 1) * kRingTabs;
        const double *src = K.ring_tab + (size_t)P.row0 * kRingTabs;
        double *dst = const_cast<double *>(P.rows);
        for (int t0 = 0; t0 < n; t0 += 64 * U) {
            double row[U];
#pragma unroll
            for (int u = 0; u < U; ++u) row[u] = src[min(t0 + 64 * u + k, n - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (t0 + 64 * u + k < n) dst[t0 + 64 * u + k] = row[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (K.fold_in_kick) {
        P.dt = cfl_fold_wave(K, k, bx == 0 && i0 == 0, fold);
        if (P.kick) P.dt = P.dt / 2;
    } else {
        P.dt = kick_dt(K);
    }
    const double dt = P.dt;
    const bool diss = ADI && P.artvisc_dissipation;
    const bool emul_derived = EMUL && (P.split_emul & SPLIT_EMUL_DERIVED);
    const bool emul_stages = EMUL && (P.split_emul & SPLIT_EMUL_STAGES);
    const bool launch_ok = P.const_ok && quot_range(dt);  // the quotients' numerators are in range
    struct Ring {
        double vr, va, s, p, phi, e;  // p: pressure, phi: potential
        double sL, vaR;               // Sigma of sector j - 1, v_phi of sector j + 1
    };
    auto ring = [&](int r, const Raw &w) {
        Ring g;
        const int c = r < nr ? r : nr - 1;
        g.vr = vr.dec(r, w.vr);
        g.va = vaz.dec(c, w.va);
        g.s = S.dec(c, w.s);
        if constexpr (ADI) {
            g.e = E.dec(c, w.e);
            g.p = (P.gamma - 1.0) * g.e;
            // a LeapFrog step's second kick reads the pressure of its own drift
            if (emul_derived)
                g.p = (P.kick == 2 ? fld<SPLIT>(P, FCPT_PRESSURE) : fld_derived<SPLIT>(P, FCPT_PRESSURE)).stored(c, j, g.p);
        } else {
            g.e = 0.0;
            g.p = iso_pressure(P, c, g.s);
        }
        g.phi = w.phi;
        g.sL = from_left(g.s);
        g.vaR = from_right(g.va);
        return g;
    };
    // the reciprocals of a ring's Sigma sums with ring r - 1 and sector j - 1:
    // the denominators of the source terms, the artificial viscosity and the
    // viscous update (whose Sigma_avg is half the sum)
    struct Rcp {
        double r, p;
        bool ok;
    };
    // the source-term velocities of ring r (b) from ring r - 1 (a); rows
    // that are not updated keep their values
    auto src = [&](int r, const Ring &a, const Ring &b, double &v1r, double &v1a) {
        const double pjp = from_left(b.p), phijp = from_left(b.phi);
        const bool upd_p = r >= 1 && r < nr - 1;
        const bool upd_r = r >= 2 && upd_p;
        const Den dr = make_den<SPLIT>(b.s + a.s, launch_ok), dp = make_den<SPLIT>(b.s + b.sL, launch_ok);
        v1a = b.va;
        v1r = b.vr;
        if (upd_p) {
            v1a = src_vphi_by(P, r, dt, b.va, quot_by<SPLIT>(2.0, dp), b.p, pjp, b.phi, phijp);
            if (emul_stages) v1a = vaz_o.stored(r, j, v1a);
        }
        if (upd_r) {
            v1r = src_vr_by(P, r, dt, b.vr, quot_by<SPLIT>(2.0, dr), b.p, a.p, b.phi, a.phi, b.va, b.vaR, a.va,
                            a.vaR);
            if (emul_stages) v1r = vr_o.stored(r, j, v1r);
        }
        return Rcp{dr.r, dp.r, dr.ok && dp.ok};
    };
    // the tensor of cell (r, j) from the source-term velocities
    struct Q {
        TwQ tw;
        SnQ sn;
        double qr, qp;
    };
    auto qcell = [&](int r, double vr0, double vr1, double va0, double va1, double sig) {
        Q q;
        if constexpr (SN) {
            q.sn = sn_q_cell(P, r, vr0, vr1, va0, va1, sig);
            q.qr = q.sn.qr;
            q.qp = q.sn.qp;
        } else {
            q.tw = tw_q_cell(P, r, vr0, vr1, va0, va1, sig);
            q.qr = q.tw.qr;
            q.qp = q.tw.qp;
        }
        return q;
    };
    // a ring after the artificial viscosity, as the viscous stage reads it
    struct Visc {
        double vr, va, s, n, e, h;
        Rcp rcp;
        bool fine;  // its E and Sigma are in range
    };
    Ring R0;                              // ring m
    double v1r0, v1a0;                    // its source-term velocities
    Rcp rcp0;
    double qr_m = 0.0, qp_m = 0.0, s_m = 0.0;  // tensor and Sigma of cell (m - 1, j)
    {
        const Ring Rm2 = ring(m0 >= 2 ? m0 - 2 : 0, x2);  // read by rings m0 - 1 >= 2 only
        const Ring Rm = ring(m0 >= 1 ? m0 - 1 : 0, x1);
        R0 = ring(m0, x0);
        rcp0 = src(m0, Rm, R0, v1r0, v1a0);  // ring 0 is passed through
        if (m0 >= 1) {
            double v1rm, v1am;
            src(m0 - 1, Rm2, Rm, v1rm, v1am);
            const Q qm = qcell(m0 - 1, v1rm, v1r0, v1am, from_right(v1am), Rm.s);
            qr_m = qm.qr;
            qp_m = qm.qp;
            s_m = Rm.s;
        }
    }
    Visc A{};                              // ring m - 1
    StressDiag dprev{0.0, 0.0, 0.0};       // its predecessor's diagonal
    double trp_c = 0.0, s_prev = 0.0;      // tau_rp(m - 1, j), Sigma(m - 2, j)
    for (int m = m0; m <= i1; ++m) {
        // the artificial viscosity at ring m (ring nr holds only v_r)
        Visc B;
        if (m < nr) {
            const Ring R1 = ring(m + 1, X);
            if (m < i1) X = load(m + 2 <= nr ? m + 2 : nr);  // before this ring's stores
            double v1r1, v1a1;
            const Rcp rcp1 = src(m + 1, R0, R1, v1r1, v1a1);
            const double v1aR = from_right(v1a0);  // v_phi of sector j + 1
            const Q q = qcell(m, v1r0, v1r1, v1a0, v1aR, R0.s);
            const double qpj = from_left(q.qp);  // tensor of cell (m, j - 1)
            const bool inner = m >= 1 && m < nr - 1;
            const bool radial = m >= 2 && inner;
            B.s = R0.s;
            if constexpr (ADI) {
                // compression_heating (rings 0 .. nr-2), then the dissipation
                double e = R0.e;
                if (m < nr - 1) e = E.stored(m, j, src_energy_new(P, m, dt, e, v1r0, v1r1, v1a0, v1aR));
                const bool s_ok = launch_ok && quot_range(R0.s);
                if (diss) {
                    if constexpr (SN) e = sn_heat(P, m, q.sn, dt, e);
                    else e = tw_heat(P, m, q.tw, R0.s, dt, e);
                    // the limits are FP64 quotients in both storage modes
                    e = E.stored(m, j, temperature_floor_in<false>(P, m, e, R0.s, s_ok));
                } else if (!emul_stages && m < nr - 1) {
                    e = E.stored(m, j, e);
                }
                // recalculate_viscosity
                B.fine = s_ok && quot_range(e);
                const AdiDerived d = adi_derived_in<SPLIT>(P, m, e, R0.s, B.fine);
                B.e = e;
                B.h = emul_derived ? fld<SPLIT>(P, FCPT_SCALE_HEIGHT).stored(m, j, d.h) : d.h;
                B.n = fld<SPLIT>(P, FCPT_VISCOSITY).stored(m, j, d.nu);
                // the second kick of a LeapFrog step smooths its potential with this H
                if (P.integrator == FCPT_INTEGRATOR_LEAPFROG && own && m >= i0 && m < i1)
                    fld<SPLIT>(P, FCPT_SCALE_HEIGHT).set(m, j, d.h);
            } else {
                B.e = B.h = 0.0;
                B.n = cst(P.iso_nu)[m];
                B.fine = false;
            }
            B.rcp = rcp0;
            B.va = v1a0;
            if (inner) {
                if constexpr (SN) {
                    B.va = sn_vphi_by(P, m, v1a0, quot_by<SPLIT>(dt * 2.0, Den{R0.s + R0.sL, rcp0.p, rcp0.ok}), q.qp, qpj);
                } else {
                    const Den D = make_den<SPLIT>(ring_tab(P, TAB_RSUP_RINF, m) * (0.5 * (R0.s + R0.sL)), rcp0.ok);
                    B.va = tw_vphi_by(P, v1a0, quot_by<SPLIT>(2.0 * dt, D), q.qp, qpj);
                }
                B.va = vaz_o.stored(m, j, B.va);
            }
            B.vr = v1r0;
            if (radial) {
                const Den D{R0.s + s_m, rcp0.r, rcp0.ok};
                if constexpr (SN) {
                    B.vr = sn_vr_by(P, m, v1r0, quot_by<SPLIT>(dt * 2.0, D), q.qr, qr_m);
                } else {
                    const Den R2{ring_tab(P, TAB_RMED_SQ_DIFF, m), ring_tab(P, TAB_RMED_SQ_DIFF_RCP, m), rcp0.ok};
                    const double c = quot_by<SPLIT>(2.0 * (P.radial_viscosity_factor * dt), D) * 2.0;
                    B.vr = tw_vr_by(P, m, v1r0, quot_by<SPLIT>(c, R2), q.qr, qr_m, q.qp, qp_m);
                }
                B.vr = vr_o.stored(m, j, B.vr);
            }
            qr_m = q.qr;
            qp_m = q.qp;
            s_m = R0.s;
            R0 = R1;
            v1r0 = v1r1;
            v1a0 = v1a1;
            rcp0 = rcp1;
        } else {
            B = Visc{R0.vr, 0.0, 0.0, 0.0, 0.0, 0.0, {0.0, 0.0, false}, false};
        }
        // the viscous stage at ring i = m - 1 (A), from rings i and i + 1 (B)
        const int i = m - 1;
        if (i >= m0) {
            const StressDiag d = stress_diag(P, i, A.vr, B.vr, A.va, from_right(A.va), A.n, A.s);
            double trp1 = 0.0;  // tau_rp at corner (i + 1, j)
            if (m <= nr - 1) {
                const double nB = ADI ? from_left(B.n) : B.n, nA = ADI ? from_left(A.n) : A.n;
                trp1 = stress_rp(P, m, B.va, A.va, B.vr, from_left(B.vr), B.n, A.n, nB, nA, B.s, A.s,
                                 from_left(B.s), from_left(A.s));
            }
            const bool upd_p = i >= 1 && i < nr - 1;
            const bool upd_r = i >= 2 && upd_p;
            const double tppj = from_left(d.tpp);    // diagonal of (i, j - 1)
            const double trp_n = from_right(trp_c);  // corner (i, j + 1)
            double qplus = 0.0, qminus = 0.0;
            if constexpr (ADI) {
                if (upd_p) {
                    qminus = cooling_beta_cell<SPLIT>(P, i, j, kick_time(P), A.e, A.s);
                    if (P.heating_viscous) {
                        double trr = d.trr, tpp = d.tpp, dv = d.divv, c0 = trp_c, c1 = trp1;
                        if (emul_stages) {
                            trr = fld<SPLIT>(P, FCPT_TAU_R_R).stored(i, j, trr);
                            tpp = fld<SPLIT>(P, FCPT_TAU_PHI_PHI).stored(i, j, tpp);
                            dv = fld<SPLIT>(P, FCPT_DIV_V).stored(i, j, dv);
                            c0 = fld<SPLIT>(P, FCPT_TAU_R_PHI).stored(i, j, c0);
                            c1 = fld<SPLIT>(P, FCPT_TAU_R_PHI).stored(m, j, c1);
                        }
                        const double c0n = emul_stages ? from_right(c0) : trp_n;
                        const double c1n = from_right(c1);  // corner (i + 1, j + 1)
                        if (A.n != 0.0)
                            qplus = viscous_heating_q<SPLIT>(P, A.n, A.s, trr, tpp, dv, 0.25 * (c0 + c1 + c0n + c1n),
                                                             A.fine);
                    }
                }
            }
            const double sAL = from_left(A.s);
            if (own && i >= i0) {
                if (upd_p) {
                    const Den D{A.s + sAL, A.rcp.p, A.rcp.ok};
                    const double inv = quot_by<SPLIT>(2.0 * (dt * ring_tab(P, TAB_INV_RMED, i)), D);
                    vaz_o.set(i, j, visc_vphi_by(P, i, A.va, inv, trp_c, trp1, d.tpp, tppj));
                }
                if (upd_r) {
                    const Den D{A.s + s_prev, A.rcp.r, A.rcp.ok};
                    const Den R{ring_tab(P, TAB_RMED_SUM, i), ring_tab(P, TAB_RMED_SUM_RCP, i), A.rcp.ok};
                    const double c = quot_by<SPLIT>(quot_by<SPLIT>(2.0 * dt, D) * P.radial_viscosity_factor * 2.0, R);
                    vr_o.set(i, j, visc_vr_by(P, i, A.vr, c, d.trr, dprev.trr, trp_c, trp_n, d.tpp, dprev.tpp));
                }
                if constexpr (ADI) {
                    const Fld<SPLIT> Eo = buf<SPLIT>(P, P.ealt, P.bg[FCPT_ENERGY], FCPT_ENERGY);
                    substep3_cell<SPLIT>(P, Eo, i, j, A.e, A.s, A.h, qplus, qminus, A.fine);
                }
            }
            dprev = d;
            trp_c = trp1;
            s_prev = A.s;
        }
        A = B;
    }
    // the rows that are not updated, copied as stored (here and not in the
    // loop: a load there would make every ring wait for its prefetch)
    if (!own) return;
    if (i0 == 0) {
        vr_o.set_raw(0, j, vr.raw(0, j));
        vaz_o.set_raw(0, j, vaz.raw(0, j));
    }
    if (i0 <= 1 && i1 > 1) vr_o.set_raw(1, j, vr.raw(1, j));
    if (i1 == nr) {
        vr_o.set_raw(nr - 1, j, vr.raw(nr - 1, j));
        vaz_o.set_raw(nr - 1, j, vaz.raw(nr - 1, j));
        vr_o.set_raw(nr, j, vr.raw(nr, j));
    }
}
template <bool SPLIT, bool ADI, bool SN, bool EMUL>
__global__ void __launch_bounds__(64, ADI ? 3 : 4) k_kv_walk(KParams P, int tile)
{
    const BlockXY bb = xcd_block();
    b_kv_walk<SPLIT, ADI, SN, EMUL>(P, bb.x, bb.y, tile, kv_lds);
}
// batched form: each disk's tile is its kv_tile
template <bool SPLIT, bool ADI, bool SN>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(ADI ? 3 : 4))) kb_kv_walk(const KParams *Ps, const BatchEntry *map)
{
    const BatchEntry e = batch_entry(map);
    const KParams &P = batch_disk(Ps, e.disk);
    b_kv_walk<SPLIT, ADI, SN, SPLIT>(P, (int)(e.yx & 0xffffu), (int)(e.yx >> 16), P.kv_tile, kv_lds);
}

// ---------------------------------------------------------------------------
// damping (boundary_conditions/damping.cpp:311-427, 754-776): whether ring i of
// a vector (v_r) or scalar field lies in a damping zone, the relaxation of its
// values over dt (the inner zone's, then the outer one's), and a value relaxed
// towards its reference x0.  Ramp and time scale are per-ring constants
// (k_ring_tables): a damped ring costs one division and one exponential,
// shared by its scalar fields.
__device__ __forceinline__ bool damped_ring(const KParams &P, bool vector, int i)
{
    return i <= P.zone_in[vector] || i >= P.zone_out[vector];
}
struct Damp {
    bool in, out;
    double f_in, f_out;
};
__device__ __forceinline__ Damp damp_ring(const KParams &P, bool vector, int i, double dt)
{
    const auto t = cst(P.damp_tab) + 8 * i + (vector ? 4 : 0);
    Damp d{i <= P.zone_in[vector], i >= P.zone_out[vector], 1.0, 1.0};
    if (d.in) d.f_in = exp(-dt * t[0] / t[1]);
    if (d.out) d.f_out = exp(-dt * t[2] / t[3]);
    return d;
}
__device__ __forceinline__ double damp_value(double x, double x0, const Damp &d)
{
    if (d.in) x = (x - x0) * d.f_in + x0;
    if (d.out) x = (x - x0) * d.f_out + x0;
    return x;
}

// damping: block row y maps to an inner-zone ring (y < n_inner) or an
// outer-zone ring
template <bool SPLIT>
__device__ __forceinline__ void b_damping(const KParams &P, int bx, int by)
{
    const int n_inner = (P.damp_ids[0] > P.damp_ids[1] ? P.damp_ids[0] : P.damp_ids[1]) + 1;
    const int ns = P.ns;
    const int j = bx * blockDim.x + threadIdx.x;
    const int y = wave_ring(0, by);
    if (j >= ns) return;
    const double dt = P.s->dt;
    int i;
    if (y < n_inner) {
        i = y;
    } else {
        // outer zone starts at the smaller of the scalar / vector limits
        const int o0 = P.damp_ids[2] < P.damp_ids[3] ? P.damp_ids[2] : P.damp_ids[3];
        i = o0 + (y - n_inner);
        if (i < n_inner || i > P.nr) return;  // a ring of both zones is the inner row's
    }
    const int F0[4] = {FCPT_VRAD0, FCPT_VAZI0, FCPT_SIGMA0, FCPT_ENERGY0};
    const int F[4] = {FCPT_VRAD, FCPT_VAZI, FCPT_SIGMA, FCPT_ENERGY};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool vector = q == 0;
        if (i >= (vector ? P.nr + 1 : P.nr) || !damped_ring(P, vector, i)) continue;
        const Fld<SPLIT> X = fld<SPLIT>(P, F[q]), X0 = fld<SPLIT>(P, F0[q]);
        X.set(i, j, damp_value(X(i, j), X0(i, j), damp_ring(P, vector, i, dt)));
    }
}
FCPT_ONE0(damping, 256)

// ghost rings: zero-gradient Sigma/E, reflecting / zero-gradient / outflow v_r,
// Keplerian v_phi (boundary_conditions.cpp:67-97 and the BC files it dispatches to)
// end of a sim::run iteration: time += dt and the monitor counter
// (simulation.cpp:244, 545-551); nothing else in the kernels that call it
// reads them.  A step whose caller waits for it writes the clock to the pinned
// mirror from here: a copy after the step costs 6 to 8 us.
__device__ __forceinline__ void advance_clock(const KParams &P, int advance_time)
{
    DevScalars *s = P.s;
    const double time_next_monitor = (s->n_monitor + 1) * P.monitor_timestep;
    s->time = s->time + s->dt;
    s->last_prev = s->last_dt;
    s->count_next = s->step_count + 1u;
    s->count_derived = s->step_count;
    if (advance_time == 2 && fabs(time_next_monitor - s->time) < 1e-6 * s->last_dt) s->n_monitor++;
    if (DevScalars *out = P.s_out) {
        out->dt = s->dt;
        out->time = s->time;
        out->last_dt = s->last_dt;
        out->cfl_dt = s->cfl_dt;
        out->n_monitor = s->n_monitor;
        out->error_flags = s->error_flags;
        out->step_count = s->step_count;
    }
}

// the inner / outer ghost rings of sector j (rows 2 and nr-2 are never
// written here, nr >= 8)
// the ghost values of v_r: rows 0 and 1 from v_r(2), rows nr and nr-1 from
// v_r(nr-2), and the Keplerian v_phi of a ghost ring
__device__ __forceinline__ void ghost_vr_inner(const KParams &P, double v2, double &v0, double &v1)
{
    if (P.bc_inner == FCPT_BC_REFLECTING) {
        v0 = -v2;
        v1 = 0;
    } else if (P.bc_inner == FCPT_BC_ZEROGRADIENT) {
        v0 = v2;
        v1 = v2;
    } else {
        v0 = v1 = v2 > 0.0 ? 0.0 : v2;
    }
}
__device__ __forceinline__ void ghost_vr_outer(const KParams &P, double vn2, double &vn, double &vn1)
{
    if (P.bc_outer == FCPT_BC_REFLECTING) {
        vn = -vn2;
        vn1 = 0;
    } else if (P.bc_outer == FCPT_BC_ZEROGRADIENT) {
        vn = vn2;
        vn1 = vn2;
    } else {
        vn = vn1 = vn2 < 0.0 ? 0.0 : vn2;
    }
}
__device__ __forceinline__ double ghost_vaz(const KParams &P, int r)
{
    const double vk = sqrt(P.G * P.mstar / cst(P.Rmed)[r]);
    return 1.0 * vk - cst(P.Rmed)[r] * P.omega_frame;
}

template <bool SPLIT>
__device__ __forceinline__ void ghost_inner(const KParams &P, int j)
{
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const double s1 = S(1, j), e1 = E(1, j), v2 = vr(2, j);
    S.set(0, j, s1);
    E.set(0, j, e1);
    double v0, v1;
    ghost_vr_inner(P, v2, v0, v1);
    vr.set(0, j, v0);
    vr.set(1, j, v1);
    vaz.set(0, j, ghost_vaz(P, 0));
}

template <bool SPLIT>
__device__ __forceinline__ void ghost_outer(const KParams &P, int j)
{
    const int nr = P.nr;
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const double s2 = S(nr - 2, j), e2 = E(nr - 2, j), vn2 = vr(nr - 2, j);
    S.set(nr - 1, j, s2);
    E.set(nr - 1, j, e2);
    double vn, vn1;
    ghost_vr_outer(P, vn2, vn, vn1);
    vr.set(nr, j, vn);
    vr.set(nr - 1, j, vn1);
    vaz.set(nr - 1, j, ghost_vaz(P, nr - 1));
}

template <bool SPLIT>
__device__ __forceinline__ void b_ghost_bc(const KParams &P, int bx, int by, int advance_time)
{
    const int j = bx * blockDim.x + threadIdx.x;
    if (advance_time && j == 0) advance_clock(P, advance_time);
    if (j >= P.ns) return;
    ghost_inner<SPLIT>(P, j);
    ghost_outer<SPLIT>(P, j);
}
FCPT_ONE1(ghost_bc, 256, int, advance_time)

// the boundary call before the transport (ghost rings, b_ghost_bc) and the
// transport's ring mean with the FARGO shift (b_ring_mean, mode 1) in one
// launch: the first blocks set the ghost rings (one thread per sector), the
// other blocks (one of 256 threads per ring) form the ring means.  The ghost
// rings' v_phi is one Keplerian value per ring, so their blocks sum that value
// as stored in place of a load (the same sums, the same tree) and no block
// reads what another writes.  Only the sweeps read the ring means.
template <bool SPLIT>
__device__ __forceinline__ void b_ghost_ring_mean(const KParams &P, int bx)
{
    const int ghost_blocks = (P.ns + 255) / 256;
    if (bx < ghost_blocks) {
        const int j = bx * 256 + (int)threadIdx.x;
        if (j < P.ns) {
            ghost_inner<SPLIT>(P, j);
            ghost_outer<SPLIT>(P, j);
        }
        return;
    }
    const int i = bx - ghost_blocks;
    if (i == 0 || i == P.nr - 1) {
        __shared__ double2 sh[256];
        // the ghost ring's v_phi as stored by ghost_inner / ghost_outer in
        // this launch (split storage with stochastic rounding: per sector)
        const Fld<SPLIT> vaz = fld<SPLIT>(P, FCPT_VAZI);
        const double g = ghost_vaz(P, i);
        const MeanConst c = mean_const(P, i);
        double acc = 0.0, aacc = 0.0;
        for (int j = (int)threadIdx.x; j < P.ns; j += 256) {
            const double gj = vaz.stored(i, j, g);
            acc += gj;
            aacc += fabs(gj);
        }
        const double2 r = block_sum_abs(acc, aacc, sh);
        ring_mean_store(P, i, r.x, r.y, 1, c, [&]() {
            double seq = 0.0;
            for (int j = 0; j < P.ns; ++j) seq += vaz.stored(i, j, g);
            return seq;
        });
        return;
    }
    b_ring_mean<SPLIT>(P, i, 0, 1);
}
template <bool SPLIT>
__global__ void __launch_bounds__(256) k_ghost_ring_mean(KParams P)
{
    b_ghost_ring_mean<SPLIT>(P, (int)blockIdx.x);
}
template <bool SPLIT>
__global__ void __launch_bounds__(256) kb_ghost_ring_mean(const KParams *Ps, const BatchEntry *map)
{
    const BatchEntry e = batch_entry(map);
    b_ghost_ring_mean<SPLIT>(batch_disk(Ps, e.disk), (int)(e.yx & 0xffffu));
}

// the final boundary call's ghost rings (b_ghost_bc, after the damping) and
// recalculate_derived_disk_quantities in one pass: a ghost-ring cell first
// takes its neighbour ring's values, then forms its derived fields from what
// it stored, exactly as the two separate kernels would
template <bool SPLIT>
__device__ __forceinline__ void b_final_derived(const KParams &P, int bx, int by, int advance_time)
{
    CELL_LOOP_HEAD(0, P.nr)
    if (advance_time && i == 0 && j == 0) advance_clock(P, advance_time);
    if (i == 0) ghost_inner<SPLIT>(P, j);
    if (i == P.nr - 1) ghost_outer<SPLIT>(P, j);
    derived_store<SPLIT>(P, i, j, derived_load<SPLIT>(P, i, j, true), true, true);
}
FCPT_ONE1(final_derived, 256, int, advance_time)

// The end of the fused LeapFrog step in one launch: the second kick's
// velocities and E, in the partner buffers of view P, damped into the fields
// with Sigma, then the ghost rings, the clock and the derived fields: what
// copying them back, b_damping and b_final_derived do (three launches, 18 us
// of a 307 x 1021 step; this one 10).  One thread per cell of the active rings;
// a ghost ring's cells are written by the thread of the ring they copy, so
// that no thread reads what another writes.
template <bool SPLIT>
__device__ __forceinline__ void b_final_leapfrog(const KParams &P, int bx, int by, int advance_time)
{
    CELL_LOOP_HEAD(1, P.nr - 1)
    using T = typename Fld<SPLIT>::T;
    const int nr = P.nr;
    const double dt = P.s->dt;
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const Fld<SPLIT> vr_s = alt_vr<SPLIT>(P), vaz_s = alt_vaz<SPLIT>(P);
    const Fld<SPLIT> E_s = P.adiabatic ? buf<SPLIT>(P, P.ealt, P.bg[FCPT_ENERGY]) : E;
    // the stored form of (r, j) of a field after the damping
    const int rv = i == 1 ? 2 : i;  // v_r(1) is a ghost value, from v_r(2)
    const bool zs = damped_ring(P, false, i), zv = damped_ring(P, true, rv);
    T s = S.raw(i, j), e = E_s.raw(i, j), va = vaz_s.raw(i, j), v = vr_s.raw(rv, j);
    if (zs) {
        const double s0 = fld<SPLIT>(P, FCPT_SIGMA0)(i, j), e0 = fld<SPLIT>(P, FCPT_ENERGY0)(i, j);
        const double va0 = fld<SPLIT>(P, FCPT_VAZI0)(i, j);
        const Damp f = damp_ring(P, false, i, dt);
        s = S.enc(i, j, damp_value(S.dec(i, s), s0, f));
        e = E.enc(i, j, damp_value(E.dec(i, e), e0, f));
        va = vaz.enc(i, j, damp_value(vaz.dec(i, va), va0, f));
    }
    if (zv) v = vr.enc(rv, j, damp_value(vr.dec(rv, v), fld<SPLIT>(P, FCPT_VRAD0)(rv, j), damp_ring(P, true, rv, dt)));
    S.set_raw(i, j, s);
    E.set_raw(i, j, e);
    vaz.set_raw(i, j, va);
    const double sv = S.dec(i, s), ev = E.dec(i, e);
    derived_store<SPLIT>(P, i, j, DerivedIn{ev, sv, 0.0, 0.0}, false, false);
    double v0, v1;
    if (i == 1) {
        ghost_vr_inner(P, vr.dec(2, v), v0, v1);
        vr.set(0, j, v0);
        vr.set(1, j, v1);
    } else {
        vr.set_raw(i, j, v);
    }
    if (i == nr - 2) {
        ghost_vr_outer(P, vr.dec(i, v), v0, v1);
        vr.set(nr, j, v0);
        vr.set(nr - 1, j, v1);
    }
    if (i == 1 || i == nr - 2) {
        const int g = i == 1 ? 0 : nr - 1;  // the ghost ring
        const double sg = S.set_get(g, j, sv), eg = E.set_get(g, j, ev);
        vaz.set(g, j, ghost_vaz(P, g));
        derived_store<SPLIT>(P, g, j, DerivedIn{eg, sg, 0.0, 0.0}, false, false);
    }
    if (advance_time && i == 1 && j == 0) advance_clock(P, advance_time);
}
FCPT_ONE1(final_leapfrog, 256, int, advance_time)

// ---------------------------------------------------------------------------
// Transport

// The ring's stored values, loaded a ring ahead of their use so that the
// loads are in flight while the previous ring is processed.  Loads go to a
// clamped ring and the results are selected, so the loop body has no branch.
template <bool SPLIT, bool ADI>
struct RingRaw {
    using T = typename Fld<SPLIT>::T;
    T sig, va, vaj, e, v0, v1;
    int r;
};

template <bool SPLIT, bool ADI>
__device__ __forceinline__ void raw_ring(const KParams &P, int r, int j, int jn, RingRaw<SPLIT, ADI> &X)
{
    const bool in = r >= 0 && r < P.nr;
    const int rc = in ? r : 0;
    const int rv = r < 0 ? 0 : (r > P.nr ? P.nr : r);
    const int rv1 = rv < P.nr ? rv + 1 : P.nr;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    X.r = r;
    X.sig = fld<SPLIT>(P, FCPT_SIGMA).raw(rc, j);
    X.va = vaz.raw(rc, j);
    X.vaj = vaz.raw(rc, jn);
    if constexpr (ADI) X.e = fld<SPLIT>(P, FCPT_ENERGY).raw(rc, j);
    X.v0 = vr.raw(rv, j);
    X.v1 = vr.raw(rv1, j);
}

// ---------------------------------------------------------------------------
// Both sweeps of the transport as one walk: OneWindRad and VanLeerRadial
// (TransportEuler.cpp:138-168, 545-619), then OneWindTheta (:270-289) with
// QuantitiesAdvection of the residual velocity v - <v> and of the ring's
// uniform residual (:292-304, VanLeerTheta :630-664) and AdvectSHIFT (:238-268).
// A wavefront owns 57 sectors (64 with the halo) and walks `tile` rings
// outward, a sector per lane.  Its window holds the rings k-1 and k with their
// slopes and ring k+1: each ring is loaded once, each slope and each interface
// flux formed once.  Ring k-1, once updated by its two radial fluxes, goes
// through both azimuthal passes in registers, a sector's neighbours being the
// adjacent lanes (DPP moves), and is written to its shifted place.
// Why one kernel: two kernels wrote the radially swept Sigma, E and momenta and
// read them back (96 of 176 bytes per cell).  Those bytes bound them on large
// grids (4.7 and 4.3 TB/s), and a launch bounds them on small ones; this walk
// is bound by FP64 instructions (three wavefronts per SIMD).  Step times with
// two kernels and now: 128x384 isothermal 36.5 -> 29.6 us, 307x1021 beta 80.0
// -> 69.8, 1024x3072 adiabatic 345.7 -> 306, 2048x6144 isothermal 877 -> 769,
// 4096x12288 beta 5034 -> 4550, split 4052 -> 3731.
// Rings at and beyond the edges take branches of their own: a select per value
// on every ring was 6 % of the instructions (2048x6144 split 697 -> 684 us per
// step).  Prefetching the ring constants an iteration ahead costs scalar
// registers (2 to 4 % slower), the loop unrolled by three so that the window
// needs no copies vector ones (4096x12288 FP64 4390 -> 4882 us).
__device__ __forceinline__ double sweep_tab(const KParams &P, int t, int i)
{
    return cst(P.sweep_tab)[i * kSweepTabs + t];
}

// half the van Leer limiter of the differences a and b: a b / (a + b) where
// they have one sign, else zero.  FINE: both below 2^500 in magnitude, so the
// quotient by the refined reciprocal is the IEEE one (of products below
// 2^-900 but for its last place)
template <bool SPLIT, bool FINE>
__device__ __forceinline__ double vl_half(double a, double b)
{
    if constexpr (SPLIT || !FINE) {
        return 0.5 * vl_lim<SPLIT>(a, b);
    } else {
        const double p = a * b;
        const double q = quot_fast(p, shared_den(a + b));
        return p > 0.0 ? q : 0.0;
    }
}
// magnitude below 2^400 (false for NaN)
__device__ __forceinline__ bool sweep_range(double x) { return fabs(x) < 0x1p400; }

// One ring of the walk's window: Sigma, v_phi, NQ advected quantities, their
// specific values, v_r at the inner interface and the half slopes.  The
// momenta are formed with the expressions of compute_momenta_from_velocities
// (TransportEuler.cpp:471-495).  Rings outside the grid hold Sigma = 1 and
// zero quantities; the reference's interface values never reach them.  The
// density's own specific value Sigma / Sigma is exactly 1 for the positive
// Sigma the floor guarantees, so its interface value is 1 on interior
// interfaces and 0 on the two edge interfaces.
template <int NQ>
struct SweepRing {
    double s, va, v, ds;
    double w[NQ], q[NQ], dw[NQ];
    bool fine;  // of the whole wavefront: Sigma and the specific values are in the fast quotients' range
};

// quantities Q0 .. Q0 + NQ - 1 of (four momenta, E)
template <bool SPLIT, bool ADI, int Q0, int NQ>
__device__ __forceinline__ void sweep_decode(const KParams &P, const RingRaw<SPLIT, ADI> &X, SweepRing<NQ> &R)
{
    const int r = X.r;
    const bool in = r >= 0 && r < P.nr;
    const int rc = in ? r : 0;
    const int rv = r < 0 ? 0 : (r > P.nr ? P.nr : r);
    const int rv1 = rv < P.nr ? rv + 1 : P.nr;
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const double sig = fld<SPLIT>(P, FCPT_SIGMA).dec(rc, X.sig);
    const double rr = sweep_tab(P, SW_RMED, rc);
    const double OmegaF = P.omega_frame;
    const double v0 = vr.dec(rv, X.v0);  // v_r(r), r inside the grid or r == nr
    R.va = vaz.dec(rc, X.va);
    double all[5];
    all[0] = sig * vr.dec(rv1, X.v1);    // v_r(r + 1) for r inside the grid
    all[1] = sig * v0;
    all[2] = sig * (vaz.dec(rc, X.vaj) + rr * OmegaF) * rr;
    all[3] = sig * (R.va + rr * OmegaF) * rr;
    if constexpr (ADI) all[4] = fld<SPLIT>(P, FCPT_ENERGY).dec(rc, X.e);
    R.v = v0;
    R.s = sig;
    const double *q = all + Q0;
    double w[NQ];
    R.fine = true;
    if constexpr (SPLIT) {
        const double inv_sig = recip<true>(sig);
#pragma unroll
        for (int k = 0; k < NQ; ++k) w[k] = q[k] * inv_sig;
    } else {
        const SharedDen D = shared_den(sig);
        bool ok = quot_range(sig);
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            w[k] = quot_fast(q[k], D);
            ok = ok && sweep_range(w[k]);
        }
        R.fine = __all(ok);
        if (!R.fine) {
            __builtin_amdgcn_s_sleep(0);  // a branch: the divisions are not formed and selected
#pragma unroll
            for (int k = 0; k < NQ; ++k) w[k] = q[k] / sig;
        }
    }
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        R.q[k] = q[k];
        R.w[k] = w[k];
    }
    if (!in) {
        __builtin_amdgcn_s_sleep(0);  // a branch: selects on every ring are 6 % of the walk's instructions
        R.s = 1.0;
        if (r != P.nr) R.v = 0.0;
#pragma unroll
        for (int k = 0; k < NQ; ++k) R.q[k] = R.w[k] = 0.0;
    }
}

// half the van Leer slopes of ring k from rings k-1, k, k+1
// (compute_star_radial first loop, TransportEuler.cpp:355-371); zero on the ghost rings
template <bool SPLIT, bool FINE, int NQ>
__device__ __forceinline__ void sweep_slopes_of(double im, double ip, const SweepRing<NQ> &M,
                                                SweepRing<NQ> &C, const SweepRing<NQ> &N)
{
    C.ds = vl_half<SPLIT, FINE>((N.s - C.s) * ip, (C.s - M.s) * im);
#pragma unroll
    for (int q = 0; q < NQ; ++q) C.dw[q] = vl_half<SPLIT, FINE>((N.w[q] - C.w[q]) * ip, (C.w[q] - M.w[q]) * im);
}
template <bool SPLIT, int NQ>
__device__ __forceinline__ void sweep_slopes(const KParams &P, int k, const SweepRing<NQ> &M, SweepRing<NQ> &C,
                                             const SweepRing<NQ> &N)
{
    const bool act = k > 0 && k < P.nr - 1;
    const int kc = act ? k : 1;
    const double im = sweep_tab(P, SW_INV_DIFF_RMED, kc), ip = sweep_tab(P, SW_INV_DIFF_RMED, kc + 1);
    if (SPLIT || (M.fine && C.fine && N.fine)) {
        sweep_slopes_of<SPLIT, true, NQ>(im, ip, M, C, N);
    } else {
        __builtin_amdgcn_s_sleep(0);
        sweep_slopes_of<SPLIT, false, NQ>(im, ip, M, C, N);
    }
    if (!act) {
        __builtin_amdgcn_s_sleep(0);
        C.ds = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) C.dw[q] = 0.0;
    }
}

// Upwind interface values at interface k between ring A = k-1 and ring B = k
// (compute_star_radial second loop, TransportEuler.cpp:376-405; zero on the
// edge interfaces k = 0 and k = nr) and the flux dt dphi Rinf[k] Q* Sigma* v_r
// of each quantity through it (VanLeerRadial, :545-619).  The reference's
// varq_sup of ring k-1 and varq_inf of ring k are this same product, Rsup[k-1]
// and Rinf[k] being the same radius.  The slopes are halved, so the distances
// are not.
template <int NQ>
__device__ __forceinline__ void sweep_flux(const KParams &P, int k, const SweepRing<NQ> &A, const SweepRing<NQ> &B,
                                           double dt, double *f, double &fs)
{
    const bool act = k > 0 && k < P.nr;
    const int kc = act ? k : 1;
    const double v = B.v;
    const double fpos = sweep_tab(P, SW_RMED, kc) - sweep_tab(P, SW_RMED, kc - 1) - v * dt;
    const double fneg = sweep_tab(P, SW_RMED, kc + 1) - sweep_tab(P, SW_RMED, kc) + v * dt;
    const bool up = v > 0.0;
    const double ds = up ? A.s + fpos * A.ds : B.s - fneg * B.ds;
    const double c = dt * P.dphi * sweep_tab(P, SW_RINF, k);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double qs = up ? A.w[q] + fpos * A.dw[q] : B.w[q] - fneg * B.dw[q];
        f[q] = c * qs * ds * v;
    }
    fs = c * ds * v;
    if (!act) {
        __builtin_amdgcn_s_sleep(0);
        fs = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q) f[q] = 0.0;
    }
}

// Both FARGO passes, with the residual and with the uniform velocity
// (TransportEuler.cpp:292-304, 630-664), for this lane's sector of one ring, the
// neighbour sectors in the adjacent lanes: s0, q0 the radially swept density
// and quantities, v0 = v_phi - <v_phi>; s2, q2 the results.  The second pass
// has one velocity vu, so each sector's interface value on its downstream
// side is formed where its slope is, and only the flux moves between lanes.
// Returns whether the quotients were in the fast form's range.
template <bool SPLIT, bool FINE, bool UP, int NQ>
__device__ __forceinline__ bool sweep_theta(double dt, double v0, double vu, double dxtheta, double invdx,
                                            double dxrad, double invsurf, double s0, const double *q0, double &s2,
                                            double *q2)
{
    auto slope = [&](double x) {
        const double b = x - from_left(x);
        return vl_half<SPLIT, FINE>(from_right(b), b) * invdx;
    };
    const double ks0 = v0 * dt, ksu = vu * dt;
    const double lo_d = dxtheta - ks0, hi_d = dxtheta + ks0;
    const bool up0 = ks0 > 0.0;
    auto star0 = [&](double x) {  // the first pass's value at the interface to the left
        const double d = slope(x);
        const double lo = from_left(x) + lo_d * from_left(d), hi = x - hi_d * d;
        return up0 ? lo : hi;
    };
    auto star1 = [&](double x) {  // the second pass's value at the downstream interface
        const double d = slope(x);
        return UP ? x + (dxtheta - ksu) * d : x - (dxtheta + ksu) * d;
    };
    auto div1 = [&](double F) { return UP ? from_left(F) - F : F - from_right(F); };
    bool ok = true;
    const double ds0 = star0(s0);
    const double f0 = dxrad * ds0 * v0;
    const double s1 = s0 + (f0 - from_right(f0)) * invsurf;
    const double ds1 = star1(s1);
    s2 = s1 + div1(dxrad * ds1 * vu) * invsurf;
    const SharedDen D0 = SPLIT ? SharedDen{s0, recip<true>(s0), true} : shared_den(s0);
    const SharedDen D1 = SPLIT ? SharedDen{s1, recip<true>(s1), true} : shared_den(s1);
    if (!SPLIT) ok = quot_range(s0) && quot_range(s1);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double w0 = SPLIT ? q0[q] * D0.r : FINE ? quot_fast(q0[q], D0) : q0[q] / s0;
        const double fq = dxrad * star0(w0) * ds0 * v0;
        const double q1 = q0[q] + (fq - from_right(fq)) * invsurf;
        const double w1 = SPLIT ? q1 * D1.r : FINE ? quot_fast(q1, D1) : q1 / s1;
        q2[q] = q1 + div1(dxrad * star1(w1) * ds1 * vu) * invsurf;
        if (!SPLIT) ok = ok && sweep_range(w0) && sweep_range(w1);
    }
    return ok;
}

constexpr int kSweepSegW = 57;  // sectors written per wavefront

template <bool SPLIT, bool ADI, int Q0, int NQ>
__device__ __forceinline__ void b_sweeps(const KParams &P, int bx, int by, int tile)
{
    const int ns = P.ns, nr = P.nr;
    const int lane = (int)threadIdx.x;
    const int j0 = bx * kSweepSegW;
    const int i0 = by * tile;
    if (j0 >= ns || i0 >= nr) return;
    const int Ls = ns - j0 < kSweepSegW ? ns - j0 : kSweepSegW;
    int j = (j0 - 4 + lane) % ns;
    if (j < 0) j += ns;
    const int jn = j == ns - 1 ? 0 : j + 1;
    const double dt = *cst(&P.s->dt);
    SweepRing<NQ> A, B, C, D;
    {
        RingRaw<SPLIT, ADI> X0, X1, X2, X3;
        raw_ring<SPLIT, ADI>(P, i0 - 2, j, jn, X0);
        raw_ring<SPLIT, ADI>(P, i0 - 1, j, jn, X1);
        raw_ring<SPLIT, ADI>(P, i0, j, jn, X2);
        raw_ring<SPLIT, ADI>(P, i0 + 1, j, jn, X3);
        sweep_decode<SPLIT, ADI, Q0, NQ>(P, X0, D);
        sweep_decode<SPLIT, ADI, Q0, NQ>(P, X1, A);
        sweep_decode<SPLIT, ADI, Q0, NQ>(P, X2, B);
        sweep_decode<SPLIT, ADI, Q0, NQ>(P, X3, C);
    }
    sweep_slopes<SPLIT, NQ>(P, i0 - 1, D, A, B);
    sweep_slopes<SPLIT, NQ>(P, i0, A, B, C);
    double f_prev[NQ], fs_prev;
    sweep_flux<NQ>(P, i0, A, B, dt, f_prev, fs_prev);
    const int iend = i0 + tile < nr ? i0 + tile : nr;
    RingRaw<SPLIT, ADI> X;
    raw_ring<SPLIT, ADI>(P, i0 + 2, j, jn, X);
    const Fld<false> Sc = buf<false>(P, P.sig_c, nullptr), Ec = buf<false>(P, P.en_c, nullptr);
    for (int k = i0 + 1; k <= iend; ++k) {
        sweep_decode<SPLIT, ADI, Q0, NQ>(P, X, D);     // ring k+1
        raw_ring<SPLIT, ADI>(P, k + 2, j, jn, X);  // in flight during this iteration
        sweep_slopes<SPLIT, NQ>(P, k, B, C, D);    // ring k
        A = B;
        B = C;
        C = D;
        double f[NQ], fs;
        sweep_flux<NQ>(P, k, A, B, dt, f, fs);
        // ring k-1 lies between interfaces k-1 and k
        const int i = k - 1;
        const double invs = sweep_tab(P, SW_INV_SURF, i);
        double q0[NQ], q2[NQ], s2;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            q0[q] = A.q[q] + (f_prev[q] - f[q]) * invs;
            if (SPLIT && Q0 + q < 4)
                q0[q] = buf<SPLIT>(P, nullptr, P.bgm[Q0 + q], kBufMom + Q0 + q).stored(i, j, q0[q]);
            f_prev[q] = f[q];
        }
        const double s0 = A.s + (fs_prev - fs) * invs;
        fs_prev = fs;
        const double v0 = A.va - cst(P.vmean)[i], vu = cst(P.vuni)[i];
        const double dxtheta = sweep_tab(P, SW_DXTHETA, i), invdx = sweep_tab(P, SW_INV_DXTHETA, i);
        const double dxrad = sweep_tab(P, SW_WIDTH, i) * dt;
        const bool up = vu * dt > 0.0;
        bool ok = up ? sweep_theta<SPLIT, true, true, NQ>(dt, v0, vu, dxtheta, invdx, dxrad, invs, s0, q0, s2, q2)
                     : sweep_theta<SPLIT, true, false, NQ>(dt, v0, vu, dxtheta, invdx, dxrad, invs, s0, q0, s2, q2);
        // lanes 0, 1, 62 and 63 hold no exact second pass and no result depends on it
        if (!SPLIT && !__all(ok || lane < 2 || lane > 61)) {
            __builtin_amdgcn_s_sleep(0);
            if (up) sweep_theta<SPLIT, false, true, NQ>(dt, v0, vu, dxtheta, invdx, dxrad, invs, s0, q0, s2, q2);
            else sweep_theta<SPLIT, false, false, NQ>(dt, v0, vu, dxtheta, invdx, dxrad, invs, s0, q0, s2, q2);
        }
        // the upstream side loses four lanes, the downstream one three
        const int k0 = lane - (up ? 4 : 3);
        int nsh = cst(P.nshift)[i];
        if (nsh >= ns || nsh <= -ns) nsh %= ns;
        int jd = j + nsh;
        if (jd >= ns) jd -= ns;
        if (jd < 0) jd += ns;
        if (k0 >= 0 && k0 < Ls) {
            if (Q0 == 0) Sc.set(i, jd, s2);
#pragma unroll
            for (int q = 0; q < NQ; ++q) (Q0 + q < 4 ? mom_out(P, Q0 + q) : Ec).set(i, jd, q2[q]);
        }
    }
}
template <bool SPLIT, bool ADI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) k_sweeps(KParams P, int tile)
{
    const BlockXY bb = xcd_block();
    b_sweeps<SPLIT, ADI, 0, ADI ? 5 : 4>(P, bb.x, bb.y, tile);
}
template <bool SPLIT, bool ADI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) kb_sweeps(const KParams *Ps, const BatchEntry *map)
{
    const BatchEntry e = batch_entry(map);
    const KParams &P = batch_disk(Ps, e.disk);
    b_sweeps<SPLIT, ADI, 0, ADI ? 5 : 4>(P, (int)(e.yx & 0xffffu), (int)(e.yx >> 16), P.radial_tile);
}
// one quantity per block (the grid's z; the first one's blocks also write Sigma)
template <bool SPLIT, bool ADI>
__global__ void __launch_bounds__(64) k_sweeps_each(KParams P, int tile)
{
    const int bx = (int)blockIdx.x, by = (int)blockIdx.y;
    switch (blockIdx.z) {
    case 0: b_sweeps<SPLIT, ADI, 0, 1>(P, bx, by, tile); break;
    case 1: b_sweeps<SPLIT, ADI, 1, 1>(P, bx, by, tile); break;
    case 2: b_sweeps<SPLIT, ADI, 2, 1>(P, bx, by, tile); break;
    case 3: b_sweeps<SPLIT, ADI, 3, 1>(P, bx, by, tile); break;
    default:
        if constexpr (ADI) b_sweeps<SPLIT, ADI, 4, 1>(P, bx, by, tile);
    }
}

// compute_velocities_from_momenta (TransportEuler.cpp:498-535), then
// assure_minimum_value(Sigma) (SourceEuler.cpp:102-131) and, adiabatic,
// SetTemperatureFloorCeilValues (TransportEuler.cpp:127-131)
template <bool SPLIT>
__device__ __forceinline__ void b_velocities(const KParams &P, int bx, int by)
{
    CELL_LOOP_HEAD(0, P.nr)
    const Fld<false> Sb = buf<false>(P, P.sig_c, nullptr);
    const Fld<false> m0 = mom_out(P, 0);
    const Fld<false> m1 = mom_out(P, 1);
    const Fld<false> m2 = mom_out(P, 2);
    const Fld<false> m3 = mom_out(P, 3);
    const Fld<false> Eb = buf<false>(P, P.en_c, nullptr);
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    const int jm = j == 0 ? ns - 1 : j - 1;
    const int im = i >= 1 ? i - 1 : 0;
    const double s0 = Sb(i, j), sm = Sb(im, j), sjm = Sb(i, jm);
    const double m0v = m0(im, j), m1v = m1(i, j), m2v = m2(i, jm), m3v = m3(i, j);
    const double e = P.adiabatic ? Eb(i, j) : 0.0;
    if (i == 0) {
        vr.set(i, j, 0.0);
    } else {
        vr.set(i, j, (m0v + m1v) / (sm + s0));
    }
    vaz.set(i, j, (m2v + m3v) / (sjm + s0) * cst(P.InvRmed)[i] - cst(P.Rmed)[i] * P.omega_frame);
    const double floor_value = P.sigma_floor * P.sigma0;
    double sig = s0;
    if (sig < floor_value) sig = floor_value;
    fld<SPLIT>(P, FCPT_SIGMA).set(i, j, sig);
    if (P.adiabatic) fld<SPLIT>(P, FCPT_ENERGY).set(i, j, temperature_floor<SPLIT>(P, e, sig));
}
FCPT_ONE0(velocities, 256)

// The end of the fused Euler step in one launch: the velocity kernel, the
// final boundary call (damping, ghost rings, the clock) and
// recalculate_derived_disk_quantities.  A thread owns one cell of an active
// ring: it forms the velocities, Sigma and E as the velocity kernel and the
// damping store them, and the derived fields from the stored values, as
// k_final_derived reads them.  Every load is issued before the first use (the
// damping references behind wave-uniform tests), so a wavefront waits once
// and not at each damping branch.  The cells of a ghost ring are written by
// the thread of the ring they copy, and v_r(1), a ghost value from v_r(2), by
// that of ring 1: no thread reads what another writes.
// Large grids are bound by bytes (88 per cell, adiabatic FP64), small ones by
// the load latency.  Several rings per thread share the density and the
// outward momentum of the ring inside, but lose more to fewer wavefronts:
// 128x384 isothermal 36.7 us/step with one, 37.7 with two, 39.9 with four;
// 2048x6144 split 1068, 1084, 1089; 4096x12288 FP64 5121, 5129, 5127.  With
// the loads behind the branches and per-cell damping ramps the steps took
// 37.7, 1141 and 5221 us.
template <bool SPLIT>
__device__ __forceinline__ void b_velocities_final(const KParams &P, int bx, int by, int advance_time)
{
    CELL_LOOP_HEAD(1, P.nr - 1)
    const int nr = P.nr;
    const int jm = j == 0 ? ns - 1 : j - 1;
    const double dt = *cst(&P.s->dt);
    const Fld<false> Sb = buf<false>(P, P.sig_c, nullptr), Eb = buf<false>(P, P.en_c, nullptr);
    const Fld<false> m0 = mom_out(P, 0), m1 = mom_out(P, 1), m2 = mom_out(P, 2), m3 = mom_out(P, 3);
    FLD(vr, FCPT_VRAD);
    FLD(vaz, FCPT_VAZI);
    FLD(S, FCPT_SIGMA);
    FLD(E, FCPT_ENERGY);
    // v_r between rings r - 1 and r, as the velocity kernel and the damping
    // pass it to set()
    auto v_r = [&](int r, double p0, double p1, double sm, double s0, double x0) {
        const double v = SPLIT ? (p0 + p1) * recip<true>(sm + s0) : (p0 + p1) / (sm + s0);
        return damped_ring(P, true, r) ? damp_value(vr.stored(r, j, v), x0, damp_ring(P, true, r, dt)) : v;
    };
    auto v_r0 = [&](int r) { return damped_ring(P, true, r) ? fld<SPLIT>(P, FCPT_VRAD0)(r, j) : 0.0; };
    const bool z = damped_ring(P, false, i);
    const double sm = Sb(i - 1, j), s0 = Sb(i, j), sj = Sb(i, jm);
    const double p0 = m0(i - 1, j), p1 = m1(i, j), p2 = m2(i, jm), p3 = m3(i, j);
    const double e0 = P.adiabatic ? Eb(i, j) : 0.0;
    double x_s = 0.0, x_e = 0.0, x_va = 0.0;
    if (z) {
        x_s = fld<SPLIT>(P, FCPT_SIGMA0)(i, j);
        x_va = fld<SPLIT>(P, FCPT_VAZI0)(i, j);
        if (P.adiabatic) x_e = fld<SPLIT>(P, FCPT_ENERGY0)(i, j);
    }
    const double x_vr = v_r0(i);
    const bool ghost = i == 1 || i == nr - 2;
    // an isothermal disk's E is only copied to the ghost rings
    const double e_ghost = ghost && !P.adiabatic ? E(i, j) : 0.0;
    double v2 = 0.0;
    if (i == 1) v2 = vr.stored(2, j, v_r(2, m0(1, j), m1(2, j), s0, Sb(2, j), v_r0(2)));

    const double floor_value = P.sigma_floor * P.sigma0;
    double sig = s0;
    if (sig < floor_value) sig = floor_value;
    double en = P.adiabatic ? temperature_floor<SPLIT>(P, e0, sig) : 0.0;
    double va = (SPLIT ? (p2 + p3) * recip<true>(sj + s0) : (p2 + p3) / (sj + s0)) * cst(P.InvRmed)[i] -
                cst(P.Rmed)[i] * P.omega_frame;
    const double v = v_r(i, p0, p1, sm, s0, x_vr);
    if (z) {
        const Damp f = damp_ring(P, false, i, dt);
        sig = damp_value(S.stored(i, j, sig), x_s, f);
        if (P.adiabatic) en = damp_value(E.stored(i, j, en), x_e, f);
        va = damp_value(vaz.stored(i, j, va), x_va, f);
    }
    const double s_stored = S.set_get(i, j, sig);
    const double e_stored = P.adiabatic ? E.set_get(i, j, en) : e_ghost;
    vaz.set(i, j, va);
    double g0, g1;  // ghost values of v_r
    if (i == 1) {
        ghost_vr_inner(P, v2, g0, g1);
        vr.set(0, j, g0);
        vr.set(1, j, g1);
    } else {
        vr.set(i, j, v);
    }
    if (i == nr - 2) {
        ghost_vr_outer(P, vr.stored(i, j, v), g0, g1);
        vr.set(nr, j, g0);
        vr.set(nr - 1, j, g1);
    }
    auto derived = [&](int r, double e, double sv) {
        DerivedIn d{e, sv, 0.0, 0.0};
        if (!P.adiabatic) {
            d.cs = cst(P.iso_cs)[r];
            d.h = cst(P.iso_h)[r];
        }
        derived_store<SPLIT>(P, r, j, d, true, true);
    };
    derived(i, e_stored, s_stored);
    if (ghost) {
        const int g = i == 1 ? 0 : nr - 1;  // the ghost ring
        const double sg = S.set_get(g, j, s_stored), eg = E.set_get(g, j, e_stored);
        vaz.set(g, j, ghost_vaz(P, g));
        derived(g, eg, sg);
    }
    if (advance_time && i == 1 && j == 0) advance_clock(P, advance_time);
}
FCPT_PAIR1(velocities_final, 256, int, advance_time)

// ---------------------------------------------------------------------------
// totals with Neumaier compensation: per ring (sum, compensation) pairs, then
// one block folds the rings in order (quantities.cpp:51-78, 242-279)
__device__ __forceinline__ void neumaier_add(double &s, double &c, double x)
{
    const double t = s + x;
    c += fabs(s) >= fabs(x) ? (s - t) + x : (x - t) + s;
    s = t;
}

template <bool SPLIT>
__global__ void __launch_bounds__(64) k_totals_rings(KParams P, double radius, double *ring_out)
{
    const int ns = P.ns;
    const int i = blockIdx.x;  // ring
    const int t = threadIdx.x;
    double m = 0.0, mc = 0.0, l = 0.0, lc = 0.0;
    const bool active = i >= 1 && i < P.nr - 1 && cst(P.Rmed)[i] <= radius;
    if (active) {
        FLD(S, FCPT_SIGMA);
        FLD(vaz, FCPT_VAZI);
        for (int j = t; j < ns; j += 64) {
            const int jm = j == 0 ? ns - 1 : j - 1;
            const double s = S(i, j);
            neumaier_add(m, mc, cst(P.Surf)[i] * s);
            neumaier_add(l, lc, cst(P.Surf)[i] * 0.5 * (s + S(i, jm)) * cst(P.Rmed)[i] *
                                    (vaz(i, j) + P.omega_frame * cst(P.Rmed)[i]));
        }
    }
    __shared__ double sh[4][64];
    sh[0][t] = m;
    sh[1][t] = mc;
    sh[2][t] = l;
    sh[3][t] = lc;
    __syncthreads();
    if (t == 0) {
        double M = 0.0, MC = 0.0, L = 0.0, LC = 0.0;
        for (int k = 0; k < 64; ++k) {
            neumaier_add(M, MC, sh[0][k]);
            MC += sh[1][k];
            neumaier_add(L, LC, sh[2][k]);
            LC += sh[3][k];
        }
        ring_out[4 * i + 0] = M;
        ring_out[4 * i + 1] = MC;
        ring_out[4 * i + 2] = L;
        ring_out[4 * i + 3] = LC;
    }
}

__global__ void k_totals_final(KParams P, const double *ring_out, double *out2)
{
    double M = 0.0, MC = 0.0, L = 0.0, LC = 0.0;
    for (int i = 0; i < P.nr; ++i) {
        neumaier_add(M, MC, ring_out[4 * i + 0]);
        MC += ring_out[4 * i + 1];
        neumaier_add(L, LC, ring_out[4 * i + 2]);
        LC += ring_out[4 * i + 3];
    }
    out2[0] = M + MC;
    out2[1] = L + LC;
}

// streaming copy of four work arrays (bandwidth probe)
__global__ void __launch_bounds__(256) k_copy4(KParams P, size_t n8)
{
    // one 8-byte element of each of the four arrays per thread, every load
    // before the stores: the load and store forms of the step kernels (on
    // MI355X this form copies ~25 % faster than a grid-stride loop of 16-byte
    // elements)
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n8) return;
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = static_cast<const double *>(P.mom[q])[k];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        void *const to = q == 0 ? P.sig_c : q == 1 ? P.en_c : P.valt[q - 2];
        static_cast<double *>(to)[k] = v[q];
    }
}

// split storage: re-express a field's deviations about a new ring background
__global__ void __launch_bounds__(256) k_rebase(float *d, const double *oldbg, const double *newbg,
                                                int ns, int rows)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * blockDim.y + threadIdx.y));
    if (j >= ns || i >= rows) return;
    const size_t c = IX(i, j);
    d[c] = (float)((oldbg[i] + (double)d[c]) - newbg[i]);
}

// split storage: the ring means of a field, background + mean deviation (one
// block per row; the deviations summed in FP64, pairwise tree order)
__global__ void __launch_bounds__(256) k_split_ring_mean(const float *d, const double *bg, int ns,
                                                         double *out)
{
    __shared__ double sh[256];
    const int i = blockIdx.x;
    const float *row = d + (size_t)i * (size_t)ns;
    double acc = 0.0;
    strided_row<256>(ns, (int)threadIdx.x, [&](int j) { return (double)row[j]; }, [&](double x) { acc += x; });
    const double sum = block_sum(acc, sh);
    if (threadIdx.x == 0) out[i] = bg[i] + sum / ns;
}

// ---------------------------------------------------------------------------
// launch helpers: each dispatches on the storage mode

#define LAUNCH(kern, grid, block, st, ...)                                               \
    do {                                                                                 \
        if (P.split) hipLaunchKernelGGL(kern<true>, grid, block, 0, st, __VA_ARGS__);    \
        else hipLaunchKernelGGL(kern<false>, grid, block, 0, st, __VA_ARGS__);           \
    } while (0)

static inline dim3 cell_grid(const KParams &P, int rows)
{
    return dim3((unsigned)((P.ns + 63) / 64), (unsigned)((rows + 3) / 4));
}
static const dim3 kBlock(64, 4);

size_t element_size(const KParams &P) { return P.split ? sizeof(float) : sizeof(double); }
size_t field_element_size(const KParams &P, int field)
{
    return field == FCPT_POTENTIAL ? sizeof(double) : element_size(P);
}

void launch_ring_mean(const KParams &P, hipStream_t st, int mode)
{
    LAUNCH(k_ring_mean, dim3(P.nr), dim3(256), st, P, mode);
}

template <bool POT>
static void launch_cfl_ring(const KParams &P, hipStream_t st)
{
    const dim3 g((unsigned)P.nr), b(512);
    if (P.split) hipLaunchKernelGGL((k_cfl_ring<true, POT>), g, b, 0, st, P);
    else hipLaunchKernelGGL((k_cfl_ring<false, POT>), g, b, 0, st, P);
}
void launch_cfl(const KParams &P, hipStream_t st, int mode)
{
    launch_cfl_ring<false>(P, st);
    hipLaunchKernelGGL(k_cfl_fold, dim3(1), dim3(256), 0, st, P, mode);
}

void launch_cfl_potential(const KParams &P, hipStream_t st)
{
    launch_cfl_ring<true>(P, st);
}

void launch_cfl_cells(const KParams &P, hipStream_t st)
{
    launch_cfl_ring<false>(P, st);
}

void launch_set_dt(const KParams &P, hipStream_t st, double dt)
{
    hipLaunchKernelGGL(k_set_dt, dim3(1), dim3(1), 0, st, P, dt);
}
void launch_set_clock(const KParams &P, hipStream_t st, double t)
{
    hipLaunchKernelGGL(k_set_clock, dim3(1), dim3(1), 0, st, P, t);
}
void launch_set_time(const KParams &P, hipStream_t st, double t, double last_dt, int n_monitor)
{
    hipLaunchKernelGGL(k_set_time, dim3(1), dim3(1), 0, st, P, t, last_dt, n_monitor);
}
void launch_set_params(const KParams &P, hipStream_t st, const fcpt_step_params &sp,
                       const BodySmoothing &sm)
{
    hipLaunchKernelGGL(k_set_params, dim3(1), dim3(1), 0, st, P, sp, sm);
}
void launch_set_mid_params(const KParams &P, hipStream_t st, const fcpt_step_params &sp,
                           const BodySmoothing &sm)
{
    hipLaunchKernelGGL(k_set_mid_params, dim3(1), dim3(1), 0, st, P, sp, sm);
}
void launch_leapfrog_phase(const KParams &P, hipStream_t st, int phase)
{
    hipLaunchKernelGGL(k_leapfrog_phase, dim3(1), dim3(1), 0, st, P, phase);
}
void launch_pressure(const KParams &P, hipStream_t st) { LAUNCH(k_pressure, cell_grid(P, P.nr), kBlock, st, P); }

// a 2-D field whose rows are constant: row i = ring[i] (split storage: the
// deviation from bg[i])
template <bool SPLIT>
__global__ void __launch_bounds__(256) k_fill_rows(void *dst, const double *ring, const double *bg,
                                                   int ns, int rows)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = wave_ring(0, (int)blockIdx.y);
    if (j >= ns || i >= rows) return;
    const size_t c = (size_t)i * (size_t)ns + (size_t)j;
    if constexpr (SPLIT) static_cast<float *>(dst)[c] = (float)(ring[i] - bg[i]);
    else static_cast<double *>(dst)[c] = ring[i];
}

void launch_fill_rows(const KParams &P, hipStream_t st, void *dst, const double *ring,
                      const double *bg, int rows)
{
    const dim3 g((unsigned)((P.ns + 63) / 64), (unsigned)((rows + 3) / 4));
    if (P.split) hipLaunchKernelGGL(k_fill_rows<true>, g, kBlock, 0, st, dst, ring, bg, P.ns, rows);
    else hipLaunchKernelGGL(k_fill_rows<false>, g, kBlock, 0, st, dst, ring, bg, P.ns, rows);
}
// one block row of 64 x 4 threads per four rings, blockIdx.z the field
template <bool SPLIT>
__global__ void __launch_bounds__(256) k_export(KParams P, ExportFields x)
{
    const int j = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int i = wave_ring(0, (int)blockIdx.y), k = (int)blockIdx.z, f = x.field[k];
    if (j >= P.ns || i >= x.rows[k]) return;
    const double v = f == FCPT_POTENTIAL ? phi_fld(P)(i, j) : fld<SPLIT>(P, f)(i, j);
    x.out[k][(size_t)i * (size_t)P.ns + (size_t)j] = v;
}
void launch_export(const KParams &P, hipStream_t st, const ExportFields &x)
{
    const dim3 c = cell_grid(P, P.nr + 1);
    LAUNCH(k_export, dim3(c.x, c.y, (unsigned)x.n), kBlock, st, P, x);
}
void launch_copy_velocities(const KParams &P, hipStream_t st)
{
    LAUNCH(k_copy_velocities, cell_grid(P, P.nr + 1), kBlock, st, P);
}

void launch_potential(const KParams &P, hipStream_t st) { launch_potential_fold(P, st, -1); }

void launch_potential_fold(const KParams &P, hipStream_t st, int fold_mode)
{
    const dim3 g = cell_grid(P, P.nr);
    const unsigned gx = (unsigned)((P.ns + 64 * kPotCells - 1) / (64 * kPotCells));
    LAUNCH(k_potential_fold, dim3(gx, g.y + 1), kBlock, st, P, fold_mode);
}

void launch_sources(const KParams &P, hipStream_t st)
{
    LAUNCH(k_src_vr, cell_grid(P, P.nr - 3), kBlock, st, P);
    LAUNCH(k_src_vphi, cell_grid(P, P.nr - 2), kBlock, st, P);
    if (P.adiabatic) LAUNCH(k_src_energy, cell_grid(P, P.nr - 1), kBlock, st, P);
}

// returns true when the viscosity recalculation was folded in
bool launch_artificial_viscosity(const KParams &P, hipStream_t st, int with_viscosity)
{
    if (P.artvisc == FCPT_ARTVISC_TW) {
        LAUNCH(k_tw_q, cell_grid(P, P.nr), kBlock, st, P);
        LAUNCH(k_tw_vel, cell_grid(P, P.nr), kBlock, st, P, with_viscosity);
        return with_viscosity != 0;
    }
    if (P.artvisc == FCPT_ARTVISC_SN) {
        LAUNCH(k_sn_q, cell_grid(P, P.nr), kBlock, st, P);
        LAUNCH(k_sn_vel, cell_grid(P, P.nr), kBlock, st, P, with_viscosity);
        return with_viscosity != 0;
    }
    if (P.adiabatic && P.artvisc_dissipation) LAUNCH(k_temperature_floor, cell_grid(P, P.nr), kBlock, st, P);
    return false;
}

void launch_recalc_viscosity(const KParams &P, hipStream_t st)
{
    LAUNCH(k_recalc_viscosity, cell_grid(P, P.nr), kBlock, st, P);
}
void launch_stress(const KParams &P, hipStream_t st) { LAUNCH(k_stress, cell_grid(P, P.nr), kBlock, st, P); }
void launch_visc_update(const KParams &P, hipStream_t st)
{
    LAUNCH(k_visc_update, cell_grid(P, P.nr - 2), kBlock, st, P);
}
void launch_substep3(const KParams &P, hipStream_t st) { LAUNCH(k_substep3, cell_grid(P, P.nr), kBlock, st, P); }
void launch_heatcool_cfl(const KParams &P, hipStream_t st)
{
    LAUNCH(k_heatcool_cfl, cell_grid(P, P.nr), kBlock, st, P);
}

void launch_boundaries(const KParams &P, hipStream_t st, int final_call, int advance_time)
{
    if (final_call && P.damping) {
        const int n_inner = (P.damp_ids[0] > P.damp_ids[1] ? P.damp_ids[0] : P.damp_ids[1]) + 1;
        const int o0 = P.damp_ids[2] < P.damp_ids[3] ? P.damp_ids[2] : P.damp_ids[3];
        const int n_outer = P.nr + 1 - o0;
        LAUNCH(k_damping, cell_grid(P, n_inner + n_outer), kBlock, st, P);
    }
    LAUNCH(k_ghost_bc, dim3((unsigned)((P.ns + 255) / 256)), dim3(256), st, P, advance_time);
}

// Rings per walk of the transport's sweeps: a walk of t rings costs about
// t + 1.5 ring times (its window start), and a ring time with n wavefronts on a
// SIMD is 0.7 n + 1.2 us up to the three its registers allow, as latency is
// left over, and 1.1 n beyond; one disk's walks are alike, so n rounds up.
// Measured step times at 512x1536 (tiles 1, 3, 5, 8, 16): 116, 107, 103, 109,
// 120 us; at 1024x3072 (3, 8, 16, 19, 32): 316, 306, 318, 303, 325; at
// 4096x12288 (8, 16, 32, 48): 4646, 4567, 4550, 4623.  A batch's walks end at
// different times, so one full round leaves SIMDs idle and n gets one more
// instead: the sweeps of 16 disks of 128 to 512 rings (4, 8, 12, 16, 32): 188,
// 171, 174, 177, 206.
template <class Waves>
static int sweep_best_tile(Waves &&waves, bool batch)
{
    int best = 1;
    double best_cost = 1e300;
    for (int t = 1; t <= 32; ++t) {
        const double w = (double)waves(t) / 1024.0, n = std::ceil(w);
        const double ring = batch ? std::max(1.9, 1.1 * (w + 1.0)) : n <= 3.0 ? 0.7 * n + 1.2 : 1.1 * n;
        if ((t + 1.5) * ring < best_cost) {
            best_cost = (t + 1.5) * ring;
            best = t;
        }
    }
    return best;
}
static long sweep_waves(const KParams &P, int tile)
{
    return (long)((P.ns + kSweepSegW - 1) / kSweepSegW) * ((P.nr + tile - 1) / tile);
}
int resolve_sweep_tile(const KParams &P)
{
    return P.radial_tile > 0 ? P.radial_tile : sweep_best_tile([&](int t) { return sweep_waves(P, t); }, false);
}
int resolve_sweep_tile(const std::vector<KParams> &D)
{
    return sweep_best_tile([&](int t) {
        long w = 0;
        for (const KParams &P : D) w += sweep_waves(P, P.radial_tile > 0 ? P.radial_tile : t);
        return w;
    }, true);
}

void launch_sweeps(const KParams &P, hipStream_t st)
{
    const int tile = resolve_sweep_tile(P);
    dim3 g((unsigned)((P.ns + kSweepSegW - 1) / kSweepSegW), (unsigned)((P.nr + tile - 1) / tile));
    // One quantity per block where every SIMD still gets at most one walk:
    // each walk is then a third as long (32x64 isothermal step 26.2 -> 25.1 us),
    // while on more walks the shared work repeated in each block costs more
    // (128x384: 29.8 -> 32.1)
    const int quantities = P.adiabatic ? 5 : 4;
    const bool each = sweep_waves(P, tile) * quantities <= 1024;
    if (each) g.z = (unsigned)quantities;
#define SW(SP, AD)                                                                                \
    do {                                                                                          \
        if (each) hipLaunchKernelGGL((k_sweeps_each<SP, AD>), g, dim3(64), 0, st, P, tile);       \
        else hipLaunchKernelGGL((k_sweeps<SP, AD>), g, dim3(64), 0, st, P, tile);                 \
    } while (0)
    if (P.split) {
        if (P.adiabatic) SW(true, true);
        else SW(true, false);
    } else {
        if (P.adiabatic) SW(false, true);
        else SW(false, false);
    }
#undef SW
}

void launch_copy4(const KParams &P, hipStream_t st)
{
    // the bytes of four fields, as doubles
    const size_t n8 = (size_t)P.nr * P.ns * element_size(P) / 8;
    const size_t blocks = (n8 + 255) / 256;
    hipLaunchKernelGGL(k_copy4, dim3((unsigned)(blocks > 0 ? blocks : 1)), dim3(256), 0, st, P, n8);
}

void launch_transport(const KParams &P, hipStream_t st) { launch_transport_to(P, P, st); }

// the sweeps read the velocities of view P; the velocity kernel reads only the
// transported density and momenta and writes the velocities of view out
void launch_transport_to(const KParams &P, const KParams &out, hipStream_t st)
{
    launch_ring_mean(P, st, 1);
    launch_sweeps(P, st);
    LAUNCH(k_velocities, cell_grid(out, out.nr), kBlock, st, out);
}

void launch_transport_ghost(const KParams &P, const KParams &out, hipStream_t st, int final_advance)
{
    const int gb = (P.ns + 255) / 256;
    LAUNCH(k_ghost_ring_mean, dim3((unsigned)(gb + P.nr)), dim3(256), st, P);
    launch_sweeps(P, st);
    if (final_advance) LAUNCH(k_velocities_final, cell_grid(out, out.nr - 2), kBlock, st, out, final_advance);
    else LAUNCH(k_velocities, cell_grid(out, out.nr), kBlock, st, out);
}

KParams swapped_view(const KParams &P)
{
    KParams Q = P;
    Q.f[FCPT_VRAD] = P.valt[0];
    Q.valt[0] = P.f[FCPT_VRAD];
    Q.f[FCPT_VAZI] = P.valt[1];
    Q.valt[1] = P.f[FCPT_VAZI];
    if (P.lazy_derived && P.adiabatic) {  // the kick walk writes E to its partner too
        Q.f[FCPT_ENERGY] = P.ealt;
        Q.ealt = P.f[FCPT_ENERGY];
    }
    return Q;
}

void launch_src_fused(const KParams &P, hipStream_t st)
{
    LAUNCH(k_src_fused, cell_grid(P, P.nr + 1), kBlock, st, P);
}
void launch_src_energy(const KParams &P, hipStream_t st)
{
    LAUNCH(k_src_energy, cell_grid(P, P.nr - 1), kBlock, st, P);
}
void launch_av_fused(const KParams &P, hipStream_t st, int with_viscosity)
{
    LAUNCH(k_av_fused, cell_grid(P, P.nr + 1), kBlock, st, P, with_viscosity);
}
// rings per thread of the viscous walk: 8, or 4, while that gives 3072
// wavefronts (the window start costs two extra rings per walk), else 1 (the
// cell-parallel form)
static int visc_tile(const KParams &P)
{
    if (P.visc_tile > 0) return P.visc_tile;
    const long segs = (P.ns + kViscSegW - 1) / kViscSegW;
    int tile = 8;
    while (tile > 1 && segs * ((P.nr + tile - 1) / tile) < 3072) tile = tile > 4 ? tile / 2 : 1;
    return tile;
}

static void launch_visc_walk(const KParams &P, int tile, bool energy, hipStream_t st)
{
    const int tiles = (P.nr + tile - 1) / tile;
    const dim3 g((unsigned)((P.ns + kViscSegW - 1) / kViscSegW), (unsigned)((tiles + 3) / 4));
    if (P.split) {
        if (energy) hipLaunchKernelGGL((k_visc_walk<true, true>), g, kBlock, 0, st, P, tile);
        else hipLaunchKernelGGL((k_visc_walk<true, false>), g, kBlock, 0, st, P, tile);
    } else {
        if (energy) hipLaunchKernelGGL((k_visc_walk<false, true>), g, kBlock, 0, st, P, tile);
        else hipLaunchKernelGGL((k_visc_walk<false, false>), g, kBlock, 0, st, P, tile);
    }
}

void launch_visc_fused(const KParams &P, hipStream_t st)
{
    const int tile = visc_tile(P);
    if (tile == 1) LAUNCH(k_visc_fused, cell_grid(P, P.nr + 1), kBlock, st, P);
    else launch_visc_walk(P, tile, false, st);
}

void launch_visc_energy(const KParams &P, hipStream_t st)
{
    const int tile = visc_tile(P);
    if (tile == 1) {
        LAUNCH(k_visc_fused, cell_grid(P, P.nr + 1), kBlock, st, P);
        launch_substep3(P, st);
    } else {
        launch_visc_walk(P, tile, true, st);
    }
}

// Split storage's rounding points.  A disk large enough for 3072 wavefronts
// of ring walks hands the source-term velocities on in FP64; a smaller one
// rounds them, the viscous heating's tensor and the derived fields to their
// stored form, as the separate passes store them.
static bool walk_rounding(const KParams &P)
{
    auto tile = [&](int set, int seg) {
        if (set > 0) return set;
        const long segs = (P.ns + seg - 1) / seg;
        int t = 8;
        while (t > 1 && segs * ((P.nr + t - 1) / t) < 3072) t = t > 4 ? t / 2 : 1;
        return t;
    };
    return tile(P.kick_tile, 60) > 1 && tile(P.visc_tile, 62) > 1;
}

bool kv_walk_applies(const KParams &P)
{
    return (P.artvisc == FCPT_ARTVISC_TW || P.artvisc == FCPT_ARTVISC_SN) && P.kick_tile != 1 && P.visc_tile != 1;
}

// whether the kick walk folds the ring minima of launch_cfl_potential itself
int fold_in_kick(const KParams &P) { return P.cfl_pot && P.nr <= kFoldRings; }

void set_step_modes(KParams &P, bool fused)
{
    P.lazy_derived = fused && kv_walk_applies(P) ? 1 : 0;
    // The CFL limits and the potential in one launch where that is the faster:
    // in FP64 storage on adiabatic disks, which then store and load no scale
    // height (4096x12288 beta step 4513 -> 4322 us, 1024x3072 307.9 -> 304.9),
    // and on grids whose kick folds the ring minima, a launch less (128x384
    // isothermal 29.5 -> 28.0; 2048x6144 isothermal 769 -> 774 is left apart);
    // in split storage on small grids only.  There an isothermal disk gains up to
    // about 1.2e5 cells (128x384 30.9 -> 30.1 us, 181x543 36.2 -> 35.6, 200x600 40.0
    // either way, 209x627 41.0 -> 41.3, 256x768 45.9 -> 46.5, 512x1536 81.4 -> 82.7),
    // an adiabatic one 4 % there and 1 % still at 512x1536 (128x384 41.7 -> 40.0,
    // 209x627 57.9 -> 56.6, 256x768 64.3 -> 62.3, 512x1536 107.0 -> 105.8).
    const bool folds = P.nr <= kFoldRings;
    P.cfl_pot = P.lazy_derived && (P.split ? folds && (long)P.nr * P.ns <= 131072 : P.adiabatic || folds);
    // LeapFrog's second kick reads the H of the step's start
    P.h_lazy = P.cfl_pot && P.adiabatic && P.integrator == FCPT_INTEGRATOR_EULER;
    P.fold_in_kick = 0;
    P.split_emul = 0;
    if (P.split && P.lazy_derived) {
        const bool walk = walk_rounding(P);
        if (!walk || P.integrator == FCPT_INTEGRATOR_LEAPFROG) P.split_emul |= SPLIT_EMUL_DERIVED;
        if (!walk) P.split_emul |= SPLIT_EMUL_STAGES;
    }
}

// Rings per thread of the kick walk: a walk of t rings costs about t + 3.5
// (its window start), and the device holds `slots` of them at once, so the
// tile with the fewest rounds of walks times their length.
template <class Rounds>
static int kv_best_tile(Rounds &&rounds_of)
{
    int best = 1;
    double best_cost = 1e300;
    for (int t = 1; t <= 24; ++t) {
        const double rounds = rounds_of(t);
        const double cost = (t + 3.5) * (rounds <= 3.0 ? std::ceil(rounds) : rounds + 0.5);
        if (cost < best_cost) {
            best_cost = cost;
            best = t;
        }
    }
    return best;
}
// walks resident at once: 3 wavefronts per SIMD of an adiabatic walk's
// registers, 4 of an isothermal one's
static double kv_slots(bool adiabatic) { return adiabatic ? 3072.0 : 4096.0; }
static int kv_tile(const KParams &P)
{
    if (P.kick_tile > 1) return P.kick_tile;
    if (P.visc_tile > 1) return P.visc_tile;
    return kv_best_tile([&](int t) { return (double)kv_waves(P, t) / kv_slots(P.adiabatic); });
}
// a batch's walks run in rounds too, each member's in slots of its kind
void resolve_kv_tiles(std::vector<KParams> &D)
{
    const int t = kv_best_tile([&](int tile) {
        long waves[2] = {0, 0};  // of isothermal and of adiabatic members
        for (const KParams &P : D)
            if (kv_walk_applies(P)) waves[P.adiabatic ? 1 : 0] += kv_waves(P, tile);
        return (double)waves[0] / kv_slots(false) + (double)waves[1] / kv_slots(true);
    });
    for (KParams &P : D)
        if (kv_walk_applies(P)) P.kv_tile = P.kick_tile > 1 ? P.kick_tile : P.visc_tile > 1 ? P.visc_tile : t;
}
long kv_waves(const KParams &P, int tile)
{
    return (long)((P.ns + kKvSegW - 1) / kKvSegW) * ((P.nr + tile - 1) / tile);
}

int resolve_kick_tile(const KParams &P) { return kv_walk_applies(P) ? kv_tile(P) : 1; }
int resolve_visc_tile(const KParams &P) { return kv_walk_applies(P) ? kv_tile(P) : visc_tile(P); }
bool walks_tunable(const KParams &P) { return kv_walk_applies(P) && (!P.split || walk_rounding(P)); }

void launch_kick(const KParams &P, hipStream_t st, int fold_mode)
{
    const int tile = kv_tile(P);
    // one wavefront per block: with four, a block's registers and LDS stay
    // taken until its last wavefront ends (1024 x 3072 adiabatic step 406 us
    // with four, 370 with one)
    const dim3 g((unsigned)((P.ns + kKvSegW - 1) / kKvSegW), (unsigned)((P.nr + tile - 1) / tile)), b(64);
    const size_t lds = kv_lds_doubles(tile) * sizeof(double);
    if (fold_mode == kFoldDone) {  // launch_cfl_potential before it
        if (!P.fold_in_kick) hipLaunchKernelGGL(k_cfl_fold, dim3(1), dim3(256), 0, st, P, 2);
    } else {
        launch_potential_fold(P, st, fold_mode);
    }
#define KV(SP, EM)                                                                                        \
    do {                                                                                                  \
        const bool sn = P.artvisc == FCPT_ARTVISC_SN;                                                     \
        if (P.adiabatic && sn) hipLaunchKernelGGL((k_kv_walk<SP, true, true, EM>), g, b, lds, st, P, tile);   \
        else if (P.adiabatic) hipLaunchKernelGGL((k_kv_walk<SP, true, false, EM>), g, b, lds, st, P, tile);   \
        else if (sn) hipLaunchKernelGGL((k_kv_walk<SP, false, true, EM>), g, b, lds, st, P, tile);            \
        else hipLaunchKernelGGL((k_kv_walk<SP, false, false, EM>), g, b, lds, st, P, tile);                   \
    } while (0)
    if (!P.split) KV(false, false);
    else if (P.split_emul) KV(true, true);
    else KV(true, false);
#undef KV
}

void launch_derived(const KParams &P, hipStream_t st) { LAUNCH(k_derived, cell_grid(P, P.nr), kBlock, st, P); }

// the final boundary call (damping, ghost rings, the clock) and the derived
// fields: damping, then one pass for the rest
void launch_final_boundaries_derived(const KParams &P, hipStream_t st, int advance_time)
{
    if (P.damping) {
        const int n_inner = (P.damp_ids[0] > P.damp_ids[1] ? P.damp_ids[0] : P.damp_ids[1]) + 1;
        const int o0 = P.damp_ids[2] < P.damp_ids[3] ? P.damp_ids[2] : P.damp_ids[3];
        const int n_outer = P.nr + 1 - o0;
        LAUNCH(k_damping, cell_grid(P, n_inner + n_outer), kBlock, st, P);
    }
    LAUNCH(k_final_derived, cell_grid(P, P.nr), kBlock, st, P, advance_time);
}
void launch_final_leapfrog(const KParams &P, hipStream_t st, int advance_time)
{
    LAUNCH(k_final_leapfrog, cell_grid(P, P.nr - 2), kBlock, st, P, advance_time);
}
void launch_iso_rings(const KParams &P, hipStream_t st)
{
    hipLaunchKernelGGL(k_iso_rings, dim3((unsigned)((P.nr + 255) / 256)), dim3(256), 0, st, P);
}

void launch_iso_profile(const KParams &P, hipStream_t st)
{
    LAUNCH(k_iso_profile, cell_grid(P, P.nr), kBlock, st, P);
}

void launch_rebase(const KParams &P, hipStream_t st, void *field, const double *oldbg,
                   const double *newbg, int rows)
{
    hipLaunchKernelGGL(k_rebase, cell_grid(P, rows), kBlock, 0, st, static_cast<float *>(field), oldbg,
                       newbg, P.ns, rows);
}

void launch_split_ring_mean(const KParams &P, hipStream_t st, const void *field, const double *bg,
                            int rows, double *out)
{
    hipLaunchKernelGGL(k_split_ring_mean, dim3((unsigned)rows), dim3(256), 0, st,
                       static_cast<const float *>(field), bg, P.ns, out);
}

void launch_totals(const KParams &P, hipStream_t st, double radius, double *ring_scratch,
                   double *out2)
{
    LAUNCH(k_totals_rings, dim3(P.nr), dim3(64), st, P, radius, ring_scratch);
    hipLaunchKernelGGL(k_totals_final, dim3(1), dim3(1), 0, st, P, ring_scratch, out2);
}

// ---------------------------------------------------------------------------
// The disk's gravity on the N bodies (ComputeDiskOnPlanetAccel, Force.cpp:23-122)

// Per cell and body, the reference's expression (the smoothing of
// compute_smoothing, Force.cpp:145-159, chosen by the flags; the Klahr-Kley
// factor 4q^3 - 3q^4 inside r_cubic); inner (Rmed < r_body) and outer sums
// kept apart as in the reference.  NB bodies per launch (a template argument,
// so only their accumulators live in registers).  One block per active ring:
// it first forms the ring's mean Sigma where the flags ask for it
// (ComputeAverageDensity, Pframeforce.cpp:174-187, pairwise tree order), with
// the first cells' loads in flight, then a thread adds every 256th cell,
// loading the next one before it works on the current one; 1 / d^3 comes from
// the reciprocal square root with two Newton steps (a few ulp from the
// reference's sqrt and division).  Each block folds its 4 NB partial sums with
// wavefront shuffles and LDS into its own slot (component-major, slot = ring),
// and k_disk_force_final sums each component's slots in a fixed order:
// deterministic, no atomics.
// What bounds it: latency on the grids that follow every step with it.  With
// the means in a launch of their own and threads that walk several rings, the
// force took 10.0 us for four bodies at 48x144 and 24.4 at 512x1536; now 7.7
// and 11.2.  The result goes straight to pinned memory: the call took 35 us at
// 48x144 with a copy, 24 without.
template <bool SPLIT, int NB>
__global__ void __launch_bounds__(256) k_disk_force(KParams P, ForceBodies B, double *part)
{
    const int ns = P.ns;
    const int t = (int)threadIdx.x;
    const int i = 1 + (int)blockIdx.x;  // rings 1 .. nr - 2
    const int nslots = (int)gridDim.x;
    double acc[NB][4];
#pragma unroll
    for (int k = 0; k < NB; ++k) acc[k][0] = acc[k][1] = acc[k][2] = acc[k][3] = 0.0;
    FLD(S, FCPT_SIGMA);
    const Fld<SPLIT> Hf = fld_derived<SPLIT>(P, FCPT_SCALE_HEIGHT);
    const double G = P.G;
    const double thick = P.thickness_smoothing;
    const double rmed = cst(P.Rmed)[i], surf = cst(P.Surf)[i];
    const double H_ring = P.adiabatic ? 0.0 : cst(P.iso_h)[i];
    const int j0 = t < ns ? t : 0;
    double sig = S(i, j0), cphi = P.cosphi[j0], sphi = P.sinphi[j0];
    // a step that forms its derived fields where it needs them stores no H
    auto height = [&](int j, double sg) {
        if (!P.adiabatic) return H_ring;
        if (!P.h_lazy) return Hf(i, j);
        return Hf.stored(i, j, adi_derived<SPLIT>(P, i, fld<SPLIT>(P, FCPT_ENERGY)(i, j), sg).h);
    };
    double H = height(j0, sig);
    double mean = 0.0;
    if (B.flags & FCPT_FORCE_CORRECT_SELFGRAVITY) {
        __shared__ double sh[256];
        double sum = 0.0;
        strided_row<256>(ns, t, [&](int j) { return S(i, j); }, [&](double x) { sum += x; });
        mean = block_sum(sum, sh) / ns;
    }
    for (int j = t; j < ns; j += 256) {
        const int jn = j + 256 < ns ? j + 256 : j;
        const double sig_n = S(i, jn), cphi_n = P.cosphi[jn], sphi_n = P.sinphi[jn];
        const double H_n = height(jn, sig_n);
        const double xc = rmed * cphi;
        const double yc = rmed * sphi;
        const double gm = G * (surf * (sig - mean));
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const double smooth = B.smooth_fixed[k] >= 0.0 ? B.smooth_fixed[k] : thick * H;
            const double dx = xc - B.x[k];
            const double dy = yc - B.y[k];
            const double d2 = (dx * dx + dy * dy) + smooth * smooth;
            const double inv_d = inv_sqrt<true>(d2);
            const double inv_d3 = inv_d * inv_d * inv_d;
            double fx = gm * dx * inv_d3;
            double fy = gm * dy * inv_d3;
            const double r_sm = B.r_cubic[k];
            if (r_sm > 0.0) {  // uniform: the body's cubic smoothing radius
                const double q = (d2 * inv_d) / r_sm;
                const double klahr = q < 1.0 ? q * q * q * (4.0 - 3.0 * q) : 1.0;
                fx *= klahr;
                fy *= klahr;
            }
            if (rmed < B.r[k]) {  // uniform: one ring against one body
                acc[k][0] += fx;
                acc[k][1] += fy;
            } else {
                acc[k][2] += fx;
                acc[k][3] += fy;
            }
        }
        sig = sig_n;
        cphi = cphi_n;
        sphi = sphi_n;
        H = H_n;
    }
    __shared__ double wsum[4][NB * 4];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            double v = acc[k][c];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
            if ((t & 63) == 0) wsum[t >> 6][4 * k + c] = v;
        }
    }
    __syncthreads();
    if (t < NB * 4)
        part[(size_t)t * nslots + blockIdx.x] = (wsum[0][t] + wsum[1][t]) + (wsum[2][t] + wsum[3][t]);
}

// one block per component: the slots summed with a 256-wide stride, then a
// pairwise tree over the 256 partial sums; out may be pinned host memory
__global__ void __launch_bounds__(256) k_disk_force_final(const double *part, int nslots, double *out)
{
    __shared__ double sh[256];
    const double *p = part + (size_t)blockIdx.x * nslots;
    double s = 0.0;
    for (int b = threadIdx.x; b < nslots; b += 256) s += p[b];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

template <bool SPLIT>
static void launch_force_split(const KParams &P, hipStream_t st, const ForceBodies &B, double *part, dim3 g)
{
#define FORCE(N) hipLaunchKernelGGL((k_disk_force<SPLIT, N>), g, dim3(256), 0, st, P, B, part)
    switch (B.n) {
    case 1: FORCE(1); break;
    case 2: FORCE(2); break;
    case 3: FORCE(3); break;
    case 4: FORCE(4); break;
    case 5: FORCE(5); break;
    case 6: FORCE(6); break;
    case 7: FORCE(7); break;
    default: FORCE(8); break;
    }
#undef FORCE
}

void launch_disk_force(const KParams &P, hipStream_t st, const ForceBodies &B, double *part, double *out4)
{
    static_assert(kForceMaxBodies == 8, "launch_force_split dispatches 1 .. 8 bodies");
    if (B.n < 1 || B.n > kForceMaxBodies) return;
    const dim3 g((unsigned)(P.nr - 2));
    if (P.split) launch_force_split<true>(P, st, B, part, g);
    else launch_force_split<false>(P, st, B, part, g);
    hipLaunchKernelGGL(k_disk_force_final, dim3((unsigned)(4 * B.n)), dim3(256), 0, st, part, (int)g.x, out4);
}

// ---------------------------------------------------------------------------
// Batched step: many disks per launch.  Each stage of one sim::run iteration
// is one launch over a work table listing, for every disk that takes part in
// the stage, every block of that disk's own grid.  A disk's blocks do exactly
// what its single-disk launch does, so a batched disk evolves bit for bit like
// the same disk stepped alone.

static void add_grid(std::vector<BatchEntry> &v, unsigned d, unsigned gx, unsigned gy)
{
    for (unsigned y = 0; y < gy; ++y)
        for (unsigned x = 0; x < gx; ++x) v.push_back(BatchEntry{d, (y << 16) | x});
}

static unsigned rows_grid(const KParams &P, int rows) { return (unsigned)((rows + 3) / 4); }
static unsigned sector_grid(const KParams &P) { return (unsigned)((P.ns + 63) / 64); }

std::vector<BatchStageHost> plan_batch_step(const std::vector<KParams> &D)
{
    std::vector<BatchStageHost> st;
    // parameter block of disk d: d (the fields hold the velocities) or n + d
    // (its swapped view: the partner buffers hold them, between fused passes)
    const unsigned n = (unsigned)D.size();
    std::vector<unsigned> view(n, 0);
    auto stage_v = [&](int kind, int arg, auto pred, auto grid, bool flips, bool fields) {
        BatchStageHost s{kind, arg, {}};
        for (unsigned d = 0; d < n; ++d) {
            if (!pred(D[d])) continue;
            grid(s.entries, (fields || !view[d]) ? d : n + d, D[d]);
            if (flips) view[d] ^= 1u;
        }
        if (!s.entries.empty()) st.push_back(std::move(s));
    };
    auto stage = [&](int kind, int arg, auto pred, auto grid) { stage_v(kind, arg, pred, grid, false, false); };
    auto all = [](const KParams &) { return true; };
    auto adi = [](const KParams &P) { return P.adiabatic != 0; };
    auto iso = [](const KParams &P) { return P.adiabatic == 0; };
    auto rows = [](int off) {
        return [off](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
            add_grid(v, d, sector_grid(P), rows_grid(P, P.nr - off));
        };
    };
    auto rings = [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        add_grid(v, d, (unsigned)P.nr, 1);
    };
    auto sweeps = [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        add_grid(v, d, (unsigned)((P.ns + kSweepSegW - 1) / kSweepSegW),
                 (unsigned)((P.nr + P.radial_tile - 1) / P.radial_tile));
    };
    auto one = [](std::vector<BatchEntry> &v, unsigned d, const KParams &) { add_grid(v, d, 1, 1); };
    // sim::CalculateTimeStep and the monitor clip (simulation.cpp:100-118, 526-542):
    // the per-ring CFL blocks and the fold, as launch_cfl
    auto merged = [](const KParams &P) { return P.cfl_pot != 0; };
    auto apart = [](const KParams &P) { return P.cfl_pot == 0; };
    stage(B_CFL_POT, 0, merged, rings);
    stage(B_CFL_RINGS, 0, apart, rings);
    stage(B_CFL_FINAL_RINGS, 2, [](const KParams &P) { return !P.fold_in_kick; }, one);
    // step_Euler (simulation.cpp:148-267), in the order of enqueue_euler
    stage(B_POTENTIAL, 0, apart, [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        add_grid(v, d, (unsigned)((P.ns + 64 * kPotCells - 1) / (64 * kPotCells)), rows_grid(P, P.nr));
    });
    // the kick: the walk where the disk's own launch uses it (its tile in
    // kv_tile), else the cell-parallel fused passes; each pass flips the
    // disk's view
    auto flip = [&](int kind, int arg, auto pred, auto grid) { stage_v(kind, arg, pred, grid, true, false); };
    auto walk = [](const KParams &P) { return kv_walk_applies(P); };
    auto kick_grid = [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        const int tiles = (P.nr + P.kv_tile - 1) / P.kv_tile;
        add_grid(v, d, (unsigned)((P.ns + kKvSegW - 1) / kKvSegW), (unsigned)tiles);
    };
    auto visc_grid = [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        const int tiles = (P.nr + P.visc_tile - 1) / P.visc_tile;
        add_grid(v, d, (unsigned)((P.ns + kViscSegW - 1) / kViscSegW), (unsigned)((tiles + 3) / 4));
    };
    int kv_most = 1;  // the longest walk, which sizes the launch's LDS
    for (const KParams &P : D)
        if (walk(P)) kv_most = std::max(kv_most, P.kv_tile);
    for (int a = 0; a < 2; ++a)
        for (int sn = 0; sn < 2; ++sn)
            flip(B_KV_WALK, 2 * a + sn + 4 * kv_most,
                 [&](const KParams &P) {
                     return walk(P) && P.adiabatic == a && (P.artvisc == FCPT_ARTVISC_SN) == (sn != 0);
                 },
                 kick_grid);
    auto cell = [&](const KParams &P) { return !walk(P); };
    flip(B_SRC_FUSED, 0, cell, rows(-1));
    stage(B_SRC_ENERGY, 0, [&](const KParams &P) { return cell(P) && P.adiabatic; }, rows(1));
    auto av = [&](const KParams &P) {
        return cell(P) && (P.artvisc == FCPT_ARTVISC_TW || P.artvisc == FCPT_ARTVISC_SN);
    };
    auto none = [](const KParams &P) { return P.artvisc == FCPT_ARTVISC_NONE; };
    flip(B_AV_FUSED, 1, av, rows(-1));
    stage(B_TEMP_FLOOR, 0,
          [](const KParams &P) {
              return P.artvisc == FCPT_ARTVISC_NONE && P.adiabatic && P.artvisc_dissipation;
          },
          rows(0));
    stage(B_RECALC_VISC, 0, none, rows(0));
    // the viscous pass: the walk (with SubStep3 when adiabatic) where the
    // disk's tile is above 1, as launch_visc_fused / launch_visc_energy
    auto vwalk = [&](const KParams &P) { return cell(P) && P.visc_tile > 1; };
    for (int a = 0; a < 2; ++a)
        flip(B_VISC_WALK, a, [&](const KParams &P) { return vwalk(P) && P.adiabatic == a; }, visc_grid);
    flip(B_VISC_FUSED, 0, [&](const KParams &P) { return cell(P) && !vwalk(P); }, rows(-1));
    stage(B_SUBSTEP3, 0, [&](const KParams &P) { return cell(P) && !vwalk(P) && P.adiabatic; }, rows(0));
    // the boundary call before the transport with the FARGO ring means
    stage(B_GHOST_MEAN, 0, all, [](std::vector<BatchEntry> &v, unsigned d, const KParams &P) {
        add_grid(v, d, (unsigned)((P.ns + 255) / 256 + P.nr), 1);
    });
    stage(B_SWEEPS_ISO, 0, iso, sweeps);
    stage(B_SWEEPS_ADI, 0, adi, sweeps);
    // the velocity kernel with the final boundary call and the derived
    // fields writes the fields of every disk
    stage_v(B_VEL_FINAL, 2, all, rows(2), false, true);
    return st;
}

#define LAUNCHB(kern, block, ...)                                                              \
    do {                                                                                       \
        if (split) hipLaunchKernelGGL(kern<true>, dim3(S.n), block, 0, st, Ps, S.map, ##__VA_ARGS__);  \
        else hipLaunchKernelGGL(kern<false>, dim3(S.n), block, 0, st, Ps, S.map, ##__VA_ARGS__);       \
    } while (0)

void launch_batch_stage(const KParams *Ps, const BatchStageDev &S, int split, hipStream_t st)
{
    const dim3 b256(256);
    switch (S.kind) {
    case B_POTENTIAL: LAUNCHB(kb_potential, kBlock); break;
    case B_SRC_FUSED: LAUNCHB(kb_src_fused, kBlock); break;
    case B_AV_FUSED: LAUNCHB(kb_av_fused, kBlock, S.arg); break;
    case B_VISC_FUSED: LAUNCHB(kb_visc_fused, kBlock); break;
    case B_SRC_ENERGY: LAUNCHB(kb_src_energy, kBlock); break;
    case B_TEMP_FLOOR: LAUNCHB(kb_temperature_floor, kBlock); break;
    case B_RECALC_VISC: LAUNCHB(kb_recalc_viscosity, kBlock); break;
    case B_SUBSTEP3: LAUNCHB(kb_substep3, kBlock); break;
    case B_CFL_RINGS:
        if (split) hipLaunchKernelGGL((kb_cfl_ring<true, false>), dim3(S.n), b256, 0, st, Ps, S.map);
        else hipLaunchKernelGGL((kb_cfl_ring<false, false>), dim3(S.n), b256, 0, st, Ps, S.map);
        break;
    case B_CFL_POT:
        if (split) hipLaunchKernelGGL((kb_cfl_ring<true, true>), dim3(S.n), b256, 0, st, Ps, S.map);
        else hipLaunchKernelGGL((kb_cfl_ring<false, true>), dim3(S.n), b256, 0, st, Ps, S.map);
        break;
    case B_CFL_FINAL_RINGS:
        hipLaunchKernelGGL(kb_cfl_fold, dim3(S.n), b256, 0, st, Ps, S.map, S.arg);
        break;
    case B_GHOST_MEAN: LAUNCHB(kb_ghost_ring_mean, b256); break;
    case B_VEL_FINAL: LAUNCHB(kb_velocities_final, kBlock, S.arg); break;
    case B_KV_WALK: {
        const dim3 g(S.n);
#define KWB(SP, AD, SN)                                                                            hipLaunchKernelGGL((kb_kv_walk<SP, AD, SN>), g, dim3(64), lds, st, Ps, S.map)
        const int v = (split ? 4 : 0) + (S.arg & 3);
        const size_t lds = kv_lds_doubles(S.arg >> 2) * sizeof(double);
        if (v == 0) KWB(false, false, false);
        else if (v == 1) KWB(false, false, true);
        else if (v == 2) KWB(false, true, false);
        else if (v == 3) KWB(false, true, true);
        else if (v == 4) KWB(true, false, false);
        else if (v == 5) KWB(true, false, true);
        else if (v == 6) KWB(true, true, false);
        else KWB(true, true, true);
#undef KWB
        break;
    }
    case B_VISC_WALK: {
        const dim3 g(S.n);
        if (split) {
            if (S.arg) hipLaunchKernelGGL((kb_visc_walk<true, true>), g, kBlock, 0, st, Ps, S.map);
            else hipLaunchKernelGGL((kb_visc_walk<true, false>), g, kBlock, 0, st, Ps, S.map);
        } else {
            if (S.arg) hipLaunchKernelGGL((kb_visc_walk<false, true>), g, kBlock, 0, st, Ps, S.map);
            else hipLaunchKernelGGL((kb_visc_walk<false, false>), g, kBlock, 0, st, Ps, S.map);
        }
        break;
    }
    case B_SWEEPS_ISO:
    case B_SWEEPS_ADI: {
        const bool a = S.kind == B_SWEEPS_ADI;
        const dim3 g(S.n);
        if (split) {
            if (a) hipLaunchKernelGGL((kb_sweeps<true, true>), g, dim3(64), 0, st, Ps, S.map);
            else hipLaunchKernelGGL((kb_sweeps<true, false>), g, dim3(64), 0, st, Ps, S.map);
        } else {
            if (a) hipLaunchKernelGGL((kb_sweeps<false, true>), g, dim3(64), 0, st, Ps, S.map);
            else hipLaunchKernelGGL((kb_sweeps<false, false>), g, dim3(64), 0, st, Ps, S.map);
        }
        break;
    }
    default: break;
    }
}

}  // namespace fcpt
