// pps_kernels.hip -- hand-written gfx950 kernels of the Krylov hot path.
//
// Two kernel skeletons carry every operation:
//  * k_stencil: 2.5-D z-marching tile.  A block of 64x8 threads owns a 64x32
//    column tile (kTX x kTH: each thread four rows) of one x-y slab and marches
//    through kz planes (the longest of 64/32/16/8 that still gives 2048
//    blocks; 4 or 2 on grids too small for 1024 blocks of 8).  Each thread keeps its columns' (k-1, k, k+1) values in
//    registers; the plane-k tile and its one-point halo are staged in LDS
//    (double-buffered, one barrier per plane), so x- and y-neighbours come from
//    LDS and every value of the input field is produced once per plane (this is
//    what lets the CG search direction p = z + beta*p be formed on the fly
//    inside the stencil).  The loads of planes k+1 and k+2 are in flight while
//    plane k is computed, so the barrier never waits on HBM latency.
//    The 7-point operator is the reference's +Laplacian
//    (matrixFreeOperatorA.hpp:33-38) written in difference form,
//    cx((x[i-1]-x)+(x[i+1]-x)) + cy(..) + cz(..), which keeps FP32 accurate
//    for smooth fields.
//  * k_vector: one-shot blocks over consecutive points of an x-row (512 x 1
//    for FP64 operands, 128 threads x 4 points for FP32) for the fused
//    axpy/dot updates: all of a thread's loads are issued before its store,
//    and consecutive blocks stream consecutive addresses.
// k_cg_pass runs one CG iteration and k_cheb_multi two or three Chebyshev
// sweeps per pass.
//
// Reductions are FP64 in every precision and deterministic: DPP row
// butterflies inside each wavefront, LDS across the wavefronts, one partial
// per block, then a one-block epilogue kernel (after a level of span sums when
// there are many blocks) sums the partials in a fixed order and runs the
// solver's scalar update (alpha, beta, omega, convergence flag) on the device.
// The epilogue runs as its own launch instead of a last-block-arrives scheme:
// on gfx950 the agent-scope release fence that scheme needs in every block
// writes back the XCD's L2, which costs more than the whole reduction.
//
// Blocks are remapped so that consecutive tiles land on the same XCD (the
// hardware deals blocks round-robin over the 8 XCDs, each with its own L2):
// the y-halo rows a tile reads from its neighbour are then L2 hits.
#include "pps_kernels.hpp"

#include <algorithm>
#include <type_traits>

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>

namespace pps {


// tiling of one launch: 64-wide tiles of `th` rows, z-chunks of kz planes
static Geo retile(const Geo& in, int th, int kz)
{
    Geo g = in;
    g.kz = kz > 0 ? kz : 1;
    g.ntx = (g.hi0 - g.lo0 + kTX - 1) / kTX;
    g.nty = (g.hi1 - g.lo1 + th - 1) / th;
    const int ntz = (g.hi2 - g.lo2 + g.kz - 1) / g.kz;
    g.nblocks = g.ntx * g.nty * ntz;
    return g;
}

Geo make_geo(const Layout& L, const Region& R, const double coef[3], int kz_st, int nt)
{
    Geo g{};
    g.plane = L.plane;
    g.px = L.px;
    g.ox = L.ox;
    g.lo0 = R.lo[0]; g.hi0 = R.hi[0];
    g.lo1 = R.lo[1]; g.hi1 = R.hi[1];
    g.lo2 = R.lo[2]; g.hi2 = R.hi[2];
    g.kz_st = kz_st;
    g.nt = nt;
    g.cx = coef[0];
    g.cy = coef[1];
    g.cz = coef[2];
    return retile(g, kTH, kz_st);
}

// stores of the field outputs: non-temporal (NT) when the fields exceed the
// caches.  NT is a template argument so that each kernel body holds one kind
// of store: with a run-time flag the compiler merges the two stores of an
// if/else into one plain store and the non-temporal hint is lost.
template <typename T> struct NoDeduce { using type = T; };
// loads of fields read once per pass (the vector kernels' operands):
// non-temporal in the same mode, so streamed inputs do not evict the caches'
// useful lines (measured at 512^3: FP64 update 5.6-5.7 -> 5.8-6.1 TB/s, FP32
// update 5.4 -> 5.9)
template <bool NT, typename T>
__device__ __forceinline__ T ld(const T* p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT, typename T>
__device__ __forceinline__ void put(T* p, typename NoDeduce<T>::type v)
{
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// ------------------------------------------------------------ common pieces

__device__ __forceinline__ int xcd_remap(int b, int nb)
{
    const int full = nb & ~7;
    if (b >= full) return b;
    return (b & 7) * (full >> 3) + (b >> 3);
}

// one DPP lane exchange of a double (two 32-bit moves); CTRL is the DPP control
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// sum over the wavefront, the same value in every lane, in a fixed order:
// butterflies inside each row of 16 lanes (quad_perm [1,0,3,2], quad_perm
// [2,3,0,1], row_half_mirror, row_mirror), then the four row sums read out
// and added as (r0 + r1) + (r2 + r3).  DPP moves stay in the VALU, where a
// shuffle is a round trip through the LDS crossbar per step; in a one-shot
// reducing kernel over FP32 fields that round trip was the bottleneck.
__device__ __forceinline__ double wave_sum(double v)
{
    v += dpp_mov<0xB1>(v);
    v += dpp_mov<0x4E>(v);
    v += dpp_mov<0x141>(v);
    v += dpp_mov<0x140>(v);
    const long long b = __double_as_longlong(v);
    double r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int lo = __builtin_amdgcn_readlane((int)b, 16 * q);
        const int hi = __builtin_amdgcn_readlane((int)(b >> 32), 16 * q);
        r[q] = __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
    }
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// sum over the block in a fixed order; result valid in thread 0
template <int NQ, int NTHREADS = kThreads>
__device__ __forceinline__ void block_sum(double (&v)[NQ], double (&tot)[NQ])
{
    constexpr int NW = NTHREADS / 64;
    __shared__ double sm[NQ][NW];
    const int tid = threadIdx.x + blockDim.x * threadIdx.y;
    const int lane = tid & 63, w = tid >> 6;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double t = wave_sum(v[q]);
        if (lane == 0) sm[q][w] = t;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        double t = 0.0;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) t += sm[q][ww];
        tot[q] = t;
    }
}

// the block's sums as partial number `slot` of the launch
template <int NQ, int NTHREADS = kThreads>
__device__ __forceinline__ void block_partials(double (&v)[NQ], const RedBuf& rb, int slot)
{
    double tot[NQ];
    block_sum<NQ, NTHREADS>(v, tot);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) rb.partials[(size_t)q * rb.cap + slot] = tot[q];
    }
}

// one block: sums the partials of the preceding launch and runs op.finish.
// Thread t owns partials t, t+1024, ... summed in that order with two
// interleaved accumulators (more loads in flight), then a fixed tree.
constexpr int kFinThreads = 1024;
template <int NQ, class Op>
__device__ __forceinline__ void finish_block(Op& op, const RedBuf& rb, int nblocks)
{
    double a0[NQ], a1[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) a0[q] = a1[q] = 0.0;
    int b = threadIdx.x;
    for (; b + kFinThreads < nblocks; b += 2 * kFinThreads) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            a0[q] += rb.partials[(size_t)q * rb.cap + b];
            a1[q] += rb.partials[(size_t)q * rb.cap + b + kFinThreads];
        }
    }
    if (b < nblocks) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) a0[q] += rb.partials[(size_t)q * rb.cap + b];
    }
    double acc[NQ], tot[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = a0[q] + a1[q];
    block_sum<NQ, kFinThreads>(acc, tot);
    if (threadIdx.x == 0) op.finish(tot);
}
template <int NQ, class Op>
__global__ __launch_bounds__(kFinThreads) void k_finish(Op op, RedBuf rb, int nblocks)
{
    if (op.gated()) return;
    finish_block<NQ>(op, rb, nblocks);
}
// the same of nalt partials while *alt != 0
template <int NQ, class Op>
__global__ __launch_bounds__(kFinThreads) void k_finish_alt(Op op, RedBuf rb, int nblocks, int nalt, const int* alt)
{
    if (op.gated()) return;
    finish_block<NQ>(op, rb, *alt ? nalt : nblocks);
}

struct Gate {
    const int* gate;
    __device__ __forceinline__ bool gated() const { return gate != nullptr && *gate != 0; }
};

// record the end of one iteration of a main/inner Krylov loop
__device__ __forceinline__ void finish_iteration(Scal* S, double err, bool history)
{
    S->v[S_ERR] = err;
    const int it = S->iter + 1;
    S->iter = it;
    if (history && S->hist != nullptr && it < S->hist_cap) S->hist[it] = err;
    if (err < S->v[S_TOL] || it >= S->maxit) S->done = 1;
}

// --------------------------------------------------------- kernel skeletons

// Stencil op hooks.  A plain op has in(c) (the staged value, a plain load) and
// out(c, v, Av, acc).  An op whose staged value is computed from several
// fields, or whose output reads more fields, declares
//   struct Raw; Raw in_raw(c); T in_value(const Raw&)   -- loads, and their combination
//   struct Ox;  Ox out_raw(c)                            -- the output's extra loads
//   out(c, v, Av, const Raw& centre, const Ox&, acc)
// (Raw defaults to T, Ox to NoRaw).  The kernel issues the raw loads planes
// ahead and combines them only when needed, so no load is waited on as soon
// as it is issued.
struct NoRaw {};
template <class Op, typename T, class = void> struct RawOf { using type = T; };
template <class Op, typename T> struct RawOf<Op, T, std::void_t<typename Op::Raw>> { using type = typename Op::Raw; };
template <class Op, class = void> struct OxOf { using type = NoRaw; };
template <class Op> struct OxOf<Op, std::void_t<typename Op::Ox>> { using type = typename Op::Ox; };
template <class Op, typename T>
constexpr bool kHooks = !std::is_same_v<typename RawOf<Op, T>::type, T> || !std::is_same_v<typename OxOf<Op>::type, NoRaw>;

template <class Op, typename T>
__device__ __forceinline__ typename RawOf<Op, T>::type st_raw(const Op& op, long long c)
{
    if constexpr (std::is_same_v<typename RawOf<Op, T>::type, T>) return op.in(c);
    else return op.in_raw(c);
}
template <class Op, typename T>
__device__ __forceinline__ T st_value(const Op& op, const typename RawOf<Op, T>::type& r)
{
    if constexpr (std::is_same_v<typename RawOf<Op, T>::type, T>) return r;
    else return op.in_value(r);
}
// the output's extra operands are read once per pass: non-temporal loads in
// the streaming mode (the staged field's loads stay cached: neighbouring tiles
// re-read its halo)
template <bool NT, class Op>
__device__ __forceinline__ typename OxOf<Op>::type st_ox(const Op& op, long long c)
{
    if constexpr (std::is_same_v<typename OxOf<Op>::type, NoRaw>) return NoRaw{};
    else return op.template out_raw<NT>(c);
}
template <bool NT, class Op, typename T>
__device__ __forceinline__ void st_out(const Op& op, long long c, T v, T Av, const typename RawOf<Op, T>::type& r,
                                       const typename OxOf<Op>::type& o, double* acc)
{
    if constexpr (kHooks<Op, T>) op.template out<NT>(c, v, Av, r, o, acc);
    else op.template out<NT>(c, v, Av, acc);
}

template <typename T, int NQ, class Op, bool NT>
__global__ __launch_bounds__(kSThreads) void k_stencil(Geo g, Op op, RedBuf rb)
{
    if (op.gated()) return;
    op.load();
    // tile: 64 columns x kTH rows; thread (lx, ly) owns rows ly, ly+kSTY, ...
    __shared__ T lds[2][kTH + 2][kTX + 2];
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int tx0 = b % g.ntx;
    const int rr = b / g.ntx;
    const int ty0 = rr % g.nty;
    const int tz0 = rr / g.nty;
    const int lx = threadIdx.x, ly = threadIdx.y, tid = lx + kTX * ly;
    const int i = g.lo0 + tx0 * kTX + lx;
    const int jt = g.lo1 + ty0 * kTH;  // first row of the tile
    const int k0 = g.lo2 + tz0 * g.kz;
    const int k1 = min(k0 + g.kz, g.hi2);

    // halo producers: 128 threads for the two y-halo rows, 2*kTH for the x-halo columns
    static_assert(2 * kTX + 2 * kTH <= kSThreads, "one thread per halo point of a plane");
    int hr = 0, hc_ = 0, hi = 0, hj = 0;
    bool hv = false;
    if (tid < 2 * kTX) {
        const int col = tid % kTX;
        const bool top = tid >= kTX;
        hr = top ? kTH + 1 : 0;
        hc_ = col + 1;
        hi = g.lo0 + tx0 * kTX + col;
        hj = jt + (top ? kTH : -1);
        hv = true;
    } else if (tid < 2 * kTX + 2 * kTH) {
        const int t = tid - 2 * kTX;
        const int row = t % kTH;
        const bool right = t >= kTH;
        hr = row + 1;
        hc_ = right ? kTX + 1 : 0;
        hi = g.lo0 + tx0 * kTX + (right ? kTX : -1);
        hj = jt + row;
        hv = true;
    }
    const bool hin = hv && hi <= g.hi0 && hj <= g.hi1;
    // where a point's input is read: itself, or the mirror point of a ghost (g.mir)
    auto mx = [&](int v) { return (g.mir & 1) && v == g.lo0 - 1 ? v + 2 : (g.mir & 2) && v == g.hi0 ? v - 2 : v; };
    auto my = [&](int v) { return (g.mir & 4) && v == g.lo1 - 1 ? v + 2 : (g.mir & 8) && v == g.hi1 ? v - 2 : v; };
    auto mz = [&](int v) { return (g.mir & 16) && v == g.lo2 - 1 ? v + 2 : (g.mir & 32) && v == g.hi2 ? v - 2 : v; };
    const long long hbase = (long long)g.ox + mx(hi) + (long long)g.px * my(hj);
    const T cx = (T)g.cx, cy = (T)g.cy, cz = (T)g.cz;

    using Raw = typename RawOf<Op, T>::type;
    using Ox = typename OxOf<Op>::type;
    bool act[kRY], inb[kRY];
    long long base[kRY];
    // per row q: values of planes k-1, k, k+1; raw loads of planes k (centre,
    // for the output), k+1 and k+2; the output's extra loads for planes k, k+1
    T vm[kRY], vc[kRY], vp[kRY];
    Raw rc[kRY], r1[kRY], r2[kRY];
    Ox oc[kRY], on[kRY];
#pragma unroll
    for (int q = 0; q < kRY; ++q) {
        const int j = jt + ly + q * kSTY;
        act[q] = (i < g.hi0) && (j < g.hi1);
        inb[q] = (i <= g.hi0) && (j <= g.hi1);
        base[q] = (long long)g.ox + mx(i) + (long long)g.px * my(j);
        vm[q] = inb[q] ? st_value<Op, T>(op, st_raw<Op, T>(op, base[q] + g.plane * mz(k0 - 1))) : T(0);
        rc[q] = inb[q] ? st_raw<Op, T>(op, base[q] + g.plane * k0) : Raw{};
        r1[q] = inb[q] ? st_raw<Op, T>(op, base[q] + g.plane * mz(k0 + 1)) : Raw{};
        if (act[q]) oc[q] = st_ox<NT>(op, base[q] + g.plane * k0);
        vc[q] = inb[q] ? st_value<Op, T>(op, rc[q]) : T(0);
    }
    double acc[NQ > 0 ? NQ : 1];
#pragma unroll
    for (int q = 0; q < (NQ > 0 ? NQ : 1); ++q) acc[q] = 0.0;

    Raw hc = hin ? st_raw<Op, T>(op, hbase + g.plane * k0) : Raw{};
    Raw h1 = (hin && k0 + 1 < k1) ? st_raw<Op, T>(op, hbase + g.plane * (k0 + 1)) : Raw{};
    int buf = 0;
    for (int k = k0; k < k1; ++k) {
        // loads first: plane k+2 (used from the next step on), the output's
        // loads of plane k+1, the halo of plane k+2
        const bool more = k + 1 < k1;
#pragma unroll
        for (int q = 0; q < kRY; ++q) {
            if (inb[q] && more) r2[q] = st_raw<Op, T>(op, base[q] + g.plane * mz(k + 2));
            if (act[q] && more) on[q] = st_ox<NT>(op, base[q] + g.plane * (k + 1));
        }
        Raw h2{};
        if (hin && k + 2 < k1) h2 = st_raw<Op, T>(op, hbase + g.plane * (k + 2));
        // plane k+1's values: its loads were issued one step ago
#pragma unroll
        for (int q = 0; q < kRY; ++q) vp[q] = inb[q] ? st_value<Op, T>(op, r1[q]) : T(0);
#pragma unroll
        for (int q = 0; q < kRY; ++q) lds[buf][ly + q * kSTY + 1][lx + 1] = vc[q];
        if (hv) lds[buf][hr][hc_] = hin ? st_value<Op, T>(op, hc) : T(0);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kRY; ++q) {
            if (act[q]) {
                const int r = ly + q * kSTY + 1;
                const T v = vc[q];
                const T Av = cx * ((lds[buf][r][lx] - v) + (lds[buf][r][lx + 2] - v)) +
                             cy * ((lds[buf][r - 1][lx + 1] - v) + (lds[buf][r + 1][lx + 1] - v)) +
                             cz * ((vm[q] - v) + (vp[q] - v));
                st_out<NT, Op, T>(op, base[q] + g.plane * k, v, Av, rc[q], oc[q], acc);
            }
            vm[q] = vc[q];
            vc[q] = vp[q];
            rc[q] = r1[q];
            r1[q] = r2[q];
            oc[q] = on[q];
        }
        hc = h1;
        h1 = h2;
        buf ^= 1;
    }
    if constexpr (NQ > 0) block_partials<NQ, kSThreads>(acc, rb, (int)blockIdx.x);
}

// Vector kernels: one-shot blocks on a 3-D grid (segment of an x-row, y, z).
// A block of BT threads covers BT * E consecutive points of one row, thread t
// taking points t, t + BT, ... (coalesced for every e); all of a thread's
// loads are issued before its first store, and consecutive blocks cover
// consecutive addresses, so the blocks in flight stream one compact window of
// memory.  The grid coordinates are the row and segment, so a block spends no
// instructions finding them.  With a few hundred bytes per wave, the per-wave
// prologue, the bytes in flight per thread and the block reduction are what
// separate these kernels from a flat copy: ops that fetch 16 bytes or more per
// point run 512 x 1, ops that fetch 8 bytes or less (FP32 fields) 128 x 4.
// (Measured on a 512^3 update r -= a Ap with r.r and r.(jac r) partials:
// FP64 256 x 1 5.6 TB/s, 512 x 1 5.8, where z-marching 64 x 4 x 32 tiles
// reached 5.1-5.35; FP32 128 x 4 5.2 TB/s where 256 x 1 reached 3.9.)
template <class Op>
struct VecShape {
    static constexpr int E = sizeof(typename Op::R) <= 8 ? 4 : 1;
    static constexpr int BT = E == 1 ? 512 : 128;
};

// segment `seg` of row (j, k): the block's BT * E points
template <bool NT, class Op>
__device__ __forceinline__ void vector_segment(const Geo& g, const Op& op, int seg, int j, int k, double* acc)
{
    constexpr int E = VecShape<Op>::E, BT = VecShape<Op>::BT;
    const int i0 = g.lo0 + seg * (BT * E) + (int)threadIdx.x;
    const long long row = (long long)g.ox + (long long)g.px * j + g.plane * k;
    typename Op::R r[E];
#pragma unroll
    for (int e = 0; e < E; ++e)
        if (i0 + e * BT < g.hi0) r[e] = op.template fetch<NT>(row + i0 + e * BT);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = i0 + e * BT;
        if (i < g.hi0) op.template apply<NT>(row + i, r[e], i, j, k, acc);
    }
}

template <int NQ, class Op, bool NT>
__global__ __launch_bounds__(VecShape<Op>::BT) void k_vector(Geo g, Op op, RedBuf rb)
{
    if (op.gated()) return;
    op.load();
    double acc[NQ > 0 ? NQ : 1];
#pragma unroll
    for (int q = 0; q < (NQ > 0 ? NQ : 1); ++q) acc[q] = 0.0;
    vector_segment<NT>(g, op, (int)blockIdx.x, g.lo1 + (int)blockIdx.y, g.lo2 + (int)blockIdx.z, acc);
    if constexpr (NQ > 0)
        block_partials<NQ, VecShape<Op>::BT>(acc, rb,
                                             (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)));
}

// sums of kSpan consecutive block partials, one block per span, fixed order
template <int NQ, class Op>
__global__ __launch_bounds__(kThreads) void k_span(Op op, RedBuf rb, int nblocks)
{
    if (op.gated()) return;
    const int b0 = blockIdx.x * kSpan, b1 = min(nblocks, b0 + kSpan);
    double acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
    for (int b = b0 + (int)threadIdx.x; b < b1; b += kThreads) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[q] += rb.partials[(size_t)q * rb.cap + b];
    }
    double tot[NQ];
    block_sum<NQ, kThreads>(acc, tot);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) rb.partials2[(size_t)q * rb.cap2 + blockIdx.x] = tot[q];
    }
}

// the epilogue of a reducing launch of nblocks blocks: one level of span sums
// first when there are many partials and the workspace has room for them
template <int NQ, class Op>
static void launch_finish(hipStream_t s, const Op& op, RedBuf rb, int nblocks)
{
    const int nspan = (nblocks + kSpan - 1) / kSpan;
    if (nblocks > 4 * kSpan && rb.partials2 != nullptr && nspan <= rb.cap2) {
        hipLaunchKernelGGL((k_span<NQ, Op>), dim3(nspan), dim3(kThreads), 0, s, op, rb, nblocks);
        RedBuf r2 = rb;
        r2.partials = rb.partials2;
        r2.cap = rb.cap2;
        hipLaunchKernelGGL((k_finish<NQ, Op>), dim3(1), dim3(kFinThreads), 0, s, op, r2, nspan);
    } else {
        hipLaunchKernelGGL((k_finish<NQ, Op>), dim3(1), dim3(kFinThreads), 0, s, op, rb, nblocks);
    }
}

template <int NQ, class Op>
static bool check_capacity(const Geo& g, const RedBuf& rb)
{
    if (NQ > 0 && g.nblocks > rb.cap) {
        std::fprintf(stderr, "pps: %d blocks exceed the reduction workspace (%d); launch skipped\n", g.nblocks, rb.cap);
        return false;
    }
    return true;
}

// tiling of a stencil launch: the z-chunk set on the context, or (kz_st = 0)
// the longest of 64, 32, 16, 8 planes that still gives 2048 blocks (a longer
// chunk re-reads fewer halo planes; 2048 blocks keep every CU busy to the end);
// below 1024 blocks of 8 planes, 4 or 2 planes (a small grid's time is the
// planes that one block marches through)
static Geo stencil_geo(const Geo& g0)
{
    if (g0.kz_st > 0) return retile(g0, kTH, g0.kz_st);
    int kz = 64;
    Geo g = retile(g0, kTH, kz);
    while ((kz > 8 && g.nblocks < 2048) || (kz > 2 && g.nblocks < 1024)) {
        kz /= 2;
        g = retile(g0, kTH, kz);
    }
    return g;
}

template <typename T, int NQ, class Op>
static void run_stencil(const Geo& g0, hipStream_t s, const Op& op, RedBuf rb)
{
    const Geo g = stencil_geo(g0);
    if (g.nblocks <= 0 || !check_capacity<NQ, Op>(g, rb)) return;
    if (g.nt) hipLaunchKernelGGL((k_stencil<T, NQ, Op, true>), dim3(g.nblocks), dim3(kTX, kSTY), 0, s, g, op, rb);
    else hipLaunchKernelGGL((k_stencil<T, NQ, Op, false>), dim3(g.nblocks), dim3(kTX, kSTY), 0, s, g, op, rb);
    if constexpr (NQ > 0) launch_finish<NQ>(s, op, rb, g.nblocks);
}

template <int NQ, class Op>
static void run_vector(const Geo& g0, hipStream_t s, const Op& op, RedBuf rb)
{
    const int nx = g0.hi0 - g0.lo0, ny = g0.hi1 - g0.lo1, nz = g0.hi2 - g0.lo2;
    if (nx <= 0 || ny <= 0 || nz <= 0) return;
    constexpr int W = VecShape<Op>::BT * VecShape<Op>::E;
    const int nseg = (nx + W - 1) / W;
    const long long nb = (long long)nseg * ny * nz;
    if (nb > 0x7FFFFFFFll || ny > 65535 || nz > 65535) {
        std::fprintf(stderr, "pps: a %d x %d x %d region exceeds a vector launch; launch skipped\n", nx, ny, nz);
        return;
    }
    Geo g = g0;
    g.nblocks = (int)nb;
    if (!check_capacity<NQ, Op>(g, rb)) return;
    const dim3 grid(nseg, ny, nz);
    const dim3 block(VecShape<Op>::BT);
    if (g.nt) hipLaunchKernelGGL((k_vector<NQ, Op, true>), grid, block, 0, s, g, op, rb);
    else hipLaunchKernelGGL((k_vector<NQ, Op, false>), grid, block, 0, s, g, op, rb);
    if constexpr (NQ > 0) launch_finish<NQ>(s, op, rb, g.nblocks);
}

static const RedBuf kNoRed{nullptr, nullptr, 0, nullptr, 0};

struct Empty {};

// ------------------------------------------------------------ basic kernels

template <typename T>
struct OpApply : Gate {
    const T* __restrict__ x;
    T* __restrict__ y;
    __device__ void load() {}
    __device__ T in(long long c) const { return x[c]; }
    template <bool NT> __device__ void out(long long c, T, T Av, double*) const { put<NT>(y + c, Av); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_apply_A(const Geo& g, hipStream_t s, const T* x, T* y)
{
    OpApply<T> op;
    op.gate = nullptr;
    op.x = x;
    op.y = y;
    run_stencil<T, 0>(g, s, op, kNoRed);
}

template <typename T>
struct OpCopy : Gate {
    const T* __restrict__ x;
    T* __restrict__ y;
    struct R { T a; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(x + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& r, int, int, int, double*) const { put<NT>(y + c, r.a); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_copy(const Geo& g, hipStream_t s, const T* x, T* y)
{
    OpCopy<T> op;
    op.gate = nullptr;
    op.x = x;
    op.y = y;
    run_vector<0>(g, s, op, kNoRed);
}

// plain copy of n contiguous doubles, 16 bytes per lane with non-temporal
// loads and stores: the HBM ceiling the field kernels are measured against
typedef double d2_t __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(256) void k_copy_flat(const double* __restrict__ x, double* __restrict__ y, long long n)
{
    const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 2;
    if (i + 1 < n) {
        const d2_t v = __builtin_nontemporal_load(reinterpret_cast<const d2_t*>(x + i));
        __builtin_nontemporal_store(v, reinterpret_cast<d2_t*>(y + i));
    } else if (i < n) {
        y[i] = x[i];
    }
}

void launch_copy_flat(hipStream_t s, const double* x, double* y, long long n)
{
    const long long blocks = (n + 511) / 512;
    if (blocks > 0) hipLaunchKernelGGL(k_copy_flat, dim3((unsigned)blocks), dim3(256), 0, s, x, y, n);
}

template <typename T>
struct OpDot : Gate {
    const T* __restrict__ a;
    const T* __restrict__ b;
    double* out;
    struct R { T a, b; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(a + c), ld<NT>(b + c)}; }
    template <bool NT> __device__ void apply(long long, const R& r, int, int, int, double* acc) const { acc[0] += (double)r.a * (double)r.b; }
    __device__ void finish(const double* t) { *out = t[0]; }
};

template <typename T>
void launch_dot(const Geo& g, hipStream_t s, RedBuf rb, const T* a, const T* b, double* out, const int* gate)
{
    OpDot<T> op;
    op.gate = gate;
    op.a = a;
    op.b = b;
    op.out = out;
    run_vector<1>(g, s, op, rb);
}

template <typename T>
struct OpFill : Gate {
    T* __restrict__ a;
    T v;
    using R = Empty;
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long) const { return {}; }
    template <bool NT> __device__ void apply(long long c, const R&, int, int, int, double*) const { put<NT>(a + c, v); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_fill(const Geo& g, hipStream_t s, T* a, T v)
{
    OpFill<T> op;
    op.gate = nullptr;
    op.a = a;
    op.v = v;
    run_vector<0>(g, s, op, kNoRed);
}

template <typename T>
struct OpScaleBox : Gate {
    T* __restrict__ a;
    const Scal* S;
    int mode;
    double nrm;
    struct R { T a; };
    __device__ void load() { nrm = S->v[S_NORM]; }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(a + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& r, int, int, int, double*) const
    {
        // normalizeProblemToFieldBNorm divides (iterativeSolverBase.hpp:227-231);
        // the solvers' epilogues multiply (baseCG.hpp:248-252)
        if (mode == 0) put<NT>(a + c, (T)((double)r.a / nrm));
        else put<NT>(a + c, (T)((double)r.a * nrm));
    }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_scale_box(const Geo& gbox, hipStream_t s, T* a, const Scal* S, int mode)
{
    OpScaleBox<T> op;
    op.gate = nullptr;
    op.a = a;
    op.S = S;
    op.mode = mode;
    run_vector<0>(gbox, s, op, kNoRed);
}

template <typename T>
struct OpPointwise : Gate {
    const T* __restrict__ in;
    T* __restrict__ out;
    T c;
    struct R { T a; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long p) const { return {ld<NT>(in + p)}; }
    template <bool NT> __device__ void apply(long long p, const R& r, int, int, int, double*) const { put<NT>(out + p, c * r.a); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_pointwise(const Geo& gbox, hipStream_t s, const T* in, T* out, double c, const int* gate)
{
    OpPointwise<T> op;
    op.gate = gate;
    op.in = in;
    op.out = out;
    op.c = (T)c;
    run_vector<0>(gbox, s, op, kNoRed);
}

template <typename TS, typename TD>
struct OpCast : Gate {
    const TS* __restrict__ src;
    TD* __restrict__ dst;
    struct R { TS a; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(src + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& r, int, int, int, double*) const { put<NT>(dst + c, (TD)r.a); }
    __device__ void finish(const double*) {}
};

template <typename TS, typename TD>
void launch_cast(const Geo& gbox, hipStream_t s, const TS* src, TD* dst, const int* gate)
{
    OpCast<TS, TD> op;
    op.gate = gate;
    op.src = src;
    op.dst = dst;
    run_vector<0>(gbox, s, op, kNoRed);
}

// ---------------------------------------------------- residual and b-norm

// r = b - A x (iterativeSolverBase.hpp:257-268)
struct OpResidual : Gate {
    const double* __restrict__ x;
    const double* __restrict__ b;
    double* __restrict__ r;
    Scal* S;
    int mode;
    __device__ void load() {}
    struct Ox { double b; };
    __device__ double in(long long c) const { return x[c]; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(b + c)}; }
    template <bool NT> __device__ void out(long long c, double, double Av, const double&, const Ox& o, double* acc) const
    {
        const double rv = o.b - Av;
        put<NT>(r + c, rv);
        acc[0] += rv * rv;
    }
    __device__ void finish(const double* t)
    {
        const double e = sqrt(t[0]);
        if (mode == 0) {
            S->v[S_ERR0] = e;
            S->v[S_ERR] = e;
            S->v[S_ERR_OP] = e;
            S->v[S_RR] = t[0];
            S->v[S_BETA] = 0.0;
            S->v[S_RHO0] = 1.0;
            S->v[S_ALPHA] = 0.0;  // no pending x update before the first iteration
            S->iter = 0;
            if (S->hist != nullptr && S->hist_cap > 0) S->hist[0] = e;
            S->done = (e < S->v[S_TOL]) ? 2 : 0;
        } else if (mode == 1) {
            S->v[S_ERR_OP] = e;
        } else {
            // residual replacement after a recursive stop: r now holds the true
            // residual of the complete x; the loop resumes from it unless it is
            // below the tolerance or the iteration cap is reached
            S->v[S_ERR_OP] = e;
            S->v[S_RR] = t[0];
            S->v[S_ALPHA] = 0.0;  // x is complete: no pending update
            if (mode == 3) S->v[S_RHO0] = t[0]; // BiCGSTAB restarted with r0 = r: rho = r0.r
            S->done = (e < S->v[S_TOL] || S->iter >= S->maxit) ? 1 : 0;
        }
    }
};

void launch_residual(const Geo& g, hipStream_t s, RedBuf rb, const double* x, const double* b, double* r, Scal* S, int mode)
{
    OpResidual op;
    op.gate = nullptr;
    op.x = x;
    op.b = b;
    op.r = r;
    op.S = S;
    op.mode = mode;
    run_stencil<double, 1>(g, s, op, rb);
}

// r = b - A x and ||r|| into one device double: the residual above without a
// solver's scalar block, for callers that bring their own fields and partials
struct OpResidualNorm : Gate {
    const double* __restrict__ x;
    const double* __restrict__ b;
    double* __restrict__ r;
    double* norm;
    __device__ void load() {}
    struct Ox { double b; };
    __device__ double in(long long c) const { return x[c]; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(b + c)}; }
    template <bool NT> __device__ void out(long long c, double, double Av, const double&, const Ox& o, double* acc) const
    {
        const double rv = o.b - Av;
        put<NT>(r + c, rv);
        acc[0] += rv * rv;
    }
    __device__ void finish(const double* t) { *norm = sqrt(t[0]); }
};

int launch_residual_norm(const Geo& g, hipStream_t s, RedBuf rb, const double* x, const double* b, double* r, double* out)
{
    const Geo gt = stencil_geo(g);
    if (gt.nblocks > rb.cap) return -1;
    OpResidualNorm op;
    op.gate = nullptr;
    op.x = x;
    op.b = b;
    op.r = r;
    op.norm = out;
    run_stencil<double, 1>(g, s, op, rb);
    return 0;
}

// boundary adjustment of b at one point (adjustFieldBForDirichletNeumanBCs,
// iterativeSolverBase.hpp:429-534): Dirichlet faces subtract the boundary value
// of x over ds^2 on the first interior layer, Neumann faces add -+ 2 du/dn / ds
// on the boundary layer; applied in the reference's face order x- x+ y- y+ z- z+
struct BAdjust {
    const double* __restrict__ x;
    const double* flux[6];
    int bc[6], ld[6], fng[6][2];
    double ds[3];
    long long stride[3];
    __device__ long long fpos(int d, int i, int j, int k) const
    {
        const int f = 2 * d;
        if (d == 0) return j + (long long)fng[f][0] * k;
        if (d == 1) return i + (long long)fng[f][0] * k;
        return i + (long long)fng[f][0] * j;
    }
    __device__ double adjust(double v, long long c, int i, int j, int k) const
    {
        const int idx[3] = {i, j, k};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double dd = ds[d] * ds[d];
            if (bc[2 * d] == 0) {
                if (idx[d] == ld[2 * d] + 1) v -= x[c - stride[d]] / dd;
            } else if (bc[2 * d] == 1 && flux[2 * d] != nullptr) {
                if (idx[d] == ld[2 * d]) v += 2 * flux[2 * d][fpos(d, i, j, k)] / ds[d];
            }
            if (bc[2 * d + 1] == 0) {
                if (idx[d] == ld[2 * d + 1] - 2) v -= x[c + stride[d]] / dd;
            } else if (bc[2 * d + 1] == 1 && flux[2 * d + 1] != nullptr) {
                if (idx[d] == ld[2 * d + 1] - 1) v -= 2 * flux[2 * d + 1][fpos(d, i, j, k)] / ds[d];
            }
        }
        return v;
    }
};

static BAdjust make_badjust(const Geo& g, const double* x, const int bc[6], const int lim_data[6],
                            const double* const flux[6], const int fng[6][2], const double ds[3])
{
    BAdjust a;
    a.x = x;
    for (int f = 0; f < 6; ++f) {
        a.flux[f] = flux[f];
        a.bc[f] = bc[f];
        a.ld[f] = lim_data[f];
        a.fng[f][0] = fng[f][0];
        a.fng[f][1] = fng[f][1];
    }
    for (int d = 0; d < 3; ++d) a.ds[d] = ds[d];
    a.stride[0] = 1;
    a.stride[1] = g.px;
    a.stride[2] = g.plane;
    return a;
}

// ||b_adj||^2 over the solver region (iterativeSolverBase.hpp:171-201)
struct OpBNorm : Gate {
    const double* __restrict__ b;
    BAdjust adj;
    Scal* S;
    struct R { double b; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(b + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& r, int i, int j, int k, double* acc) const
    {
        const double v = adj.adjust(r.b, c, i, j, k);
        acc[0] += v * v;
    }
    __device__ void finish(const double* t) { S->v[S_NORM] = sqrt(t[0]); }
};

void launch_bnorm(const Geo& g, hipStream_t s, RedBuf rb, const double* x, const double* b, const int bc[6],
                  const int lim_data[6], const int lim_solver[6], const double* const flux[6], const int fng[6][2],
                  const double ds[3], Scal* S)
{
    (void)lim_solver;
    OpBNorm op;
    op.gate = nullptr;
    op.b = b;
    op.adj = make_badjust(g, x, bc, lim_data, flux, fng, ds);
    op.S = S;
    run_vector<1>(g, s, op, rb);
}

// the adjusted right-hand side written in place over the data region (the
// main-loop Chebyshev works on this copy; chebyshevIteration.hpp:61-67)
struct OpAdjustB : Gate {
    double* __restrict__ b;
    BAdjust adj;
    struct R { double b; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(b + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& r, int i, int j, int k, double*) const { put<NT>(b + c, adj.adjust(r.b, c, i, j, k)); }
    __device__ void finish(const double*) {}
};

void adjust_b_field(const Geo& gdata, hipStream_t s, const double* x, double* b, const int bc[6], const int lim_data[6],
                    const double* const flux[6], const int fng[6][2], const double ds[3])
{
    OpAdjustB op;
    op.gate = nullptr;
    op.b = b;
    op.adj = make_badjust(gdata, x, bc, lim_data, flux, fng, ds);
    run_vector<0>(gdata, s, op, kNoRed);
}

// ------------------------------------------------------- Neumann ghost fill

// iterativeSolverBase.hpp:62-169 (orderNeumanBcs == 2): the guard point of a
// Neumann face takes the value of the data point mirrored through the face
// point; data fields add -+ 2 ds du/dn / normFieldB_.
template <typename T>
__global__ __launch_bounds__(256) void k_ghost(Layout L, Faces F, T* field, int with_flux, const Scal* S, const int* gate)
{
    if (gate != nullptr && *gate != 0) return;
    const int slot = blockIdx.y;
    const int f = F.face[slot];
    const int d = f >> 1, side = f & 1;
    const int d1 = d == 0 ? 1 : 0, d2 = d == 2 ? 1 : 2;
    const int n1 = F.lim_data[2 * d1 + 1] - F.lim_data[2 * d1];
    const int n2 = F.lim_data[2 * d2 + 1] - F.lim_data[2 * d2];
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n1 * n2) return;
    int idx[3];
    idx[d1] = F.lim_data[2 * d1] + (int)(t % n1);
    idx[d2] = F.lim_data[2 * d2] + (int)(t / n1);
    idx[d] = side == 0 ? F.lim_data[2 * d] : F.lim_data[2 * d + 1] - 1;
    const long long e = d == 0 ? 1 : (d == 1 ? (long long)L.px : L.plane);
    const long long p = L.at(idx[0], idx[1], idx[2]);
    const long long guard = side == 0 ? p - e : p + e;
    const long long data = side == 0 ? p + e : p - e;
    if (with_flux && F.flux[slot] != nullptr) {
        const double nrm = S != nullptr ? S->v[S_NORM] : 1.0;
        const double q = F.flux[slot][idx[d1] + (long long)F.fng[f][0] * idx[d2]];
        const double v = (double)field[data];
        field[guard] = (T)(side == 0 ? v - 2 * F.ds[d] * q / nrm : v + 2 * F.ds[d] * q / nrm);
    } else {
        field[guard] = field[data];
    }
}

template <typename T>
void launch_ghost(hipStream_t s, const Layout& L, const Faces& F, T* field, int with_flux, const Scal* S, const int* gate)
{
    if (F.n == 0) return;
    int maxpts = 0;
    for (int q = 0; q < F.n; ++q) {
        const int f = F.face[q], d = f >> 1;
        const int d1 = d == 0 ? 1 : 0, d2 = d == 2 ? 1 : 2;
        const int pts = (F.lim_data[2 * d1 + 1] - F.lim_data[2 * d1]) * (F.lim_data[2 * d2 + 1] - F.lim_data[2 * d2]);
        if (pts > maxpts) maxpts = pts;
    }
    dim3 grid((maxpts + 255) / 256, F.n);
    hipLaunchKernelGGL(k_ghost<T>, grid, dim3(256), 0, s, L, F, field, with_flux, S, gate);
}

// ------------------------------------ pieces of the multi-level marching kernels
// (k_cg_pass, k_cheb_multi: several applications of A per pass, on a tile and rings around it)

template <typename T>
__device__ __forceinline__ T lap7(T v, T xm, T xp, T ym, T yp, T zm, T zp, T cx, T cy, T cz)
{
    const T dx = (xm - v) + (xp - v), dy = (ym - v) + (yp - v), dz = (zm - v) + (zp - v);
    return fma(cx, dx, fma(cy, dy, cz * dz));
}

// Raw buffer access to one plane of a field, relative to a tile's origin: a load
// whose byte offset is at or beyond num_records returns 0 and such a store is
// dropped, so points off the solver region (offset kOob) and planes off it
// (num_records 0) need no branch and no mask around the access.  The aux bit
// stores non-temporally.
constexpr unsigned kOob = 0x80000000u;
constexpr int kInRange = 0x7fffffff;
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const T* p, bool ok)
{
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    void* q = (void*)(((unsigned long long)hi << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(q, (short)0, ok ? kInRange : 0, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t r, unsigned off)
{
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <bool NT, typename T>
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t r, unsigned off, T v)
{
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), r, off, 0, NT ? 2 : 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, NT ? 2 : 0);
}

// point t of the ring around a box of W x H points -> (row, col) in the box's frame
template <int W, int H>
__device__ __forceinline__ void ring_point(int t, int& r, int& c)
{
    if (t < W + 2) { r = -1; c = t - 1; }
    else if (t < 2 * (W + 2)) { r = H; c = t - (W + 2) - 1; }
    else if (t < 2 * (W + 2) + H) { r = t - 2 * (W + 2); c = -1; }
    else { r = t - 2 * (W + 2) - H; c = W; }
}

int cu_count()
{
    static const int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            return v;
        return 256;
    }();
    return n;
}

// z-chunk of a marching kernel whose blocks take kz + extra steps and of which
// per_cu (1 or 2) fit on a CU: the one with the least time on the busiest CU (the
// longest of equals, up to 128 planes).  Two blocks that share a CU take 1.5 times
// as long as one alone (Chebyshev(11), Dirichlet, us per BiCGSTAB iteration, chunk
// of one / two blocks per CU: 98^3 200 / 215, 130^3 258 / 270).
static int pick_kz(long long tiles, int nz, int per_cu, int extra)
{
    int best = 1;
    double cost = -1.0;
    const int cus = cu_count();
    for (int kz = 1; kz <= 128; ++kz) {
        if (kz > 1 && kz > nz) break;
        const long long n = (tiles * ((nz + kz - 1) / kz) + cus - 1) / cus;  // blocks of the busiest CU
        const double c = (per_cu == 2 ? (n / 2) * 1.5 + n % 2 : (double)n) * (std::min(kz, nz) + extra);
        if (cost < 0.0 || c <= cost) {
            cost = c;
            best = kz;
        }
    }
    return best;
}

// ------------------------------------------------------------------- CG

// One CG iteration in one pass over the grid (pointwise preconditioner M = jac I;
// baseCG.hpp:126-207 has two reductions and a pass for each):
//   r = r_old - alpha_old A p_old      the previous iteration's update
//   p = jac r + beta p_old             the new direction
//   sums r.r, p.Ap, r.Ap, Ap.Ap        finish: alpha = jac r.r / p.Ap and
//   ||r - alpha Ap||^2 = r.r - 2 alpha r.Ap + alpha^2 Ap.Ap, hence beta and the
//   convergence test, before the next residual has been formed.
// A p_old is recomputed from p_old instead of being stored, so a pass reads
// r_old and p_old and writes r and p: 4 words per point and iteration where a
// stencil pass plus an update pass move 7.  r.r is summed from the residual
// itself in every pass; the expansion only predicts the next one.  It loses
// digits when one step removes most of r: below kCgRecheck r.r the next pass
// only forms r (p is kept, no iteration is counted) and beta and the
// convergence test take its sum.
//
// Measured at 512^3 FP64: 0.85 ms for its 4 words (5.06 TB/s; 5.4 with the rings'
// re-reads that miss L2, 1.14x on the reads), where the stencil and update
// passes took 0.83 + 0.53 ms; 1.10 against 1.60 ms per iteration with x's
// deferred updates.  The HBM rate is that of the other marching stencils.  FP32:
// 0.47 ms (4.6 TB/s; 5.7 with the re-reads, 1.52x on the reads).
//
// A block owns a 64 x (8 RY) tile and marches z.  It forms p on the tile and a
// one-point ring, from p_old on the tile and a two-point ring; a thread owns RY
// consecutive rows of one column (their y-neighbours are its own registers)
// and at most one point of each ring.  Per plane: p_old of plane s goes to
// LDS, one barrier, then p of plane s (to the other LDS array) and A p of plane
// s - 1, whose neighbours went to LDS one plane earlier.  Both arrays alternate
// between two planes, so one barrier separates every write from its readers:
// p_old's buffer is rewritten two steps later, after the barrier that all its
// readers have passed, and p of plane s - 1 was written before this plane's
// barrier.  Every rounding is spelled out (explicit fma, or none) so that a ring
// point and the tile point it mirrors in the neighbouring block round alike.
constexpr double kCgRecheck = 1e-2;  // beta's relative error stays near eps / kCgRecheck
constexpr int kCgW = 8;              // wavefronts per block

// p = z + beta p_old with z = jac r, each product rounded, as the reference
// forms it (baseCG.hpp:139,199-203)
template <typename T>
__device__ __forceinline__ T cg_direction(T r, T p_old, T jac, T beta)
{
#pragma clang fp contract(off)
    const T z = jac * r, bp = beta * p_old;
    return z + bp;
}

template <typename T>
struct CgPassArgs {
    const T* __restrict__ r_in;
    const T* __restrict__ pin;
    T* __restrict__ r_out;
    T* __restrict__ pout;
    T* __restrict__ x;  // null: x's updates are deferred to the ring's flush
    const Scal* S;
};

template <typename T, int RY, bool XUPD, bool NT>
__global__ __launch_bounds__(kTX* kCgW) void k_cg_pass(Geo g, CgPassArgs<T> A, RedBuf rb)
{
    if (A.S->done) return;
    constexpr int TY = kCgW * RY;
    constexpr int N1 = 2 * (kTX + 2) + 2 * TY, N2 = 2 * (kTX + 4) + 2 * (TY + 2);
    static_assert(N1 <= kTX * kCgW && N2 <= kTX * kCgW, "ring points need one thread each");
    __shared__ T ysl[2][TY + 4][kTX + 4];  // p_old, tile and two-point ring
    __shared__ T wsl[2][TY + 2][kTX + 2];  // p, tile and one-point ring
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int tx0 = b % g.ntx, rr = b / g.ntx;
    const int ty0 = rr % g.nty, tz0 = rr / g.nty;
    const int i0 = g.lo0 + tx0 * kTX, j0 = g.lo1 + ty0 * TY;
    const int k0 = g.lo2 + tz0 * g.kz, k1 = min(k0 + g.kz, g.hi2);
    const int lx = threadIdx.x, ly = threadIdx.y, tid = lx + kTX * ly;
    const T cx = (T)g.cx, cy = (T)g.cy, cz = (T)g.cz;
    const bool recheck = A.S->recheck != 0;
    const T alpha = (T)A.S->v[S_ALPHA];
    const T beta = recheck ? T(1) : (T)A.S->v[S_BETA];
    const T jac = recheck ? T(0) : (T)A.S->v[S_JAC];

    // points of this thread: RY tile rows, one point of each ring; a point off
    // the solver region holds 0 and is never loaded
    const long long px = g.px;
    const long long t0 = (long long)g.ox + (i0 + lx) + px * (j0 + ly * RY);
    bool in[RY];
#pragma unroll
    for (int q = 0; q < RY; ++q) in[q] = i0 + lx < g.hi0 && j0 + ly * RY + q < g.hi1;
    int r1 = 0, c1 = 0, r2 = 0, c2 = 0;
    const bool has1 = tid < N1, has2 = tid < N2;
    if (has1) ring_point<kTX, TY>(tid, r1, c1);
    if (has2) {
        ring_point<kTX + 2, TY + 2>(tid, r2, c2);
        r2 -= 1;
        c2 -= 1;
    }
    auto inxy = [&](int i, int j) { return i >= g.lo0 && i < g.hi0 && j >= g.lo1 && j < g.hi1; };
    const bool in1 = has1 && inxy(i0 + c1, j0 + r1), in2 = has2 && inxy(i0 + c2, j0 + r2);
    const long long o1 = (long long)g.ox + (i0 + c1) + px * (j0 + r1);
    const long long o2 = (long long)g.ox + (i0 + c2) + px * (j0 + r2);

    T pm[RY], pc[RY], pp[RY], pn[RY], rc[RY], rn[RY], rv[RY], wm[RY], wc[RY], wn[RY], xc[RY], xn[RY];
    T qm = 0, qc = 0, qp = 0, qn = 0, qr = 0, qrn = 0, oc = 0, on = 0;
    auto zin = [&](int k) { return k >= g.lo2 && k < g.hi2; };
    const int s0 = k0 - 1;
    {
        const bool za = zin(s0 - 1), zb = zin(s0), zc = zin(s0 + 1);
        const long long fa = g.plane * (s0 - 1), fb = g.plane * s0, fc = g.plane * (s0 + 1);
#pragma unroll
        for (int q = 0; q < RY; ++q) {
            pm[q] = in[q] && za ? A.pin[t0 + px * q + fa] : T(0);
            pc[q] = in[q] && zb ? A.pin[t0 + px * q + fb] : T(0);
            pp[q] = in[q] && zc ? A.pin[t0 + px * q + fc] : T(0);
            rc[q] = in[q] && zb ? A.r_in[t0 + px * q + fb] : T(0);
            pn[q] = rn[q] = rv[q] = wm[q] = wc[q] = wn[q] = xc[q] = xn[q] = T(0);
        }
        if (in1) {
            qm = za ? A.pin[o1 + fa] : T(0);
            qc = zb ? A.pin[o1 + fb] : T(0);
            qp = zc ? A.pin[o1 + fc] : T(0);
            qr = zb ? A.r_in[o1 + fb] : T(0);
        }
        if (in2 && zb) oc = A.pin[o2 + fb];
    }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int s = s0; s <= k1; ++s) {
        const int buf = s & 1;
        const long long fs = g.plane * s;
#pragma unroll
        for (int q = 0; q < RY; ++q) ysl[buf][ly * RY + q + 2][lx + 2] = pc[q];
        if (has1) ysl[buf][r1 + 2][c1 + 2] = qc;
        if (has2) ysl[buf][r2 + 2][c2 + 2] = oc;
        // loads for the next step: p_old of plane s + 2 (s + 1 on the outer ring), r_old (and x) of plane s + 1
        const bool z1 = s < k1 && zin(s + 1), z2 = s < k1 && zin(s + 2);
        const long long f1 = fs + g.plane, f2 = f1 + g.plane;
#pragma unroll
        for (int q = 0; q < RY; ++q) {
            pn[q] = in[q] && z2 ? A.pin[t0 + px * q + f2] : T(0);
            rn[q] = in[q] && z1 ? A.r_in[t0 + px * q + f1] : T(0);
            if constexpr (XUPD) xn[q] = in[q] && z1 && s + 1 < k1 ? ld<NT>(A.x + t0 + px * q + f1) : T(0);
        }
        if (in1) {
            qn = z2 ? A.pin[o1 + f2] : T(0);
            qrn = z1 ? A.r_in[o1 + f1] : T(0);
        }
        if (in2) on = z1 ? A.pin[o2 + f1] : T(0);
        __syncthreads();
        const bool zs = zin(s), own = s >= k0 && s < k1;
        T rs[RY];
#pragma unroll
        for (int q = 0; q < RY; ++q) {
            const int r = ly * RY + q + 2, c = lx + 2;
            T w = T(0), v = T(0);
            if (in[q] && zs) {
                const T ym = q > 0 ? pc[q > 0 ? q - 1 : 0] : ysl[buf][r - 1][c];
                const T yp = q + 1 < RY ? pc[q + 1 < RY ? q + 1 : 0] : ysl[buf][r + 1][c];
                const T Ap = lap7(pc[q], ysl[buf][r][c - 1], ysl[buf][r][c + 1], ym, yp, pm[q], pp[q], cx, cy, cz);
                v = fma(-alpha, Ap, rc[q]);
                w = cg_direction(v, pc[q], jac, beta);
                if (own) {
                    put<NT>(A.r_out + t0 + px * q + fs, v);
                    put<NT>(A.pout + t0 + px * q + fs, w);
                    if constexpr (XUPD) put<NT>(A.x + t0 + px * q + fs, fma(alpha, pc[q], xc[q]));
                    acc[0] += (double)v * (double)v;
                }
            }
            rs[q] = v;
            wn[q] = w;
            wsl[buf][r - 1][c - 1] = w;
        }
        if (has1) {
            T w = T(0);
            if (in1 && zs) {
                const int r = r1 + 2, c = c1 + 2;
                const T Ap = lap7(qc, ysl[buf][r][c - 1], ysl[buf][r][c + 1], ysl[buf][r - 1][c], ysl[buf][r + 1][c], qm,
                                  qp, cx, cy, cz);
                w = cg_direction(fma(-alpha, Ap, qr), qc, jac, beta);
            }
            wsl[buf][r1 + 1][c1 + 1] = w;
        }
        // A p of plane s - 1
        if (s > k0) {
            const int pb = buf ^ 1;
#pragma unroll
            for (int q = 0; q < RY; ++q) {
                if (!in[q]) continue;
                const int r = ly * RY + q + 1, c = lx + 1;
                const T ym = q > 0 ? wc[q > 0 ? q - 1 : 0] : wsl[pb][r - 1][c];
                const T yp = q + 1 < RY ? wc[q + 1 < RY ? q + 1 : 0] : wsl[pb][r + 1][c];
                const double Ap = (double)lap7(wc[q], wsl[pb][r][c - 1], wsl[pb][r][c + 1], ym, yp, wm[q], wn[q], cx, cy, cz);
                acc[1] += (double)wc[q] * Ap;
                acc[2] += (double)rv[q] * Ap;
                acc[3] += Ap * Ap;
            }
        }
#pragma unroll
        for (int q = 0; q < RY; ++q) {
            pm[q] = pc[q];
            pc[q] = pp[q];
            pp[q] = pn[q];
            rc[q] = rn[q];
            rv[q] = rs[q];
            wm[q] = wc[q];
            wc[q] = wn[q];
            xc[q] = xn[q];
        }
        qm = qc;
        qc = qp;
        qp = qn;
        qr = qrn;
        oc = on;
    }
    block_partials<4, kTX * kCgW>(acc, rb, (int)blockIdx.x);
}

struct OpCgPass {
    Scal* S;
    bool history;
    int slot;
    __device__ __forceinline__ bool gated() const { return S->done != 0; }
    __device__ void end_iteration(int it, double rr) const
    {
        const double err = sqrt(rr);
        S->v[S_RR] = rr;
        S->v[S_ERR] = err;
        if (history && S->hist != nullptr && it < S->hist_cap) S->hist[it] = err;
        if (err < S->v[S_TOL] || it >= S->maxit) S->done = 1;
    }
    __device__ void finish(const double* t) const
    {
        const double rr = t[0];
        S->passes += 1;
        if (S->recheck) {
            // the pass formed r (x has its step already) and kept p
            S->recheck = 0;
            S->v[S_BETA] = rr > 0.0 ? rr / S->v[S_RR] : 0.0;
            S->v[S_ALPHA] = 0.0;
            if (slot >= 0) S->ahist[slot] = 0.0;
            end_iteration(S->iter, rr);
            return;
        }
        // r = 0: x is exact and no step follows
        const double rz = S->v[S_JAC] * rr, a = rr == 0.0 ? 0.0 : rz / t[1];
        S->v[S_RZ] = rz;
        S->v[S_PAP] = t[1];
        S->v[S_ALPHA] = a;
        if (slot >= 0) S->ahist[slot] = a;
        S->iter += 1;
        const double next = rr - 2.0 * a * t[2] + a * a * t[3];
        if (next > kCgRecheck * rr) {
            S->v[S_BETA] = next / rr;
            end_iteration(S->iter, next);
        } else {
            S->v[S_RR] = rr;
            S->recheck = 1;
        }
    }
};

template <typename T, int RY>
static void run_cg_pass(const Geo& g, hipStream_t s, const CgPassArgs<T>& A, const OpCgPass& op, RedBuf rb)
{
    if (!check_capacity<4, OpCgPass>(g, rb)) return;
    const dim3 grid(g.nblocks), block(kTX, kCgW);
    if (g.nt && A.x) hipLaunchKernelGGL((k_cg_pass<T, RY, true, true>), grid, block, 0, s, g, A, rb);
    else if (g.nt) hipLaunchKernelGGL((k_cg_pass<T, RY, false, true>), grid, block, 0, s, g, A, rb);
    else if (A.x) hipLaunchKernelGGL((k_cg_pass<T, RY, true, false>), grid, block, 0, s, g, A, rb);
    else hipLaunchKernelGGL((k_cg_pass<T, RY, false, false>), grid, block, 0, s, g, A, rb);
    launch_finish<4>(s, op, rb, g.nblocks);
}

template <typename T>
void launch_cg_pass(const Geo& g0, hipStream_t s, RedBuf rb, const T* r_in, const T* pin, T* r_out, T* pout, T* x,
                    Scal* S, bool history, int ring_slot)
{
    const CgPassArgs<T> A{r_in, pin, r_out, pout, ring_slot < 0 ? x : nullptr, S};
    const OpCgPass op{S, history, ring_slot};
    const int nx = g0.hi0 - g0.lo0, ny = g0.hi1 - g0.lo1, nz = g0.hi2 - g0.lo2;
    if (nx <= 0 || ny <= 0 || nz <= 0) return;
    auto tiles = [&](int th) { return (long long)((nx + kTX - 1) / kTX) * ((ny + th - 1) / th); };
    auto tiling = [&](int th, int per_cu) {
        return retile(g0, th, g0.kz_st > 0 ? g0.kz_st : pick_kz(tiles(th), nz, per_cu, 4));
    };
    // 32-row tiles (one block per CU: 158 VGPRs) read fewer ring points and win
    // where there is enough work for two 16-plane chunks per CU, 16-row tiles (two
    // blocks per CU) below that.  us per iteration, 32 / 16 rows, FP64: 514^3
    // 1110 / 1169, 258^3 145 / 148, 194^3 77.5 / 71.5, 130^3 32.8 / 27.1, 66^3 15.5 / 13.9
    // (and where the last row of 32-row tiles is more than half full)
    const bool tall = tiles(4 * kCgW) * nz >= 2ll * 16 * cu_count() && (ny - 1) % (4 * kCgW) + 1 > 2 * kCgW;
    if (tall) run_cg_pass<T, 4>(tiling(4 * kCgW, 1), s, A, op, rb);
    else run_cg_pass<T, 2>(tiling(2 * kCgW, 2), s, A, op, rb);
}

// buffer-preconditioned CG: p_new = z + beta*p_old, Ap = A p_new, p.Ap ; alpha = rz / pAp
// (baseCG.hpp:126-150,197-207).  The reference updates x and r together after alpha is
// known (baseCG.hpp:154-165); here x's update for iteration k-1 rides along with iteration
// k's stencil pass, which reads p_{k-1} anyway: the same x after every iteration, one
// fewer field pass per iteration.  The last update runs after the loop.
template <typename T>
struct OpCgA : Gate {
    const T* __restrict__ src;
    const T* __restrict__ pin;
    T* __restrict__ pout;
    T* __restrict__ Ap;
    T* __restrict__ x;
    Scal* S;
    int slot;  // >= 0: deferred x updates (x untouched; alpha to S->ahist[slot])
    T beta, alpha_prev;
    __device__ void load()
    {
        beta = (T)S->v[S_BETA];
        alpha_prev = (T)S->v[S_ALPHA];
    }
    struct Raw { T src, pold; };  // p_old at the point also feeds the folded x update
    struct Ox { T x; };
    __device__ Raw in_raw(long long c) const { return {src[c], pin[c]}; }
    __device__ T in_value(const Raw& r) const { return r.src + beta * r.pold; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {slot < 0 ? ld<NT>(x + c) : T(0)}; }
    template <bool NT> __device__ void out(long long c, T vc, T Av, const Raw& r, const Ox& o, double* acc) const
    {
        put<NT>(pout + c, vc);
        put<NT>(Ap + c, Av);
        if (slot < 0) put<NT>(x + c, o.x + alpha_prev * r.pold);
        acc[0] += (double)vc * (double)Av;
    }
    __device__ void finish(const double* t)
    {
        S->v[S_PAP] = t[0];
        S->v[S_ALPHA] = S->v[S_RZ] / t[0];
        if (slot >= 0) S->ahist[slot] = S->v[S_ALPHA];
    }
};

// pin/pout double-buffer the search direction: neighbouring tiles rebuild
// p_new on their halo from p_old, so p_old must stay intact during the launch.
template <typename T>
void launch_cg_A2(const Geo& g, hipStream_t s, RedBuf rb, const T* z, const T* pin, T* pout, T* Ap, T* x, Scal* S,
                  int ring_slot)
{
    OpCgA<T> op;
    op.gate = &S->done;
    op.src = z;
    op.pin = pin;
    op.pout = pout;
    op.Ap = Ap;
    op.x = x;
    op.S = S;
    op.slot = ring_slot;
    run_stencil<T, 1>(g, s, op, rb);
}

template <typename T>
struct OpCgFinalX : Gate {
    T* __restrict__ x;
    const T* __restrict__ p;
    const Scal* S;
    T alpha;
    struct R { T x, p; };
    __device__ void load() { alpha = (T)S->v[S_ALPHA]; }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(x + c), ld<NT>(p + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const { put<NT>(x + c, v.x + alpha * v.p); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_cg_final_x(const Geo& g, hipStream_t s, T* x, const T* p, const Scal* S)
{
    OpCgFinalX<T> op;
    op.gate = nullptr;
    op.x = x;
    op.p = p;
    op.S = S;
    run_vector<0>(g, s, op, kNoRed);
}

// r -= alpha Ap, r.r  (baseCG.hpp:154-194)
template <typename T>
struct OpCgB : Gate {
    T* __restrict__ r;
    const T* __restrict__ Ap;
    Scal* S;
    bool history;
    T alpha;
    struct R { T r, ap; };
    __device__ void load() { alpha = (T)S->v[S_ALPHA]; }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(r + c), ld<NT>(Ap + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double* acc) const
    {
        const T rv = v.r - alpha * v.ap;
        put<NT>(r + c, rv);
        acc[0] += (double)rv * (double)rv;
    }
    __device__ void finish(const double* t)
    {
        S->v[S_RR] = t[0];
        finish_iteration(S, sqrt(t[0]), history);
    }
};

template <typename T>
void launch_cg_B(const Geo& g, hipStream_t s, RedBuf rb, T* r, const T* Ap, Scal* S, bool history)
{
    OpCgB<T> op;
    op.gate = &S->done;
    op.r = r;
    op.Ap = Ap;
    op.S = S;
    op.history = history;
    run_vector<1>(g, s, op, rb);
}

template <typename T>
struct OpCgRz : Gate {
    const T* __restrict__ r;
    const T* __restrict__ z;
    Scal* S;
    struct R { T r, z; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(r + c), ld<NT>(z + c)}; }
    template <bool NT> __device__ void apply(long long, const R& v, int, int, int, double* acc) const { acc[0] += (double)v.r * (double)v.z; }
    __device__ void finish(const double* t)
    {
        S->v[S_BETA] = S->iter == 0 ? 0.0 : t[0] / S->v[S_RZ];
        S->v[S_RZ] = t[0];
    }
};

template <typename T>
void launch_cg_rz(const Geo& g, hipStream_t s, RedBuf rb, const T* r, const T* z, Scal* S)
{
    OpCgRz<T> op;
    op.gate = &S->done;
    op.r = r;
    op.z = z;
    op.S = S;
    run_vector<1>(g, s, op, rb);
}

// ------------------------------------------------------------- BiCGSTAB

// AMp = A (amp*Mp), r0.AMp ; alpha = rho0 / r0.AMp   (BiCGSTAB.hpp:142-164)
template <typename T>
struct OpBiK1 : Gate {
    const T* __restrict__ Mp;
    T* __restrict__ AMp;
    const T* __restrict__ r0;
    Scal* S;
    T amp;
    __device__ void load() {}
    struct Raw { T m; };
    struct Ox { T r0; };
    __device__ Raw in_raw(long long c) const { return {Mp[c]}; }
    __device__ T in_value(const Raw& r) const { return amp * r.m; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(r0 + c)}; }
    template <bool NT> __device__ void out(long long c, T, T Av, const Raw&, const Ox& o, double* acc) const
    {
        put<NT>(AMp + c, Av);
        acc[0] += (double)o.r0 * (double)Av;
    }
    __device__ void finish(const double* t) { S->v[S_ALPHA] = S->v[S_RHO0] / t[0]; }
};

template <typename T>
void launch_bicg_k1(const Geo& g0, hipStream_t s, RedBuf rb, int mir, const T* Mp, double amp, T* AMp, const T* r0, Scal* S)
{
    OpBiK1<T> op;
    op.gate = &S->done;
    op.Mp = Mp;
    op.AMp = AMp;
    op.r0 = r0;
    op.S = S;
    op.amp = (T)amp;
    Geo g = g0;
    g.mir = mir;
    run_stencil<T, 1>(g, s, op, rb);
}

template <typename T>
struct OpBiK2 : Gate {
    T* __restrict__ r;
    const T* __restrict__ AMp;
    const Scal* S;
    T alpha;
    struct R { T r, a; };
    __device__ void load() { alpha = (T)S->v[S_ALPHA]; }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(r + c), ld<NT>(AMp + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const { put<NT>(r + c, v.r - alpha * v.a); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_bicg_k2(const Geo& g, hipStream_t s, T* r, const T* AMp, const Scal* S)
{
    OpBiK2<T> op;
    op.gate = &S->done;
    op.r = r;
    op.AMp = AMp;
    op.S = S;
    run_vector<0>(g, s, op, kNoRed);
}

// Az = A (az*z), r.Az, Az.Az ; omega   (BiCGSTAB.hpp:189-225)
template <typename T>
struct OpBiK3 : Gate {
    const T* __restrict__ z;
    T* __restrict__ Az;
    const T* __restrict__ r;
    Scal* S;
    T az;
    __device__ void load() {}
    struct Raw { T z; };
    struct Ox { T r; };
    __device__ Raw in_raw(long long c) const { return {z[c]}; }
    __device__ T in_value(const Raw& v) const { return az * v.z; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(r + c)}; }
    template <bool NT> __device__ void out(long long c, T, T Av, const Raw&, const Ox& o, double* acc) const
    {
        put<NT>(Az + c, Av);
        acc[0] += (double)o.r * (double)Av;
        acc[1] += (double)Av * (double)Av;
    }
    __device__ void finish(const double* t) { S->v[S_OMEGA] = t[0] / t[1]; }
};

template <typename T>
void launch_bicg_k3(const Geo& g0, hipStream_t s, RedBuf rb, int mir, const T* z, double az, T* Az, const T* r, Scal* S)
{
    OpBiK3<T> op;
    op.gate = &S->done;
    op.z = z;
    op.Az = Az;
    op.r = r;
    op.S = S;
    op.az = (T)az;
    Geo g = g0;
    g.mir = mir;
    run_stencil<T, 2>(g, s, op, rb);
}

// x += alpha Mp + omega z ; r -= omega Az ; r0.r, r.r ; beta   (BiCGSTAB.hpp:227-259)
template <typename T>
struct OpBiK45 : Gate {
    T* __restrict__ x;
    const T* __restrict__ Mp;
    const T* __restrict__ z;
    T* __restrict__ r;
    const T* __restrict__ Az;
    const T* __restrict__ r0;
    Scal* S;
    T amp, az, alpha, omega;
    bool history;
    struct R { T x, mp, z, r, az, r0; };
    __device__ void load()
    {
        alpha = (T)S->v[S_ALPHA];
        omega = (T)S->v[S_OMEGA];
    }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(x + c), ld<NT>(Mp + c), ld<NT>(z + c), ld<NT>(r + c), ld<NT>(Az + c), ld<NT>(r0 + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double* acc) const
    {
        put<NT>(x + c, v.x + alpha * (amp * v.mp) + omega * (az * v.z));
        const T rv = v.r - omega * v.az;
        put<NT>(r + c, rv);
        acc[0] += (double)v.r0 * (double)rv;
        acc[1] += (double)rv * (double)rv;
    }
    __device__ void finish(const double* t)
    {
        const double rho1 = t[0];
        S->v[S_BETA] = rho1 / S->v[S_RHO0] * S->v[S_ALPHA] / S->v[S_OMEGA];
        S->v[S_RHO0] = rho1;
        finish_iteration(S, sqrt(t[1]), history);
    }
};

template <typename T>
void launch_bicg_k45(const Geo& g, hipStream_t s, RedBuf rb, T* x, const T* Mp, double amp, const T* z, double az, T* r,
                     const T* Az, const T* r0, Scal* S, bool history)
{
    OpBiK45<T> op;
    op.gate = &S->done;
    op.x = x;
    op.Mp = Mp;
    op.z = z;
    op.r = r;
    op.Az = Az;
    op.r0 = r0;
    op.S = S;
    op.amp = (T)amp;
    op.az = (T)az;
    op.history = history;
    run_vector<2>(g, s, op, rb);
}

// p = r + beta (p - omega AMp)   (BiCGSTAB.hpp:262-272)
template <typename T>
struct OpBiK6 : Gate {
    T* __restrict__ p;
    const T* __restrict__ r;
    const T* __restrict__ AMp;
    const Scal* S;
    T beta, omega;
    struct R { T p, r, a; };
    __device__ void load()
    {
        beta = (T)S->v[S_BETA];
        omega = (T)S->v[S_OMEGA];
    }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(p + c), ld<NT>(r + c), ld<NT>(AMp + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const { put<NT>(p + c, v.r + beta * (v.p - omega * v.a)); }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_bicg_k6(const Geo& g, hipStream_t s, T* p, const T* r, const T* AMp, const Scal* S)
{
    OpBiK6<T> op;
    op.gate = &S->done;
    op.p = p;
    op.r = r;
    op.AMp = AMp;
    op.S = S;
    run_vector<0>(g, s, op, kNoRed);
}

// ------------------------------------------------------------ Chebyshev

// one level: a v + b (B + A v) - c z
template <typename T>
__device__ __forceinline__ T cheb_level(T a, T v, T b, T rhs, T Av, T c, T z)
{
    return fma(-c, z, fma(b, rhs + Av, a * v));
}
// the recurrence's start: c1 (2 B + c0 A B)
template <typename T>
__device__ __forceinline__ T cheb_start(T c1, T c0, T v, T Av)
{
    return c1 * fma(c0, Av, T(2) * v);
}

// Z = c0 B ; Y = c1 (2B + c0 A B)   (chebyshevIteration.hpp:79-90)
template <typename T>
struct OpChebFirst : Gate {
    const T* __restrict__ B;
    T* __restrict__ Z;
    T* __restrict__ Y;
    T c0, c1;
    __device__ void load() {}
    __device__ T in(long long c) const { return B[c]; }
    template <bool NT> __device__ void out(long long c, T vc, T Av, double*) const
    {
        put<NT>(Z + c, c0 * vc);
        put<NT>(Y + c, cheb_start(c1, c0, vc, Av));
    }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_cheb_first(const Geo& g, hipStream_t s, const T* B, T* Z, T* Y, double c0, double c1, const int* gate)
{
    OpChebFirst<T> op;
    op.gate = gate;
    op.B = B;
    op.Z = Z;
    op.Y = Y;
    op.c0 = (T)c0;
    op.c1 = (T)c1;
    run_stencil<T, 0>(g, s, op, kNoRed);
}

template <typename T, typename TO>
struct OpChebFirstOut : Gate {
    const T* __restrict__ B;
    TO* __restrict__ X;
    T c0, c1;
    int which;
    double sign;
    __device__ void load() {}
    __device__ T in(long long c) const { return B[c]; }
    template <bool NT> __device__ void out(long long c, T vc, T Av, double*) const
    {
        const T y = which == 0 ? c0 * vc : cheb_start(c1, c0, vc, Av);
        put<NT>(X + c, (TO)(sign * (double)y));
    }
    __device__ void finish(const double*) {}
};

template <typename T, typename TO>
void launch_cheb_first_out(const Geo& g, hipStream_t s, const T* B, TO* X, double c0, double c1, int which, double sign,
                           const int* gate)
{
    OpChebFirstOut<T, TO> op;
    op.gate = gate;
    op.B = B;
    op.X = X;
    op.c0 = (T)c0;
    op.c1 = (T)c1;
    op.which = which;
    op.sign = sign;
    run_stencil<T, 0>(g, s, op, kNoRed);
}

// W = rho (2 sigma Y + 2/delta (B + A Y) - rho_old Z)   (chebyshevIteration.hpp:103-113)
template <typename T, typename TO>
struct OpChebSweep : Gate {
    const T* __restrict__ Y;
    const T* __restrict__ B;
    const T* __restrict__ Z;
    TO* __restrict__ W;
    T a, b, cz;
    double sign;
    __device__ void load() {}
    struct Ox { T b, z; };
    __device__ T in(long long c) const { return Y[c]; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(B + c), ld<NT>(Z + c)}; }
    template <bool NT> __device__ void out(long long c, T vc, T Av, const T&, const Ox& o, double*) const
    {
        const T w = cheb_level(a, vc, b, o.b, Av, cz, o.z);
        if constexpr (sizeof(TO) == sizeof(T)) put<NT>(W + c, sign < 0 ? -w : w);
        else put<NT>(W + c, (TO)(sign * (double)w));
    }
    __device__ void finish(const double*) {}
};

template <typename T, typename TO>
void launch_cheb_sweep(const Geo& g, hipStream_t s, const T* Y, const T* B, const T* Z, TO* W, double a, double b,
                       double c, double sign, const int* gate)
{
    OpChebSweep<T, TO> op;
    op.gate = gate;
    op.Y = Y;
    op.B = B;
    op.Z = Z;
    op.W = W;
    op.a = (T)a;
    op.b = (T)b;
    op.cz = (T)c;
    op.sign = sign;
    run_stencil<T, 0>(g, s, op, kNoRed);
}

// ---------------------------------------------- fused Chebyshev sweeps
// S = 2 or 3 consecutive sweeps of the three-term recurrence in one pass over
// the grid (temporal blocking of chebyshevIteration.hpp:103-113 / the alpaka
// Chebyshev2Kernel, kernelsAlpakaChebyshev.hpp:191-273):
//   W1 = a1 Y  + b1 (B + A Y)  - c1 Z      sweep c      (Y = y_c, Z = y_{c-1})
//   W2 = a2 W1 + b2 (B + A W1) - c2 Y      sweep c + 1
//   W3 = a3 W2 + b3 (B + A W2) - c3 W1     sweep c + 2
// The stage's first pass reads only B: Z = c0 B, Y-stream B, and its first level
// is the recurrence's start W1 = c1 (2 B + c0 A B).  A pass reads Y, Z, B and
// writes the last two levels (the stage's last pass only its result): 5 words
// per point for 2 or 3 sweeps, where separate sweeps move 4 each.
//
// A block owns a 64 x (8 RY) tile and marches z.  Level l is formed on the tile
// and S - l rings of points around it, at plane s - (l - 1) of step s; a thread
// owns RY consecutive rows of one column (their y-neighbours are its own
// registers) and at most one point of each ring, with each point's z-history in
// registers.  The x-y neighbours of every level go through LDS, two planes per
// level used in turn, with one barrier per plane: level l of a plane is read
// one step after it was written, and its buffer is rewritten a step later.
//
// Neumann ghosts (the data point two cells inward) are never stored: the thread
// that owns a ghost position loads and evaluates its mirror point instead and
// puts the value at the ghost's place in LDS; ghosts in z are a choice of
// register.  A level's other points off the solver region are 0; B's, which the
// first pass's start reads, are whatever the field holds there.
//
// Measured at 512^3 FP64: three sweeps in 1.24 ms (4.3 TB/s of its 5 words; 4.7
// with the rings' re-reads that miss L2, 1.16x on the reads; vector pipe 22 % busy,
// LDS 16 %), 0.41 ms per sweep, where the pair took
// 1.08 ms and needed a ghost fill per pass with Neumann faces.  On grids that stay
// in the caches the steps' instructions are half of the time, so plane pointers
// are advanced instead of formed from the plane's number and two steps make a trip
// of the loop, which makes the LDS planes constants: 2-5 % at every size (us per
// BiCGSTAB + Chebyshev(24) iteration: 66^3 231 -> 226, mixed 130^3 756 -> 715,
// 258^3 3000 -> 2905, 514^3 23450 -> 22920).
constexpr int kChW = 8;   // wavefronts per block

template <typename T, typename TO>
struct ChebArgs {
    const T* __restrict__ Y;   // first pass: B
    const T* __restrict__ Z;   // null: first pass
    const T* __restrict__ B;
    T* __restrict__ Wp;        // level S - 1 (null: the stage's last pass)
    TO* __restrict__ W;        // level S
    T a[3], b[3], c[3], c0, c1;
    T sign;                    // of W
    const int* gate;
};

// registers of one owned point: Y of planes s-1..s+2, Z of s, s+1, B of s-2..s+1, levels 1 and 2
template <typename T>
struct ChebPoint {
    T ym, yc, yp, yn, zc, zn, b2, b1, bc, bn, um, uc, un, vm, vc, vn;
};

// NEU: the grid has Neumann faces
template <typename T, typename TO, int S, int RY, bool NEU, bool NT>
__global__ __launch_bounds__(kTX* kChW, RY == 2 && !(NEU && S == 3) ? 4 : 2) void k_cheb_multi(Geo g, ChebPairGeo cg, ChebArgs<T, TO> A)
{
    if (A.gate != nullptr && *A.gate != 0) return;
    constexpr int TY = kChW * RY;
    // points of ring d around the tile
    constexpr int NR[3] = {2 * (kTX + 2) + 2 * TY, 2 * (kTX + 4) + 2 * (TY + 2), 2 * (kTX + 6) + 2 * (TY + 4)};
    static_assert(NR[2] <= kTX * kChW, "ring points need one thread each");
    __shared__ T ysl[2][TY + 2 * S][kTX + 2 * S];
    __shared__ T usl[2][TY + 2 * (S - 1)][kTX + 2 * (S - 1)];                                  // level 1
    __shared__ T vsl[S == 3 ? 2 : 1][S == 3 ? TY + 2 : 1][S == 3 ? kTX + 2 : 1];               // level 2
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int tx0 = bid % g.ntx, rr = bid / g.ntx;
    const int ty0 = rr % g.nty, tz0 = rr / g.nty;
    const int i0 = g.lo0 + tx0 * kTX, j0 = g.lo1 + ty0 * TY;
    const int k0 = g.lo2 + tz0 * g.kz, k1 = min(k0 + g.kz, g.hi2);
    const int lx = threadIdx.x, ly = threadIdx.y, tid = lx + kTX * ly;
    const T cx = (T)g.cx, cy = (T)g.cy, cz = (T)g.cz;
    const bool first = A.Z == nullptr;

    // a ghost position stands for its mirror point
    auto mirx = [&](int i) {
        if constexpr (!NEU) return 0;
        return (cg.neu & 1) && i == cg.lo_d[0] - 1 ? 2 : (cg.neu & 2) && i == cg.hi_d[0] ? -2 : 0;
    };
    auto miry = [&](int j) {
        if constexpr (!NEU) return 0;
        return (cg.neu & 4) && j == cg.lo_d[1] - 1 ? 2 : (cg.neu & 8) && j == cg.hi_d[1] ? -2 : 0;
    };
    auto inxy = [&](int i, int j) { return i >= g.lo0 && i < g.hi0 && j >= g.lo1 && j < g.hi1; };
    auto ybox = [&](int i, int j) { return i >= 0 && i < cg.ng[0] && j >= 0 && j < cg.ng[1]; };
    // byte offset of tile point (r, c) from the fields' tile origin (row -S, column -S)
    auto off = [&](int r, int c) { return (unsigned)(g.px * (r + S) + c + S) * (unsigned)sizeof(T); };
    const long long org = (long long)g.ox + (i0 - S) + (long long)g.px * (j0 - S);

    // tile rows: row q at j0 + ly RY + q; `val` = the (mirrored) point is in the
    // solver region; `to` its offset for loads (kOob where nothing is read), `so`
    // the point's own offset for stores (kOob off the solver region)
    const int jr = ly * RY, dc = mirx(i0 + lx);
    int dr[RY];
    bool val[RY];
    unsigned to[RY], so[RY];
#pragma unroll
    for (int q = 0; q < RY; ++q) {
        dr[q] = miry(j0 + jr + q);
        const int i = i0 + lx + dc, j = j0 + jr + q + dr[q];
        val[q] = inxy(i, j);
        to[q] = (first ? ybox(i, j) : val[q]) ? off(jr + q + dr[q], lx + dc) : kOob;
        so[q] = inxy(i0 + lx, j0 + jr + q) ? off(jr + q, lx) : kOob;
    }
    // whether the tile or its rings hold a ghost in x or y (uniform)
    const bool ghosts = NEU && (((cg.neu & 1) && i0 == g.lo0) || ((cg.neu & 2) && i0 + kTX + S > cg.hi_d[0]) ||
                                ((cg.neu & 4) && j0 == g.lo1) || ((cg.neu & 8) && j0 + TY + S > cg.hi_d[1]));
    // ring points: position, mirrored centre, validity
    int pr[3] = {0, 0, 0}, pc[3] = {0, 0, 0}, mr[3], mc[3];
    bool has[3], rv[3];
    unsigned ro[3];
#pragma unroll
    for (int d = 0; d < S; ++d) {
        has[d] = tid < NR[d];
        if (has[d]) {
            if (d == 0) ring_point<kTX, TY>(tid, pr[d], pc[d]);
            else if (d == 1) ring_point<kTX + 2, TY + 2>(tid, pr[d], pc[d]);
            else ring_point<kTX + 4, TY + 4>(tid, pr[d], pc[d]);
            pr[d] -= d;
            pc[d] -= d;
        }
        mr[d] = pr[d] + miry(j0 + pr[d]);
        mc[d] = pc[d] + mirx(i0 + pc[d]);
        rv[d] = has[d] && inxy(i0 + mc[d], j0 + mr[d]);
        ro[d] = has[d] && (first ? ybox(i0 + mc[d], j0 + mr[d]) : rv[d]) ? off(mr[d], mc[d]) : kOob;
    }

    ChebPoint<T> t[RY], r[2];  // r[d]: ring d + 1 where it forms a level (d < S - 1)
    T oc, on = T(0);           // outermost ring: Y of planes s, s + 1
    auto zin = [&](int k) { return k >= g.lo2 && k < g.hi2; };
    auto yin = [&](int k) { return first ? k >= 0 && k < cg.ng[2] : zin(k); };
    const T* Yo = A.Y + org;
    const T* Zo = first ? Yo : A.Z + org;
    const T* Bo = A.B + org;
    auto yrs = [&](int k) { return plane_rsrc(Yo + g.plane * k, yin(k)); };
    auto zrs = [&](int k) { return plane_rsrc(Zo + g.plane * k, !first && zin(k)); };
    auto brs = [&](int k) { return plane_rsrc(Bo + g.plane * k, !first && zin(k)); };
    const int s0 = k0 - (S - 1), s1 = k1 + S - 2;  // steps s0 .. s1
    {
        const auto ya = yrs(s0 - 1), yb = yrs(s0), yc = yrs(s0 + 1), za = zrs(s0), ba = brs(s0);
        auto start = [&](ChebPoint<T>& P, unsigned o) {
            P = ChebPoint<T>{};
            P.ym = buf_ld<T>(ya, o);
            P.yc = buf_ld<T>(yb, o);
            P.yp = buf_ld<T>(yc, o);
            P.zc = buf_ld<T>(za, o);
            P.bc = buf_ld<T>(ba, o);
        };
#pragma unroll
        for (int q = 0; q < RY; ++q) start(t[q], to[q]);
#pragma unroll
        for (int d = 0; d < S - 1; ++d) start(r[d], ro[d]);
        oc = buf_ld<T>(yb, ro[S - 1]);
    }

    // plane k of a field with bound n: in [lo, lo + n) it is read or written
    const long long pb = g.plane * (long long)sizeof(T);
    const int ylo = first ? 0 : g.lo2, yend = min(first ? cg.ng[2] : g.hi2, s1 + 2);  // no step after s1 reads
    const int zend = first ? g.lo2 : min(g.hi2, s1 + 1);                             // the first pass reads only Y
    auto within = [](int k, int lo, int hi) { return (unsigned)(k - lo) < (unsigned)max(hi - lo, 0); };
    const char *y2p = (const char*)(Yo + g.plane * (s0 + 2)), *z1p = (const char*)(Zo + g.plane * (s0 + 1)),
               *b1p = (const char*)(Bo + g.plane * (s0 + 1));
    char* wpp = (char*)((A.Wp ? A.Wp : (T*)A.Y) + org + g.plane * (s0 - (S - 2)));  // plane of level S - 1
    char* wp = (char*)(A.W + org + g.plane * (s0 - (S - 1)));                       // plane of level S
    const T c0 = first ? A.c0 : T(1);  // Z of the second sweep is c0 B on the first pass

    // one step; BUF: the LDS planes that it writes, a constant so that the LDS addresses are
    auto one = [&](const int s, auto BUF) __attribute__((always_inline)) {
        const int buf = BUF, alt = buf ^ 1;
        // Y of plane s into LDS
#pragma unroll
        for (int q = 0; q < RY; ++q) ysl[buf][jr + q + S][lx + S] = t[q].yc;
#pragma unroll
        for (int d = 0; d < S - 1; ++d)
            if (has[d]) ysl[buf][pr[d] + S][pc[d] + S] = r[d].yc;
        if (has[S - 1]) ysl[buf][pr[S - 1] + S][pc[S - 1] + S] = oc;
        // loads for the next step: Y of plane s + 2 (s + 1 on the outermost ring), Z and B of plane s + 1
        {
            const auto y1 = plane_rsrc(y2p - pb, within(s + 1, ylo, yend));
            const auto y2 = plane_rsrc(y2p, within(s + 2, ylo, yend));
            const auto z1 = plane_rsrc(z1p, within(s + 1, g.lo2, zend));
            const auto b1 = plane_rsrc(b1p, within(s + 1, g.lo2, zend));
            auto fetch = [&](ChebPoint<T>& P, unsigned o) {
                P.yn = buf_ld<T>(y2, o);
                P.zn = buf_ld<T>(z1, o);
                P.bn = buf_ld<T>(b1, o);
            };
#pragma unroll
            for (int q = 0; q < RY; ++q) fetch(t[q], to[q]);
#pragma unroll
            for (int d = 0; d < S - 1; ++d) fetch(r[d], ro[d]);
            on = buf_ld<T>(y1, ro[S - 1]);
        }
        __syncthreads();

        // Neumann ghosts in z of the planes whose level is formed in this step: the
        // register of the plane beyond the face takes the mirror plane's value
        // (what it held belongs to a plane off the solver region, where every
        // level is 0)
        if constexpr (NEU) {
            const int lo = cg.lo_d[2], hi = cg.hi_d[2] - 1;
            auto each = [&](auto f) {
#pragma unroll
                for (int q = 0; q < RY; ++q) f(t[q]);
#pragma unroll
                for (int d = 0; d < S - 1; ++d) f(r[d]);
            };
            if ((cg.neu & 16) && s == lo) each([](ChebPoint<T>& P) { P.ym = P.yp; });
            if ((cg.neu & 32) && s == hi) each([](ChebPoint<T>& P) { P.yp = P.ym; });
        }
        // level 1 of plane s
        {
            const bool zs = zin(s);
            auto level1 = [&](ChebPoint<T>& P, T Av, bool in) {
                T w;
                if (first) {
                    P.bc = P.yc;
                    w = cheb_start(A.c1, A.c0, P.yc, Av);
                } else {
                    w = cheb_level(A.a[0], P.yc, A.b[0], P.bc, Av, A.c[0], P.zc);
                }
                P.un = in ? w : T(0);
            };
            auto at = [&](const ChebPoint<T>& P, int row, int col) {
                const T(*y)[kTX + 2 * S] = ysl[buf];
                return lap7(P.yc, y[row][col - 1], y[row][col + 1], y[row - 1][col], y[row + 1][col], P.ym, P.yp, cx, cy, cz);
            };
            T Av[RY];
            if (!NEU || !ghosts) {
#pragma unroll
                for (int q = 0; q < RY; ++q) {
                    const int row = jr + q + S, col = lx + S;
                    const T ym = q > 0 ? t[q > 0 ? q - 1 : 0].yc : ysl[buf][row - 1][col];
                    const T yp = q + 1 < RY ? t[q + 1 < RY ? q + 1 : 0].yc : ysl[buf][row + 1][col];
                    Av[q] = lap7(t[q].yc, ysl[buf][row][col - 1], ysl[buf][row][col + 1], ym, yp, t[q].ym, t[q].yp, cx, cy, cz);
                }
            } else {
#pragma unroll
                for (int q = 0; q < RY; ++q) Av[q] = at(t[q], jr + q + dr[q] + S, lx + dc + S);
            }
            const auto wr = plane_rsrc(wpp, S == 2 && A.Wp && within(s, k0, k1));
#pragma unroll
            for (int q = 0; q < RY; ++q) {
                if (zs) level1(t[q], Av[q], val[q]);
                else t[q].un = T(0);
            }
#pragma unroll
            for (int q = 0; q < RY; ++q) {
                usl[buf][jr + q + S - 1][lx + S - 1] = t[q].un;
                if constexpr (S == 2) buf_st<NT>(wr, so[q], t[q].un);
            }
#pragma unroll
            for (int d = 0; d < S - 1; ++d) {
                if (!has[d]) continue;
                if (zs) level1(r[d], at(r[d], mr[d] + S, mc[d] + S), rv[d]);
                else r[d].un = T(0);
                usl[buf][pr[d] + S - 1][pc[d] + S - 1] = r[d].un;
            }
        }
        // level 2 of plane s - 1 (level 1 of that plane is in the other LDS buffer)
        if (s >= s0 + 2) {
            const int p = s - 1;
            const bool zs = zin(p), own = within(p, k0, k1);
            if constexpr (NEU) {
                const bool zlo = (cg.neu & 16) && p == cg.lo_d[2], zhi = (cg.neu & 32) && p == cg.hi_d[2] - 1;
                auto mirror = [&](ChebPoint<T>& P) {
                    if (zlo) P.um = P.un;
                    else P.un = P.um;
                };
                if (zlo || zhi) {
#pragma unroll
                    for (int q = 0; q < RY; ++q) mirror(t[q]);
                    if constexpr (S == 3) mirror(r[0]);
                }
            }
            auto level2 = [&](const ChebPoint<T>& P, T Av) {
                return cheb_level(A.a[1], P.uc, A.b[1], P.b1, Av, A.c[1], c0 * P.ym);
            };
            auto at = [&](const ChebPoint<T>& P, int row, int col) {
                const T(*u)[kTX + 2 * (S - 1)] = usl[alt];
                return lap7(P.uc, u[row][col - 1], u[row][col + 1], u[row - 1][col], u[row + 1][col], P.um, P.un, cx, cy, cz);
            };
            T Av[RY];
            // the pass's last level is wanted on the solver region only: ghost positions
            // take no mirror there (a mirrored centre may lie a column or row before the
            // tile, whose neighbours level 1 of a two-sweep pass does not hold)
            constexpr bool kMir2 = NEU && S == 3;
            static_assert(!kMir2 || S - 1 >= 2, "a mirrored centre's neighbours lie in level 1's planes");
            if (!kMir2 || !ghosts) {
#pragma unroll
                for (int q = 0; q < RY; ++q) {
                    const int row = jr + q + S - 1, col = lx + S - 1;
                    const T ym = q > 0 ? t[q > 0 ? q - 1 : 0].uc : usl[alt][row - 1][col];
                    const T yp = q + 1 < RY ? t[q + 1 < RY ? q + 1 : 0].uc : usl[alt][row + 1][col];
                    Av[q] = lap7(t[q].uc, usl[alt][row][col - 1], usl[alt][row][col + 1], ym, yp, t[q].um, t[q].un, cx, cy, cz);
                }
            } else {
#pragma unroll
                for (int q = 0; q < RY; ++q) Av[q] = at(t[q], jr + q + dr[q] + S - 1, lx + dc + S - 1);
            }
            const auto wr = plane_rsrc((T*)wpp, S == 3 && A.Wp && own);
            const auto xr = plane_rsrc((TO*)wp, S == 2 && own);
#pragma unroll
            for (int q = 0; q < RY; ++q) {
                T w = level2(t[q], Av[q]);
                if constexpr (S == 2) {
                    buf_st<NT>(xr, so[q] == kOob ? kOob : so[q] * (unsigned)(sizeof(TO) / sizeof(T)), (TO)(A.sign * w));
                } else {
                    w = val[q] && zs ? w : T(0);
                    t[q].vn = w;
                    vsl[alt][jr + q + 1][lx + 1] = w;
                    buf_st<NT>(wr, so[q], w);
                }
            }
            if constexpr (S == 3) {
                if (has[0]) {
                    T w = level2(r[0], at(r[0], mr[0] + S - 1, mc[0] + S - 1));
                    if (!(rv[0] && zs)) w = T(0);
                    vsl[alt][pr[0] + 1][pc[0] + 1] = w;
                }
            }
        }
        // level 3 of plane s - 2
        if constexpr (S == 3) {
            if (s >= s0 + 4) {
                const int p = s - 2;
                if constexpr (NEU) {
                    const bool zlo = (cg.neu & 16) && p == cg.lo_d[2], zhi = (cg.neu & 32) && p == cg.hi_d[2] - 1;
                    if (zlo || zhi) {
#pragma unroll
                        for (int q = 0; q < RY; ++q) {
                            if (zlo) t[q].vm = t[q].vn;
                            else t[q].vn = t[q].vm;
                        }
                    }
                }
                const auto xr = plane_rsrc((TO*)wp, true);
#pragma unroll
                for (int q = 0; q < RY; ++q) {
                    const int row = jr + q + 1, col = lx + 1;
                    const T ym = q > 0 ? t[q > 0 ? q - 1 : 0].vc : vsl[buf][row - 1][col];
                    const T yp = q + 1 < RY ? t[q + 1 < RY ? q + 1 : 0].vc : vsl[buf][row + 1][col];
                    const T Av = lap7(t[q].vc, vsl[buf][row][col - 1], vsl[buf][row][col + 1], ym, yp, t[q].vm, t[q].vn, cx,
                                      cy, cz);
                    const T w = cheb_level(A.a[2], t[q].vc, A.b[2], t[q].b2, Av, A.c[2], t[q].um);
                    buf_st<NT>(xr, so[q] == kOob ? kOob : so[q] * (unsigned)(sizeof(TO) / sizeof(T)), (TO)(A.sign * w));
                }
            }
        }
        // advance one plane
        auto step = [&](ChebPoint<T>& P) {
            P.ym = P.yc;
            P.yc = P.yp;
            P.yp = P.yn;
            P.zc = P.zn;
            P.b2 = P.b1;
            P.b1 = P.bc;
            P.bc = P.bn;
            P.um = P.uc;
            P.uc = P.un;
            P.vm = P.vc;
            P.vc = P.vn;
        };
#pragma unroll
        for (int q = 0; q < RY; ++q) step(t[q]);
#pragma unroll
        for (int d = 0; d < S - 1; ++d) step(r[d]);
        oc = on;
        y2p += pb;
        z1p += pb;
        b1p += pb;
        wpp += pb;
        wp += g.plane * (long long)sizeof(TO);
    };
    if constexpr (sizeof(T) == 8 && S == 3 && RY == 2 && !NEU) {
        // 128 registers, all in use: two steps per trip spill 15 (130^3 506 -> 586 us)
        for (int s = s0; s <= s1; ++s) one(s, (s - s0) & 1);
    } else {
        for (int s = s0;;) {
            one(s, std::integral_constant<int, 0>{});
            if (++s > s1) break;
            one(s, std::integral_constant<int, 1>{});
            if (++s > s1) break;
        }
    }
}

template <typename T, typename TO, int S, int RY>
static void run_cheb_multi(const Geo& g0, const ChebPairGeo& cg, hipStream_t s, const ChebArgs<T, TO>& A, int per_cu)
{
    constexpr int TY = kChW * RY;
    const int nx = g0.hi0 - g0.lo0, ny = g0.hi1 - g0.lo1, nz = g0.hi2 - g0.lo2;
    const long long tiles = (long long)((nx + kTX - 1) / kTX) * ((ny + TY - 1) / TY);
    const Geo g = retile(g0, TY, cg.kz > 0 ? cg.kz : pick_kz(tiles, nz, per_cu, 2 * S));
    const dim3 grid(g.nblocks), block(kTX, kChW);
    if (cg.neu && g.nt) hipLaunchKernelGGL((k_cheb_multi<T, TO, S, RY, true, true>), grid, block, 0, s, g, cg, A);
    else if (cg.neu) hipLaunchKernelGGL((k_cheb_multi<T, TO, S, RY, true, false>), grid, block, 0, s, g, cg, A);
    else if (g.nt) hipLaunchKernelGGL((k_cheb_multi<T, TO, S, RY, false, true>), grid, block, 0, s, g, cg, A);
    else hipLaunchKernelGGL((k_cheb_multi<T, TO, S, RY, false, false>), grid, block, 0, s, g, cg, A);
}

template <typename T, typename TO>
void launch_cheb_multi(const Geo& g, const ChebPairGeo& cg, hipStream_t s, int sweeps, const T* Y, const T* Z, const T* B,
                       T* Wp, TO* W, const double* a, const double* b, const double* c, double c0, double c1, double sign,
                       const int* gate)
{
    if (g.hi0 <= g.lo0 || g.hi1 <= g.lo1 || g.hi2 <= g.lo2) return;
    ChebArgs<T, TO> A{};
    A.Y = Y;
    A.Z = Z;
    A.B = B;
    A.Wp = Wp;
    A.W = W;
    for (int l = 0; l < sweeps; ++l) {
        A.a[l] = (T)a[l];
        A.b[l] = (T)b[l];
        A.c[l] = (T)c[l];
    }
    A.c0 = (T)c0;
    A.c1 = (T)c1;
    A.sign = (T)sign;
    A.gate = gate;
    // 32-row tiles read fewer ring points (one block per CU); 16-row tiles (two per
    // CU; one with Neumann faces, whose FP64 form for three sweeps needs more
    // registers) where the 32-row ones do not give every CU 8 planes of work or
    // where the last row of tiles is at most half full.  us per BiCGSTAB +
    // Chebyshev(24) iteration, 32 / 16 rows: Dirichlet 130^3 621 / 573, 194^3
    // 1461 / 1503, 514^3 24500 / 24730; mixed faces 130^3 (129 rows) 807 / 762,
    // 131x257x190 (256 rows) 1796 / 1859, 258^3 (257 rows) 4334 / 3997
    const int nx = g.hi0 - g.lo0, ny = g.hi1 - g.lo1, nz = g.hi2 - g.lo2, tail = (ny - 1) % (4 * kChW) + 1;
    const long long tiles = (long long)((nx + kTX - 1) / kTX) * ((ny + 4 * kChW - 1) / (4 * kChW));
    const bool tall = tiles * nz >= 8ll * cu_count() && tail > 2 * kChW;
    if (sweeps == 3 && tall) run_cheb_multi<T, TO, 3, 4>(g, cg, s, A, 1);
    else if (sweeps == 3) run_cheb_multi<T, TO, 3, 2>(g, cg, s, A, cg.neu && sizeof(T) == 8 ? 1 : 2);
    else if (tall) run_cheb_multi<T, TO, 2, 4>(g, cg, s, A, 1);
    else run_cheb_multi<T, TO, 2, 2>(g, cg, s, A, 2);
}

// ------------------------------------------------------------------ FCG

// end of an FCG iteration once ||r||^2 of the updated residual is known
__device__ inline void update_finish(Scal* S, double rr, bool history)
{
    S->v[S_PAP_OLD] = S->v[S_PAP];
    S->v[S_RR] = rr;
    const double err = sqrt(rr);
    finish_iteration(S, err, history);
    // stall monitor: every stall_window iterations the residual must have
    // dropped by the factor v[S_AUX1], else the fallback preconditioner takes over
    if (S->stall_window > 0 && !S->fallback && S->iter % S->stall_window == 0) {
        if (err > S->v[S_AUX1] * S->v[S_AUX2]) S->fallback = 1;
        S->v[S_AUX2] = err;
    }
}

// gamma = z.Apold and beta.  Where the preconditioner sums z.Apold itself (the
// learned one in its output kernel, its fallback in its update), only the finish
// runs.  With a pass over z and Apold and a second finish for the fallback, gated
// off in nearly every iteration, an iteration had two launches more (learned FCG
// solves, us: FP64 66^3 2999 / 2906 without them, 130^3 4770 / 4701; under
// refinement 34^3 3862 / 3655).
template <typename T>
struct OpFcgGamma : Gate {
    const T* __restrict__ z;
    const T* __restrict__ Apold;
    Scal* S;
    struct R { T z, a; };
    __device__ void load() {}
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(z + c), ld<NT>(Apold + c)}; }
    template <bool NT> __device__ void apply(long long, const R& v, int, int, int, double* acc) const { acc[0] += (double)v.z * (double)v.a; }
    __device__ void finish(const double* t)
    {
        S->v[S_GAM] = t[0];
        // restart after a discarded step: the old direction may hold non-finite values
        S->v[S_BETA] = (S->iter == 0 || S->restart) ? 0.0 : t[0] / S->v[S_PAP_OLD];
    }
};

template <typename T>
void launch_fcg_gamma(const Geo& g, hipStream_t s, RedBuf rb, const T* z, const T* Apold, Scal* S)
{
    OpFcgGamma<T> op;
    op.gate = &S->done;
    op.z = z;
    op.Apold = Apold;
    op.S = S;
    run_vector<1>(g, s, op, rb);
}

template <typename T>
void launch_fcg_gamma_finish(hipStream_t s, RedBuf rb, int nblocks, int nfallback, Scal* S)
{
    OpFcgGamma<T> op;
    op.gate = &S->done;
    op.z = nullptr;
    op.Apold = nullptr;
    op.S = S;
    if (nblocks <= 0 || nblocks > rb.cap) return;
    hipLaunchKernelGGL((k_finish_alt<1, OpFcgGamma<T>>), dim3(1), dim3(kFinThreads), 0, s, op, rb, nblocks, nfallback,
                       &S->fallback);
}

// p = z - beta pold ; Ap = A p ; p.Ap, p.r ; alpha = p.r / p.Ap ; and the
// previous iteration's x += alpha_prev pold (folded in: this pass reads pold
// anyway), unless that step was discarded (restart).
// FUSED: the residual update r -= alpha Ap has no pass of its own; the next
// iteration's preconditioner forms it while reading r.  This pass then also
// sums r.Ap, Ap.Ap and r.r, and its finish takes over the update's:
// ||r - alpha Ap||^2 = r.r - 2 alpha r.Ap + alpha^2 Ap.Ap, the convergence
// test and the stall monitor.
template <typename T, bool FUSED = false>
struct OpFcgP : Gate {
    const T* __restrict__ z;
    const T* __restrict__ pold;
    T* __restrict__ p;
    T* __restrict__ Ap;
    const T* __restrict__ r;
    T* __restrict__ x;
    Scal* S;
    bool history;  // FUSED: record the residual history
    T beta, alpha_prev;
    bool upd;  // apply the previous step to x
    int slot;  // >= 0: deferred x updates (x untouched; alpha to S->ahist[slot])
    __device__ void load()
    {
        beta = (T)S->v[S_BETA];
        alpha_prev = (T)S->v[S_ALPHA];
        upd = slot < 0 && !S->restart && alpha_prev != (T)0;
    }
    // beta = 0 takes z as it is, and pold is read only when it is used, so a
    // restart never multiplies a non-finite pold
    struct Raw { T z, pold; };
    struct Ox { T r, x; };
    __device__ Raw in_raw(long long c) const { return {z[c], (beta == (T)0 && !upd) ? (T)0 : pold[c]}; }
    __device__ T in_value(const Raw& v) const { return beta == (T)0 ? v.z : v.z - beta * v.pold; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(r + c), upd ? ld<NT>(x + c) : (T)0}; }
    template <bool NT> __device__ void out(long long c, T vc, T Av, const Raw& v, const Ox& o, double* acc) const
    {
        put<NT>(p + c, vc);
        put<NT>(Ap + c, Av);
        if (upd) put<NT>(x + c, o.x + alpha_prev * v.pold);
        acc[0] += (double)vc * (double)Av;
        acc[1] += (double)vc * (double)o.r;
        if constexpr (FUSED) {
            acc[2] += (double)o.r * (double)Av;
            acc[3] += (double)Av * (double)Av;
            acc[4] += (double)o.r * (double)o.r;
        }
    }
    __device__ void finish(const double* t)
    {
        S->v[S_PAP] = t[0];
        const double a = t[1] / t[0];
        double rr_next = 0.0;
        // a non-finite step (the preconditioner returned inf/NaN or a null
        // direction): discard it, switch to the fallback preconditioner, restart
        if (!isfinite(a)) {
            S->restart = 1;
            S->fallback = 1;
            S->v[S_ALPHA] = 0.0;
            if constexpr (FUSED) rr_next = t[4];  // r stays
        } else {
            S->restart = 0;
            S->v[S_ALPHA] = a;
            // the expansion cancels when one step removes almost all of r: its
            // error is a few eps * r.r, so below 1e-8 r.r it is noise.  Clamping
            // there over-estimates the next residual (the loop runs on, and the
            // next pass sums r.r exactly) and never gives the next network input
            // a zero scale
            if constexpr (FUSED) rr_next = fmax(t[4] - 2.0 * a * t[2] + a * a * t[3], 1e-8 * t[4]);
        }
        if (slot >= 0) S->ahist[slot] = S->v[S_ALPHA];
        if constexpr (FUSED) update_finish(S, rr_next, history);
    }
};

template <typename T>
void launch_fcg_p(const Geo& g, hipStream_t s, RedBuf rb, const T* z, const T* pold, T* p, T* Ap, const T* r, T* x,
                  Scal* S)
{
    OpFcgP<T> op;
    op.gate = &S->done;
    op.z = z;
    op.pold = pold;
    op.p = p;
    op.Ap = Ap;
    op.r = r;
    op.x = x;
    op.S = S;
    op.history = false;
    op.slot = -1;
    run_stencil<T, 2>(g, s, op, rb);
}

template <typename T>
void launch_fcg_p_fused(const Geo& g, hipStream_t s, RedBuf rb, const T* z, const T* pold, T* p, T* Ap, const T* r,
                        T* x, Scal* S, bool history, int ring_slot)
{
    OpFcgP<T, true> op;
    op.gate = &S->done;
    op.z = z;
    op.pold = pold;
    op.p = p;
    op.Ap = Ap;
    op.r = r;
    op.x = x;
    op.S = S;
    op.history = history;
    op.slot = ring_slot;
    run_stencil<T, 5>(g, s, op, rb);
}

// deferred x updates: x += ahist[j] * ring[j] over the slots in order, the
// slots with alpha 0 (unused, or a discarded step whose direction may hold
// non-finite values) neither read nor added
template <typename T>
struct OpFcgFlush : Gate {
    T* __restrict__ x;
    const T* ring[kFcgRing];
    const Scal* S;
    T a[kFcgRing];
    unsigned used;
    struct R { T x, p[kFcgRing]; };
    __device__ void load()
    {
        used = 0u;
#pragma unroll
        for (int j = 0; j < kFcgRing; ++j) {
            a[j] = (T)S->ahist[j];
            if (S->ahist[j] != 0.0) used |= 1u << j;
        }
    }
    template <bool NT> __device__ R fetch(long long c) const
    {
        R v;
        v.x = ld<NT>(x + c);
#pragma unroll
        for (int j = 0; j < kFcgRing; ++j) v.p[j] = ((used >> j) & 1u) ? ld<NT>(ring[j] + c) : (T)0;
        return v;
    }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const
    {
        T acc = v.x;
#pragma unroll
        for (int j = 0; j < kFcgRing; ++j)
            if ((used >> j) & 1u) acc = acc + a[j] * v.p[j];
        put<NT>(x + c, acc);
    }
    __device__ void finish(const double*) {}
};

__global__ void k_fcg_ring_reset(Scal* S)
{
    if (threadIdx.x < kFcgRing) S->ahist[threadIdx.x] = 0.0;
}

void launch_fcg_ring_reset(hipStream_t s, Scal* S)
{
    hipLaunchKernelGGL(k_fcg_ring_reset, dim3(1), dim3(64), 0, s, S);
}

template <typename T>
void launch_fcg_flush(const Geo& g, hipStream_t s, T* x, T* const ring[kFcgRing], Scal* S)
{
    OpFcgFlush<T> op;
    op.gate = nullptr;
    op.x = x;
    for (int j = 0; j < kFcgRing; ++j) op.ring[j] = ring[j];
    op.S = S;
    run_vector<0>(g, s, op, kNoRed);
    launch_fcg_ring_reset(s, S);
}

// the last step of an FCG solve: x += alpha p unless it was discarded
template <typename T>
struct OpFcgFinalX : Gate {
    T* __restrict__ x;
    const T* __restrict__ p;
    const Scal* S;
    T alpha;
    int skip;
    struct R { T x, p; };
    __device__ void load()
    {
        alpha = (T)S->v[S_ALPHA];
        skip = S->restart;
    }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(x + c), skip ? (T)0 : ld<NT>(p + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const
    {
        if (!skip) put<NT>(x + c, v.x + alpha * v.p);
    }
    __device__ void finish(const double*) {}
};

template <typename T>
void launch_fcg_final_x(const Geo& g, hipStream_t s, T* x, const T* p, const Scal* S)
{
    OpFcgFinalX<T> op;
    op.gate = nullptr;
    op.x = x;
    op.p = p;
    op.S = S;
    run_vector<0>(g, s, op, kNoRed);
}

template <typename T>
struct OpFcgUpdate : Gate {
    T* __restrict__ r;
    const T* __restrict__ Ap;
    Scal* S;
    bool history;
    T alpha;
    int skip;
    struct R { T r, ap; };
    __device__ void load()
    {
        alpha = (T)S->v[S_ALPHA];
        skip = S->restart;
    }
    // r -= alpha Ap; x takes alpha p in the next stencil pass (or in the final
    // x kernel after the last iteration)
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(r + c), skip ? (T)0 : ld<NT>(Ap + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double* acc) const
    {
        T rv = v.r;
        if (!skip) {
            rv = v.r - alpha * v.ap;
            put<NT>(r + c, rv);
        }
        acc[0] += (double)rv * (double)rv;
    }
    __device__ void finish(const double* t) { update_finish(S, t[0], history); }
};

template <typename T>
void launch_fcg_update(const Geo& g, hipStream_t s, RedBuf rb, T* r, const T* Ap, Scal* S, bool history)
{
    OpFcgUpdate<T> op;
    op.gate = &S->done;
    op.r = r;
    op.Ap = Ap;
    op.S = S;
    op.history = history;
    run_vector<1>(g, s, op, rb);
}

// --------------------------------------------------- iterative refinement

struct OpIrRes : Gate {
    const double* __restrict__ x;
    const double* __restrict__ b;
    float* __restrict__ r32;
    Scal* So;
    Scal* SI;
    double itol, itol0;  // inner tolerance: first outer step, later ones
    double adapt;        // > 0: no less than adapt * tol / ||r||
    __device__ void load() {}
    struct Ox { double b; };
    __device__ double in(long long c) const { return x[c]; }
    template <bool NT> __device__ Ox out_raw(long long c) const { return {ld<NT>(b + c)}; }
    template <bool NT> __device__ void out(long long c, double, double Av, const double&, const Ox& o, double* acc) const
    {
        const double rv = o.b - Av;
        const float rf = (float)rv;
        put<NT>(r32 + c, rf);
        acc[0] += rv * rv;
        acc[1] += (double)rf * (double)rf;
    }
    __device__ void finish(const double* t)
    {
        const double e = sqrt(t[0]);
        So->v[S_ERR] = e;
        So->v[S_ERR_OP] = e;
        const int o = So->outer;
        if (So->hist != nullptr && o < So->hist_cap) So->hist[o] = e;
        if (o == 0) So->v[S_ERR0] = e;
        So->done = e < So->v[S_TOL] ? 1 : 0;
        SI->v[S_INNER_NORM] = sqrt(t[1]);
        const double base = o == 0 ? itol0 : itol;
        SI->v[S_TOL] = (adapt > 0.0 && e > 0.0) ? fmax(base, adapt * So->v[S_TOL] / e) : base;
    }
};

void launch_ir_residual(const Geo& g, hipStream_t s, RedBuf rb, const double* x, const double* b, float* r32, Scal* So,
                        Scal* SI, double itol, double itol0, double adapt)
{
    OpIrRes op;
    op.gate = nullptr;
    op.x = x;
    op.b = b;
    op.r32 = r32;
    op.So = So;
    op.SI = SI;
    op.itol = itol;
    op.itol0 = itol0;
    op.adapt = adapt;
    run_stencil<double, 2>(g, s, op, rb);
}

struct OpIrUpdate : Gate {
    double* __restrict__ x;
    const float* __restrict__ d;
    const Scal* SI;
    float sc;
    struct R { double x; float d; };
    __device__ void load() { sc = (float)SI->v[S_INNER_NORM]; }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(x + c), ld<NT>(d + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double*) const { put<NT>(x + c, v.x + (double)(v.d * sc)); }
    __device__ void finish(const double*) {}
};

void launch_ir_update(const Geo& g, hipStream_t s, double* x, const float* d, const Scal* SI)
{
    OpIrUpdate op;
    op.gate = nullptr;
    op.x = x;
    op.d = d;
    op.SI = SI;
    run_vector<0>(g, s, op, kNoRed);
}

// inner solve start: the non-main normalisation of BaseCG (x = 0, b /= ||b||,
// r0 = b) applied to r32 in place
struct OpIrInit : Gate {
    float* __restrict__ r;
    float* __restrict__ x;
    float* __restrict__ p;
    Scal* SI;
    float inv;
    struct R { float r; };
    __device__ void load() { inv = (float)(1.0 / SI->v[S_INNER_NORM]); }
    template <bool NT> __device__ R fetch(long long c) const { return {ld<NT>(r + c)}; }
    template <bool NT> __device__ void apply(long long c, const R& v, int, int, int, double* acc) const
    {
        const float rv = v.r * inv;
        put<NT>(r + c, rv);
        put<NT>(x + c, 0.0f);
        put<NT>(p + c, 0.0f);
        acc[0] += (double)rv * (double)rv;
    }
    __device__ void finish(const double* t)
    {
        const double e = sqrt(t[0]);
        SI->v[S_ERR0] = e;
        SI->v[S_ERR] = e;
        SI->v[S_RR] = t[0];
        SI->v[S_BETA] = 0.0;
        SI->v[S_PAP_OLD] = 1.0;
        SI->v[S_ALPHA] = 0.0;
        SI->v[S_AUX2] = 1e300;
        SI->fallback = 0;
        SI->restart = 0;
        SI->passes = 0;
        SI->recheck = 0;
        SI->iter = 0;
        SI->done = e < SI->v[S_TOL] ? 2 : 0;
    }
};

void launch_ir_inner_init(const Geo& g, hipStream_t s, RedBuf rb, float* r, float* x, float* p, Scal* SI)
{
    OpIrInit op;
    op.gate = nullptr;
    op.r = r;
    op.x = x;
    op.p = p;
    op.SI = SI;
    run_vector<1>(g, s, op, rb);
}

// ------------------------------------------------------ instantiations

#define PPS_INST_T(T)                                                                                          \
    template void launch_apply_A<T>(const Geo&, hipStream_t, const T*, T*);                                    \
    template void launch_copy<T>(const Geo&, hipStream_t, const T*, T*);                                       \
    template void launch_dot<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, double*, const int*);      \
    template void launch_scale_box<T>(const Geo&, hipStream_t, T*, const Scal*, int);                          \
    template void launch_fill<T>(const Geo&, hipStream_t, T*, T);                                              \
    template void launch_ghost<T>(hipStream_t, const Layout&, const Faces&, T*, int, const Scal*, const int*);  \
    template void launch_cg_pass<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, T*, T*, T*, Scal*, bool, \
                                    int);                                                                          \
    template void launch_cg_A2<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, T*, T*, T*, Scal*, int);    \
    template void launch_cg_final_x<T>(const Geo&, hipStream_t, T*, const T*, const Scal*);                      \
    template void launch_cg_B<T>(const Geo&, hipStream_t, RedBuf, T*, const T*, Scal*, bool);                  \
    template void launch_cg_rz<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, Scal*);                 \
    template void launch_pointwise<T>(const Geo&, hipStream_t, const T*, T*, double, const int*);              \
    template void launch_bicg_k1<T>(const Geo&, hipStream_t, RedBuf, int, const T*, double, T*, const T*, Scal*);   \
    template void launch_bicg_k2<T>(const Geo&, hipStream_t, T*, const T*, const Scal*);                       \
    template void launch_bicg_k3<T>(const Geo&, hipStream_t, RedBuf, int, const T*, double, T*, const T*, Scal*);   \
    template void launch_bicg_k45<T>(const Geo&, hipStream_t, RedBuf, T*, const T*, double, const T*, double, T*, \
                                     const T*, const T*, Scal*, bool);                                         \
    template void launch_bicg_k6<T>(const Geo&, hipStream_t, T*, const T*, const T*, const Scal*);             \
    template void launch_cheb_first<T>(const Geo&, hipStream_t, const T*, T*, T*, double, double, const int*); \
    template void launch_fcg_gamma<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, Scal*);             \
    template void launch_fcg_gamma_finish<T>(hipStream_t, RedBuf, int, int, Scal*);                             \
    template void launch_fcg_p<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, T*, T*, const T*, T*, Scal*); \
    template void launch_fcg_p_fused<T>(const Geo&, hipStream_t, RedBuf, const T*, const T*, T*, T*, const T*, T*,    \
                                        Scal*, bool, int);                                                         \
    template void launch_fcg_final_x<T>(const Geo&, hipStream_t, T*, const T*, const Scal*);                      \
    template void launch_fcg_flush<T>(const Geo&, hipStream_t, T*, T* const[kFcgRing], Scal*);                    \
    template void launch_fcg_update<T>(const Geo&, hipStream_t, RedBuf, T*, const T*, Scal*, bool);

PPS_INST_T(double)
PPS_INST_T(float)

#define PPS_INST_CHEB(T, TO)                                                                                     \
    template void launch_cheb_multi<T, TO>(const Geo&, const ChebPairGeo&, hipStream_t, int, const T*, const T*,  \
                                           const T*, T*, TO*, const double*, const double*, const double*, double, \
                                           double, double, const int*);
PPS_INST_CHEB(double, double)
PPS_INST_CHEB(float, float)
PPS_INST_CHEB(float, double)
template void launch_cheb_sweep<double, double>(const Geo&, hipStream_t, const double*, const double*, const double*,
                                                double*, double, double, double, double, const int*);
template void launch_cheb_sweep<float, float>(const Geo&, hipStream_t, const float*, const float*, const float*, float*,
                                              double, double, double, double, const int*);
template void launch_cheb_sweep<float, double>(const Geo&, hipStream_t, const float*, const float*, const float*,
                                               double*, double, double, double, double, const int*);
template void launch_cheb_first_out<double, double>(const Geo&, hipStream_t, const double*, double*, double, double, int,
                                                    double, const int*);
template void launch_cheb_first_out<float, float>(const Geo&, hipStream_t, const float*, float*, double, double, int,
                                                  double, const int*);
template void launch_cheb_first_out<float, double>(const Geo&, hipStream_t, const float*, double*, double, double, int,
                                                   double, const int*);
template void launch_cast<double, float>(const Geo&, hipStream_t, const double*, float*, const int*);
template void launch_cast<float, double>(const Geo&, hipStream_t, const float*, double*, const int*);

}  // namespace pps
