// dslash_direct.hip -- the operator on the caller's own vectors: one [site][spin]
// [colour] array per right-hand side, FP32 or FP64, Nc <= 4, without the copies to
// and from the RHS-innermost layout.
//
// The hops of dslash_lane.h, one lane per (site, RHS).  Consecutive lanes hold consecutive sites of one
// right-hand side and read their spinors as 16-byte pieces, so that a wavefront walks runs of whole lines
// of a few vectors (with consecutive right-hand sides, as in the RHS-innermost layout, every load touches
// the same offset of R vectors: 24^3 x 48, 16 RHS, FP32 1436 us, against 1128).  Both parities of
// M = A - kappa D go into one launch.
//
// Against copies to the RHS-innermost layout, two hops and copies back (whole calls): FP32 24^3 x 48 1964 ->
// 1128 us at 16 RHS, 705 -> 389 at 4, 16^3 x 32, 32 RHS 1108 -> 563, 20 x 14 x 10 x 18, 5 RHS with clover
// 105 -> 72; FP64 16^3 x 32, 12 RHS 575 -> 470, 24^3 x 48, 1 RHS 1237 -> 1135, 8^4, 4 RHS 42 -> 29; faster
// at every size timed, so no size is kept on the copies.  A hop by itself is slower than the RHS-innermost
// one (FP32 24^3 x 48, 16 RHS: 550 against 325 us), so solvers keep that layout.
#include <algorithm>

#include "dslash_direct.h"
#include "dslash_lane.h"
#include "geom.h"

namespace qcu {
namespace {

using namespace lane;

extern __shared__ __align__(16) unsigned char direct_smem[];

// one spinor of one right-hand side: 4 NC complex numbers, 16-byte aligned
template <typename C, int NC>
struct Spinor {
    static constexpr int kPieces = 4 * NC * int(sizeof(C)) / 16;
    u32x4 q[kPieces];
};
template <typename C, int NC>
__device__ __forceinline__ const u32x4 *pieces(const C *base, unsigned site) {
    unsigned k = site * unsigned(Spinor<C, NC>::kPieces);
    asm volatile("" : "+v"(k));  // as MrhsRows::fetch
    return reinterpret_cast<const u32x4 *>(base) + k;
}

template <typename C, int NC>
struct VectorRows {
    static constexpr bool kSiteFast = true;  // consecutive lanes: consecutive sites of one vector
    const C *base;                           // this lane's vector, input parity
    __device__ __forceinline__ void fetch(Vec<C, 1> (&w)[4][NC], int site) const {
        const u32x4 *q = pieces<C, NC>(base, unsigned(site));
        Spinor<C, NC> sp;
#pragma unroll
        for (int i = 0; i < Spinor<C, NC>::kPieces; ++i) sp.q[i] = q[i];
        __builtin_memcpy(&w, &sp, sizeof(sp));
    }
};

// FULL: out_p = x_p + coef D_p x_{1-p} (CLOV: A_pp x_p) for parity p = blockIdx.y of full vectors; else
// out = coef D x, parity `parity`, of half vectors
template <typename S, int NC, bool DAG, bool FULL, bool CLOV>
__global__ __launch_bounds__(256, sizeof(S) == 8 ? (NC == 4 ? 2 : 3) : 4) void k_operator_direct(
    PtrTable out, PtrTable in, const Cx<S> *__restrict__ gauge, const Cx<S> *__restrict__ clover, S coef, int Vh, int R,
    int spb, int lds_blocks, int parity, const int *__restrict__ walk) {
    using C = Cx<S>;
    const int par = FULL ? int(blockIdx.y) : parity;
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * spb;
    const long half = long(Vh) * 4 * NC;
    const int rv = min(int(threadIdx.x) / spb, R - 1);
    const C *x = static_cast<const C *>(in.p[rv]);
    const VectorRows<C, NC> src{FULL ? x + (1 - par) * half : x};
    Cx<S> acc[4][NC][1];
    Place p;
    Clover<S, NC> cl{nullptr, nullptr};
    if constexpr (CLOV) {
        cl = {clover + long(par) * Vh * (8 * NC * NC), reinterpret_cast<Cx<S> *>(direct_smem + lds_blocks)};
        p = hops_from<S, NC, 1, DAG, false, false>(acc, direct_smem, src, gauge, Vh, R, spb, pos0, par, walk, cl);
    } else {
        p = hops_from<S, NC, 1, DAG, false, false>(acc, direct_smem, src, gauge, Vh, R, spb, pos0, par, walk, NoExtra{});
    }
    if (!p.active) return;
    Vec<C, 1> xw[4][NC], ow[4][NC];
    if constexpr (FULL) VectorRows<C, NC>{x + par * half}.fetch(xw, p.site);
    if constexpr (CLOV) {
        cl.template rows_of<1>(
            acc, true, false, coef, p.local, [&](int k) { return xw[k / NC][k % NC]; },
            [&](int k, const Cx<S>(&o)[1], const Cx<S>(&)[1]) { ow[k / NC][k % NC].c[0] = o[0]; });
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const Cx<S> h = acc[s][c][0];
                if constexpr (FULL) {
                    const Cx<S> v = xw[s][c].c[0];
                    ow[s][c].c[0] = {fma(coef, h.re, v.re), fma(coef, h.im, v.im)};
                } else {
                    ow[s][c].c[0] = coef * h;
                }
            }
    }
    Spinor<C, NC> sp;
    __builtin_memcpy(&sp, &ow, sizeof(sp));
    C *o = static_cast<C *>(const_cast<void *>(out.p[rv])) + (FULL ? par * half : 0L);
    u32x4 *q = reinterpret_cast<u32x4 *>(o) + unsigned(p.site) * unsigned(Spinor<C, NC>::kPieces);
#pragma unroll
    for (int i = 0; i < Spinor<C, NC>::kPieces; ++i) q[i] = sp.q[i];
}

// Small lattices: a wavefront per direction, 64 / R sites per workgroup (direction(), dslash_lane.h);
// wavefront mu finishes spin mu.
template <typename S, int NC, bool DAG, bool FULL, bool CLOV>
__global__ __launch_bounds__(256) void k_operator_direct_split(
    PtrTable out, PtrTable in, const Cx<S> *__restrict__ gauge, const Cx<S> *__restrict__ clover, S coef, int Vh, int R,
    int spb, int parity, const int *__restrict__ walk) {
    using C = Cx<S>;
    constexpr int n = 2 * NC;
    auto *part = reinterpret_cast<C *>(direct_smem);
    const int par = FULL ? int(blockIdx.y) : parity;
    const int lane = threadIdx.x & 63;
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * spb;
    const int ns = min(spb, Vh - pos0);
    const int r = lane / spb, local = lane - r * spb, rv = min(r, R - 1);
    const int *row = walk + (long(par) * Vh + pos0 + min(local, ns - 1)) * 9;
    const long half = long(Vh) * 4 * NC;
    const C *x = static_cast<const C *>(in.p[rv]);
    Cx<S> acc[4][NC][1];
    direction_of<S, NC, DAG>(mu, acc, VectorRows<C, NC>{FULL ? x + (1 - par) * half : x}, gauge, Vh, par, row);
    put_parts<S, NC>(part, mu, lane, acc);
    const long site = row[0];
    // this spin's rows: of the chirality's spinor where the blocks mix its two spins
    constexpr int nx = CLOV ? n : NC;
    C xv[nx];
    if constexpr (FULL) {
        const C *xs = x + par * half + site * 4 * NC + (CLOV ? (mu >> 1) * n : mu * NC);
#pragma unroll
        for (int k = 0; k < nx; ++k) xv[k] = xs[k];
    }
    __syncthreads();
    if (local >= ns || r >= R) return;
    C *o = static_cast<C *>(const_cast<void *>(out.p[rv])) + (FULL ? par * half : 0L) + site * 4 * NC + mu * NC;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const Cx<S> h = sum_parts<S, NC>(part, mu, lane, c);
        if constexpr (CLOV) {
            const C *b = clover + ((long(par) * Vh + site) * 2 + (mu >> 1)) * n * n + ((mu & 1) * NC + c) * n;
            Cx<S> v{S(0), S(0)};
#pragma unroll
            for (int k = 0; k < n; ++k) cfma(v, b[k], xv[k]);
            o[c] = {fma(coef, h.re, v.re), fma(coef, h.im, v.im)};
        } else if constexpr (FULL) {
            o[c] = {fma(coef, h.re, xv[c].re), fma(coef, h.im, xv[c].im)};
        } else {
            o[c] = coef * h;
        }
    }
}

template <typename S, int NC>
hipError_t launch_split(const OperatorArgs &a, const GeomTables &tab, hipStream_t stream) {
    const int spb = 64 / a.R;
    auto k = a.clover ? (a.dagger ? k_operator_direct_split<S, NC, true, true, true> : k_operator_direct_split<S, NC, false, true, true>)
             : a.full ? (a.dagger ? k_operator_direct_split<S, NC, true, true, false> : k_operator_direct_split<S, NC, false, true, false>)
                      : (a.dagger ? k_operator_direct_split<S, NC, true, false, false> : k_operator_direct_split<S, NC, false, false, false>);
    hipLaunchKernelGGL(k, dim3(div_up(a.g.Vh, spb), a.full ? 2 : 1), dim3(256), size_t(16) * NC * 64 * sizeof(Cx<S>), stream,
                       a.out, a.in, static_cast<const Cx<S> *>(a.gauge), static_cast<const Cx<S> *>(a.clover), S(a.coef),
                       a.g.Vh, a.R, spb, a.parity, tab.walk);
    return hipGetLastError();
}

template <typename S, int NC>
hipError_t launch_t(const OperatorArgs &a, int by, int bz, hipStream_t stream) {
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, by, bz, tab, stream));
    constexpr int links = kSiteLds<S, NC>, blocks = kCloverRow<NC> * int(sizeof(Cx<S>));
    const int per_site = links + (a.clover ? blocks : 0);
    const int par = a.full ? 2 : 1;
    if (split_over_directions(double(par) * a.g.Vh, a.R)) return launch_split<S, NC>(a, tab, stream);
    // as the RHS-innermost launch: 256 lanes, fewer where the grid would leave compute units idle
    int threads = 256;
    while (threads > 64 && threads / 2 >= a.R && par * div_up(a.g.Vh, std::max(1, threads / a.R)) < 2 * num_cus())
        threads /= 2;
    int spb = std::max(1, threads / a.R);
    spb = std::min(spb, std::max(1, 65520 / per_site));
    threads = (spb * a.R + 63) / 64 * 64;
    const int off = (spb * links + 15) / 16 * 16;
    const size_t lds = size_t(off) + (a.clover ? size_t(spb) * blocks : 0);
    auto k = a.clover ? (a.dagger ? k_operator_direct<S, NC, true, true, true> : k_operator_direct<S, NC, false, true, true>)
             : a.full ? (a.dagger ? k_operator_direct<S, NC, true, true, false> : k_operator_direct<S, NC, false, true, false>)
                      : (a.dagger ? k_operator_direct<S, NC, true, false, false> : k_operator_direct<S, NC, false, false, false>);
    hipLaunchKernelGGL(k, dim3(div_up(a.g.Vh, spb), par), dim3(threads), lds, stream, a.out, a.in,
                       static_cast<const Cx<S> *>(a.gauge), static_cast<const Cx<S> *>(a.clover), S(a.coef), a.g.Vh,
                       a.R, spb, off, a.parity, tab.walk);
    return hipGetLastError();
}

template <typename S>
hipError_t launch_s(const OperatorArgs &a, int by, int bz, hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_t<S, 2>(a, by, bz, stream);
        case 3: return launch_t<S, 3>(a, by, bz, stream);
        case 4: return launch_t<S, 4>(a, by, bz, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool operator_direct_supported(const OperatorArgs &a) {
    if ((a.prec != kSingle && a.prec != kDouble) || a.R < 1 || a.R > kMaxPtrs || a.g.Vh < 1 || (a.clover && !a.full) ||
        !dslash_lane_supported(a.g, a.Nc, a.R, a.prec))
        return false;
    // the kernel named for this shape, or forced, is another one: keep to it
    DslashArgs h{nullptr, nullptr, nullptr, nullptr, 1.0, a.g, a.Nc, a.R, a.parity, a.dagger, a.prec};
    if (dslash_resolve(h).variant != kDslashLaneRhs) return false;
    // A site's results are written while others still read their neighbours: no output may overlap an
    // input or another output.  16-byte pieces: as aligned as the caller's vectors are
    const uintptr_t bytes = uintptr_t(a.g.Vh) * 4 * a.Nc * 2 * prec_bytes(a.prec) * (a.full ? 2 : 1);
    uintptr_t lo[2 * kMaxPtrs];
    for (int r = 0; r < a.R; ++r) {
        lo[r] = reinterpret_cast<uintptr_t>(a.out.p[r]);
        lo[a.R + r] = reinterpret_cast<uintptr_t>(a.in.p[r]);
        if ((lo[r] | lo[a.R + r]) % 16) return false;
    }
    std::sort(lo, lo + a.R);                // outputs
    std::sort(lo + a.R, lo + 2 * a.R);      // inputs, which may coincide
    for (int r = 0; r + 1 < a.R; ++r)
        if (lo[r + 1] - lo[r] < bytes) return false;
    for (int o = 0, i = a.R; o < a.R && i < 2 * a.R;) {
        if (lo[o] < lo[i]) {
            if (lo[i] - lo[o] < bytes) return false;
            ++o;
        } else {
            if (lo[o] - lo[i] < bytes) return false;
            ++i;
        }
    }
    return true;
}

hipError_t launch_operator_direct(const OperatorArgs &a, hipStream_t stream) {
    if (!operator_direct_supported(a)) return hipErrorInvalidValue;
    DslashArgs h{nullptr, nullptr, nullptr, nullptr, 1.0, a.g, a.Nc, a.R, a.parity, a.dagger, a.prec};
    const DslashTune t = dslash_resolve(h);
    if (t.by <= 0 || t.bz <= 0 || a.g.L[1] % t.by || a.g.L[2] % t.bz) return hipErrorInvalidValue;
    return a.prec == kDouble ? launch_s<double>(a, t.by, t.bz, stream) : launch_s<float>(a, t.by, t.bz, stream);
}

}  // namespace qcu
