// dslash_lane.hip -- lane-per-(site, RHS) Wilson hopping term (variants
// kDslashLaneRhs and, in 16 bits, kDslashLane16; dslash_lane.h), every storage
// precision, Nc <= 4.
//
// What bounds it: the bytes that miss the XCD's L2 (FP64, FP32: 4.9 and 2.2 GB
// per hop at 24^3 x 48, 16 RHS, at 6-7 TB/s, against 2.4 and 1.2 GB that the
// operator needs) and, in 16 bits, the L2 -> L1 fill of the neighbour spinors
// (48 lines per site; the same loads without the arithmetic take the same time).
// Against the wave-per-site kernel, whose 16 lanes per direction idle when R is
// no multiple of 16 and whose cross-lane sums cost 3.5 times the instructions
// per site: FP64 24^3 x 48, 16 RHS 1012 -> 636 us, 16^3 x 32, 12 RHS 190 -> 79 us,
// 8^4, 4 RHS 22 -> 9 us; FP32 592 -> 323 us, 109 -> 57 us, 20 -> 9 us; SU(4) 16^4,
// 17 RHS FP32 131 -> 62 us.
#include <algorithm>

#include "dslash_lane.h"
#include "geom.h"

namespace qcu {
namespace {

using namespace lane;

extern __shared__ __align__(16) unsigned char lane_smem[];

// out = coef acc (+ xpay) at this lane's place
template <typename S, int NC, int V>
__device__ __forceinline__ void store_lane(const Cx<typename Arith<S>::T> (&acc)[4][NC][V], typename Arith<S>::C *out,
                                           const typename Arith<S>::C *xpay, typename Arith<S>::T coef, const Place &p,
                                           int R, unsigned vec_bytes) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    using RW = Raw<V * int(sizeof(C))>;
    using W = Vec<C, V>;
    const unsigned rb = unsigned(R) * unsigned(sizeof(C));
    const auto r_out = rsrc(out, vec_bytes);
    if (xpay) {
        const auto r_x = rsrc(xpay, vec_bytes);
        W xw[4][NC];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) xw[s][c] = __builtin_bit_cast(W, RW::load(r_x, p.vo, unsigned(s * NC + c) * rb));
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                W o;
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    Cx<T> x = load_cx<T>(&xw[s][c].c[v]);
                    x.re = fma(coef, acc[s][c][v].re, x.re);
                    x.im = fma(coef, acc[s][c][v].im, x.im);
                    store_cx(&o.c[v], x);
                }
                RW::store(r_out, __builtin_bit_cast(typename RW::type, o), p.vo, unsigned(s * NC + c) * rb);
            }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                W o;
#pragma unroll
                for (int v = 0; v < V; ++v) store_cx(&o.c[v], coef * acc[s][c][v]);
                RW::store(r_out, __builtin_bit_cast(typename RW::type, o), p.vo, unsigned(s * NC + c) * rb);
            }
    }
}

// out = coef D in (+ xpay)
template <typename S, int NC, int V, bool DAG, bool ORD = false>
__global__ __launch_bounds__(256, ORD ? 2 : (kMinWaves<S, NC, V>)) void k_dslash_lane(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *xpay, typename Arith<S>::T coef, int Vh,
    int R, int RV, int spb, int parity, const int *__restrict__ walk, unsigned vec_bytes) {
    Cx<typename Arith<S>::T> acc[4][NC][V];
    const Place p = hops<S, NC, V, DAG, ORD, !ORD && kAhead<S, NC>>(acc, lane_smem, in, gauge, Vh, R, RV, spb,
                                             xcd_remap(blockIdx.x, gridDim.x) * spb, parity, walk, vec_bytes);
    if (p.active) store_lane<S, NC, V>(acc, out, xpay, coef, p, R, vec_bytes);
}

// With the clover blocks of the output sites: out = A x + coef D in, or (x null) out = A (coef D in + xpay).
// The hop's sums never leave the registers in between; a separate pass over the vector reads and writes it
// once more (16^3 x 32, SU(3), 12 RHS: FP16 64 -> 47.5 us, FP64 185 -> 134 us against hop and pass).  The
// blocks' LDS reads and products are most of what is left over the bare hop (35 us in FP16).
template <typename S, int NC, int V, bool DAG>
__global__ __launch_bounds__(256, (kMinWaves<S, NC, V>)) void k_dslash_lane_clover(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *__restrict__ x,
    const typename Arith<S>::C *xpay, const Cx<typename Arith<S>::T> *__restrict__ blocks, typename Arith<S>::T coef,
    int Vh, int R, int RV, int spb, int parity, const int *__restrict__ walk, unsigned vec_bytes) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    using RW = Raw<V * int(sizeof(C))>;
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * spb;
    const Clover<S, NC> cl = clover_lds<S, NC>(blocks, lane_smem, spb);
    Cx<T> acc[4][NC][V];
    const Place p =
        hops<S, NC, V, DAG, false, kAhead<S, NC>>(acc, lane_smem, in, gauge, Vh, R, RV, spb, pos0, parity, walk, vec_bytes, cl);
    if (!p.active) return;
    const unsigned rb = unsigned(R) * unsigned(sizeof(C));
    const auto r_out = rsrc(out, vec_bytes);
    cl.template rows<V>(acc, x, xpay, coef, p, min(spb, Vh - pos0), rb, vec_bytes,
                        [&](int row, const Cx<T>(&o)[V], const Cx<T>(&)[V]) {
                            Vec<C, V> w;
#pragma unroll
                            for (int i = 0; i < V; ++i) store_cx(&w.c[i], o[i]);
                            RW::store(r_out, __builtin_bit_cast(typename RW::type, w), p.vo, unsigned(row) * rb);
                        });
}

// Small lattices: a wavefront per direction (direction(), dslash_lane.h), summed through LDS; wavefront mu
// finishes spin mu.
template <typename S, int NC, bool DAG>
__global__ __launch_bounds__(256) void k_dslash_lane_split(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *xpay, typename Arith<S>::T coef, int Vh,
    int R, int spb, int parity, const int *__restrict__ walk, unsigned vec_bytes) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    using RW = Raw<int(sizeof(C))>;
    auto *part = reinterpret_cast<Cx<T> *>(lane_smem);  // [spin][wavefront][colour][lane]
    const int lane = threadIdx.x & 63;
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * spb;
    const int ns = min(spb, Vh - pos0);
    const int local = lane / R, r = lane - local * R;
    const int *row = walk + (long(parity) * Vh + pos0 + min(local, ns - 1)) * 9;
    const unsigned rb = unsigned(R) * unsigned(sizeof(C)), lo = unsigned(r) * unsigned(sizeof(C));
    Cx<T> acc[4][NC][1];
    direction_of<S, NC, DAG>(mu, acc, MrhsRows<C, NC, 1>{rsrc(in, vec_bytes), rb, lo}, gauge, Vh, parity, row);
    put_parts<T, NC>(part, mu, lane, acc);
    const bool active = local < ns;
    const unsigned vo = unsigned(row[0]) * 4u * NC * rb + unsigned(mu) * NC * rb + lo;
    C xw[NC];
    if (xpay) {
        const auto r_x = rsrc(xpay, vec_bytes);
#pragma unroll
        for (int c = 0; c < NC; ++c) xw[c] = __builtin_bit_cast(C, RW::load(r_x, vo, unsigned(c) * rb));
    }
    __syncthreads();
    if (!active) return;
    const auto r_out = rsrc(out, vec_bytes);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        Cx<T> v = sum_parts<T, NC>(part, mu, lane, c);
        if (xpay) {
            Cx<T> x = load_cx<T>(&xw[c]);
            x.re = fma(coef, v.re, x.re);
            x.im = fma(coef, v.im, x.im);
            v = x;
        } else {
            v = coef * v;
        }
        C o;
        store_cx(&o, v);
        RW::store(r_out, __builtin_bit_cast(typename RW::type, o), vo, unsigned(c) * rb);
    }
}

// Reliable-update residual (FP64 hop): d = b - (xpay + coef D in) is not stored; lo = scale_r d in the inner
// storage and part[block][r] = sum over the workgroup's sites of |d|^2.  CLOV: A xpay (clover blocks) in
// place of xpay.
template <int NC, typename LO, bool CLOV>
__global__ __launch_bounds__(256, (kMinWaves<double, NC, 1>)) void k_dslash_lane_residual(
    LO *__restrict__ lo, const Cx<double> *__restrict__ in, const Cx<double> *__restrict__ gauge,
    const Cx<double> *__restrict__ xpay, const Cx<double> *__restrict__ blocks, const Cx<double> *__restrict__ b,
    const double *__restrict__ scale, double *__restrict__ part, double coef, int Vh, int R, int spb, int parity, const int *__restrict__ walk,
    unsigned vec_bytes) {
    using RL = Raw<int(sizeof(LO))>;
    using W = Vec<Cx<double>, 1>;
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    Cx<double> acc[4][NC][1];
    const Clover<double, NC> cl = clover_lds<double, NC>(blocks, lane_smem, spb);
    Place p;
    if constexpr (CLOV)
        p = hops<double, NC, 1, false>(acc, lane_smem, in, gauge, Vh, R, R, spb, blk * spb, parity, walk, vec_bytes, cl);
    else
        p = hops<double, NC, 1, false>(acc, lane_smem, in, gauge, Vh, R, R, spb, blk * spb, parity, walk, vec_bytes);
    double a2[1][1] = {{0.0}};
    if (p.active) {
        const unsigned rb = unsigned(R) * 16u;
        const auto r_x = rsrc(xpay, vec_bytes), r_b = rsrc(b, vec_bytes);
        const auto r_lo = rsrc(lo, vec_bytes / 16u * unsigned(sizeof(LO)));
        const double sc = scale[p.rv];
        const auto finish = [&](int row, Cx<double> v, Cx<double> bv) {
            const Cx<double> d = bv - v;
            a2[0][0] = fma(d.re, d.re, fma(d.im, d.im, a2[0][0]));
            LO o;
            store_cx(&o, sc * d);
            RL::store(r_lo, __builtin_bit_cast(typename RL::type, o), p.vo / 16u * unsigned(sizeof(LO)),
                      unsigned(row) * unsigned(R) * unsigned(sizeof(LO)));
        };
        if constexpr (CLOV) {
            cl.template rows<1>(acc, xpay, nullptr, coef, p, min(spb, Vh - blk * spb), rb, vec_bytes,
                                [&](int row, const Cx<double>(&v)[1], const Cx<double>(&)[1]) {
                                    finish(row, v[0], __builtin_bit_cast(W, Raw<16>::load(r_b, p.vo, unsigned(row) * rb)).c[0]);
                                });
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                W xw[NC], bw[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    xw[c] = __builtin_bit_cast(W, Raw<16>::load(r_x, p.vo, unsigned(s * NC + c) * rb));
                    bw[c] = __builtin_bit_cast(W, Raw<16>::load(r_b, p.vo, unsigned(s * NC + c) * rb));
                }
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    Cx<double> v = xw[c].c[0];
                    v.re = fma(coef, acc[s][c][0].re, v.re);
                    v.im = fma(coef, acc[s][c][0].im, v.im);
                    finish(s * NC + c, v, bw[c].c[0]);
                }
            }
        }
    }
    sum_sites<1, 1>(a2, reinterpret_cast<double *>(lane_smem), p, R, min(spb, Vh - blk * spb));
    if (int(threadIdx.x) < R) part[long(blockIdx.x) * R + threadIdx.x] = a2[0][0];
}

// Every group of a batch in one launch (blockIdx.y = group, SegTab layout); spb[g] sites per workgroup.
struct GroupSites {
    int spb[kMaxGroups];
};
template <typename S, int NC, bool DAG>
__global__ __launch_bounds__(256, (kMinWaves<S, NC, 1>)) void k_dslash_lane_groups(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *__restrict__ xpay,
    typename Arith<S>::T coef, int Vh, int parity, const int *__restrict__ walk, SegTab tab, GroupSites gs) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    const int grp = blockIdx.y;
    if (tab.done && tab.done[grp]) return;
    const int spb = gs.spb[grp], R = tab.R[grp];
    const int nblk = (Vh + spb - 1) / spb;
    if (int(blockIdx.x) >= nblk) return;
    const long off = tab.n * tab.base[grp];
    const unsigned vec_bytes = unsigned(tab.n * R * long(sizeof(C)));
    Cx<T> acc[4][NC][1];
    const Place p = hops<S, NC, 1, DAG, false, kAhead<S, NC>>(acc, lane_smem, in + off, gauge, Vh, R, R, spb,
                                        xcd_remap(blockIdx.x, nblk) * spb, parity, walk, vec_bytes);
    if (p.active) store_lane<S, NC, 1>(acc, out + off, xpay ? xpay + off : nullptr, coef, p, R, vec_bytes);
}

// fewest sites per workgroup of the forms that leave a partial sum per workgroup
template <typename S>
int min_sites(int Nc, int Vh, int R) {
    const auto least = [&](auto nc) {
        return std::min(lane_shape<S, decltype(nc)::value>(Vh, R, 1).spb, lane_shape<S, decltype(nc)::value>(Vh, R, 1, true).spb);
    };
    return Nc == 2   ? least(std::integral_constant<int, 2>{})
           : Nc == 3 ? least(std::integral_constant<int, 3>{})
                     : least(std::integral_constant<int, 4>{});
}

template <int NC, typename LO>
hipError_t launch_residual(const DslashArgs &a, const DslashTune &t, const void *b, void *lo, const double *scale,
                           double *partials, int &nblk, hipStream_t stream) {
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, t.by, t.bz, tab, stream));
    const Shape sh = lane_shape<double, NC>(a.g.Vh, a.R, 1, a.clover != nullptr);
    nblk = div_up(a.g.Vh, sh.spb);
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * 16);
    auto k = a.clover ? k_dslash_lane_residual<NC, LO, true> : k_dslash_lane_residual<NC, LO, false>;
    hipLaunchKernelGGL(k, dim3(nblk), dim3(sh.threads), sh.lds, stream,
                       static_cast<LO *>(lo), static_cast<const Cx<double> *>(a.in),
                       static_cast<const Cx<double> *>(a.gauge),
                       static_cast<const Cx<double> *>(a.clover ? a.clover_in : a.xpay),
                       static_cast<const Cx<double> *>(a.clover),
                       static_cast<const Cx<double> *>(b), scale, partials, a.coef, a.g.Vh, a.R, sh.spb, a.parity,
                       tab.walk, vec_bytes);
    return hipGetLastError();
}

template <int NC>
hipError_t launch_residual_lo(const DslashArgs &a, const DslashTune &t, const void *b, void *lo, int lo_prec,
                              const double *scale, double *partials, int &nblk, hipStream_t stream) {
    switch (lo_prec) {
        case kSingle: return launch_residual<NC, Cx<float>>(a, t, b, lo, scale, partials, nblk, stream);
        case kHalf: return launch_residual<NC, Half2Store>(a, t, b, lo, scale, partials, nblk, stream);
        case kBF16: return launch_residual<NC, Bf162Store>(a, t, b, lo, scale, partials, nblk, stream);
        default: return hipErrorInvalidValue;
    }
}

template <typename S, int NC>
hipError_t launch_groups(const DslashArgs &a, const SegTab &seg, int by, int bz, hipStream_t stream) {
    using C = typename Arith<S>::C;
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, by, bz, tab, stream));
    GroupSites gs{};
    int nmax = 1, smax = 1;
    for (int k = 0; k < seg.G; ++k) {
        gs.spb[k] = std::min(std::max(1, 256 / seg.R[k]), std::max(1, 40960 / kSiteLds<S, NC>));
        nmax = std::max(nmax, div_up(a.g.Vh, gs.spb[k]));
        smax = std::max(smax, gs.spb[k]);
    }
    auto k = a.dagger ? k_dslash_lane_groups<S, NC, true> : k_dslash_lane_groups<S, NC, false>;
    constexpr int per_site = kSiteLds<S, NC>;
    hipLaunchKernelGGL(k, dim3(nmax, seg.G), dim3(256), size_t(smax) * per_site, stream,
                       static_cast<C *>(a.out), static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.xpay), typename Arith<S>::T(a.coef), a.g.Vh, a.parity, tab.walk, seg,
                       gs);
    return hipGetLastError();
}

template <typename S>
hipError_t launch_groups_s(const DslashArgs &a, const SegTab &seg, int by, int bz, hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_groups<S, 2>(a, seg, by, bz, stream);
        case 3: return launch_groups<S, 3>(a, seg, by, bz, stream);
        case 4: return launch_groups<S, 4>(a, seg, by, bz, stream);
        default: return hipErrorInvalidValue;
    }
}

template <typename S, int NC, int V, bool DAG, bool ORD = false>
hipError_t launch_v(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    using C = typename Arith<S>::C;
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, t.by, t.bz, tab, stream));
    const Shape sh = lane_shape<S, NC>(a.g.Vh, a.R, V);
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * sizeof(C));
    hipLaunchKernelGGL((k_dslash_lane<S, NC, V, DAG, ORD>), dim3(div_up(a.g.Vh, sh.spb)), dim3(sh.threads), sh.lds, stream,
                       static_cast<C *>(a.out), static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.xpay), typename Arith<S>::T(a.coef), a.g.Vh, a.R, sh.RV, sh.spb,
                       a.parity, tab.walk, vec_bytes);
    return hipGetLastError();
}

template <typename S, int NC, int V, bool DAG>
hipError_t launch_clover_v(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    using C = typename Arith<S>::C;
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, t.by, t.bz, tab, stream));
    const Shape sh = lane_shape<S, NC>(a.g.Vh, a.R, V, true);
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * sizeof(C));
    hipLaunchKernelGGL((k_dslash_lane_clover<S, NC, V, DAG>), dim3(div_up(a.g.Vh, sh.spb)), dim3(sh.threads), sh.lds,
                       stream, static_cast<C *>(a.out), static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.clover_in), static_cast<const C *>(a.xpay),
                       static_cast<const Cx<typename Arith<S>::T> *>(a.clover), typename Arith<S>::T(a.coef), a.g.Vh,
                       a.R, sh.RV, sh.spb, a.parity, tab.walk, vec_bytes);
    return hipGetLastError();
}

template <typename S, int NC>
hipError_t launch_split(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    using C = typename Arith<S>::C;
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, t.by, t.bz, tab, stream));
    const int spb = 64 / a.R;
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * sizeof(C));
    auto k = a.dagger ? k_dslash_lane_split<S, NC, true> : k_dslash_lane_split<S, NC, false>;
    hipLaunchKernelGGL(k, dim3(div_up(a.g.Vh, spb)), dim3(256), size_t(16) * NC * 64 * sizeof(Cx<typename Arith<S>::T>),
                       stream, static_cast<C *>(a.out), static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.xpay), typename Arith<S>::T(a.coef), a.g.Vh, a.R, spb, a.parity,
                       tab.walk, vec_bytes);
    return hipGetLastError();
}

template <typename S, int NC, int V>
hipError_t launch_dag(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    if constexpr (kWide<S>) {
        if (a.clover) return hipErrorInvalidValue;
    } else if (a.clover)
        return a.dagger ? launch_clover_v<S, NC, V, true>(a, t, stream) : launch_clover_v<S, NC, V, false>(a, t, stream);
    return a.dagger ? launch_v<S, NC, V, true>(a, t, stream) : launch_v<S, NC, V, false>(a, t, stream);
}

template <typename S, int NC>
hipError_t launch_nc(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    if (!a.clover && split_over_directions(a.g.Vh, a.R)) return launch_split<S, NC>(a, t, stream);
    if constexpr (std::is_same<S, float>::value)
        if (a.keep_order)
            return a.dagger ? launch_v<S, NC, 1, true, true>(a, t, stream)
                            : launch_v<S, NC, 1, false, true>(a, t, stream);
    if constexpr (std::is_same<S, float>::value && NC <= 3)
        if (two_per_lane<S, NC>(a)) return launch_dag<S, NC, 2>(a, t, stream);
    return launch_dag<S, NC, 1>(a, t, stream);
}

template <typename S>
hipError_t launch_s(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_nc<S, 2>(a, t, stream);
        case 3: return launch_nc<S, 3>(a, t, stream);
        case 4: return launch_nc<S, 4>(a, t, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// one buffer resource spans a vector: below 4 GiB
bool dslash_lane_supported(const Geom &g, int Nc, int R, int prec) {
    return Nc <= 4 && double(g.Vh) * 4.0 * Nc * R * 2.0 * double(prec_bytes(prec)) < 4294967296.0;
}

// Traversal tile: rows of x and a (by, bz) tile of them per t slice.  The input rows outside the tile
// (2 / by + 2 / bz + the t faces of an XCD's share, per site) are read again by the neighbouring tile,
// so the tile is as large as the XCD's 4 MB L2 lets three slices of it survive: up to 900 sites and
// 2.75 MB per slice; a whole number of tile columns per XCD where there are 8 or more (24^3 x 48,
// 16 RHS: (6, 12) 323 us FP32, 641 us FP64, (8, 8) -- 9 columns -- 364 and 661 us, (4, 4) 380 and
// 708 us, untiled 398 and 839 us).
void dslash_lane_tile(const Geom &g, int Nc, int R, int prec, int &by, int &bz) {
    const double site_bytes = 4.0 * Nc * R * 2.0 * double(prec_bytes(prec));
    const int Ly = g.L[1], Lz = g.L[2], Lt = g.L[3];
    const bool keep_y = by > 0 && Ly % by == 0, keep_z = bz > 0 && Lz % bz == 0;
    const int want_y = by, want_z = bz;
    double best = 1e30;
    by = bz = 1;
    for (int y = 1; y <= Ly; ++y) {
        if (Ly % y || (keep_y && y != want_y)) continue;
        for (int z = 1; z <= Lz; ++z) {
            if (Lz % z || (keep_z && z != want_z)) continue;
            const double sites = double(g.Lxh) * y * z;
            const int cols = (Ly / y) * (Lz / z);
            double cost = (y < Ly ? 1.0 / y : 0.0) + (z < Lz ? 1.0 / z : 0.0);
            if (cols < kNumXcd) cost += double(kNumXcd) / (double(cols) * Lt);
            else if (cols % kNumXcd) cost += 0.05;
            if (sites > 900.0 || sites * site_bytes > 2.75e6) cost += 100.0 * sites * y * z;
            if (cost < best) {
                best = cost;
                by = y;
                bz = z;
            }
        }
    }
}

bool dslash_lane_split(const Geom &g, int R) { return split_over_directions(g.Vh, R); }

bool dslash_lane_clover_fused(const DslashArgs &a, const DslashTune &t) {
    return dslash_lane_forms(a, t) && !a.keep_order && !split_over_directions(a.g.Vh, a.R);
}

hipError_t launch_dslash_lane(const DslashArgs &a, const DslashTune &t, hipStream_t stream) {
    if (!dslash_lane_supported(a.g, a.Nc, a.R, a.prec) || t.by <= 0 || t.bz <= 0 || a.g.L[1] % t.by ||
        a.g.L[2] % t.bz)
        return hipErrorInvalidValue;
    const bool wide = t.variant == kDslashLaneRhs;
    switch (a.prec) {
        case kDouble: return launch_s<double>(a, t, stream);
        case kSingle: return launch_s<float>(a, t, stream);
        case kHalf: return wide ? launch_s<WideHalf>(a, t, stream) : launch_s<__half>(a, t, stream);
        case kBF16: return wide ? launch_s<WideBf16>(a, t, stream) : launch_s<__hip_bfloat16>(a, t, stream);
        default: return hipErrorInvalidValue;
    }
}

int dslash_lane_blocks(const Geom &g, int Nc, int R, int prec) {
    return div_up(g.Vh, prec == kDouble   ? min_sites<double>(Nc, g.Vh, R)
                        : prec == kSingle ? min_sites<float>(Nc, g.Vh, R)
                                          : min_sites<__half>(Nc, g.Vh, R));
}

hipError_t launch_dslash_lane_residual(const DslashArgs &a, const DslashTune &t, const void *b, void *lo, int lo_prec,
                                       const double *scale, double *partials, int &nblk, hipStream_t stream) {
    if (a.prec != kDouble || !dslash_lane_supported(a.g, a.Nc, a.R, a.prec) || t.by <= 0 || t.bz <= 0 ||
        a.g.L[1] % t.by || a.g.L[2] % t.bz)
        return hipErrorInvalidValue;
    switch (a.Nc) {
        case 2: return launch_residual_lo<2>(a, t, b, lo, lo_prec, scale, partials, nblk, stream);
        case 3: return launch_residual_lo<3>(a, t, b, lo, lo_prec, scale, partials, nblk, stream);
        case 4: return launch_residual_lo<4>(a, t, b, lo, lo_prec, scale, partials, nblk, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_dslash_lane_groups(const DslashArgs &a, const SegTab &tab, int by, int bz, hipStream_t stream) {
    if (tab.G < 1 || tab.G > kMaxGroups || by <= 0 || bz <= 0 || a.g.L[1] % by || a.g.L[2] % bz)
        return hipErrorInvalidValue;
    for (int k = 0; k < tab.G; ++k)
        if (tab.R[k] < 1 || !dslash_supported(a.Nc, tab.R[k]) || !dslash_lane_supported(a.g, a.Nc, tab.R[k], a.prec))
            return hipErrorInvalidValue;
    switch (a.prec) {
        case kDouble: return launch_groups_s<double>(a, tab, by, bz, stream);
        case kSingle: return launch_groups_s<float>(a, tab, by, bz, stream);
        case kHalf: return launch_groups_s<WideHalf>(a, tab, by, bz, stream);
        case kBF16: return launch_groups_s<WideBf16>(a, tab, by, bz, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qcu
