// dslash_dots.hip -- hops of the lane-per-(site, RHS) kernels whose epilogue also forms the inner
// products that a BiCGStab step takes of their result: <r0, v> of v = A p for alpha, <t, s> and
// <t, t> of t = A s for omega.
//
// A separate reduction reads the stored vector and the other one again (two vectors of traffic and a
// launch); here the result is in registers, and s is the hop's own xpay vector.  The sums are of the
// stored (rounded) values, in FP64 for every storage type as in the separate reductions, over a
// workgroup's sites in order, then over workgroups by the reductions' finisher.
// Hop and reduction before -> now: alpha FP16 24^3 x 48, 16 RHS 319 -> 263 us, FP32 16^3 x 32, 12 RHS 102 ->
// 93 us; omega FP32 94 -> 74 us (16 bits had it); FP64 8^4, 4 RHS 9.6 -> 7.1 and 10.1 -> 7.9 us.
#include <algorithm>

#include "blas.h"
#include "dslash_lane.h"
#include "geom.h"

namespace qcu {
namespace {

using namespace lane;

extern __shared__ __align__(16) unsigned char dots_smem[];

template <int KIND>
constexpr int kNumDots = KIND == kDotsOmega ? 3 : 2;

// KIND's products of one stored entry o with u (alpha: of r0, omega: of s)
template <int KIND, typename C>
__device__ __forceinline__ void add_products(double (&q)[kNumDots<KIND>], const C &o, const C &u) {
    const Cx<double> t = load_cx<double>(&o), w = load_cx<double>(&u);
    if constexpr (KIND == kDotsAlpha) {  // <r0, v>
        q[0] = fma(w.re, t.re, fma(w.im, t.im, q[0]));
        q[1] = fma(w.re, t.im, fma(-w.im, t.re, q[1]));
    } else {  // <t, s>, <t, t>
        q[0] = fma(w.re, t.re, fma(w.im, t.im, q[0]));
        q[1] = fma(t.re, w.im, fma(-t.im, w.re, q[1]));
        q[2] = fma(t.re, t.re, fma(t.im, t.im, q[2]));
    }
}

// part[block][r][4]: the workgroup's sums for right-hand side r
template <int KIND>
__device__ __forceinline__ void put_row(double *part, int R, int r, const double (&q)[kNumDots<KIND>]) {
    double *row = part + (long(blockIdx.x) * R + r) * 4;
#pragma unroll
    for (int k = 0; k < kNumDots<KIND>; ++k) row[k] = q[k];
}

// out = xpay + coef D in, or with clover blocks A xpay + coef D in, from traversal position pos0 on
template <typename S, int NC, int V, int KIND, bool CLOV>
__device__ __forceinline__ void dots_body(typename Arith<S>::C *out, const typename Arith<S>::C *in,
                                          const typename Arith<S>::C *gauge, const typename Arith<S>::C *xpay,
                                          const typename Arith<S>::C *r0, const Cx<typename Arith<S>::T> *blocks,
                                          typename Arith<S>::T coef, int Vh, int R, int RV, int spb, int pos0,
                                          int parity, const int *walk, unsigned vec_bytes, double *part) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    using RW = Raw<V * int(sizeof(C))>;
    using W = Vec<C, V>;
    constexpr int NA = kNumDots<KIND>, N = 4 * NC;
    const int ns = min(spb, Vh - pos0);
    Cx<T> acc[4][NC][V];
    const Clover<S, NC> cl = clover_lds<S, NC>(blocks, dots_smem, spb);
    Place p;
    if constexpr (CLOV)
        p = hops<S, NC, V, false, false, kAhead<S, NC>>(acc, dots_smem, in, gauge, Vh, R, RV, spb, pos0, parity, walk,
                                                        vec_bytes, cl);
    else
        p = hops<S, NC, V, false, false, kAhead<S, NC>>(acc, dots_smem, in, gauge, Vh, R, RV, spb, pos0, parity, walk,
                                                        vec_bytes);
    double q[V][NA];
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
        for (int k = 0; k < NA; ++k) q[i][k] = 0.0;
    if (p.active) {
        const unsigned rb = unsigned(R) * unsigned(sizeof(C));
        const auto r_out = rsrc(out, vec_bytes), r_x = rsrc(xpay, vec_bytes), r_r = rsrc(r0, vec_bytes);
        // all loads before the first store
        W x[N], u[KIND == kDotsAlpha ? N : 1];
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] = __builtin_bit_cast(W, RW::load(r_x, p.vo, unsigned(k) * rb));
        if constexpr (KIND == kDotsAlpha) {
#pragma unroll
            for (int k = 0; k < N; ++k) u[k] = __builtin_bit_cast(W, RW::load(r_r, p.vo, unsigned(k) * rb));
        }
        const auto finish = [&](int row, const Cx<T>(&v)[V]) {
            W o;
#pragma unroll
            for (int i = 0; i < V; ++i) {
                store_cx(&o.c[i], v[i]);
                add_products<KIND>(q[i], o.c[i], KIND == kDotsAlpha ? u[KIND == kDotsAlpha ? row : 0].c[i] : x[row].c[i]);
            }
            RW::store(r_out, __builtin_bit_cast(typename RW::type, o), p.vo, unsigned(row) * rb);
        };
        if constexpr (CLOV) {
            cl.template rows_of<V>(
                acc, true, false, coef, min(p.local, ns - 1), [&](int k) { return x[k]; },
                [&](int row, const Cx<T>(&v)[V], const Cx<T>(&)[V]) { finish(row, v); });
        } else {
#pragma unroll
            for (int row = 0; row < N; ++row) {
                Cx<T> v[V];
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const Cx<T> h = acc[row / NC][row % NC][i], xv = load_cx<T>(&x[row].c[i]);
                    v[i] = {fma(coef, h.re, xv.re), fma(coef, h.im, xv.im)};
                }
                finish(row, v);
            }
        }
    }
    double w[NA][V];
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
        for (int k = 0; k < NA; ++k) w[k][i] = q[i][k];
    sum_sites<NA, V>(w, reinterpret_cast<double *>(dots_smem), p, RV, ns);
    if (int(threadIdx.x) < RV) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
            double row[NA];
#pragma unroll
            for (int k = 0; k < NA; ++k) row[k] = w[k][i];
            put_row<KIND>(part, R, int(threadIdx.x) * V + i, row);
        }
    }
}

template <typename S, int NC, int V, int KIND, bool CLOV>
__global__ __launch_bounds__(256, (kMinWaves<S, NC, V>)) void k_dslash_dots(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *__restrict__ xpay,
    const typename Arith<S>::C *__restrict__ r0, const Cx<typename Arith<S>::T> *__restrict__ blocks,
    typename Arith<S>::T coef, int Vh, int R, int RV, int spb, int parity, const int *__restrict__ walk,
    unsigned vec_bytes, double *__restrict__ part) {
    dots_body<S, NC, V, KIND, CLOV>(out, in, gauge, xpay, r0, blocks, coef, Vh, R, RV, spb,
                                    xcd_remap(blockIdx.x, gridDim.x) * spb, parity, walk, vec_bytes, part);
}

// Every running group of a batch in one launch (blockIdx.y = group, SegTab layout)
template <typename S, int NC, int KIND>
__global__ __launch_bounds__(256, (kMinWaves<S, NC, 1>)) void k_dslash_dots_groups(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *__restrict__ xpay,
    const typename Arith<S>::C *__restrict__ r0, typename Arith<S>::T coef, int Vh, int parity,
    const int *__restrict__ walk, SegTab tab, SegRows rows, double *__restrict__ part) {
    const int grp = blockIdx.y;
    if (tab.done && tab.done[grp]) return;
    const int nblk = rows.n[grp], R = tab.R[grp], spb = rows.sites[grp];
    if (int(blockIdx.x) >= nblk) return;
    const long off = tab.n * tab.base[grp];
    const unsigned vec_bytes = unsigned(tab.n * R * long(sizeof(typename Arith<S>::C)));
    dots_body<S, NC, 1, KIND, false>(out + off, in + off, gauge, xpay + off, r0 ? r0 + off : nullptr, nullptr, coef, Vh,
                                     R, R, spb, xcd_remap(blockIdx.x, nblk) * spb, parity, walk, vec_bytes,
                                     part + rows.off[grp]);
}

// Small lattices: a wavefront per direction, wavefront mu finishing spin mu (direction(), dslash_lane.h)
template <typename S, int NC, int KIND>
__global__ __launch_bounds__(256) void k_dslash_dots_split(
    typename Arith<S>::C *__restrict__ out, const typename Arith<S>::C *__restrict__ in,
    const typename Arith<S>::C *__restrict__ gauge, const typename Arith<S>::C *__restrict__ xpay,
    const typename Arith<S>::C *__restrict__ r0, typename Arith<S>::T coef, int Vh, int R, int spb, int parity,
    const int *__restrict__ walk, unsigned vec_bytes, double *__restrict__ part) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    using RW = Raw<int(sizeof(C))>;
    constexpr int NA = kNumDots<KIND>;
    auto *sums = reinterpret_cast<Cx<T> *>(dots_smem);
    const int lane = threadIdx.x & 63;
    const int mu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * spb;
    const int ns = min(spb, Vh - pos0);
    const int local = lane / R, r = lane - local * R;
    const int *row = walk + (long(parity) * Vh + pos0 + min(local, ns - 1)) * 9;
    const unsigned rb = unsigned(R) * unsigned(sizeof(C)), lo = unsigned(r) * unsigned(sizeof(C));
    Cx<T> acc[4][NC][1];
    direction_of<S, NC, false>(mu, acc, MrhsRows<C, NC, 1>{rsrc(in, vec_bytes), rb, lo}, gauge, Vh, parity, row);
    put_parts<T, NC>(sums, mu, lane, acc);
    const unsigned vo = unsigned(row[0]) * 4u * NC * rb + unsigned(mu) * NC * rb + lo;
    const auto r_out = rsrc(out, vec_bytes), r_x = rsrc(xpay, vec_bytes), r_r = rsrc(r0, vec_bytes);
    C x[NC], u[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        x[c] = __builtin_bit_cast(C, RW::load(r_x, vo, unsigned(c) * rb));
        if constexpr (KIND == kDotsAlpha) u[c] = __builtin_bit_cast(C, RW::load(r_r, vo, unsigned(c) * rb));
    }
    __syncthreads();
    double q[NA];
#pragma unroll
    for (int k = 0; k < NA; ++k) q[k] = 0.0;
    Place p;
    p.active = local < ns;
    if (p.active) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const Cx<T> h = sum_parts<T, NC>(sums, mu, lane, c), xv = load_cx<T>(&x[c]);
            C o;
            store_cx(&o, Cx<T>{fma(coef, h.re, xv.re), fma(coef, h.im, xv.im)});
            RW::store(r_out, __builtin_bit_cast(typename RW::type, o), vo, unsigned(c) * rb);
            if constexpr (KIND == kDotsAlpha) add_products<KIND>(q, o, u[c]);
            else add_products<KIND>(q, o, x[c]);
        }
    }
    // sums over the sites of each spin, then over the spins
    auto *red = reinterpret_cast<double *>(dots_smem);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NA; ++k) red[k * 256 + threadIdx.x] = p.active ? q[k] : 0.0;
    __syncthreads();
    if (int(threadIdx.x) < R) {
        double t[NA];
#pragma unroll
        for (int k = 0; k < NA; ++k) {
            t[k] = 0.0;
            for (int m = 0; m < 4; ++m)
                for (int l = 0; l < ns; ++l) t[k] += red[k * 256 + m * 64 + l * R + threadIdx.x];
        }
        put_row<KIND>(part, R, threadIdx.x, t);
    }
}

template <typename S, int NC, int V, int KIND>
hipError_t launch_v(const DslashArgs &a, const void *r0, const GeomTables &tab, double *part, int &nblk,
                    hipStream_t stream) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    const Shape sh = lane_shape<S, NC>(a.g.Vh, a.R, V, a.clover != nullptr);
    nblk = div_up(a.g.Vh, sh.spb);
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * sizeof(C));
    auto k = a.clover ? k_dslash_dots<S, NC, V, KIND, true> : k_dslash_dots<S, NC, V, KIND, false>;
    hipLaunchKernelGGL(k, dim3(nblk), dim3(sh.threads), sh.lds, stream, static_cast<C *>(a.out),
                       static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.clover ? a.clover_in : a.xpay), static_cast<const C *>(r0),
                       static_cast<const Cx<T> *>(a.clover), T(a.coef), a.g.Vh, a.R, sh.RV, sh.spb, a.parity, tab.walk,
                       vec_bytes, part);
    return hipGetLastError();
}

template <typename S, int NC, int KIND>
hipError_t launch_split(const DslashArgs &a, const void *r0, const GeomTables &tab, double *part, int &nblk,
                        hipStream_t stream) {
    using T = typename Arith<S>::T;
    using C = typename Arith<S>::C;
    const int spb = 64 / a.R;
    nblk = div_up(a.g.Vh, spb);
    const unsigned vec_bytes = unsigned(size_t(a.g.Vh) * 4 * NC * a.R * sizeof(C));
    const size_t lds = std::max(size_t(16) * NC * 64 * sizeof(Cx<T>), size_t(3) * 256 * sizeof(double));
    hipLaunchKernelGGL((k_dslash_dots_split<S, NC, KIND>), dim3(nblk), dim3(256), lds, stream, static_cast<C *>(a.out),
                       static_cast<const C *>(a.in), static_cast<const C *>(a.gauge), static_cast<const C *>(a.xpay),
                       static_cast<const C *>(r0), T(a.coef), a.g.Vh, a.R, spb, a.parity, tab.walk, vec_bytes, part);
    return hipGetLastError();
}

template <typename S, int NC, int KIND>
hipError_t launch_kind(const DslashArgs &a, const void *r0, const GeomTables &tab, double *part, int &nblk,
                       hipStream_t stream) {
    if (!a.clover && split_over_directions(a.g.Vh, a.R)) return launch_split<S, NC, KIND>(a, r0, tab, part, nblk, stream);
    if constexpr (std::is_same<S, float>::value && NC <= 3)
        if (two_per_lane<S, NC>(a)) return launch_v<S, NC, 2, KIND>(a, r0, tab, part, nblk, stream);
    return launch_v<S, NC, 1, KIND>(a, r0, tab, part, nblk, stream);
}

template <typename S, int NC>
hipError_t launch_nc(const DslashArgs &a, DotsKind kind, const void *r0, const GeomTables &tab, double *part, int &nblk,
                     hipStream_t stream) {
    return kind == kDotsAlpha ? launch_kind<S, NC, kDotsAlpha>(a, r0, tab, part, nblk, stream)
                              : launch_kind<S, NC, kDotsOmega>(a, r0, tab, part, nblk, stream);
}

template <typename S>
hipError_t launch_s(const DslashArgs &a, DotsKind kind, const void *r0, const GeomTables &tab, double *part, int &nblk,
                    hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_nc<S, 2>(a, kind, r0, tab, part, nblk, stream);
        case 3: return launch_nc<S, 3>(a, kind, r0, tab, part, nblk, stream);
        case 4: return launch_nc<S, 4>(a, kind, r0, tab, part, nblk, stream);
        default: return hipErrorInvalidValue;
    }
}

template <typename S, int NC>
hipError_t launch_groups(const DslashArgs &a, DotsKind kind, const void *r0, const SegTab &seg, const SegRows &rows,
                         const GeomTables &tab, double *part, hipStream_t stream) {
    using C = typename Arith<S>::C;
    constexpr int per_site = kSiteLds<S, NC>;
    int nmax = 1, smax = 1;
    for (int k = 0; k < seg.G; ++k) {
        nmax = std::max(nmax, rows.n[k]);
        smax = std::max(smax, rows.sites[k]);
    }
    auto k = kind == kDotsAlpha ? k_dslash_dots_groups<S, NC, kDotsAlpha> : k_dslash_dots_groups<S, NC, kDotsOmega>;
    hipLaunchKernelGGL(k, dim3(nmax, seg.G), dim3(256), std::max(size_t(smax) * per_site, size_t(256) * 3 * 8), stream,
                       static_cast<C *>(a.out), static_cast<const C *>(a.in), static_cast<const C *>(a.gauge),
                       static_cast<const C *>(a.xpay), static_cast<const C *>(r0), typename Arith<S>::T(a.coef), a.g.Vh,
                       a.parity, tab.walk, seg, rows, part);
    return hipGetLastError();
}

template <typename S>
hipError_t launch_groups_s(const DslashArgs &a, DotsKind kind, const void *r0, const SegTab &seg, const SegRows &rows,
                           const GeomTables &tab, double *part, hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_groups<S, 2>(a, kind, r0, seg, rows, tab, part, stream);
        case 3: return launch_groups<S, 3>(a, kind, r0, seg, rows, tab, part, stream);
        case 4: return launch_groups<S, 4>(a, kind, r0, seg, rows, tab, part, stream);
        default: return hipErrorInvalidValue;
    }
}

int site_lds(int Nc, int prec) {
    const auto of = [&](auto nc) {
        constexpr int NC = decltype(nc)::value;
        return prec == kDouble ? kSiteLds<double, NC> : prec == kSingle ? kSiteLds<float, NC> : kSiteLds<__half, NC>;
    };
    return Nc == 2   ? of(std::integral_constant<int, 2>{})
           : Nc == 3 ? of(std::integral_constant<int, 3>{})
                     : of(std::integral_constant<int, 4>{});
}

}  // namespace

bool dslash_dots_rows(const Geom &g, int Nc, int prec, const SegTab &tab, SegRows &rows) {
    if (tab.G < 1 || tab.G > kMaxGroups || Nc > 4) return false;
    rows = SegRows{};
    for (int k = 0; k < tab.G; ++k) {
        if (tab.R[k] < 1 || tab.R[k] > 256 || !dslash_lane_supported(g, Nc, tab.R[k], prec)) return false;
        rows.sites[k] = std::min(std::max(1, 256 / tab.R[k]), std::max(1, 40960 / site_lds(Nc, prec)));
        rows.n[k] = div_up(g.Vh, rows.sites[k]);
        if (rows.n[k] > kMaxFinishRows) return false;
        rows.off[k] = rows.total;
        rows.total += long(rows.n[k]) * tab.R[k] * 4;
    }
    return true;
}

hipError_t launch_dslash_lane_dots_groups(const DslashArgs &a, DotsKind kind, const void *r0, const SegTab &tab,
                                          const SegRows &rows, double *partials, int by, int bz, hipStream_t stream) {
    SegRows check;
    if (!dslash_dots_rows(a.g, a.Nc, a.prec, tab, check) || check.total != rows.total || !partials || a.dagger ||
        !a.xpay || by <= 0 || bz <= 0 || a.g.L[1] % by || a.g.L[2] % bz)
        return hipErrorInvalidValue;
    GeomTables g;
    QCU_HIP_TRY(geom_tables(a.g, by, bz, g, stream));
    switch (a.prec) {
        case kDouble: return launch_groups_s<double>(a, kind, r0, tab, rows, g, partials, stream);
        case kSingle: return launch_groups_s<float>(a, kind, r0, tab, rows, g, partials, stream);
        case kHalf: return launch_groups_s<WideHalf>(a, kind, r0, tab, rows, g, partials, stream);
        case kBF16: return launch_groups_s<WideBf16>(a, kind, r0, tab, rows, g, partials, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_dslash_lane_dots(const DslashArgs &a, const DslashTune &t, DotsKind kind, const void *r0,
                                   double *partials, hipStream_t stream, int &nblk) {
    if (!dslash_lane_supported(a.g, a.Nc, a.R, a.prec) || t.by <= 0 || t.bz <= 0 || a.g.L[1] % t.by || a.g.L[2] % t.bz)
        return hipErrorInvalidValue;
    GeomTables tab;
    QCU_HIP_TRY(geom_tables(a.g, t.by, t.bz, tab, stream));
    switch (a.prec) {
        case kDouble: return launch_s<double>(a, kind, r0, tab, partials, nblk, stream);
        case kSingle: return launch_s<float>(a, kind, r0, tab, partials, nblk, stream);
        case kHalf: return launch_s<__half>(a, kind, r0, tab, partials, nblk, stream);
        case kBF16: return launch_s<__hip_bfloat16>(a, kind, r0, tab, partials, nblk, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qcu
