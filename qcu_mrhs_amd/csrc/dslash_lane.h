// dslash_lane.h -- device body of the lane-per-(site, RHS) hopping kernels
// (dslash_lane.hip has the launches and the measurements).
//
// A workgroup takes `spb` consecutive traversal positions; lane l of it holds
// one output site and V consecutive right-hand sides, and runs all eight hops
// of them, so nothing is reduced across lanes and no lane idles whatever R is.
// The walk-table rows and the 8 links of every site go through LDS (each is
// read once by the workgroup and then broadcast to the lanes of its site); the
// neighbour spinors are buffer loads whose (spin, colour) row offset is scalar.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dslash_common.h"

namespace qcu {
namespace lane {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}

// The output of a hop is read by a later kernel only, after the caches have turned over: stored with
// the non-temporal policy it leaves the XCD's L2 to the input spinors (24^3 x 48, 16 RHS: FP64
// 730 -> 699 us, FP32 380 -> 363 us; 16^3 x 32, 12 RHS, FP64: 124 -> 97 us).
constexpr int kStorePolicy = 2;  // gfx950 cache-policy bit nt

// one load / store of B bytes at voffset + soffset
template <int B> struct Raw;
template <> struct Raw<4> {
    using type = uint32_t;
    __device__ __forceinline__ static type load(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        return uint32_t(__builtin_amdgcn_raw_buffer_load_b32(r, int(v), int(s), 0));
    }
    __device__ __forceinline__ static void store(__amdgpu_buffer_rsrc_t r, type w, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b32(int(w), r, int(v), int(s), kStorePolicy);
    }
};
template <> struct Raw<8> {
    using type = u32x2;
    __device__ __forceinline__ static type load(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, int(v), int(s), 0));
    }
    __device__ __forceinline__ static void store(__amdgpu_buffer_rsrc_t r, type w, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b64(w, r, int(v), int(s), kStorePolicy);
    }
};
template <> struct Raw<16> {
    using type = u32x4;
    __device__ __forceinline__ static type load(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, int(v), int(s), 0));
    }
    // The row offset goes into the vector register: after a store of more than 8 bytes the compiler keeps two
    // wait states before its data registers are written again, but not if the store has a scalar offset, and
    // there rows have been stored with the next row's values in part (FP32, two per lane, 12 RHS at 24^4)
    __device__ __forceinline__ static void store(__amdgpu_buffer_rsrc_t r, type w, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b128(w, r, int(v + s), 0, kStorePolicy);
    }
};

// Arithmetic of one storage type: C = stored complex, T = accumulation, Link = what LDS holds of a
// link entry, H = one projected spinor entry.
//   proj<K>(a, b) = a + i^K b;  madd(s, u, h): s += u h
// FP32 / FP64 storage: everything in the storage type.
template <typename S>
struct Arith {
    using T = S;
    using C = Cx<S>;
    using Link = Cx<S>;
    using H = Cx<S>;
    __device__ __forceinline__ static Link link(C u, bool fwd) { return fwd ? u : conj(u); }
    template <int K>
    __device__ __forceinline__ static H proj(C a, C b) { return a + ipow<K>(b); }
    __device__ __forceinline__ static void madd(Cx<T> &s, const Link &u, H h) { cfma(s, u, h); }
};
// FP16 / BF16 storage: the projected entry is rounded to the storage type (as the matrix-core kernel
// does) and a complex product is two 2-element dot products with FP32 accumulation (v_dot2_f32_{f16,
// bf16}: half the instructions of FP32 FMAs), the link kept in LDS as the two words (Re, -Im) and
// (Im, Re) they multiply.
template <>
struct Arith<__half> {
    using T = float;
    using C = Half2Store;
    using Link = u32x2;
    using H = uint32_t;
    __device__ __forceinline__ static Link link(C u, bool fwd) {
        const uint32_t w = __builtin_bit_cast(uint32_t, u);
        const uint32_t sw = __builtin_amdgcn_perm(w, w, 0x01000302u);
        return fwd ? Link{w ^ 0x80000000u, sw} : Link{w, sw ^ 0x00008000u};
    }
    template <int K>
    __device__ __forceinline__ static H proj(C a, C b) {
        const f16x2 x = __builtin_bit_cast(f16x2, a), y = __builtin_bit_cast(f16x2, b);
        f16x2 r;
        if constexpr ((K & 3) == 0) r = x + y;
        else if constexpr ((K & 3) == 1) r = x + f16x2{-y[1], y[0]};
        else if constexpr ((K & 3) == 2) r = x - y;
        else r = x + f16x2{y[1], -y[0]};
        return __builtin_bit_cast(uint32_t, r);
    }
    __device__ __forceinline__ static void madd(Cx<T> &s, const Link &u, H h) {
        const f16x2 hh = __builtin_bit_cast(f16x2, h);
        s.re = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, uint32_t(u[0])), hh, s.re, false);
        s.im = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, uint32_t(u[1])), hh, s.im, false);
    }
};
template <>
struct Arith<__hip_bfloat16> {
    using T = float;
    using C = Bf162Store;
    using Link = u32x2;
    using H = uint32_t;
    __device__ __forceinline__ static Link link(C u, bool fwd) {
        const uint32_t w = __builtin_bit_cast(uint32_t, u);
        const uint32_t sw = __builtin_amdgcn_perm(w, w, 0x01000302u);
        return fwd ? Link{w ^ 0x80000000u, sw} : Link{w, sw ^ 0x00008000u};
    }
    template <int K>
    __device__ __forceinline__ static H proj(C a, C b) {
        const Cx<float> h = load_cx<float>(&a) + ipow<K>(load_cx<float>(&b));
        C o;
        store_cx(&o, h);
        return __builtin_bit_cast(uint32_t, o);
    }
    __device__ __forceinline__ static void madd(Cx<T> &s, const Link &u, H h) {
        const bf16x2 hh = __builtin_bit_cast(bf16x2, h);
        s.re = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, uint32_t(u[0])), hh, s.re, false);
        s.im = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, uint32_t(u[1])), hh, s.im, false);
    }
};

// FP16 / BF16 storage with everything from the loads on in FP32 (kDslashLaneRhs and the batches, whose other
// kernel does so too), at twice the instructions of a product: 31.7 -> 36.9 us at 16^3 x 32, SU(3), 16 RHS in
// FP16, BF16 even.
struct WideHalf {};
struct WideBf16 {};
template <typename CS>
struct ArithWide {
    using T = float;
    using C = CS;
    using Link = Cx<float>;
    using H = Cx<float>;
    __device__ __forceinline__ static Link link(C u, bool fwd) {
        const Cx<float> v = load_cx<float>(&u);
        return fwd ? v : conj(v);
    }
    template <int K>
    __device__ __forceinline__ static H proj(C a, C b) {
        return load_cx<float>(&a) + ipow<K>(load_cx<float>(&b));
    }
    __device__ __forceinline__ static void madd(Cx<T> &s, const Link &u, H h) { cfma(s, u, h); }
};
template <>
struct Arith<WideHalf> : ArithWide<Half2Store> {};
template <>
struct Arith<WideBf16> : ArithWide<Bf162Store> {};
template <typename S>
constexpr bool kWide = std::is_same<S, WideHalf>::value || std::is_same<S, WideBf16>::value;

// LDS words of one site's 8 links: one entry more than they need, so that the sites of a wavefront
// reading the same entry start in different banks
template <typename S, int NC>
constexpr int kLinkRow = 8 * NC * NC + 1;
template <typename S, int NC>
constexpr int kSiteLds = kLinkRow<S, NC> * int(sizeof(typename Arith<S>::Link)) + 9 * int(sizeof(int));

// V stored complex numbers as one register vector
template <typename C, int V>
struct Vec {
    C c[V];
};

// Keeps the accumulators live here: every hop's arithmetic is done before the next hop's loads are
// waited for.  Without it the compiler interleaves the hops until it spills (FP64, Nc = 3: 256
// registers and 106 spilled, 1741 us at 24^3 x 48, 16 RHS, instead of 130 registers and 787 us).
template <typename T, int NC, int V>
__device__ __forceinline__ void pin(Cx<T> (&acc)[4][NC][V]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < V; ++v) asm volatile("" : "+v"(acc[s][c][v].re), "+v"(acc[s][c][v].im));
}

// the 4 NC entries of one neighbour spinor
template <typename C, int NC, int V>
__device__ __forceinline__ void load_spinor(Vec<C, V> (&w)[4][NC], __amdgpu_buffer_rsrc_t r_in, unsigned vo,
                                            unsigned row_bytes) {
    using R = Raw<V * int(sizeof(C))>;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c)
            w[s][c] = __builtin_bit_cast(Vec<C, V>, R::load(r_in, vo, unsigned(s * NC + c) * row_bytes));
}

// acc += (1 -+ gamma) V w for one hop
template <typename S, int NC, int V, bool DAG, int MU, bool FWD>
__device__ __forceinline__ void hop_arith(Cx<typename Arith<S>::T> (&acc)[4][NC][V],
                                          const Vec<typename Arith<S>::C, V> (&w)[4][NC],
                                          const typename Arith<S>::Link *U) {
    using A = Arith<S>;
    using T = typename A::T;
    constexpr int sgn = (FWD != DAG) ? 2 : 0;
    constexpr int m0 = kMat2(MU, 0), m1 = kMat2(MU, 1);
    constexpr int kp0 = kProjK(MU, 0) + sgn, kp1 = kProjK(MU, 1) + sgn;
    constexpr int kr0 = kReconK(MU, 0) + sgn, kr1 = kReconK(MU, 1) + sgn;
    typename A::H h0[NC][V], h1[NC][V];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            h0[c][v] = A::template proj<kp0>(w[0][c].c[v], w[m0][c].c[v]);
            h1[c][v] = A::template proj<kp1>(w[1][c].c[v], w[m1][c].c[v]);
        }
#pragma unroll
    for (int a = 0; a < NC; ++a) {
        Cx<T> s0[V], s1[V];
#pragma unroll
        for (int v = 0; v < V; ++v) s0[v] = s1[v] = {T(0), T(0)};
#pragma unroll
        for (int b = 0; b < NC; ++b) {
            const typename A::Link u = U[a * NC + b];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                A::madd(s0[v], u, h0[b][v]);
                A::madd(s1[v], u, h1[b][v]);
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            acc[0][a][v] = acc[0][a][v] + s0[v];
            acc[m0][a][v] = acc[m0][a][v] + ipow<kr0>(s0[v]);
            acc[1][a][v] = acc[1][a][v] + s1[v];
            acc[m1][a][v] = acc[m1][a][v] + ipow<kr1>(s1[v]);
        }
    }
}

// Where the spinors come from: an RHS-innermost half vector (C [site][spin][colour][rhs]).  The loads of a
// fetch stay behind the arithmetic before them (see pin).
template <typename C, int NC, int V>
struct MrhsRows {
    static constexpr bool kSiteFast = false;  // consecutive lanes: consecutive right-hand sides
    __amdgpu_buffer_rsrc_t r;
    unsigned row_bytes, lo;  // lo: byte offset of the lane's right-hand sides in a row
    __device__ __forceinline__ void fetch(Vec<C, V> (&w)[4][NC], int site) const {
        unsigned vo = unsigned(site) * (4u * NC * row_bytes) + lo;
        asm volatile("" : "+v"(vo));
        load_spinor<C, NC, V>(w, r, vo, row_bytes);
    }
};

template <typename S, int NC, int V, bool DAG, int MU, bool FWD>
__device__ __forceinline__ void hop(Cx<typename Arith<S>::T> (&acc)[4][NC][V],
                                    const Vec<typename Arith<S>::C, V> (&w)[4][NC],
                                    const typename Arith<S>::Link *U) {
    hop_arith<S, NC, V, DAG, MU, FWD>(acc, w, U);
    pin<typename Arith<S>::T, NC, V>(acc);
    __builtin_amdgcn_sched_barrier(0);
}

// What a workgroup loads into LDS besides its links, in the same wait: nothing, or (Clover, below) the
// clover blocks of its sites.
struct NoExtra {
    __device__ __forceinline__ void load(const int *, int) const {}
};

// What a lane knows after the hops.
struct Place {
    bool active;    // holds a site of the workgroup (idle lanes repeat the last one)
    int site;       // output site
    int rv;         // RHS vector: right-hand sides rv V .. rv V + V - 1
    int local;      // site within the workgroup
    unsigned vo;    // byte offset of (site, spin 0, colour 0, rv V)
};

// acc = D (spinors of src) for the workgroup's sites, from traversal position pos0 on.  smem: kSiteLds bytes
// per site.
// ORD: the hops of each direction are summed apart and then as ((x + z) + (y + t)), the wave-per-site
// kernel's order (four sets of accumulators), instead of one after the other.
// AHEAD: the next hop's spinor is loaded before the arithmetic of this one.
template <typename S, int NC, int V, bool DAG, bool ORD, bool AHEAD, typename SRC, typename X>
__device__ __forceinline__ Place hops_from(Cx<typename Arith<S>::T> (&acc)[4][NC][V], unsigned char *smem,
                                           const SRC &src, const typename Arith<S>::C *gauge, int Vh, int RV, int spb,
                                           int pos0, int parity, const int *walk, const X &extra) {
    using A = Arith<S>;
    using T = typename A::T;
    using C = typename A::C;
    constexpr int NN = NC * NC, LR = kLinkRow<S, NC>;
    auto *sl = reinterpret_cast<typename A::Link *>(smem);
    int *sw = reinterpret_cast<int *>(sl + spb * LR);
    const int ns = min(spb, Vh - pos0);
    const int *wt = walk + (long(parity) * Vh + pos0) * 9;
    const int nt = blockDim.x;
    for (int i = threadIdx.x; i < ns * 9; i += nt) sw[i] = wt[i];
    __syncthreads();
    for (int i = threadIdx.x; i < ns * 8 * NN; i += nt) {
        const int l = i / (8 * NN), k = i / NN - l * 8, e = i - (l * 8 + k) * NN;
        const bool fwd = (k & 1) == 0;
        // V = U_mu(x) forward (parity of x), U_mu(x - mu)^+ backward
        const int a = e / NC, b = e - a * NC;
        const long li = fwd ? ((k >> 1) * 2 + parity) * long(Vh) + sw[l * 9]
                            : ((k >> 1) * 2 + 1 - parity) * long(Vh) + sw[l * 9 + 1 + k];
        sl[l * LR + k * NN + e] = A::link(gauge[li * NN + (fwd ? e : b * NC + a)], fwd);
    }
    extra.load(sw, ns);
    __syncthreads();
    Place p;
    if constexpr (SRC::kSiteFast) {
        p.rv = int(threadIdx.x) / spb;
        p.local = int(threadIdx.x) - p.rv * spb;
        p.active = p.local < ns && p.rv < RV;
    } else {
        p.local = int(threadIdx.x) / RV;
        p.rv = int(threadIdx.x) - p.local * RV;
        p.active = p.local < ns;
    }
    const int l = min(p.local, ns - 1);
    const int *row = sw + l * 9;
    const typename A::Link *U = sl + l * LR;
    constexpr int NA = ORD ? 4 : 1;
    Cx<T> sums[NA][4][NC][V];
#pragma unroll
    for (int m = 0; m < NA; ++m)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int v = 0; v < V; ++v) sums[m][s][c][v] = {T(0), T(0)};
    // Hop order t-, z-, y-, x-, x+, y+, z+, t+: the traversal sweeps upwards, so the backward neighbours
    // are the input sites about to leave the XCD's L2 and are read before the forward ones push them out
    // (24^3 x 48, 16 RHS: FP64 711 -> 636 us, FP32 350 -> 323 us against x+, x-, ..., t+, t-; 786 and
    // 393 us in the reverse order; 16^3 x 32, 12 RHS, FP64: 103 -> 79 us).
#define QCU_FETCH(W, MU, FWD) src.fetch(W, row[2 + 2 * MU - FWD]);
#define QCU_HOP(W, MU, FWD) hop<S, NC, V, DAG, MU, FWD>(sums[ORD ? MU : 0], W, U + (2 * MU + 1 - FWD) * NN);
#define QCU_STEP(MU, FWD) { Vec<C, V> w[4][NC]; QCU_FETCH(w, MU, FWD) QCU_HOP(w, MU, FWD) }
    if constexpr (AHEAD) {
        Vec<C, V> w0[4][NC], w1[4][NC];
        QCU_FETCH(w0, 3, false)
        QCU_FETCH(w1, 2, false) QCU_HOP(w0, 3, false)
        QCU_FETCH(w0, 1, false) QCU_HOP(w1, 2, false)
        QCU_FETCH(w1, 0, false) QCU_HOP(w0, 1, false)
        QCU_FETCH(w0, 0, true) QCU_HOP(w1, 0, false)
        QCU_FETCH(w1, 1, true) QCU_HOP(w0, 0, true)
        QCU_FETCH(w0, 2, true) QCU_HOP(w1, 1, true)
        QCU_FETCH(w1, 3, true) QCU_HOP(w0, 2, true)
        QCU_HOP(w1, 3, true)
    } else {
        QCU_STEP(3, false)
        QCU_STEP(2, false)
        QCU_STEP(1, false)
        QCU_STEP(0, false)
        QCU_STEP(0, true)
        QCU_STEP(1, true)
        QCU_STEP(2, true)
        QCU_STEP(3, true)
    }
#undef QCU_STEP
#undef QCU_HOP
#undef QCU_FETCH
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if constexpr (ORD)
                    acc[s][c][v] = (sums[0][s][c][v] + sums[2][s][c][v]) + (sums[1][s][c][v] + sums[3][s][c][v]);
                else
                    acc[s][c][v] = sums[0][s][c][v];
            }
    p.site = row[0];
    return p;
}

// acc = D in, `in` an RHS-innermost half vector of vec_bytes
template <typename S, int NC, int V, bool DAG, bool ORD = false, bool AHEAD = false, typename X = NoExtra>
__device__ __forceinline__ Place hops(Cx<typename Arith<S>::T> (&acc)[4][NC][V], unsigned char *smem,
                                      const typename Arith<S>::C *in, const typename Arith<S>::C *gauge, int Vh,
                                      int R, int RV, int spb, int pos0, int parity, const int *walk,
                                      unsigned vec_bytes, const X &extra = X{}) {
    using C = typename Arith<S>::C;
    const unsigned rb = unsigned(R) * unsigned(sizeof(C));
    const MrhsRows<C, NC, V> src{rsrc(in, vec_bytes), rb, unsigned(int(threadIdx.x) % RV) * V * unsigned(sizeof(C))};
    Place p = hops_from<S, NC, V, DAG, ORD, AHEAD>(acc, smem, src, gauge, Vh, RV, spb, pos0, parity, walk, extra);
    p.vo = unsigned(p.site) * (4u * NC * rb) + src.lo;
    return p;
}

// Small lattices: the two hops of each direction in a wavefront of their own, the four wavefronts' sums
// combined through LDS (wavefront mu finishes spin mu).  A lane then waits for two dependent loads (its
// walk row, then links and both spinors together) instead of ten, and a lattice that would leave most
// SIMDs without a wavefront has four times as many.
template <typename S, int NC, bool DAG, int MU, typename SRC>
__device__ __forceinline__ void direction(Cx<typename Arith<S>::T> (&acc)[4][NC][1], const SRC &src,
                                          const typename Arith<S>::C *gauge, int Vh, int parity, const int *row) {
    using A = Arith<S>;
    using C = typename A::C;
    constexpr int NN = NC * NC;
    const int site = row[0], nf = row[1 + 2 * MU], nb = row[2 + 2 * MU];
    Vec<C, 1> wf[4][NC], wb[4][NC];
    src.fetch(wb, nb);
    src.fetch(wf, nf);
    const C *gf = gauge + ((MU * 2 + parity) * long(Vh) + site) * NN, *gb = gauge + ((MU * 2 + 1 - parity) * long(Vh) + nb) * NN;
    typename A::Link uf[NN], ub[NN];
#pragma unroll
    for (int a = 0; a < NC; ++a)
#pragma unroll
        for (int b = 0; b < NC; ++b) {
            ub[a * NC + b] = A::link(gb[b * NC + a], false);
            uf[a * NC + b] = A::link(gf[a * NC + b], true);
        }
    hop_arith<S, NC, 1, DAG, MU, false>(acc, wb, ub);
    hop_arith<S, NC, 1, DAG, MU, true>(acc, wf, uf);
}

template <typename S, int NC, bool DAG, typename SRC>
__device__ __forceinline__ void direction_of(int mu, Cx<typename Arith<S>::T> (&acc)[4][NC][1], const SRC &src,
                                             const typename Arith<S>::C *gauge, int Vh, int parity, const int *row) {
    using T = typename Arith<S>::T;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[s][c][0] = {T(0), T(0)};
    if (mu == 0) direction<S, NC, DAG, 0>(acc, src, gauge, Vh, parity, row);
    else if (mu == 1) direction<S, NC, DAG, 1>(acc, src, gauge, Vh, parity, row);
    else if (mu == 2) direction<S, NC, DAG, 2>(acc, src, gauge, Vh, parity, row);
    else direction<S, NC, DAG, 3>(acc, src, gauge, Vh, parity, row);
}

// part: [spin][wavefront][colour][lane] complex, the sums of wavefront mu's two hops; combined for spin mu
template <typename T, int NC>
__device__ __forceinline__ void put_parts(Cx<T> *part, int mu, int lane, const Cx<T> (&acc)[4][NC][1]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c) part[((s * 4 + mu) * NC + c) * 64 + lane] = acc[s][c][0];
}
template <typename T, int NC>
__device__ __forceinline__ Cx<T> sum_parts(const Cx<T> *part, int mu, int lane, int c) {
    const Cx<T> *q = part + (mu * 4 * NC + c) * 64 + lane;
    return (q[0] + q[2 * NC * 64]) + (q[NC * 64] + q[3 * NC * 64]);  // the wave-per-site kernel's order
}

// Four wavefronts per (site, RHS) pay while a launch holds fewer lanes than four wavefronts per SIMD
// (65536; 8^4, 4 RHS, FP64: 9.0 -> 5.6 us, 8^3 x 16, 16 RHS, FP16: 7.0 -> 5.5 us; at 98304 lanes 14.8 ->
// 15.9 us), twice that for up to 4 RHS, whose links few lanes share (16^4, 4 RHS, FP32: 19.4 -> 15.6 us),
// and with no more than a quarter of a wavefront's lanes idle.
inline bool split_over_directions(double sites, int R) {
    if (R > 64 || (64 / R) * R < 48) return false;
    return sites * R <= (R <= 4 ? 131072.0 : 65536.0);
}

// Clover blocks of a workgroup's sites, in memory [site][chirality][2 NC][2 NC], complex in the accumulation
// type and Hermitian (the term by construction, its inverse up to its rounding).  LDS holds their lower
// triangles, row by row, kCloverRow entries per site (an odd number: banks, as the links), each read once
// per lane for its row and, conjugated, for its column (16^3 x 32, SU(3), 12 RHS: FP16 hop with blocks
// 57 -> 47.5 us, FP64 143 -> 134 us against whole rows).
template <int NC>
constexpr int kCloverTri = NC * (2 * NC + 1);
template <int NC>
constexpr int kCloverRow = 2 * kCloverTri<NC> + 1;

template <typename S, int NC>
struct Clover {
    using T = typename Arith<S>::T;
    const Cx<T> *blocks;  // of the output parity
    Cx<T> *lds;

    __device__ __forceinline__ void load(const int *sw, int ns) const {
        constexpr int n = 2 * NC, tri = kCloverTri<NC>, per = 2 * tri;
        for (int i = threadIdx.x; i < ns * per; i += blockDim.x) {
            const int l = i / per, e = i - l * per, ch = e >= tri, f = e - ch * tri;
            int row = 0;
#pragma unroll
            for (int k = 1; k < n; ++k) row += f >= k * (k + 1) / 2;
            const int col = f - row * (row + 1) / 2;
            lds[l * kCloverRow<NC> + e] = blocks[((long(sw[l * 9]) * 2 + ch) * n + row) * n + col];
        }
    }

    // TERM: rows of A x + coef acc, x = read(entry); else rows of A (coef acc [+ read(entry) if have]).
    // read(spin * NC + colour) returns the stored entry; emit(entry, value[V], x_entry[V]) is called for
    // each, x_entry being what the block was applied to
    template <int V, typename G, typename F>
    __device__ __forceinline__ void rows_of(const Cx<T> (&acc)[4][NC][V], bool term, bool have, T coef, int site,
                                            G &&read, F &&emit) const {
        using W = Vec<typename Arith<S>::C, V>;
        constexpr int n = 2 * NC;
        const Cx<T> *own = lds + site * kCloverRow<NC>;
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
            Cx<T> v[n][V];
            if (term || have) {
                W w[n];
#pragma unroll
                for (int k = 0; k < n; ++k) w[k] = read(ch * n + k);
#pragma unroll
                for (int k = 0; k < n; ++k)
#pragma unroll
                    for (int i = 0; i < V; ++i) v[k][i] = load_cx<T>(&w[k].c[i]);
            }
            if (!term) {
#pragma unroll
                for (int k = 0; k < n; ++k)
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        const Cx<T> h = acc[2 * ch + k / NC][k % NC][i];
                        v[k][i] = have ? Cx<T>{fma(coef, h.re, v[k][i].re), fma(coef, h.im, v[k][i].im)} : coef * h;
                    }
            }
            Cx<T> o[n][V];
#pragma unroll
            for (int row = 0; row < n; ++row)
#pragma unroll
                for (int i = 0; i < V; ++i) o[row][i] = {T(0), T(0)};
            // every row's products in the order of its columns
#pragma unroll
            for (int row = 0; row < n; ++row)
#pragma unroll
                for (int k = 0; k <= row; ++k) {
                    const Cx<T> b = own[ch * kCloverTri<NC> + row * (row + 1) / 2 + k];
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        cfma(o[row][i], b, v[k][i]);
                        if (k < row) cfma_conj(o[k][i], b, v[row][i]);
                    }
                }
#pragma unroll
            for (int row = 0; row < n; ++row) {
                if (term) {
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        const Cx<T> h = acc[2 * ch + row / NC][row % NC][i];
                        o[row][i].re = fma(coef, h.re, o[row][i].re);
                        o[row][i].im = fma(coef, h.im, o[row][i].im);
                    }
                }
                emit(ch * n + row, o[row], v[row]);
            }
        }
    }

    // x given: A x + coef acc (xpay not read); else A (coef acc + xpay); x, xpay RHS-innermost
    template <int V, typename F>
    __device__ __forceinline__ void rows(const Cx<T> (&acc)[4][NC][V], const typename Arith<S>::C *x,
                                         const typename Arith<S>::C *xpay, T coef, const Place &p, int ns,
                                         unsigned row_bytes, unsigned vec_bytes, F &&emit) const {
        using RW = Raw<V * int(sizeof(typename Arith<S>::C))>;
        const auto r_x = rsrc(x ? x : xpay, vec_bytes);
        rows_of<V>(
            acc, x != nullptr, xpay != nullptr, coef, min(p.local, ns - 1),
            [&](int k) {
                return __builtin_bit_cast(Vec<typename Arith<S>::C, V>, RW::load(r_x, p.vo, unsigned(k) * row_bytes));
            },
            emit);
    }
};

// Wavefronts per SIMD the register budget is set for: accumulators, a hop's spinor rows and its projected
// entries fit without spilling (Nc = 3: 130 registers FP64, 67 FP32, 62 FP16).
template <typename S, int NC, int V>
constexpr int kMinWaves = NC * V * int(sizeof(typename Arith<S>::T)) >= 32 ? 2 : NC * V * int(sizeof(typename Arith<S>::T)) >= 24 ? 3 : 4;

// 16 bits, Nc <= 3: the next hop's spinor is loaded ahead, at 12 registers and no loss of occupancy (24^3 x 48:
// 104 -> 97 us at 4 RHS, 333 -> 328 at 24, equal at 32; Nc = 4: 84 -> 87 us at 16^3 x 32, 32 RHS).  Not in
// FP32 and FP64, whose lines then come into the L2 a hop too early (16^3 x 32, 12 RHS, FP64: 107 -> 111 us;
// 24^3 x 48, 16 RHS: 645 -> 683 us, FP32 325 -> 339 us).
template <typename S, int NC>
constexpr bool kAhead = sizeof(typename Arith<S>::C) == 4 && NC <= 3;

// LDS of a workgroup with clover blocks: the hops', then the blocks.
template <typename S, int NC>
__host__ __device__ constexpr int clover_offset(int spb) {
    return (spb * kSiteLds<S, NC> + 15) / 16 * 16;
}
template <typename S, int NC>
__device__ __forceinline__ Clover<S, NC> clover_lds(const Cx<typename Arith<S>::T> *blocks, unsigned char *smem,
                                                       int spb) {
    return {blocks, reinterpret_cast<Cx<typename Arith<S>::T> *>(smem + clover_offset<S, NC>(spb))};
}

// Sums N values of V right-hand sides per lane over the workgroup's sites, per RHS, in site order; the sums
// are those of the first RV lanes.  red: N V rows of blockDim.x doubles.
template <int N, int V>
__device__ __forceinline__ void sum_sites(double (&v)[N][V], double *red, const Place &p, int RV, int ns) {
    __syncthreads();  // the hops' LDS is free
    const int nt = blockDim.x;
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) red[(k * V + i) * nt + threadIdx.x] = p.active ? v[k][i] : 0.0;
    __syncthreads();
    if (int(threadIdx.x) < RV) {
#pragma unroll
        for (int k = 0; k < N; ++k)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                double t = 0.0;
                for (int l = 0; l < ns; ++l) t += red[(k * V + i) * nt + l * RV + threadIdx.x];
                v[k][i] = t;
            }
    }
}

// Launch shape: V right-hand sides per lane, `spb` sites per workgroup of `threads` lanes.
struct Shape {
    int V, RV, spb, threads;
    size_t lds;
};

template <typename S, int NC>
Shape lane_shape(int Vh, int R, int v, bool clover = false) {
    Shape s;
    s.V = v;
    s.RV = R / s.V;
    const int blocks = clover ? kCloverRow<NC> * int(sizeof(Cx<typename Arith<S>::T>)) : 0;
    const int per_site = kSiteLds<S, NC> + blocks;
    // 256 lanes, fewer where the grid would leave compute units idle (a site's hops are one serial
    // chain, so a small lattice runs at the speed of one workgroup: more, smaller ones)
    s.threads = 256;
    while (s.threads > 64 && s.threads / 2 >= s.RV && div_up(Vh, std::max(1, s.threads / s.RV)) < 2 * num_cus())
        s.threads /= 2;
    s.spb = std::max(1, s.threads / s.RV);
    s.spb = std::min(s.spb, std::max(1, (s.RV <= 2 || clover ? 65520 : 40960) / per_site));  // 64 KB of LDS at most
    s.threads = (s.spb * s.RV + 63) / 64 * 64;
    const size_t lds = clover ? clover_offset<S, NC>(s.spb) + size_t(s.spb) * blocks : size_t(s.spb) * per_site;
    s.lds = std::max(lds, size_t(s.threads) * 3 * v * sizeof(double));  // hops, then sums over sites
    return s;
}

// FP32: two right-hand sides per lane (16-byte loads, half the link reads) where the fields exceed
// the 256 MiB memory-side cache and the rows are wide enough (24^3 x 48: 400 -> 323 us at 16 RHS,
// 666 -> 574 at 24, 367 -> 357 at 12, but 243 -> 247 at 8 and 174 -> 203 at 4); inside the cache
// one per lane, at twice the wavefronts, is faster (16^3 x 32, 12 RHS: 57 against 61 us).
template <typename S, int NC>
bool two_per_lane(const DslashArgs &a) {
    if (!std::is_same<S, float>::value || NC > 3) return false;
    const double bytes = double(a.g.Vh) * (8.0 * NC * NC + 8.0 * NC * a.R) * 8.0;
    return a.R % 2 == 0 && a.R >= 12 && bytes > 268435456.0;
}

}  // namespace lane
}  // namespace qcu
