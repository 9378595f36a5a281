// dslash.hip -- one-parity multi-RHS SU(N) Wilson hopping term on gfx950.
//
// Operator (include/kernel/sun_mrhs_wilson_dslash_simt.cuh:97-181 of the
// reference; output parity p, input on 1-p):
//   out(x) = sum_mu (1 - g_mu) U_mu(x) psi(x+mu) + (1 + g_mu) U_mu(x-mu)^+ psi(x-mu)
// dagger flips the sign of every gamma (ibid. :147,176).  Spin structure via
// two projected rows per hop: h_r = psi_r + s_r psi_m(r), out_r += U h_r,
// out_m(r) += c_r U h_r (include/kernel/qcu_gamma.cuh:47-324).
//
// This file holds the dispatcher and the general lane-per-(site, rhs) VALU
// kernel: R lanes of one site read R consecutive complex numbers for every
// (spin, colour); the link is a broadcast load shared by those lanes.  It
// serves variant kDslashLaneRhs for Nc = 8, for vectors of 4 GiB and more and
// for few right-hand sides on large lattices (dslash_general_faster); the one for the
// other shapes of Nc <= 4 is in dslash_lane.hip.  The wave-per-site kernels live
// in dslash_wave.hip (VALU) and dslash_mfma.hip (matrix cores).  Every variant has an optional epilogue
// out = x + coef * D psi (Schur operator, full-lattice M, source preparation).
#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <tuple>

#include "blas.h"
#include "clover.h"
#include "dslash_common.h"

namespace qcu {
namespace {

template <typename T, typename CS, typename CG, int NC, int MU, bool FWD, bool DAG>
__device__ __forceinline__ void hop(Cx<T> (&acc)[4][NC], const CS *__restrict__ psi, int R,
                                    const CG *__restrict__ U) {
    constexpr int sgn = (FWD != DAG) ? 2 : 0;
    constexpr int m0 = kMat2(MU, 0), m1 = kMat2(MU, 1);
    constexpr int kp0 = kProjK(MU, 0) + sgn, kp1 = kProjK(MU, 1) + sgn;
    constexpr int kr0 = kReconK(MU, 0) + sgn, kr1 = kReconK(MU, 1) + sgn;
    Cx<T> h0[NC], h1[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const Cx<T> a0 = load_cx<T>(psi + (0 * NC + c) * R);
        const Cx<T> a1 = load_cx<T>(psi + (1 * NC + c) * R);
        const Cx<T> b0 = load_cx<T>(psi + (m0 * NC + c) * R);
        const Cx<T> b1 = load_cx<T>(psi + (m1 * NC + c) * R);
        h0[c] = a0 + ipow<kp0>(b0);
        h1[c] = a1 + ipow<kp1>(b1);
    }
#pragma unroll
    for (int a = 0; a < NC; ++a) {
        Cx<T> s0 = {T(0), T(0)}, s1 = {T(0), T(0)};
#pragma unroll
        for (int b = 0; b < NC; ++b) {
            if constexpr (FWD) {
                const Cx<T> u = load_cx<T>(U + a * NC + b);
                cfma(s0, u, h0[b]);
                cfma(s1, u, h1[b]);
            } else {
                const Cx<T> u = load_cx<T>(U + b * NC + a);   // (U^+)[a][b] = conj(U[b][a])
                cfma_conj(s0, u, h0[b]);
                cfma_conj(s1, u, h1[b]);
            }
        }
        acc[0][a] = acc[0][a] + s0;
        acc[m0][a] = acc[m0][a] + ipow<kr0>(s0);
        acc[1][a] = acc[1][a] + s1;
        acc[m1][a] = acc[m1][a] + ipow<kr1>(s1);
    }
}

template <typename T, typename CS, typename CG, int NC, bool DAG>
__global__ __launch_bounds__(256) void k_wilson_dslash_valu(CS *__restrict__ out,
                                                           const CS *__restrict__ in,
                                                           const CG *__restrict__ gauge,
                                                           const CS *__restrict__ xpay, T coef,
                                                           Geom g, int R, int parity) {
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int site = b * blockDim.y + threadIdx.y;
    if (site >= g.Vh) return;
    const int r = threadIdx.x;

    const int Lx = g.L[0], Ly = g.L[1], Lz = g.L[2], Lt = g.L[3], Lxh = g.Lxh;
    const int xh = site % Lxh;
    int rest = site / Lxh;
    const int y = rest % Ly;
    rest /= Ly;
    const int z = rest % Lz;
    const int t = rest / Lz;
    const int x = 2 * xh + ((y + z + t + parity) & 1);
    const int row = site - xh;
    const int sy = Lxh, sz = Lxh * Ly, st = Lxh * Ly * Lz;

    int nbf[4], nbb[4];
    nbf[0] = row + ((x + 1 == Lx ? 0 : x + 1) >> 1);
    nbb[0] = row + ((x == 0 ? Lx - 1 : x - 1) >> 1);
    nbf[1] = site + (y + 1 == Ly ? -(Ly - 1) * sy : sy);
    nbb[1] = site + (y == 0 ? (Ly - 1) * sy : -sy);
    nbf[2] = site + (z + 1 == Lz ? -(Lz - 1) * sz : sz);
    nbb[2] = site + (z == 0 ? (Lz - 1) * sz : -sz);
    nbf[3] = site + (t + 1 == Lt ? -(Lt - 1) * st : st);
    nbb[3] = site + (t == 0 ? (Lt - 1) * st : -st);

    const long site_len = 4L * NC * R;
    const long link_len = long(NC) * NC;
    const CS *inr = in + r;
    const long Vh = g.Vh;

    Cx<T> acc[4][NC];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[s][c] = {T(0), T(0)};

#define QCU_HOP(MU)                                                                          \
    hop<T, CS, CG, NC, MU, true, DAG>(acc, inr + nbf[MU] * site_len, R,                       \
                                      gauge + ((MU * 2 + parity) * Vh + site) * link_len);    \
    hop<T, CS, CG, NC, MU, false, DAG>(acc, inr + nbb[MU] * site_len, R,                      \
                                       gauge + ((MU * 2 + 1 - parity) * Vh + nbb[MU]) * link_len);
    QCU_HOP(0)
    QCU_HOP(1)
    QCU_HOP(2)
    QCU_HOP(3)
#undef QCU_HOP

    CS *o = out + site * site_len + r;
    if (xpay) {
        const CS *xp = xpay + site * site_len + r;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                Cx<T> v = load_cx<T>(xp + (s * NC + c) * R);
                v.re = fma(coef, acc[s][c].re, v.re);
                v.im = fma(coef, acc[s][c].im, v.im);
                store_cx(o + (s * NC + c) * R, v);
            }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) store_cx(o + (s * NC + c) * R, coef * acc[s][c]);
    }
}

template <typename T, typename S, int NC>
hipError_t launch_valu(const DslashArgs &a, hipStream_t stream) {
    using CS = typename CxStore<S>::type;
    const int spb = a.R >= 256 ? 1 : 256 / a.R;
    dim3 block(a.R, spb);
    dim3 grid(div_up(a.g.Vh, spb));
    auto out = static_cast<CS *>(a.out);
    auto in = static_cast<const CS *>(a.in);
    auto gauge = static_cast<const CS *>(a.gauge);
    auto xp = static_cast<const CS *>(a.xpay);
    if (a.dagger)
        hipLaunchKernelGGL((k_wilson_dslash_valu<T, CS, CS, NC, true>), grid, block, 0, stream,
                           out, in, gauge, xp, T(a.coef), a.g, a.R, a.parity);
    else
        hipLaunchKernelGGL((k_wilson_dslash_valu<T, CS, CS, NC, false>), grid, block, 0, stream,
                           out, in, gauge, xp, T(a.coef), a.g, a.R, a.parity);
    return hipGetLastError();
}

template <typename T, typename S>
hipError_t dispatch_nc(const DslashArgs &a, hipStream_t stream) {
    switch (a.Nc) {
        case 2: return launch_valu<T, S, 2>(a, stream);
        case 3: return launch_valu<T, S, 3>(a, stream);
        case 4: return launch_valu<T, S, 4>(a, stream);
        case 8: return launch_valu<T, S, 8>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool dslash_supported(int Nc, int R) {
    return (Nc == 2 || Nc == 3 || Nc == 4 || Nc == 8) && R >= 1 && R <= 256;
}

namespace {
std::mutex g_tune_mu;
std::map<std::tuple<int, int, int, int, int, int, int>, DslashTune> g_tuned;
DslashTune g_override;  // variant != auto: forced for every launch

int largest_divisor_at_most(int L, int cap) {
    for (int d = cap < L ? cap : L; d > 1; --d)
        if (L % d == 0) return d;
    return 1;
}
}  // namespace

void dslash_set_tuned(const int L[4], int Nc, int R, int prec, const DslashTune &t) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[std::make_tuple(L[0], L[1], L[2], L[3], Nc, R, prec)] = t;
}

void dslash_set_override(const DslashTune &t) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_override = t;
}

DslashTune dslash_resolve(const DslashArgs &a) {
    DslashTune t = a.tune;
    if (t.variant == kDslashAuto) {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        if (g_override.variant != kDslashAuto) {
            t = g_override;
        } else {
            auto it = g_tuned.find(std::make_tuple(a.g.L[0], a.g.L[1], a.g.L[2], a.g.L[3], a.Nc, a.R, a.prec));
            if (it != g_tuned.end()) t = it->second;
        }
    }
    return dslash_fill_defaults(a, t);
}

bool dslash_get_tuned(const int L[4], int Nc, int R, int prec, DslashTune &t) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(std::make_tuple(L[0], L[1], L[2], L[3], Nc, R, prec));
    if (it == g_tuned.end()) return false;
    t = it->second;
    return true;
}

std::vector<std::pair<std::array<int, 7>, DslashTune>> dslash_tuned_entries() {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    std::vector<std::pair<std::array<int, 7>, DslashTune>> v;
    for (const auto &e : g_tuned) {
        const auto &k = e.first;
        v.push_back({{std::get<0>(k), std::get<1>(k), std::get<2>(k), std::get<3>(k), std::get<4>(k),
                      std::get<5>(k), std::get<6>(k)},
                     e.second});
    }
    return v;
}

namespace {
// what the 16-bit matrix-core kernel addresses
bool fits_mfma16(const DslashArgs &a) {
    return double(a.g.Vh) * 16.0 * a.Nc * a.R < 2147483647.0 && double(a.g.Vh) * 32.0 * a.Nc * a.Nc < 2147483647.0;
}

// 16 bits: a lane per (site, RHS) instead of the matrix cores (lane / matrix cores below, us, FP16).
// A row of right-hand sides has to be a whole number of 16-byte pieces, or to need a second chunk of the
// matrix cores' 16 columns; otherwise the lanes' loads straddle those pieces (at 5 to 15 on lattices from 12^4 to
// 24^3 x 48 SU(3) 1.05 to 1.6 times, SU(4) 1.1 to 2.1 times the matrix cores' time, SU(2) 0.8 to 1.5 times).
bool row_fits_lanes(int R) { return R % 4 == 0 || R > 16; }

bool lane16_faster(const DslashArgs &a) {
    if (!fits_mfma16(a)) return false;
    const long sites = a.g.Vh, lanes = sites * a.R;
    const bool split = dslash_lane_split(a.g, a.R);
    // Up to 3 right-hand sides leave 13 of the matrix cores' 16 columns empty.  From 8192 sites (8^3 x 16 with
    // 4096: even) a lane per site is faster where the lattice takes a wavefront per direction (16^3 x 32,
    // SU(3): 13 / 45 at 1, 21 / 46 at 2; beyond it 24^4, SU(3): 118 / 89 at 1; SU(4) 16^4: 13 / 25 at 1, but
    // 21 / 25 at 3, where solves on SU(4) lose 5 %) and beyond it where the rows of a site still share lines
    // (SU(2): 24^3 x 48 80 / 127 at 1, 84 / 128 at 3; SU(3) at 3: 24^4 82 / 88, 24^3 x 48 145 / 205)
    if (a.R <= 3)
        return sites >= 8192 && (a.Nc == 2 || (a.Nc == 3 && (split || a.R == 3)) || (a.Nc == 4 && split && a.R == 1));
    if (!row_fits_lanes(a.R)) return false;
    // clover blocks are applied in the lane kernel's epilogue only
    if (a.clover) return true;
    // A site's arithmetic takes the matrix cores fewer cycles, the lane kernel moves fewer bytes (24^3 x 48, SU(3):
    // 100 / 181 at 8, 209 / 242 at 16, 361 / 761 at 32).  SU(2): lanes but in the smallest ragged launches
    // (at 17: 8^3 x 16 5.8 / 5.4, 12^4 9.1 / 10.5)
    if (a.Nc == 2) return a.R % 4 == 0 || lanes > 98304;
    // SU(3) beyond 8 and two chunks: more than three wavefronts per SIMD (SU(3) 12^4 8.8 / 8.1 at 16, 10.5 / 13.3
    // at 20, 16^4 18.1 / 19.0 at 16, 8^4 6.3 / 5.5 at 48; SU(4) 8^3 x 16 13.4 / 12.4 at 48, 13.6 / 15.8 at 64,
    // 12^4 18.7 / 16.4 at 17)
    if (a.R > 16 || (a.Nc == 3 && a.R > 8)) return lanes > 196608;
    if (a.Nc == 3) return true;
    // SU(4), one chunk: up to 8 a wavefront per direction (12^4 6.4 / 9.4 at 4) or four wavefronts per SIMD
    // (at 8: 12^4 11.6 / 9.6, 16^4 20.6 / 22.6); 12 and 16 once the fields exceed the 256 MiB memory-side cache
    // (at 16: 12^4 13.8 / 9.5, 16^3 x 32 48 / 43, 24^4 120 / 165)
    if (a.R <= 8) return split || lanes >= 262144;
    return double(sites) * (8.0 * a.Nc * a.Nc + 8.0 * a.Nc * a.R) * 4.0 > 268435456.0;
}

// Kernel chosen for a hop that names none.
int automatic_variant(const DslashArgs &a) {
    const bool lane = dslash_lane_supported(a.g, a.Nc, a.R, a.prec);
    if (a.keep_order && a.prec != kSingle) return dslash_mfma_supported(a.Nc, a.prec) ? kDslashMfma : kDslashWaveSite;
    if (a.keep_order && a.Nc == 8) return kDslashWaveSite;
    if (a.prec == kSingle || a.prec == kDouble) {
        // Nc = 8 fills the 16 x 16 matrix-core tile (16^4, 16 RHS: FP64 265 us against 1035 us wave per
        // site, FP32 147 against 311 us); Nc <= 4 runs a lane per (site, RHS), faster than the
        // wave-per-site and matrix-core kernels at every size timed (dslash_lane.hip)
        if (a.Nc == 8) return kDslashMfma;
        return lane ? kDslashLaneRhs : kDslashWaveSite;
    }
    if (lane && lane16_faster(a)) return kDslashLane16;
    return dslash_mfma_supported(a.Nc, a.prec) ? kDslashMfma : kDslashWaveSite;
}
}  // namespace

DslashTune dslash_fill_defaults(const DslashArgs &a, DslashTune t) {
    if (t.variant == kDslashAuto) t.variant = automatic_variant(a);
    if (t.variant == kDslashLane16) {
        if (a.prec == kSingle || a.prec == kDouble) t.variant = kDslashLaneRhs;
        else if (!dslash_lane_supported(a.g, a.Nc, a.R, a.prec))
            t.variant = dslash_mfma_supported(a.Nc, a.prec) && fits_mfma16(a) ? kDslashMfma : kDslashWaveSite;
    }
    if ((t.variant == kDslashLaneRhs || t.variant == kDslashLane16) &&
        dslash_lane_supported(a.g, a.Nc, a.R, a.prec)) {
        dslash_lane_tile(a.g, a.Nc, a.R, a.prec, t.by, t.bz);
        return t;
    }
    if (t.variant == kDslashMfma && !dslash_matrix_supported(a.Nc, a.prec)) t.variant = kDslashWaveSite;
    if (t.variant == kDslashLds && !dslash_lds_supported(a.g, a.Nc, a.prec))
        t.variant = dslash_matrix_supported(a.Nc, a.prec) ? kDslashMfma : kDslashWaveSite;
    if (t.variant == kDslashLds) {
        // t steps per workgroup and the (y, z) block of the workgroup order (measured at 24^3x48,
        // 16 RHS: blocks of 4 x 8 to 6 x 12 rows 232-235 us against 237-254 us row by row)
        if (t.spw <= 0) t.spw = 12;
        if (t.by <= 0 || a.g.L[1] % t.by) t.by = largest_divisor_at_most(a.g.L[1], 4);
        if (t.bz <= 0 || a.g.L[2] % t.bz) t.bz = largest_divisor_at_most(a.g.L[2], 8);
        return t;
    }
    if (t.variant != kDslashLaneRhs) {
        // spw < 0 (persistent grid, -spw workgroups per CU) exists for the FP16/BF16 MFMA kernel only
        if (t.spw == 0 || (t.spw < 0 && !(t.variant == kDslashMfma && dslash_mfma_supported(a.Nc, a.prec))))
            t.spw = t.variant == kDslashMfma ? 1 : 4;  // measured best at 24^3x48, R = 16
        // tile the (y, z) plane so one tile slice (the t-reuse distance) stays
        // around 256 KiB: bytes per site = 4 Nc R complex numbers (measured at
        // 24^3x48, 16 RHS: best among tiles of 0.06 - 5 MiB for FP16 and FP64)
        const double site_bytes = 4.0 * a.Nc * a.R * 2.0 * double(prec_bytes(a.prec));
        double area = (1 << 18) / (site_bytes * a.g.Lxh);
        if (area < 1) area = 1;
        if (t.by <= 0 || a.g.L[1] % t.by) {
            int cap = 1;
            while ((cap + 1) * (cap + 1) <= area) ++cap;
            t.by = largest_divisor_at_most(a.g.L[1], cap);
        }
        if (t.bz <= 0 || a.g.L[2] % t.bz) {
            int cap = int(area / t.by);
            t.bz = largest_divisor_at_most(a.g.L[2], cap < 1 ? 1 : cap);
        }
    }
    return t;
}

// kDslashLaneRhs, Nc <= 4: the general kernel of this file instead of the one of dslash_lane.hip.  There a
// workgroup holds the links of all its sites in LDS, so with few right-hand sides LDS, not registers, limits
// the wavefronts on a compute unit.  24^3 x 48, general against lane kernel: SU(3) 1 RHS FP16 54 / 207,
// FP32 76 / 235, FP64 270 / 534 us; 2 RHS 82 / 153, 112 / 189, 307 / 354 (but 158 / 152 at 24^4, SU(2) 137 /
// 127); FP32 147 / 177 at 3 but 174 / 172 at 4, FP64 397 / 282 at 3; SU(4) FP16 195 / 261 at 3, 309 / 362 at 6, 262 / 249 at 8, BF16 258 / 259 at 3, 287 /
// 209 at 4 (the general kernel spills there).  In the cache FP32 gains up to 5 (16^3 x 32, SU(3) 38 / 48 at 5).
// A wavefront per direction (dslash_lane_split) is better until the lattice fills the GPU without it (8^4, 1
// RHS, FP32 7.9 / 4.9, FP64 13.1 / 6.0 us; 16^3 x 32 14.1 / 20.3, 24.2 / 39.6; FP16 16^3 x 24 9.9 / 9.3,
// 16^3 x 32 10.5 / 11.2).
bool dslash_general_faster(const DslashArgs &a) {
    if (a.keep_order || a.Nc > 4) return false;
    const bool split = dslash_lane_split(a.g, a.R);
    const long sites = a.g.Vh, lanes = sites * a.R;
    if (a.prec == kDouble) {
        if (split || a.R != 2) return a.R == 1 && (!split || lanes >= 49152);
        return a.Nc == 4 || (a.Nc == 3 && sites > 200000);
    }
    if (a.prec == kSingle) return split ? a.R <= 2 && lanes >= 49152 : a.R <= 3 || (a.R <= 5 && sites <= 65536);
    const bool spills = a.prec == kBF16 && a.Nc == 4;
    return split ? a.R <= 2 && sites >= 65536 && !spills : a.R <= (spills ? 3 : 7);
}

hipError_t launch_dslash(const DslashArgs &a, hipStream_t stream) {
    if (!dslash_supported(a.Nc, a.R)) return hipErrorInvalidValue;
    if (a.g.Vh <= 0) return hipSuccess;
    const DslashTune t = dslash_resolve(a);
    if (t.variant == kDslashWaveSite) return launch_dslash_wave(a, t, stream);
    if (t.variant == kDslashLds) return launch_dslash_lds(a, t, stream);
    if (t.variant == kDslashLane16 ||
        (t.variant == kDslashLaneRhs && dslash_lane_supported(a.g, a.Nc, a.R, a.prec) && !dslash_general_faster(a)))
        return launch_dslash_lane(a, t, stream);
    if (t.variant == kDslashMfma)
        return (a.prec == kSingle || a.prec == kDouble) ? launch_dslash_mfma32(a, t, stream)
                                                         : launch_dslash_mfma(a, t, stream);
    switch (a.prec) {
        case kDouble: return dispatch_nc<double, double>(a, stream);
        case kSingle: return dispatch_nc<float, float>(a, stream);
        case kHalf: return dispatch_nc<float, __half>(a, stream);
        case kBF16: return dispatch_nc<float, __hip_bfloat16>(a, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_dslash_clover(const DslashArgs &a, hipStream_t stream) {
    if (!a.clover || !dslash_supported(a.Nc, a.R)) return hipErrorInvalidValue;
    if (a.g.Vh <= 0) return hipSuccess;
    const DslashTune t = dslash_resolve(a);
    if (dslash_lane_clover_fused(a, t)) return launch_dslash_lane(a, t, stream);
    DslashArgs h = a;
    h.clover = h.clover_in = nullptr;
    if (a.clover_in) {
        h.xpay = nullptr;
        h.coef = 1.0;
    }
    QCU_HIP_TRY(launch_dslash(h, stream));
    return launch_clover_apply(a.out, a.clover_in ? a.clover_in : a.out, a.clover, a.clover_in ? a.out : nullptr,
                               a.clover_in ? a.coef : 0.0, a.g.Vh, a.Nc, a.R, a.prec,
                               a.prec == kDouble ? kDouble : kSingle, stream);
}

namespace {
// no kernel is named for these arguments: by themselves, for the process or in the tuning table
bool automatic(const DslashArgs &a) {
    if (a.tune.variant != kDslashAuto) return false;
    std::lock_guard<std::mutex> lk(g_tune_mu);
    return g_override.variant == kDslashAuto &&
           !g_tuned.count(std::make_tuple(a.g.L[0], a.g.L[1], a.g.L[2], a.g.L[3], a.Nc, a.R, a.prec));
}
}  // namespace

constexpr int kDotSlices = 512;  // first-level slices of the per-workgroup partials

long dslash_dots_partials(const Geom &g, int Nc, int R, int prec) {
    // one row of R x 4 per workgroup of the forms that exist for these arguments: the lane kernel's, or a
    // wavefront's worth of sites (a wavefront per direction); matrix cores: at most one per 4 sites, or 64 per
    // CU for the persistent grid
    long nblk = 0;
    if (dslash_lane_supported(g, Nc, R, prec)) {
        nblk = dslash_lane_blocks(g, Nc, R, prec);
        if (dslash_lane_split(g, R)) nblk = std::max<long>(nblk, div_up(g.Vh, 64 / R));
    }
    if (dslash_mfma_supported(Nc, prec)) nblk = std::max<long>({nblk, long(div_up(g.Vh, 4)), 64L * num_cus()});
    return nblk ? (nblk + kDotSlices) * R * 4 : 0;
}

hipError_t launch_dslash_dots(const DslashArgs &a, DotsKind kind, const void *r0, double *partials, long cap,
                              Cx<double> *st, hipStream_t stream) {
    if (!dslash_supported(a.Nc, a.R) || a.g.Vh <= 0 || a.dagger || a.keep_order || !partials || !st ||
        !(a.clover ? a.clover_in : a.xpay) || (kind == kDotsAlpha && !r0) || a.R > kReduceThreads)
        return hipErrorNotSupported;
    DslashTune t = dslash_resolve(a);
    // alpha's products in the lane kernel's epilogue save a pass over two vectors, more than its hop is behind
    // that of the matrix cores where lane16_faster prefers those (SU(3) 12^4, 12 RHS: 0.7 us, the pass 6 us)
    if (kind == kDotsAlpha && t.variant == kDslashMfma && row_fits_lanes(a.R) && automatic(a)) {
        t = DslashTune{};
        t.variant = kDslashLane16;
        t = dslash_fill_defaults(a, t);
    }
    const bool lane = dslash_lane_forms(a, t);
    const bool mfma = t.variant == kDslashMfma && (a.prec == kHalf || a.prec == kBF16) && kind == kDotsOmega && !a.clover;
    if ((!lane && !mfma) || (a.clover && !dslash_lane_clover_fused(a, t))) return hipErrorNotSupported;
    if (cap < dslash_dots_partials(a.g, a.Nc, a.R, a.prec)) return hipErrorInvalidValue;
    int nblk = 0;
    if (lane) QCU_HIP_TRY(launch_dslash_lane_dots(a, t, kind, r0, partials, stream, nblk));
    else QCU_HIP_TRY(launch_dslash_mfma_omega(a, t, partials, stream, nblk));
    const auto finish = kind == kDotsAlpha ? launch_finish_alpha : launch_finish_omega;
    if (nblk <= kMaxFinishRows) return finish(st, a.R, partials, nblk, stream);
    // [nblk][R][4] -> [kDotSlices][R][4] (after them) -> the finisher sums the slices in order
    double *p2 = partials + long(nblk) * a.R * 4;
    QCU_HIP_TRY(launch_rows_sum(p2, partials, nblk, 4 * a.R, kDotSlices, stream));
    return finish(st, a.R, p2, kDotSlices, stream);
}

}  // namespace qcu
