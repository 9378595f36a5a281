// clover.hip -- build, block inverse and application of the clover term.
//
// Build and inverse run once per (gauge, kappa, c_sw) in FP64.  The application
// runs twice per Schur operator in the solver and is HBM-bound: a workgroup
// stages the clover blocks of its sites into LDS with contiguous loads
// (consecutive sites' blocks are adjacent in memory), then every lane owns
// one (site, chirality, RHS) triple: it reads the 2Nc spinor entries of its
// chirality (RHS-innermost, so the lanes of a wavefront read consecutive
// words), multiplies by the block read from LDS (the lanes of one block read
// the same LDS word: a broadcast) and writes 2Nc entries.  A lane reads all
// of its input before its first store and nothing else reads those entries,
// so out may alias in (A^{-1} applied in place) or y.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "clover.h"

namespace qcu {
namespace {

// sigma_{mu nu} = (i/2)[gamma_mu, gamma_nu] restricted to the two chirality
// blocks: [plane (01,02,03,12,13,23)][chirality][2][2].
struct SigmaTab {
    Cx<double> s[6][2][2][2];
};

// The chiral gamma basis of the hopping kernels (the (1 + gamma_mu) forms
// spelled out in the reference's include/kernel/qcu_gamma.cuh:10-18, 70-76,
// 126-132, 185-191), rows spin 0..3.
SigmaTab make_sigma() {
    using C = Cx<double>;
    const C o{0, 0}, p1{1, 0}, m1{-1, 0}, pi{0, 1}, mi{0, -1};
    const C gam[4][4][4] = {
        {{o, o, o, pi}, {o, o, pi, o}, {o, mi, o, o}, {mi, o, o, o}},
        {{o, o, o, m1}, {o, o, p1, o}, {o, p1, o, o}, {m1, o, o, o}},
        {{o, o, pi, o}, {o, o, o, mi}, {mi, o, o, o}, {o, pi, o, o}},
        {{o, o, p1, o}, {o, o, o, p1}, {p1, o, o, o}, {o, p1, o, o}},
    };
    SigmaTab t{};
    int q = 0;
    for (int mu = 0; mu < 4; ++mu)
        for (int nu = mu + 1; nu < 4; ++nu, ++q)
            for (int ch = 0; ch < 2; ++ch)
                for (int a = 0; a < 2; ++a)
                    for (int b = 0; b < 2; ++b) {
                        const int sa = 2 * ch + a, sb = 2 * ch + b;
                        C c{0, 0};
                        for (int k = 0; k < 4; ++k)
                            c = c + gam[mu][sa][k] * gam[nu][k][sb] - gam[nu][sa][k] * gam[mu][k][sb];
                        t.s[q][ch][a][b] = C{-0.5 * c.im, 0.5 * c.re};  // (i/2) c
                    }
    return t;
}

// coordinate c moved by d in {-1, 0, 1} on a periodic extent L
__device__ __forceinline__ int wrap(int c, int d, int L) {
    c += d;
    return c < 0 ? c + L : c >= L ? c - L : c;
}

// The four leaves of the (mu, nu) clover at x, each a path of four links:
// {direction (0 = mu, 1 = nu), offset along mu, offset along nu, daggered}.
constexpr int kLeaf[4][4][4] = {
    {{0, 0, 0, 0}, {1, 1, 0, 0}, {0, 0, 1, 1}, {1, 0, 0, 1}},        // U_mu(x) U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
    {{1, 0, 0, 0}, {0, -1, 1, 1}, {1, -1, 0, 1}, {0, -1, 0, 0}},     // U_nu(x) U_mu(x-mu+nu)^+ U_nu(x-mu)^+ U_mu(x-mu)
    {{0, -1, 0, 1}, {1, -1, -1, 1}, {0, -1, -1, 0}, {1, 0, -1, 0}},  // U_mu(x-mu)^+ U_nu(x-mu-nu)^+ U_mu(x-mu-nu) U_nu(x-nu)
    {{1, 0, -1, 1}, {0, 0, -1, 0}, {1, 1, -1, 0}, {0, 0, 0, 1}},     // U_nu(x-nu)^+ U_mu(x-nu) U_nu(x+mu-nu) U_mu(x)^+
};

// S sites per workgroup.  A thread owns one colour row of one (site, plane): row i of a path of links
// needs row i of its running product only, so the paths take one row of registers and 6 Nc times the
// threads of a site each (a thread per site held whole matrices, left 8 wavefronts on a compute unit
// and added its planes to the blocks in memory).  The rows of one site read the same links.  The
// leaves' sums of all planes then meet in LDS, and the block entries are written in memory order.
// 16^3 x 32, SU(3): 1394 -> 310 us (1.8 GB of links through the L1s, 151 MB written).
template <int NC>
struct BuildShape {
    static constexpr int S = NC == 8 ? 8 : 32;
    static constexpr int kThreads = 6 * S * NC;
};

template <int NC>
__global__ __launch_bounds__(BuildShape<NC>::kThreads) void k_clover_build(Cx<double> *__restrict__ clov,
                                                                          const Cx<double> *__restrict__ gauge, Geom g,
                                                                          double coef, SigmaTab sig) {
    constexpr int n = 2 * NC, S = BuildShape<NC>::S;
    __shared__ Cx<double> lq[6][S][NC * NC];
    const long e0 = long(blockIdx.x) * S;
    const long total = 2L * g.Vh;
    {
        const int row = threadIdx.x % NC, sl = threadIdx.x / NC % S, plane = threadIdx.x / (NC * S);
        const long e = e0 + sl;
        if (e < total) {
            const int parity = e >= g.Vh, site = int(e - (parity ? g.Vh : 0));
            int x[4];
            const int xh = site % g.Lxh;
            int rest = site / g.Lxh;
            x[1] = rest % g.L[1];
            rest /= g.L[1];
            x[2] = rest % g.L[2];
            x[3] = rest / g.L[2];
            x[0] = 2 * xh + ((x[1] + x[2] + x[3] + parity) & 1);
            // planes 01 02 03 12 13 23
            const int mu = plane < 3 ? 0 : plane < 5 ? 1 : 2;
            const int nu = plane < 3 ? plane + 1 : plane < 5 ? plane - 1 : 3;
            Cx<double> Q[NC];
#pragma unroll
            for (int j = 0; j < NC; ++j) Q[j] = Cx<double>{0.0, 0.0};
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                Cx<double> w[NC];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const int *st = kLeaf[l][h];
                    int c[4], p = 0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        c[k] = wrap(x[k], k == mu ? st[1] : k == nu ? st[2] : 0, g.L[k]);
                        p += c[k];
                    }
                    const long idx = ((long(c[3]) * g.L[2] + c[2]) * g.L[1] + c[1]) * g.Lxh + c[0] / 2;
                    const Cx<double> *u = gauge + ((long(st[0] ? nu : mu) * 2 + (p & 1)) * g.Vh + idx) * NC * NC;
                    Cx<double> t[NC];
#pragma unroll
                    for (int j = 0; j < NC; ++j) {
                        if (h == 0) {
                            t[j] = st[3] ? conj(u[j * NC + row]) : u[row * NC + j];
                            continue;
                        }
                        t[j] = Cx<double>{0.0, 0.0};
#pragma unroll
                        for (int k = 0; k < NC; ++k) cfma(t[j], w[k], st[3] ? conj(u[j * NC + k]) : u[k * NC + j]);
                    }
#pragma unroll
                    for (int j = 0; j < NC; ++j) w[j] = t[j];
                }
#pragma unroll
                for (int j = 0; j < NC; ++j) Q[j] = Q[j] + w[j];
            }
#pragma unroll
            for (int j = 0; j < NC; ++j) lq[plane][sl][row * NC + j] = Q[j];
        }
    }
    __syncthreads();
    const int ns = int(total - e0 < S ? total - e0 : S);
    for (int k = threadIdx.x; k < ns * 2 * n * n; k += BuildShape<NC>::kThreads) {
        const int c = k % n, r = k / n % n, ch = k / (n * n) & 1, sl = k / (2 * n * n);
        const int sp = r / NC, a = r % NC, t = c / NC, b = c % NC;
        // F is formed in its upper triangle; the lower one is its conjugate
        const int lo = a < b ? a : b, hi = a < b ? b : a;
        Cx<double> v{r == c ? 1.0 : 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const Cx<double> sv = sig.s[q][ch][sp][t];
            if (sv.re == 0.0 && sv.im == 0.0) continue;
            const Cx<double> *Q = lq[q][sl];
            // F = ((Q - Q^+) - tr(Q - Q^+)/NC) / (8i); tr(Q - Q^+) = 2i Im tr Q
            Cx<double> d = Q[lo * NC + hi] - conj(Q[hi * NC + lo]);  // anti-Hermitian part times 2
            if (a == b) {
                double imtr = 0.0;
#pragma unroll
                for (int i = 0; i < NC; ++i) imtr += Q[i * NC + i].im;
                d.im -= 2.0 * imtr / NC;
            }
            // F_ab = d / (8i) = (d.im, -d.re) / 8
            Cx<double> f{d.im * 0.125, -d.re * 0.125};
            if (a > b) f = conj(f);
            v = v + (-coef) * (sv * f);
        }
        clov[e0 * 2 * n * n + k] = v;
    }
}

__device__ __forceinline__ Cx<double> select(bool c, Cx<double> a, Cx<double> b) {
    return {c ? a.re : b.re, c ? a.im : b.im};
}

// In-place Gauss-Jordan inversion with partial pivoting (row interchanges
// recorded, undone as column interchanges at the end).  N lanes per block, one
// column in the registers of each: the lanes read whole rows from memory, the
// pivot column goes round by shuffles, and the column interchanges at the end are
// the address that each lane writes to (a thread per block worked in memory).
// 16^3 x 32, SU(3) (262144 blocks of 6 x 6): 2032 -> 62 us (302 MB, read and written once: 4.9 TB/s).
template <int N>
__global__ __launch_bounds__(256) void k_clover_invert(Cx<double> *inv, const Cx<double> *a, long nblocks) {
    constexpr int G = 64 / N;  // blocks per wavefront
    const int lane = threadIdx.x & 63, j = lane % N, lane0 = lane - j;
    const long e = (long(blockIdx.x) * (256 / 64) + (threadIdx.x >> 6)) * G + lane / N;
    const bool live = lane < G * N && e < nblocks;
    Cx<double> m[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        m[i] = Cx<double>{i == j ? 1.0 : 0.0, 0.0};
        if (live) m[i] = a[(e * N + i) * N + j];
    }
    int perm[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        Cx<double> col[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
            col[i] = Cx<double>{__shfl(m[i].re, lane0 + k), __shfl(m[i].im, lane0 + k)};
        int p = k;
        double best = -1.0;
#pragma unroll
        for (int i = k; i < N; ++i) {
            const double mag = fma(col[i].re, col[i].re, col[i].im * col[i].im);
            if (mag > best) {
                best = mag;
                p = i;
            }
        }
        perm[k] = p;
#pragma unroll
        for (int i = k + 1; i < N; ++i) {
            const bool sw = p == i;
            const Cx<double> t = m[k], u = col[k];
            m[k] = select(sw, m[i], t);
            m[i] = select(sw, t, m[i]);
            col[k] = select(sw, col[i], u);
            col[i] = select(sw, u, col[i]);
        }
        const Cx<double> piv = cdiv(Cx<double>{1.0, 0.0}, col[k]);
        const Cx<double> d = select(j == k, Cx<double>{1.0, 0.0}, m[k]);
        m[k] = Cx<double>{fma(d.re, piv.re, -(d.im * piv.im)), fma(d.re, piv.im, d.im * piv.re)};
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (i == k) continue;
            const Cx<double> f = col[i], r = m[k];
            m[i] = select(j == k, Cx<double>{0.0, 0.0}, m[i]) -
                   Cx<double>{fma(f.re, r.re, -(f.im * r.im)), fma(f.im, r.re, f.re * r.im)};
        }
    }
    int dst = j;
#pragma unroll
    for (int k = N - 1; k >= 0; --k) dst = dst == k ? perm[k] : dst == perm[k] ? k : dst;
    if (!live) return;
#pragma unroll
    for (int i = 0; i < N; ++i) inv[(e * N + i) * N + dst] = m[i];
}

extern __shared__ __align__(16) unsigned char qcu_clover_lds[];

// out = A in + coef * y; S sites per workgroup, lanes (site, chirality, rhs)
template <int NC, typename CS, typename TC>
__global__ __launch_bounds__(1024) void k_clover_apply(CS *out, const CS *in, const Cx<TC> *__restrict__ blocks,
                                                      const CS *y, TC coef, int Vh, int R, int S) {
    constexpr int n = 2 * NC;
    auto *lds = reinterpret_cast<Cx<TC> *>(qcu_clover_lds);
    const int site0 = blockIdx.x * S;
    const int ns = min(S, Vh - site0);
    const long base = long(site0) * 2 * n * n;
    const int total = ns * 2 * n * n;
    for (int k = threadIdx.x; k < total; k += blockDim.x) lds[k] = blocks[base + k];
    __syncthreads();
    const int tid = threadIdx.x;
    const int sl = tid / (2 * R);
    if (sl >= ns) return;
    const int ch = (tid / R) & 1, r = tid % R;
    const long site = site0 + sl;
    const long e0 = ((site * 4 + 2 * ch) * NC) * R + r;  // entry (spin 2ch, colour 0, rhs r)
    Cx<TC> v[n];
#pragma unroll
    for (int k = 0; k < n; ++k) v[k] = load_cx<TC>(in + e0 + long(k) * R);
    const Cx<TC> *L = lds + (sl * 2 + ch) * n * n;
#pragma unroll
    for (int row = 0; row < n; ++row) {
        Cx<TC> acc{TC(0), TC(0)};
#pragma unroll
        for (int col = 0; col < n; ++col) cfma(acc, L[row * n + col], v[col]);
        const long e = e0 + long(row) * R;
        if (y) {
            const Cx<TC> yv = load_cx<TC>(y + e);
            acc.re = fma(coef, yv.re, acc.re);
            acc.im = fma(coef, yv.im, acc.im);
        }
        store_cx(out + e, acc);
    }
}

template <int NC, typename CS, typename TC>
hipError_t apply_t(void *out, const void *in, const void *blocks, const void *y, double coef, int Vh, int R,
                   hipStream_t s) {
    constexpr int n = 2 * NC;
    const int per_site = 2 * n * n * int(sizeof(Cx<TC>));
    int S = 2 * R >= 256 ? 1 : 256 / (2 * R);
    S = std::min(S, std::max(1, 65536 / per_site));
    const int threads = (S * 2 * R + 63) / 64 * 64;
    if (threads > 1024) return hipErrorInvalidConfiguration;
    const int blocks_n = div_up(Vh, S);
    hipLaunchKernelGGL((k_clover_apply<NC, CS, TC>), dim3(blocks_n), dim3(threads), size_t(S) * per_site, s,
                       static_cast<CS *>(out), static_cast<const CS *>(in), static_cast<const Cx<TC> *>(blocks),
                       static_cast<const CS *>(y), TC(coef), Vh, R, S);
    return hipGetLastError();
}

template <int NC, typename TC>
hipError_t apply_prec(void *out, const void *in, const void *blocks, const void *y, double coef, int Vh, int R,
                      int prec, hipStream_t s) {
    switch (prec) {
        case kDouble: return apply_t<NC, Cx<double>, TC>(out, in, blocks, y, coef, Vh, R, s);
        case kSingle: return apply_t<NC, Cx<float>, TC>(out, in, blocks, y, coef, Vh, R, s);
        case kHalf: return apply_t<NC, Half2Store, TC>(out, in, blocks, y, coef, Vh, R, s);
        case kBF16: return apply_t<NC, Bf162Store, TC>(out, in, blocks, y, coef, Vh, R, s);
        default: return hipErrorInvalidValue;
    }
}

template <int NC>
hipError_t apply_nc(void *out, const void *in, const void *blocks, const void *y, double coef, int Vh, int R,
                    int prec, int clover_prec, hipStream_t s) {
    if (clover_prec == kDouble) return apply_prec<NC, double>(out, in, blocks, y, coef, Vh, R, prec, s);
    if (clover_prec == kSingle) return apply_prec<NC, float>(out, in, blocks, y, coef, Vh, R, prec, s);
    return hipErrorInvalidValue;
}

}  // namespace

bool clover_supported(int Nc) { return Nc == 2 || Nc == 3 || Nc == 4 || Nc == 8; }

hipError_t launch_clover_build(void *clover, const void *gauge, const Geom &g, int Nc, double csw, double kappa,
                               hipStream_t s) {
    static const SigmaTab sig = make_sigma();
    const double coef = kappa * csw;
    auto *c = static_cast<Cx<double> *>(clover);
    const auto *u = static_cast<const Cx<double> *>(gauge);
    switch (Nc) {
        case 2: hipLaunchKernelGGL(k_clover_build<2>, dim3(div_up(2L * g.Vh, BuildShape<2>::S)),
                                   dim3(BuildShape<2>::kThreads), 0, s, c, u, g, coef, sig); break;
        case 3: hipLaunchKernelGGL(k_clover_build<3>, dim3(div_up(2L * g.Vh, BuildShape<3>::S)),
                                   dim3(BuildShape<3>::kThreads), 0, s, c, u, g, coef, sig); break;
        case 4: hipLaunchKernelGGL(k_clover_build<4>, dim3(div_up(2L * g.Vh, BuildShape<4>::S)),
                                   dim3(BuildShape<4>::kThreads), 0, s, c, u, g, coef, sig); break;
        case 8: hipLaunchKernelGGL(k_clover_build<8>, dim3(div_up(2L * g.Vh, BuildShape<8>::S)),
                                   dim3(BuildShape<8>::kThreads), 0, s, c, u, g, coef, sig); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_clover_invert(void *inv, const void *clover, long nblocks, int n, hipStream_t s) {
    const int nb = div_up(nblocks, 4 * (64 / n));
    auto *o = static_cast<Cx<double> *>(inv);
    const auto *a = static_cast<const Cx<double> *>(clover);
    switch (n) {
        case 4: hipLaunchKernelGGL(k_clover_invert<4>, dim3(nb), dim3(256), 0, s, o, a, nblocks); break;
        case 6: hipLaunchKernelGGL(k_clover_invert<6>, dim3(nb), dim3(256), 0, s, o, a, nblocks); break;
        case 8: hipLaunchKernelGGL(k_clover_invert<8>, dim3(nb), dim3(256), 0, s, o, a, nblocks); break;
        case 16: hipLaunchKernelGGL(k_clover_invert<16>, dim3(nb), dim3(256), 0, s, o, a, nblocks); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_clover_apply(void *out, const void *in, const void *blocks, const void *y, double coef,
                               int Vh, int Nc, int R, int prec, int clover_prec, hipStream_t s) {
    if (R <= 0 || R > 512 || Vh <= 0) return hipErrorInvalidValue;
    switch (Nc) {
        case 2: return apply_nc<2>(out, in, blocks, y, coef, Vh, R, prec, clover_prec, s);
        case 3: return apply_nc<3>(out, in, blocks, y, coef, Vh, R, prec, clover_prec, s);
        case 4: return apply_nc<4>(out, in, blocks, y, coef, Vh, R, prec, clover_prec, s);
        case 8: return apply_nc<8>(out, in, blocks, y, coef, Vh, R, prec, clover_prec, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qcu
