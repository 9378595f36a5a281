// lgnn_stencil.hip -- FP32 kernels of the learned preconditioner on matrix
// cores (declared in lgnn.h): the transported (hop, spin) mixing on the even
// sites and the outer-product gradient of the 32 x 32 stencil.
//
// Both take the input fields themselves and transport them on the fly: per even
// site y a workgroup forms the 32 rows u_(k,s)(y) = V_k(y) f_s(nb_k(y)) of one
// chunk of right-hand sides (columns = (colour, rhs), at most 64) in LDS -- FP32,
// the same arithmetic as a transport kernel that stores them -- and the matrix
// cores read them from there.  Storing the eight hop fields instead costs 0.8 GB
// written and read again per use at 16^3 x 32, 16 RHS.
//
// k_lgnn_mix32: q = M u in FP32 (v_mfma_f32_16x16x4_f32) through the real 2 x 2
// embedding of M, whose fragments stay in registers: wavefront w computes complex
// rows 8 w .. 8 w + 7 of every column.  26 GFLOP and 0.9 GB at 16^3 x 32, 16 RHS,
// so the FP32 matrix rate (145 TFLOP/s: 178 us) and the field writes (170 us) are
// about even.
// k_lgnn_gram: G += a conj(u)^T in FP64 (v_mfma_f64_16x16x4_f64), two columns per
// instruction (k = column, re | im): G_re takes (a_re, a_im), G_im (a_im, -a_re)
// against (u_re, u_im).  The wavefronts take columns in turn, each with the whole
// 32 x 32 complex sum in 64 registers.  26 GFLOP in FP64: 360 us at 72 TFLOP/s.
//
// Measured at 16^3 x 32, 16 RHS (SU(3)): k_lgnn_mix32 342 us (transport to 8 fields and a
// VALU product before: 666 us), k_lgnn_gram 583 us (transport and a VALU FP64 sum
// through LDS before: 2960 us); a gradient pass of power 3 15.1 -> 5.97 ms.
#include <algorithm>

#include "dslash_common.h"
#include "geom.h"
#include "lgnn.h"

namespace qcu {
namespace {

using C32 = Cx<float>;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxCols = 64;                   // columns (colour, rhs) of one chunk, padded to a multiple of 16
constexpr int row_words(int cols) { return 2 * cols + 4; }  // 16 rows of one column fall into 16 bank quads

// right-hand sides per chunk: as even as the 64 columns allow, at most 32
int chunk_rhs(int Nc, int R) {
    const int most = std::min(32, kMaxCols / Nc);
    return div_up(R, div_up(R, most));
}

// What a thread stages of each site: IT of the 32 rc (row, rhs) items -- the NC colours of its neighbour
// spinor row, transported by the 8 links in LDS -- and at most ceil(8 NC^2 / 256) link entries.  The
// loads of the next site go out before the matrix-core work of this one, and the neighbour indices they
// need one site earlier still, so no load latency is waited for inside the loop.
template <int NC, int IT>
struct Items {
    static constexpr int LI = (8 * NC * NC + 255) / 256;
    int ks[IT], rr[IT];     // row (k, s) (negative: none) and rhs of the chunk
    int nb[IT];             // neighbour of the site whose spinors are loaded next
    int li[LI], lsite[LI];  // walk column of the link's site, that site
    __device__ __forceinline__ Items(int rc) {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int e = int(threadIdx.x) + 256 * i, q = e / rc;
            ks[i] = q < 32 ? q : -1;
            rr[i] = e - q * rc;
        }
#pragma unroll
        for (int i = 0; i < LI; ++i) {
            const int e = int(threadIdx.x) + 256 * i, k = e / (NC * NC);
            li[i] = k < 8 ? ((k & 1) ? 1 + k : 0) : -1;  // forward links sit at the site, backward ones at the neighbour
        }
    }
    __device__ __forceinline__ void indices(const int *__restrict__ row) {
#pragma unroll
        for (int i = 0; i < IT; ++i) nb[i] = row[1 + (max(ks[i], 0) >> 2)];
#pragma unroll
        for (int i = 0; i < LI; ++i) lsite[i] = row[max(li[i], 0)];
    }
    __device__ __forceinline__ void load_links(C32 (&l)[LI], const C32 *__restrict__ gauge, int Vh) const {
#pragma unroll
        for (int i = 0; i < LI; ++i) {
            const int e = int(threadIdx.x) + 256 * i, k = e / (NC * NC), x = e - k * NC * NC;
            if (li[i] >= 0) l[i] = gauge[((long(k >> 1) * 2 + (k & 1)) * Vh + lsite[i]) * NC * NC + x];
        }
    }
    __device__ __forceinline__ void store_links(C32 *lds, const C32 (&l)[LI]) const {
#pragma unroll
        for (int i = 0; i < LI; ++i)
            if (li[i] >= 0) lds[int(threadIdx.x) + 256 * i] = l[i];
    }
    // right-hand sides past R repeat the last one
    template <typename CS>
    __device__ __forceinline__ void load_spinors(CS (&v)[IT][NC], const CS *__restrict__ in, int R, int r0) const {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const CS *src = in + ((long(nb[i]) * 4 + (max(ks[i], 0) & 3)) * NC) * R + min(r0 + rr[i], R - 1);
#pragma unroll
            for (int b = 0; b < NC; ++b) v[i][b] = src[b * R];
        }
    }
    // rows u_(k,s) = V_k v into u[(4 k + s) * words + 2 col], col = colour * rc + rhs
    template <typename CS>
    __device__ __forceinline__ void transport(float *u, int words, const CS (&v)[IT][NC], const C32 *links, int rc,
                                              int zero_from) const {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            if (ks[i] < 0) continue;
            const int k = ks[i] >> 2;
            const bool fwd = (k & 1) == 0;
            const C32 *U = links + k * NC * NC;
            C32 p[NC];
#pragma unroll
            for (int b = 0; b < NC; ++b) {
                p[b] = load_cx<float>(&v[i][b]);
                if (rr[i] >= zero_from) p[b] = {0.f, 0.f};
            }
            float *dst = u + ks[i] * words + 2 * rr[i];
#pragma unroll
            for (int a = 0; a < NC; ++a) {
                C32 acc = {0.f, 0.f};
#pragma unroll
                for (int b = 0; b < NC; ++b) {
                    C32 l = U[fwd ? a * NC + b : b * NC + a];
                    if (!fwd) l.im = -l.im;
                    cfma(acc, l, p[b]);
                }
                *reinterpret_cast<f32x2 *>(dst + 2 * a * rc) = f32x2{acc.re, acc.im};
            }
        }
    }
};

// columns past NC rc up to `cols` hold zeros (never written by transport)
template <int NC>
__device__ __forceinline__ void zero_padding(float *u, int words, int rc, int cols) {
    const int pad = cols - NC * rc;
    for (int i = threadIdx.x; i < 32 * pad; i += 256) {
        const int row = i / pad, c = NC * rc + i - row * pad;
        *reinterpret_cast<f32x2 *>(u + row * words + 2 * c) = f32x2{0.f, 0.f};
    }
}

template <typename CS, int NC, int NT, int IT>  // NT tiles of 16 columns, IT items per thread
__global__ __launch_bounds__(256) void k_lgnn_mix32(C32 *__restrict__ q, const CS *__restrict__ in,
                                                   const C32 *__restrict__ gauge, const C32 *__restrict__ mcol,
                                                   const int *__restrict__ walk, int Vh, int R, int rc, int sites,
                                                   long fsize) {
    constexpr int words = row_words(16 * NT);
    __shared__ __align__(16) float u[32 * words];
    __shared__ __align__(16) C32 links[8 * NC * NC];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int r0 = rc * int(blockIdx.y);
    // A operand: real row 16 w + m = (complex row, re | im), k = 4 t + g = (complex column, re | im)
    float a[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const C32 c = mcol[(8 * w + (m >> 1)) * 32 + 2 * t + (g >> 1)];
        const int rho = m & 1, sig = g & 1;
        a[t] = rho == sig ? c.re : (rho == 0 ? -c.im : c.im);
    }
    Items<NC, IT> it(rc);
    // where this lane's columns 16 ct + m go (negative: nowhere)
    int col_off[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
        const int col = 16 * ct + m, c = col / rc, r = r0 + col - c * rc;
        col_off[ct] = c < NC && r < R ? c * R + r : -1;
    }
    zero_padding<NC>(u, words, rc, 16 * NT);
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * sites, pos1 = min(pos0 + sites, Vh);
    if (pos0 >= pos1) return;
    CS v[IT][NC];
    C32 l[Items<NC, IT>::LI];
    it.indices(walk + long(pos0) * 9);
    it.load_spinors(v, in, R, r0);
    it.load_links(l, gauge, Vh);
    it.indices(walk + long(min(pos0 + 1, pos1 - 1)) * 9);
    for (int pos = pos0; pos < pos1; ++pos) {
        const int site = walk[long(pos) * 9];
        it.store_links(links, l);
        __syncthreads();  // also: every wavefront has read the last site's rows
        it.transport(u, words, v, links, rc, rc);
        __syncthreads();
        it.load_spinors(v, in, R, r0);  // the last trip loads its own site again
        it.load_links(l, gauge, Vh);
        it.indices(walk + long(min(pos + 2, pos1 - 1)) * 9);
        f32x4 d[NT];
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) d[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const float *b = u + (2 * t + (g >> 1)) * words + 2 * m + (g & 1);
#pragma unroll
            for (int ct = 0; ct < NT; ++ct) d[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[32 * ct], d[ct], 0, 0, 0);
        }
        // lane (m, g) holds complex rows 8 w + 2 g, + 1 of column 16 ct + m
        const int i0 = 8 * w + 2 * g;
        C32 *dst = q + (i0 >> 2) * fsize + ((long(site) * 4 + (i0 & 3)) * NC) * R;
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
            if (col_off[ct] >= 0) {
                auto *o = reinterpret_cast<f32x2 *>(dst + col_off[ct]);
                __builtin_nontemporal_store(f32x2{d[ct][0], d[ct][1]}, o);
                __builtin_nontemporal_store(f32x2{d[ct][2], d[ct][3]}, o + long(NC) * R);
            }
    }
}

// part[block][i * 32 + j] = sum over the block's even sites and columns of a_(i)(col) conj(u_(j)(col)),
// a_(k,s) = the transported dphi of hop k ^ 1 (the adjoint of hop k), u the transported w
template <int NC, int IT>
__global__ __launch_bounds__(256) void k_lgnn_gram(Cx<double> *__restrict__ part, const C32 *__restrict__ dphi,
                                                  const C32 *__restrict__ wf, const C32 *__restrict__ gauge,
                                                  const int *__restrict__ walk, int Vh, int R, int rc, int cols,
                                                  int sites) {
    extern __shared__ __align__(16) float lds[];
    const int words = row_words(cols);
    float *sa = lds, *su = lds + 32 * words;
    C32 *links = reinterpret_cast<C32 *>(su + 32 * words);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, g = lane >> 4, im = g & 1;
    const int r0 = rc * int(blockIdx.y);
    Items<NC, IT> it(rc);
    zero_padding<NC>(sa, words, rc, cols);
    zero_padding<NC>(su, words, rc, cols);
    f64x4 gr[2][2], gi[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) gr[x][y] = gi[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
    const int pos0 = xcd_remap(blockIdx.x, gridDim.x) * sites, pos1 = min(pos0 + sites, Vh);
    const int steps = (NC * rc + 1) / 2;
    C32 vd[IT][NC], vw[IT][NC];
    C32 l[Items<NC, IT>::LI];
    if (pos0 < pos1) {
        it.indices(walk + long(pos0) * 9);
        it.load_spinors(vd, dphi, R, r0);
        it.load_spinors(vw, wf, R, r0);
        it.load_links(l, gauge, Vh);
        it.indices(walk + long(min(pos0 + 1, pos1 - 1)) * 9);
    }
    for (int pos = pos0; pos < pos1; ++pos) {
        it.store_links(links, l);
        __syncthreads();  // also: every wavefront has read the last site's rows
        it.transport(sa, words, vd, links, rc, R - r0);
        it.transport(su, words, vw, links, rc, R - r0);
        __syncthreads();
        it.load_spinors(vd, dphi, R, r0);  // the last trip loads its own site again
        it.load_spinors(vw, wf, R, r0);
        it.load_links(l, gauge, Vh);
        it.indices(walk + long(min(pos + 2, pos1 - 1)) * 9);
        for (int st = w; st < steps; st += 4) {
            const int col = 2 * (2 * st + (g >> 1));
            double ar[2], ai[2], b[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                // G row (k, s) pairs with hop k ^ 1: LDS row ^ 4
                const f32x2 av = *reinterpret_cast<const f32x2 *>(sa + ((16 * x + m) ^ 4) * words + col);
                ar[x] = im ? av[1] : av[0];
                ai[x] = im ? -av[0] : av[1];
                b[x] = su[(16 * x + m) * words + col + im];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    gr[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[x], b[y], gr[x][y], 0, 0, 0);
                    gi[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[x], b[y], gi[x][y], 0, 0, 0);
                }
        }
    }
    __syncthreads();
    // sum the four wavefronts in order; lane (m, g) holds rows 16 x + g + 4 v, column 16 y + m
    double *red = reinterpret_cast<double *>(lds);  // [32][32] complex
    for (int k = 0; k < 4; ++k) {
        if (w == k)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        double *e = red + 2 * ((16 * x + g + 4 * v) * 32 + 16 * y + m);
                        e[0] = (k ? e[0] : 0.0) + gr[x][y][v];
                        e[1] = (k ? e[1] : 0.0) + gi[x][y][v];
                    }
        __syncthreads();
    }
    Cx<double> *out = part + (long(blockIdx.y) * gridDim.x + blockIdx.x) * 1040;
    for (int i = threadIdx.x; i < 1024; i += 256) out[i] = {red[2 * i], red[2 * i + 1]};
}

// most items per thread that a chunk of 64 columns can need
template <int NC>
constexpr int kMostItems = NC == 2 ? 4 : NC == 3 ? 3 : NC == 4 ? 2 : 1;

template <typename CS, int NC, int NT>
auto mix_kernel(int rc) {
    const int it = div_up(rc, 8);
    auto k = k_lgnn_mix32<CS, NC, NT, 1>;
    if constexpr (kMostItems<NC> >= 2) if (it == 2) k = k_lgnn_mix32<CS, NC, NT, 2>;
    if constexpr (kMostItems<NC> >= 3) if (it == 3) k = k_lgnn_mix32<CS, NC, NT, 3>;
    if constexpr (kMostItems<NC> >= 4) if (it == 4) k = k_lgnn_mix32<CS, NC, NT, 4>;
    return k;
}

template <typename CS, int NC>
hipError_t mix_nc(void *q, const void *in, const void *gauge, const C32 *mcol, const int *walk, const Geom &g, int R,
                  hipStream_t s) {
    const int rc = chunk_rhs(NC, R), nt = div_up(NC * rc, 16);
    // Several sites per workgroup share the fragments of M and overlap a site's loads with the last one's
    // products: up to 16 where eight workgroups per compute unit and chunk are left, up to 4 where two are (8^4,
    // SU(3), whole application with 1 site 87 us at 32 RHS and 61 at 16, with 4 sites 65 and 50; 8^3 x 16, 32 RHS
    // with 2 sites 109, with 4 97 us; 4^4, 64 RHS, which gets 1, 38.5 against 41 us with 4)
    const int sites = std::max({1, std::min(4, g.Vh / (2 * num_cus())), std::min(16, g.Vh / (8 * num_cus()))});
    const dim3 grid(div_up(g.Vh, sites), div_up(R, rc));
    // items per thread: one for 8 right-hand sides per chunk
    auto k = nt == 1 ? mix_kernel<CS, NC, 1>(rc) : nt == 2 ? mix_kernel<CS, NC, 2>(rc)
             : nt == 3 ? mix_kernel<CS, NC, 3>(rc) : mix_kernel<CS, NC, 4>(rc);
    hipLaunchKernelGGL(k, grid, dim3(256), 0, s, static_cast<C32 *>(q), static_cast<const CS *>(in),
                       static_cast<const C32 *>(gauge), mcol, walk, g.Vh, R, rc, sites, long(g.Vh) * 4 * NC * R);
    return hipGetLastError();
}

template <typename CS>
hipError_t mix_s(void *q, const void *in, const void *gauge, const C32 *mcol, const int *walk, const Geom &g, int Nc,
                 int R, hipStream_t s) {
    switch (Nc) {
        case 2: return mix_nc<CS, 2>(q, in, gauge, mcol, walk, g, R, s);
        case 3: return mix_nc<CS, 3>(q, in, gauge, mcol, walk, g, R, s);
        case 4: return mix_nc<CS, 4>(q, in, gauge, mcol, walk, g, R, s);
        case 8: return mix_nc<CS, 8>(q, in, gauge, mcol, walk, g, R, s);
        default: return hipErrorInvalidValue;
    }
}

template <int NC>
hipError_t gram_nc(Cx<double> *part, int max_blocks, int &blocks, const void *dphi, const void *w, const void *gauge,
                   const int *walk, const Geom &g, int R, hipStream_t s) {
    const int rc = chunk_rhs(NC, R), nch = div_up(R, rc);
    const int cols = div_up(NC * rc, 16) * 16;
    const int nb = std::max(1, std::min(max_blocks / nch, g.Vh));
    if (nb * nch > max_blocks) return hipErrorInvalidValue;
    const int sites = div_up(g.Vh, nb);
    blocks = nb * nch;
    const size_t lds = std::max(size_t(2) * 32 * row_words(cols) * sizeof(float) + 8 * NC * NC * sizeof(C32),
                                size_t(2048) * sizeof(double));
    const int it = div_up(rc, 8);
    auto k = k_lgnn_gram<NC, 1>;
    if constexpr (kMostItems<NC> >= 2) if (it == 2) k = k_lgnn_gram<NC, 2>;
    if constexpr (kMostItems<NC> >= 3) if (it == 3) k = k_lgnn_gram<NC, 3>;
    if constexpr (kMostItems<NC> >= 4) if (it == 4) k = k_lgnn_gram<NC, 4>;
    hipLaunchKernelGGL(k, dim3(nb, nch), dim3(256), lds, s, part, static_cast<const C32 *>(dphi),
                       static_cast<const C32 *>(w), static_cast<const C32 *>(gauge), walk, g.Vh, R, rc, cols, sites);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_lgnn_mix32(void *q, const void *in, int prec, const void *gauge, const Cx<float> *mcol,
                             const int *walk, const Geom &g, int Nc, int R, hipStream_t s) {
    if (R < 1 || !q || !in || !gauge || !mcol || !walk) return hipErrorInvalidValue;
    switch (prec) {
        case kDouble: return mix_s<Cx<double>>(q, in, gauge, mcol, walk, g, Nc, R, s);
        case kSingle: return mix_s<Cx<float>>(q, in, gauge, mcol, walk, g, Nc, R, s);
        case kHalf: return mix_s<Half2Store>(q, in, gauge, mcol, walk, g, Nc, R, s);
        case kBF16: return mix_s<Bf162Store>(q, in, gauge, mcol, walk, g, Nc, R, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_lgnn_gram(Cx<double> *part, int max_blocks, int &blocks, const void *dphi, const void *w,
                            const void *gauge, const int *walk, const Geom &g, int Nc, int R, hipStream_t s) {
    if (R < 1 || !part || !dphi || !w || !gauge || !walk) return hipErrorInvalidValue;
    switch (Nc) {
        case 2: return gram_nc<2>(part, max_blocks, blocks, dphi, w, gauge, walk, g, R, s);
        case 3: return gram_nc<3>(part, max_blocks, blocks, dphi, w, gauge, walk, g, R, s);
        case 4: return gram_nc<4>(part, max_blocks, blocks, dphi, w, gauge, walk, g, R, s);
        case 8: return gram_nc<8>(part, max_blocks, blocks, dphi, w, gauge, walk, g, R, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qcu
