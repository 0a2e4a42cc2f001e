// Radial edge embedding: the Bessel basis times the cutoff envelope,
//   f[e][k] = c(r_e) * (phi_k(r_e) - mu_k) / sigma_k,
//   phi_k(r) = sqrt(2 / r_cut) sin(k pi r / r_cut) / (r + eps),   k = 1 .. n,
// with c the cosine envelope 0.5 (cos(pi r / r_cut) + 1) or the polynomial one
// u(x) = (1 - x)^3 sum_{j<p} C(j+2, 2) x^j, x = r / r_cut (both 0 for r >= r_cut),
// as MACE combines them (src/molrep/embedding/radial.py:36-148,
// src/molrep/embedding/cutoff.py:23-161, src/molzoo/mace.py:180-182).  One
// thread per edge: r is read once, the n values are written as one row; the
// backward reads the row's gradient and writes dL/dr (basis terms in fp64).  The torch composition
// this replaces makes ~20 passes over the (E, n) values forward and backward.
//
// k_pair_features writes the whole input row of an edge model's two-body MLP instead: those n values,
// the type embeddings of the edge's two atoms, and the envelope on its own
// (src/molzoo/allegro.py:137-249).

#include "common.h"

namespace mnx {
namespace {

constexpr int kEmbThreads = 256;
constexpr int kEmbMaxRadial = 32;

struct EmbArgs {
    int n;
    float r_cut, eps, pref, w;  // pref = sqrt(2 / r_cut), w = pi / r_cut (rounded once, as the reference's buffers)
    int cutoff;    // 0 none, 1 cosine, 2 polynomial
    int exponent;  // polynomial envelope
    const float* mu;     // [n] or null (no shift / scale)
    const float* sigma;  // [n] or null
};

// envelope and its derivative with respect to r
__device__ __forceinline__ void envelope(float r, const EmbArgs& a, float& c, float& dc) {
    if (a.cutoff == 0) {
        c = 1.f;
        dc = 0.f;
        return;
    }
    if (!(r < a.r_cut)) {
        c = 0.f;
        dc = 0.f;
        return;
    }
    if (a.cutoff == 1) {
        float s, co;
        sincosf(float(M_PI) * (r / a.r_cut), &s, &co);
        c = 0.5f * (co + 1.f);
        dc = -0.5f * float(M_PI) / a.r_cut * s;
        return;
    }
    const float x = r / a.r_cut;
    const int p = a.exponent;
    // g(x) = sum_{j<p} C(j+2, 2) x^j and g'(x), Horner, highest coefficient first
    float g = float((p + 1) * p / 2), gp = 0.f;
    for (int j = p - 2; j >= 0; --j) {
        gp = fmaf(gp, x, g);
        g = fmaf(g, x, float((j + 2) * (j + 1) / 2));
    }
    const float om = 1.f - x;
    const float om2 = om * om;
    c = om2 * om * g;
    dc = (om2 * om * gp - 3.f * om2 * g) / a.r_cut;
}

__global__ void __launch_bounds__(kEmbThreads) k_bessel_cutoff(const float* __restrict__ r, int64_t E, EmbArgs a,
                                                               float* __restrict__ out) {
    const int64_t e = int64_t(blockIdx.x) * kEmbThreads + threadIdx.x;
    if (e >= E) return;
    const float re = r[e];
    float c, dc;
    envelope(re, a, c, dc);
    const float inv = 1.f / (re + a.eps);
    float* o = out + e * a.n;
    for (int k = 0; k < a.n; ++k) {
        float phi = a.pref * sinf(re * (float(k + 1) * a.w)) * inv;
        if (a.mu) phi = (phi - a.mu[k]) / a.sigma[k];
        o[k] = phi * c;
    }
}

// SUB lanes to an edge, each every SUB-th term.  One where the gradient's rows are the n values alone
// (bound by the fp64 sines, and the division and the envelope are per lane: 2.6M edges, n = 8: 80 us,
// with four lanes 115); four where they are the first columns of longer rows, which one lane to an edge
// read a cache line per lane and load (526k edges, 8 of 40 columns: 69 us, with four lanes 28).
template <int SUB>
__global__ void __launch_bounds__(kEmbThreads) k_bessel_cutoff_bwd(const float* __restrict__ r, int64_t E, EmbArgs a,
                                                                   const float* __restrict__ grad, int ld,
                                                                   const float* __restrict__ grad_u,
                                                                   float* __restrict__ grad_r) {
    const int64_t e = (int64_t(blockIdx.x) * kEmbThreads + threadIdx.x) / SUB;
    const int sub = threadIdx.x % SUB;
    if (e >= E) return;  // an edge's lanes leave together
    const float re = r[e];
    float c, dc;
    envelope(re, a, c, dc);
    // d/dr [pref sin(f r) / (r + eps)] = pref (f cos(f r) - sin(f r) / (r + eps)) / (r + eps): the two
    // terms cancel to ~(f r)^2 / 3 of their size for small f r (about 1e-5 at r = 1e-3 A), so the
    // basis and its derivative are evaluated in fp64 here
    const double rd = double(re), inv = 1.0 / (rd + double(a.eps));
    const float* g = grad + e * ld;
    double acc = grad_u && sub == 0 ? double(grad_u[e]) * double(dc) : 0.0;
    for (int k = sub; k < a.n; k += SUB) {
        const double f = double(float(k + 1) * a.w);
        double s, co;
        sincos(rd * f, &s, &co);
        double phi = double(a.pref) * s * inv;
        double dphi = double(a.pref) * (f * co - s * inv) * inv;
        if (a.mu) {
            phi = (phi - double(a.mu[k])) / double(a.sigma[k]);
            dphi = dphi / double(a.sigma[k]);
        }
        acc += double(g[k]) * (dphi * double(c) + phi * double(dc));
    }
#pragma unroll
    for (int m = 1; m < SUB; m *= 2) acc += __shfl_xor(acc, m);
    if (sub == 0) grad_r[e] = float(acc);
}

// Rows [n radial features | table[ti] | table[tj]] and the envelope u of each edge.
//
// Bound by the row writes: a workgroup evaluates its 64 edges' n values with every lane (LDS), then
// writes the 64 rows as one contiguous run, four floats to a lane where n and dim allow it (VEC).  A
// thread to an edge would write 160-byte rows a float at a time, and a lane to four columns would
// leave the sines to a fifth of each wavefront.  526k edges, n = 8, dim = 16: 31 us (84 MB), against
// 26 elementwise kernels, a row gather and a concatenation (200 us); the backward above replaces 45 kernels
// (290 us).  A type outside the table gives a row of NaN (and is never read).
template <bool VEC>
__global__ void __launch_bounds__(kEmbThreads) k_pair_features(const float* __restrict__ r,
                                                               const int64_t* __restrict__ ti,
                                                               const int64_t* __restrict__ tj, int64_t E, EmbArgs a,
                                                               const float* __restrict__ table, int64_t types,
                                                               int dim, float* __restrict__ out,
                                                               float* __restrict__ u) {
    constexpr int kEdges = 64;
    __shared__ __attribute__((aligned(16))) float f[kEdges * kEmbMaxRadial];
    const int64_t e0 = int64_t(blockIdx.x) * kEdges;
    const int ne = int(E - e0 < kEdges ? E - e0 : kEdges);
    for (int i = threadIdx.x; i < ne * a.n; i += kEmbThreads) {
        const int le = i / a.n, k = i - le * a.n;
        const float re = r[e0 + le];
        float c, dc;
        envelope(re, a, c, dc);
        float phi = a.pref * sinf(re * (float(k + 1) * a.w)) * (1.f / (re + a.eps));
        if (a.mu) phi = (phi - a.mu[k]) / a.sigma[k];
        f[i] = phi * c;
        if (k == 0) u[e0 + le] = c;
    }
    __syncthreads();
    constexpr int kPer = VEC ? 4 : 1;
    const int w = (a.n + 2 * dim) / kPer, nq = a.n / kPer, dq = dim / kPer;
    float* __restrict__ o = out + e0 * (a.n + 2 * dim);
    for (int i = threadIdx.x; i < ne * w; i += kEmbThreads) {
        const int le = i / w, q = i - le * w;
        if (q < nq) {
            if (VEC) reinterpret_cast<float4*>(o)[i] = reinterpret_cast<const float4*>(f)[le * nq + q];
            else o[i] = f[le * nq + q];
            continue;
        }
        const bool second = q >= nq + dq;
        const int64_t t = (second ? tj : ti)[e0 + le];
        const int64_t at = t * dq + (q - nq - (second ? dq : 0));
        const bool ok = t >= 0 && t < types;
        if (VEC) {
            const float bad = __builtin_nanf("");
            reinterpret_cast<float4*>(o)[i] =
                ok ? reinterpret_cast<const float4*>(table)[at] : make_float4(bad, bad, bad, bad);
        } else {
            o[i] = ok ? table[at] : __builtin_nanf("");
        }
    }
}

int check_args(int64_t E, int n, double r_cut, double eps, int cutoff, int exponent, const float* mu,
               const float* sigma) {
    MNX_REQUIRE(E >= 0 && E < (int64_t(1) << 40), "edge count out of range");
    MNX_REQUIRE(n >= 1 && n <= kEmbMaxRadial, "num_radial %d not in [1, %d]", n, kEmbMaxRadial);
    MNX_REQUIRE(r_cut > 0.0 && eps >= 0.0, "r_cut must be positive and eps non-negative");
    MNX_REQUIRE(cutoff >= 0 && cutoff <= 2, "cutoff kind %d not in {0 none, 1 cosine, 2 polynomial}", cutoff);
    MNX_REQUIRE(cutoff != 2 || (exponent >= 1 && exponent <= 64), "polynomial exponent %d not in [1, 64]", exponent);
    MNX_REQUIRE((mu == nullptr) == (sigma == nullptr), "mu and sigma must both be given or both be null");
    return MNX_OK;
}

EmbArgs make_args(int n, double r_cut, double eps, int cutoff, int exponent, const float* mu, const float* sigma) {
    return EmbArgs{n, float(r_cut), float(eps), float(sqrt(2.0 / r_cut)), float(M_PI / r_cut), cutoff, exponent, mu,
                   sigma};
}

}  // namespace
}  // namespace mnx

using namespace mnx;

extern "C" {

int mnx_bessel_cutoff_f32(const float* r, int64_t num_edges, int32_t num_radial, double r_cut, double eps,
                          const float* mu, const float* sigma, int32_t cutoff, int32_t exponent, float* out,
                          mnx_stream_t stream) {
    clear_error();
    int rc = check_args(num_edges, num_radial, r_cut, eps, cutoff, exponent, mu, sigma);
    if (rc) return rc;
    if (num_edges == 0) return MNX_OK;
    MNX_REQUIRE(r && out, "null pointer argument");
    hipLaunchKernelGGL(k_bessel_cutoff, dim3(unsigned(ceil_div(num_edges, kEmbThreads))), dim3(kEmbThreads), 0,
                       (hipStream_t)stream, r, num_edges,
                       make_args(num_radial, r_cut, eps, cutoff, exponent, mu, sigma), out);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

int mnx_bessel_cutoff_bwd_f32(const float* r, int64_t num_edges, int32_t num_radial, double r_cut, double eps,
                              const float* mu, const float* sigma, int32_t cutoff, int32_t exponent,
                              const float* grad, float* grad_r, mnx_stream_t stream) {
    clear_error();
    int rc = check_args(num_edges, num_radial, r_cut, eps, cutoff, exponent, mu, sigma);
    if (rc) return rc;
    if (num_edges == 0) return MNX_OK;
    MNX_REQUIRE(r && grad && grad_r, "null pointer argument");
    hipLaunchKernelGGL(k_bessel_cutoff_bwd<1>, dim3(unsigned(ceil_div(num_edges, kEmbThreads))), dim3(kEmbThreads), 0,
                       (hipStream_t)stream, r, num_edges,
                       make_args(num_radial, r_cut, eps, cutoff, exponent, mu, sigma), grad, num_radial,
                       static_cast<const float*>(nullptr), grad_r);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

int mnx_pair_features_f32(const float* r, const int64_t* ti, const int64_t* tj, int64_t num_edges, int32_t num_radial,
                          double r_cut, double eps, const float* mu, const float* sigma, int32_t cutoff,
                          int32_t exponent, const float* table, int64_t num_types, int32_t dim, float* out, float* u,
                          mnx_stream_t stream) {
    clear_error();
    int rc = check_args(num_edges, num_radial, r_cut, eps, cutoff, exponent, mu, sigma);
    if (rc) return rc;
    MNX_REQUIRE(num_types >= 0 && num_types < (int64_t(1) << 40) && dim >= 0 && dim <= 4096,
                "type table %lld x %d out of range", (long long)num_types, dim);
    if (num_edges == 0) return MNX_OK;
    MNX_REQUIRE(r && ti && tj && out && u && (table || num_types == 0 || dim == 0), "null pointer argument");
    const EmbArgs a = make_args(num_radial, r_cut, eps, cutoff, exponent, mu, sigma);
    const dim3 grid(unsigned(ceil_div(num_edges, 64)));
    if (num_radial % 4 == 0 && dim % 4 == 0 && ((uintptr_t)table | (uintptr_t)out) % 16 == 0)
        hipLaunchKernelGGL(k_pair_features<true>, grid, dim3(kEmbThreads), 0, (hipStream_t)stream, r, ti, tj,
                           num_edges, a, table, num_types, dim, out, u);
    else
        hipLaunchKernelGGL(k_pair_features<false>, grid, dim3(kEmbThreads), 0, (hipStream_t)stream, r, ti, tj,
                           num_edges, a, table, num_types, dim, out, u);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

int mnx_pair_features_bwd_f32(const float* r, int64_t num_edges, int32_t num_radial, double r_cut, double eps,
                              const float* mu, const float* sigma, int32_t cutoff, int32_t exponent, const float* grad,
                              int32_t row, const float* grad_u, float* grad_r, mnx_stream_t stream) {
    clear_error();
    int rc = check_args(num_edges, num_radial, r_cut, eps, cutoff, exponent, mu, sigma);
    if (rc) return rc;
    MNX_REQUIRE(row >= num_radial, "row length %d below num_radial %d", row, num_radial);
    if (num_edges == 0) return MNX_OK;
    MNX_REQUIRE(r && grad && grad_u && grad_r, "null pointer argument");
    hipLaunchKernelGGL(k_bessel_cutoff_bwd<4>, dim3(unsigned(ceil_div(num_edges, kEmbThreads / 4))), dim3(kEmbThreads), 0,
                       (hipStream_t)stream, r, num_edges,
                       make_args(num_radial, r_cut, eps, cutoff, exponent, mu, sigma), grad, row, grad_u, grad_r);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

}  // extern "C"
