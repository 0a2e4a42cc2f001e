// Particle-mesh Ewald on gfx950: B-spline charge spreading, reciprocal-space
// convolution with the energy sum, force / charge-derivative gathering, and the
// real-space pair sum.  The 3-D FFTs between spread and convolve (forward) and
// between convolve and gather (backward) are rocFFT transforms issued by the
// caller on the same stream (torch.fft on ROCm).
//
// Follows the reference's CPU op (src/molix/op/src/pme/pme_cpu.cpp) term by
// term: box inversion (:22-35), grid index and B-spline recursion (:37-91),
// spreading (:240-256), influence function and energy (:263-294), gather
// (:311-343), direct sum with exclusions (:95-164).  The reference's CUDA path
// (pme_cuda.cu:394,460) supports spline orders 4 and 5; these kernels take any
// order 3..8.  The spread is a gather over mesh bricks (no atomics, fixed
// summation order); the direct-space derivatives use fp32 / fp64 atomics, and
// energies are reduced deterministically in fp64.

#include <math.h>

#include <type_traits>

#include "common.h"
#include "scan.h"
#include "wave.h"

namespace mnx {
namespace {

constexpr int kMaxOrder = 8;

template <typename T>
struct Recip {
    T r[3][3];
};

template <typename T>
__device__ __forceinline__ Recip<T> invert_box(const T* __restrict__ b) {
    Recip<T> R;
    const T s = T(1) / (b[0] * b[4] * b[8]);
    R.r[0][0] = b[4] * b[8] * s;
    R.r[0][1] = 0;
    R.r[0][2] = 0;
    R.r[1][0] = -b[3] * b[8] * s;
    R.r[1][1] = b[0] * b[8] * s;
    R.r[1][2] = 0;
    R.r[2][0] = (b[3] * b[7] - b[4] * b[6]) * s;
    R.r[2][1] = -b[0] * b[7] * s;
    R.r[2][2] = b[0] * b[4] * s;
    return R;
}

// Grid origin index and fractional offset of one atom along each axis (pme_cpu.cpp:37-60).
// The index is clamped into [0, grid) so that a non-finite position cannot address
// memory outside the mesh (its weights are then non-finite, as in the reference).
template <typename T>
__device__ __forceinline__ void grid_coord(const T* __restrict__ pos, int64_t atom, const T* __restrict__ box,
                                           const Recip<T>& R, const int grid[3], int gidx[3], T frac[3]) {
    T p[3] = {pos[3 * atom], pos[3 * atom + 1], pos[3 * atom + 2]};
    for (int i = 2; i >= 0; --i) {
        const T sc = floor(p[i] * R.r[i][i]);
        for (int j = 0; j < 3; ++j) p[j] -= sc * box[3 * i + j];
    }
    for (int i = 0; i < 3; ++i) {
        T t = p[0] * R.r[0][i] + p[1] * R.r[1][i] + p[2] * R.r[2][i];
        t = (t - floor(t)) * grid[i];
        const int ti = int(t);
        frac[i] = t - ti;
        const int g = ti % grid[i];
        gidx[i] = g < 0 ? 0 : (g < grid[i] ? g : grid[i] - 1);
    }
}

// B-spline weights d and (when DD) derivatives dd of a fractional offset dr along one axis.
template <typename T, int ORDER, bool DD>
__device__ __forceinline__ void spline(T dr, T (&d)[ORDER], T (&dd)[ORDER]) {
    d[ORDER - 1] = 0;
    d[1] = dr;
    d[0] = 1 - dr;
#pragma unroll
    for (int j = 3; j < ORDER; ++j) {
        const T div = T(1) / (j - 1);
        d[j - 1] = div * dr * d[j - 2];
#pragma unroll
        for (int k = 1; k < j - 1; ++k) d[j - k - 1] = div * ((dr + k) * d[j - k - 2] + (j - k - dr) * d[j - k - 1]);
        d[0] = div * (1 - dr) * d[0];
    }
    if (DD) {
        dd[0] = -d[0];
#pragma unroll
        for (int j = 1; j < ORDER; ++j) dd[j] = d[j - 1] - d[j];
    }
    const T sc = T(1) / (ORDER - 1);
    d[ORDER - 1] = sc * dr * d[ORDER - 2];
#pragma unroll
    for (int j = 1; j < ORDER - 1; ++j)
        d[ORDER - j - 1] = sc * ((dr + j) * d[ORDER - j - 2] + (ORDER - j - dr) * d[ORDER - j - 1]);
    d[0] = sc * (1 - dr) * d[0];
}

// Calls f(integral_constant ORDER) for the order, 3..kMaxOrder.
template <typename F>
void with_order(int order, F&& f) {
    switch (order) {
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        default: f(std::integral_constant<int, kMaxOrder>{}); break;
    }
}

// ---------------------------------------------------------------------------
// Spreading as a gather over mesh bricks.  The mesh is cut into bricks of
// kBrick^3 points (the last brick along an axis may be partial).  Atoms are
// binned by the brick holding their spline origin, in ascending atom order
// inside each brick, as records of origin, offset and scaled charge.  One
// workgroup owns one brick: it goes through the records of the brick and of the
// bricks that precede it within order-1 points (cyclically), keeps those whose
// support reaches it (about one in six), evaluates their splines, one axis per
// thread, straight into the brick's 8 positions along that axis (zero outside
// the support), and sums them: each lane owns one (y, z) column of the brick,
// each of the four wavefronts takes every fourth atom, and the four partial sums
// are added in wave order and stored once.  No atomics, every mesh point written
// exactly once (no clearing pass), and a fixed summation order.
// Measured, 50k atoms on 128^3, order 6: 18.5 us, bound by the per-brick passes over records; 81 us
// when every brick evaluated the splines of all candidates and one thread looked up its sources.
// ---------------------------------------------------------------------------
constexpr int kBrick = 8;          // mesh points per brick edge (>= kMaxOrder - 1)
constexpr int kBrickThreads = 256;
constexpr int kBrickStage = 128;   // atoms summed per pass
constexpr int kAxisSrc = 3;        // source bricks per axis (see axis_sources)
static_assert(kBrick * kBrick == kWave, "one lane per (y, z) column of a brick");
static_assert(kBrickStage * 3 * kBrick >= kBrickThreads * kBrick, "reduction fits the staging area");

__device__ __forceinline__ int brick_of(const int gi[3], int nby, int nbz) {
    return ((gi[0] / kBrick) * nby + gi[1] / kBrick) * nbz + gi[2] / kBrick;
}

// An atom as the spread reads it: mesh origin, offset from it, charge x sqrt(coulomb).
template <typename T>
struct alignas(16) SpreadRec {
    int32_t g[3];
    int32_t pad;
    T frac[3];
    T qs;
};

template <typename T>
__global__ void k_bin_count(const T* __restrict__ pos, const T* __restrict__ box, int64_t n, int gx, int gy, int gz,
                            int nby, int nbz, int32_t* __restrict__ brick, int32_t* __restrict__ rank,
                            int32_t* __restrict__ counts) {
    const int64_t a = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (a >= n) return;
    const int G[3] = {gx, gy, gz};
    const Recip<T> R = invert_box<T>(box);
    int gi[3];
    T frac[3];
    grid_coord<T>(pos, a, box, R, G, gi, frac);
    const int b = brick_of(gi, nby, nbz);
    brick[a] = b;
    rank[a] = atomicAdd(counts + b, 1);
}

__global__ void k_bin_place(const int32_t* __restrict__ brick, int64_t n, const int32_t* __restrict__ ptr,
                            const int32_t* __restrict__ rank, int32_t* __restrict__ slots) {
    const int64_t a = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (a < n) slots[ptr[brick[a]] + rank[a]] = int32_t(a);
}

// Ascending atom order inside each brick: the atom in slot j moves to its rank within its brick, as
// a record.
template <typename T>
__global__ void k_bin_rank(const T* __restrict__ pos, const T* __restrict__ q, const T* __restrict__ box, int gx, int gy,
                           int gz, T sqrt_k, const int32_t* __restrict__ brick, const int32_t* __restrict__ ptr,
                           const int32_t* __restrict__ slots, int64_t n, SpreadRec<T>* __restrict__ recs) {
    const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int a = slots[j];
    const int b = brick[a];
    const int lo = ptr[b], hi = ptr[b + 1];
    int r = 0;
    for (int k = lo; k < hi; ++k) r += slots[k] < a;
    const int G[3] = {gx, gy, gz};
    const Recip<T> R = invert_box<T>(box);
    SpreadRec<T> rec;
    grid_coord<T>(pos, a, box, R, G, rec.g, rec.frac);
    rec.pad = 0;
    rec.qs = q[a] * sqrt_k;
    recs[lo + r] = rec;
}

// Bricks along one axis whose atoms reach destination brick b: b itself and the
// bricks before it (cyclically) covering the order-1 points ahead of b's first
// point.  Only the last brick of an axis can be partial, so three suffice.
__device__ __forceinline__ int axis_sources(int b, int nb, int G, int order, int out[kAxisSrc]) {
    int k = 0;
    out[k++] = b;
    int need = order - 1, cur = b;
    while (need > 0 && k < kAxisSrc) {
        cur = cur == 0 ? nb - 1 : cur - 1;
        if (cur == b) break;
        out[k++] = cur;
        need -= min(kBrick, G - cur * kBrick);
    }
    return k;
}

template <typename T, int ORDER>
__global__ void __launch_bounds__(kBrickThreads)
    k_spread_bricks(int gx, int gy, int gz, int nbx, int nby, int nbz, const int32_t* __restrict__ ptr,
                    const SpreadRec<T>* __restrict__ recs, T* __restrict__ grid) {
    constexpr int kSrc = kAxisSrc * kAxisSrc * kAxisSrc;
    __shared__ int s_src[kSrc + 1];      // first record of each source brick
    __shared__ int s_end[kSrc + 1];      // candidates up to and including it
    __shared__ int s_cnt[2][4];          // reaching candidates of each wavefront, this pass and the next
    __shared__ int s_rec[kBrickStage + kBrickThreads];  // records of the reaching atoms found
    __shared__ T s_w[kBrickStage][3 * kBrick];          // [x weights * q | y weights | z weights] per position
    const int bid = blockIdx.x;
    const int bz = bid % nbz, by = (bid / nbz) % nby, bx = bid / (nbz * nby);
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    int sx[kAxisSrc], sy[kAxisSrc], sz[kAxisSrc];
    const int nx = axis_sources(bx, nbx, gx, ORDER, sx);
    const int ny = axis_sources(by, nby, gy, ORDER, sy);
    const int nz = axis_sources(bz, nbz, gz, ORDER, sz);
    const int nsrc = nx * ny * nz;
    if (wave == 0) {
        // lane s: source brick s, in (x, y, z) source order
        int first = 0, len = 0;
        if (lane < nsrc) {
            const int ix = lane / (ny * nz), iy = (lane / nz) % ny, iz = lane % nz;
            auto pick = [](const int (&v)[kAxisSrc], int k) { return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]); };
            const int s = (pick(sx, ix) * nby + pick(sy, iy)) * nbz + pick(sz, iz);
            first = ptr[s];
            len = ptr[s + 1] - first;
        }
        int incl = len;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
            const int u = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += u;
        }
        if (lane <= kSrc) {
            s_src[lane] = first;
            s_end[lane] = incl;
        }
    }
    __syncthreads();
    const int total = s_end[nsrc - 1];
    const int G[3] = {gx, gy, gz};
    const int S[3] = {bx * kBrick, by * kBrick, bz * kBrick};
    // origin relative to the brick start along axis a, cyclically in (-G, brick size); the atom
    // reaches the brick along the axis iff that offset is > -ORDER
    auto relative = [&](int g, int a) {
        int r = g - S[a];
        r += r < 0 ? G[a] : 0;
        if (r >= min(kBrick, G[a] - S[a])) r -= G[a];
        return r;
    };
    // lane -> (y, z) column of the brick; acc[x] for its 8 points along x
    const int ly = lane >> 3, lz = lane & 7;
    T acc[kBrick];
    for (int x = 0; x < kBrick; ++x) acc[x] = 0;
    int held = 0;  // reaching atoms in s_rec
    for (int base = 0, pass = 0; base < total; base += kBrickThreads, ++pass) {
        // this thread's candidate: does its support reach the brick?
        int rec = -1;
        if (base + t < total) {
            int s = 0;  // sources that end at or before it
#pragma unroll
            for (int step = 16; step > 0; step >>= 1)
                if (s + step <= nsrc - 1 && s_end[s + step - 1] <= base + t) s += step;
            rec = s_src[s] + (base + t - (s ? s_end[s - 1] : 0));
            const SpreadRec<T>& r = recs[rec];
            if (!(relative(r.g[0], 0) > -ORDER && relative(r.g[1], 1) > -ORDER && relative(r.g[2], 2) > -ORDER)) rec = -1;
        }
        const uint64_t m = __ballot(rec >= 0);
        if (lane == 0) s_cnt[pass & 1][wave] = __popcll(m);
        __syncthreads();
        int at = held + __popcll(m & ((uint64_t(1) << lane) - 1));
        for (int w = 0; w < kBrickThreads / kWave; ++w) {
            const int c = s_cnt[pass & 1][w];
            if (w < wave) at += c;
            held += c;
        }
        if (rec >= 0) s_rec[at] = rec;
        const bool last = base + kBrickThreads >= total;
        __syncthreads();
        while (held >= kBrickStage || (last && held > 0)) {
            const int cnt = min(held, kBrickStage);
            // one axis of one atom per thread
            for (int e = t; e < 3 * cnt; e += kBrickThreads) {
                const int c = e / 3, a = e - 3 * c;
                const SpreadRec<T>& r = recs[s_rec[c]];
                const int rel = relative(a == 0 ? r.g[0] : (a == 1 ? r.g[1] : r.g[2]), a);
                const T fr = a == 0 ? r.frac[0] : (a == 1 ? r.frac[1] : r.frac[2]);
                const int period = a == 0 ? gx : (a == 1 ? gy : gz);
                T d[ORDER], dd[ORDER];
                spline<T, ORDER, false>(fr, d, dd);
                const T sc = a == 0 ? r.qs : T(1);
                T* w = &s_w[c][a * kBrick];
#pragma unroll
                for (int x = 0; x < kBrick; ++x) w[x] = 0;
#pragma unroll
                for (int k = 0; k < ORDER; ++k) {
                    const int x = rel + k, y = x - period;  // y: around a mesh shorter than brick + order
                    if (x >= 0 && x < kBrick) w[x] = sc * d[k];
                    if (y >= 0 && y < kBrick) w[y] = sc * d[k];
                }
            }
            __syncthreads();
            for (int c = wave; c < cnt; c += kBrickThreads / kWave) {
                const T wyz = s_w[c][kBrick + ly] * s_w[c][2 * kBrick + lz];
#pragma unroll
                for (int x = 0; x < kBrick; ++x) acc[x] += s_w[c][x] * wyz;
            }
            __syncthreads();
            // the atoms left over move to the front
            const int keep = held - cnt;
            const int moved = t < keep ? s_rec[cnt + t] : 0;
            __syncthreads();
            if (t < keep) s_rec[t] = moved;
            held = keep;
            __syncthreads();
        }
    }
    // the four waves' partial sums, added in wave order (reuses the staging area)
    T* red = &s_w[0][0];
    for (int x = 0; x < kBrick; ++x) red[(wave * kBrick + x) * kWave + lane] = acc[x];
    __syncthreads();
    for (int i = t; i < kBrick * kWave; i += kBrickThreads) {
        const int x = i / kWave, l = i % kWave;
        T v = red[x * kWave + l];
        for (int w = 1; w < kBrickThreads / kWave; ++w) v += red[(w * kBrick + x) * kWave + l];
        const int px = S[0] + x, py = S[1] + (l >> 3), pz = S[2] + (l & 7);
        if (px < gx && py < gy && pz < gz) grid[(int64_t(px) * gy + py) * gz + pz] = v;
    }
}

constexpr int kConvThreads = 256;

// In-place multiply of the half-spectrum grid by the influence function and the
// per-block energy partial sums (pme_cpu.cpp:263-294).
template <typename T>
__global__ void __launch_bounds__(kConvThreads) k_convolve(T* __restrict__ cgrid, const T* __restrict__ box, int gx,
                                                           int gy, int gz, double alpha, const void* __restrict__ xm,
                                                           const void* __restrict__ ym, const void* __restrict__ zm,
                                                           bool mods64, double* __restrict__ partials) {
    __shared__ double red[kConvThreads];
    const int zs = gz / 2 + 1;
    const int64_t total = int64_t(gx) * gy * zs;
    const int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double e = 0.0;
    if (idx < total) {
        // the influence function and the energy's terms in fp64, rounded once: the energy is a small
        // difference from the self term, where a factor common to all terms, rounded in T, shows
        double b64[9];
        for (int k = 0; k < 9; ++k) b64[k] = double(box[k]);
        const Recip<double> R = invert_box<double>(b64);
        // the mesh has fewer than 2^31 points
        const uint32_t i32 = uint32_t(idx), plane = uint32_t(gy) * zs;
        const int kx = int(i32 / plane);
        const uint32_t rem = i32 - uint32_t(kx) * plane;
        const int ky = int(rem / uint32_t(zs));
        const int kz = int(rem - uint32_t(ky) * zs);
        const int mx = kx < (gx + 1) / 2 ? kx : kx - gx;
        const int my = ky < (gy + 1) / 2 ? ky : ky - gy;
        const int mz = kz < (gz + 1) / 2 ? kz : kz - gz;
        const double mhx = mx * R.r[0][0];
        const double mhy = mx * R.r[1][0] + my * R.r[1][1];
        const double mhz = mx * R.r[2][0] + my * R.r[2][1] + mz * R.r[2][2];
        const double m2 = mhx * mhx + mhy * mhy + mhz * mhz;
        const double scale_f = M_PI * b64[0] * b64[4] * b64[8];
        // the moduli in T or (mods64) in double
        auto mod = [&](const void* m, int k) {
            return mods64 ? static_cast<const double*>(m)[k] : double(static_cast<const T*>(m)[k]);
        };
        const double denom = m2 * (scale_f * mod(xm, kx) * mod(ym, ky)) * mod(zm, kz);
        const double rexp = M_PI * M_PI / (alpha * alpha);
        const double eterm = idx == 0 ? 0.0 : exp(-rexp * m2) / denom;
        const double s = (kz > 0 && kz <= (gz - 1) / 2) ? 2.0 : 1.0;
        T* c = cgrid + 2 * idx;
        const double re = c[0], im = c[1];
        e = s * eterm * (re * re + im * im);
        c[0] = T(re * eterm);
        c[1] = T(im * eterm);
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int off = kConvThreads / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

// energy = scale * sum(partials) + sum(more), summed by one block in a fixed order.
template <typename T>
__global__ void __launch_bounds__(1024) k_sum_partials(const double* __restrict__ partials, int64_t n, double scale,
                                                       const double* __restrict__ more, int64_t nmore,
                                                       T* __restrict__ energy) {
    __shared__ double red[1024];
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) s += partials[i];
    s *= scale;
    for (int64_t i = threadIdx.x; i < nmore; i += 1024) s += more[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *energy = T(red[0]);
}

// d/dpos and d/dq of the reciprocal energy from the back-transformed grid (pme_cpu.cpp:311-343), plus
// the given derivatives (dpos_add, dq_add) when there are any, times *grad when it is given.
//
// ORDER^2 columns of ORDER consecutive mesh points per atom: L lanes share an atom (16 up to order
// 4, else 32), each taking whole columns; three of them evaluate the atom's splines, one axis each,
// into LDS.  (One thread per atom left 50k atoms on 782 wavefronts, each with 216 dependent loads.)
// Measured, 50k atoms on 128^3, order 6: 33 us (10.8 M mesh reads from L2), 88 us before.
constexpr int kGatherThreads = 256;

template <typename T, int ORDER>
__global__ void __launch_bounds__(kGatherThreads) k_gather(const T* __restrict__ pos, const T* __restrict__ q,
                                                           const T* __restrict__ box, int64_t n,
                                                           const T* __restrict__ grid, int gx, int gy, int gz, T sqrt_k,
                                                           const T* __restrict__ grad, const T* __restrict__ dpos_add,
                                                           const T* __restrict__ dq_add, T* __restrict__ dpos,
                                                           T* __restrict__ dq) {
    constexpr int L = ORDER <= 4 ? 16 : 32, ATOMS = kGatherThreads / L;
    __shared__ T s_w[ATOMS][3][2][ORDER];  // weights and derivatives
    const int slot = threadIdx.x / L, l = threadIdx.x % L;
    const int64_t atom = int64_t(blockIdx.x) * ATOMS + slot;
    const bool in = atom < n;
    const int G[3] = {gx, gy, gz};
    const Recip<T> R = invert_box<T>(box);
    int gi[3] = {0, 0, 0};
    if (in) {
        T frac[3];
        grid_coord<T>(pos, atom, box, R, G, gi, frac);
        if (l < 3) {
            T d[ORDER], dd[ORDER];
            spline<T, ORDER, true>(l == 0 ? frac[0] : (l == 1 ? frac[1] : frac[2]), d, dd);
#pragma unroll
            for (int k = 0; k < ORDER; ++k) {
                s_w[slot][l][0][k] = d[k];
                s_w[slot][l][1][k] = dd[k];
            }
        }
    }
    __syncthreads();
    T p0 = 0, p1 = 0, p2 = 0, s = 0;
    if (in) {
        T wz[ORDER], dz[ORDER];
        int oz[ORDER];
#pragma unroll
        for (int k = 0; k < ORDER; ++k) {
            wz[k] = s_w[slot][2][0][k];
            dz[k] = s_w[slot][2][1][k];
            oz[k] = gi[2] + k < gz ? gi[2] + k : gi[2] + k - gz;
        }
#pragma unroll
        for (int c0 = 0; c0 < ORDER * ORDER; c0 += L) {
            const int c = c0 + l;
            if (c < ORDER * ORDER) {
                const int ix = c / ORDER, iy = c - ix * ORDER;
                const int x = gi[0] + ix < gx ? gi[0] + ix : gi[0] + ix - gx;
                const int y = gi[1] + iy < gy ? gi[1] + iy : gi[1] + iy - gy;
                const T* row = grid + (int64_t(x) * gy + y) * gz;
                T v = 0, dv = 0;
#pragma unroll
                for (int k = 0; k < ORDER; ++k) {
                    const T g = row[oz[k]];
                    v += wz[k] * g;
                    dv += dz[k] * g;
                }
                const T wx = s_w[slot][0][0][ix], dx = s_w[slot][0][1][ix], wy = s_w[slot][1][0][iy],
                        dy = s_w[slot][1][1][iy];
                p0 += dx * wy * v;
                p1 += wx * dy * v;
                p2 += wx * wy * dv;
                s += wx * wy * v;
            }
        }
    }
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) {
        p0 += __shfl_xor(p0, o, kWave);
        p1 += __shfl_xor(p1, o, kWave);
        p2 += __shfl_xor(p2, o, kWave);
        s += __shfl_xor(s, o, kWave);
    }
    if (!in || l) return;
    const T sc = q[atom] * sqrt_k;
    T f[3] = {sc * (p0 * gx * R.r[0][0]), sc * (p0 * gx * R.r[1][0] + p1 * gy * R.r[1][1]),
              sc * (p0 * gx * R.r[2][0] + p1 * gy * R.r[2][1] + p2 * gz * R.r[2][2])};
    T fq = s * sqrt_k;
    if (dpos_add) {
        for (int k = 0; k < 3; ++k) f[k] += dpos_add[3 * atom + k];
        fq += dq_add[atom];
    }
    if (grad) {
        const T w = *grad;
        for (int k = 0; k < 3; ++k) f[k] *= w;
        fq *= w;
    }
    for (int k = 0; k < 3; ++k) dpos[3 * atom + k] = f[k];
    dq[atom] = fq;
}

// Block-wide fp64 sum of one value per thread into partials[blockIdx.x].
__device__ __forceinline__ void block_partial(double e, double* __restrict__ partials) {
    __shared__ double red[kConvThreads];
    red[threadIdx.x] = e;
    __syncthreads();
    for (int off = kConvThreads / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

// Real-space pair sum over the given pair list minus excluded pairs (pme_cpu.cpp:110-135).
// GRAD: also dE/dq and dE/dpos (pme_cpu.cpp:195-215).  Pair lists come grouped by
// their first atom (the neighbor list's row order), so the first atom's four
// derivative terms are summed over each run of equal rows in the wavefront and
// added once per run; the second atom's terms are added per pair.  Each pair's
// terms are evaluated in fp64 whatever the storage type (erfc/exp/division in
// double cost nothing next to the pair list's memory latency), so the fp32 path
// differs from an fp64 evaluation only by its rounded inputs and the fp32
// accumulation of the derivatives.
template <typename T, bool GRAD>
__global__ void __launch_bounds__(kConvThreads) k_direct_pairs(const T* __restrict__ q, int64_t n,
                                                               const int32_t* __restrict__ nb, int64_t P, const T* __restrict__ dl,
                                                               const T* __restrict__ r, const int32_t* __restrict__ excl,
                                                               int max_excl, double alpha, double coulomb,
                                                               T* __restrict__ dpos, T* __restrict__ dq,
                                                               double* __restrict__ partials) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double e = 0.0;
    int row = -1;
    double g1[4] = {0, 0, 0, 0};  // d/dq and d/dpos of the pair's first atom
    if (i < P) {
        const int a1 = nb[i], a2 = nb[P + i];
        // -1 marks padding (reference); any other out-of-range index is skipped too
        bool include = a1 > -1 && a1 < n && a2 >= 0 && a2 < n;
        if (include) row = a1;
        for (int j = 0; include && j < max_excl && excl[int64_t(a1) * max_excl + j] >= a2; ++j)
            if (excl[int64_t(a1) * max_excl + j] == a2) include = false;
        if (include) {
            const double rr = double(r[i]);
            const double inv = 1.0 / rr;
            const double ar = alpha * rr;
            const double ec = erfc(ar);
            const double pref = coulomb * inv;
            const double c1 = double(q[a1]), c2 = double(q[a2]);
            e = pref * ec * c1 * c2;
            if (GRAD) {
                const double ex = exp(-ar * ar);
                const double dedr = pref * c1 * c2 * (ec + ar * ex * M_2_SQRTPI) * inv * inv;
                g1[0] = pref * ec * c2;
                atomicAdd(dq + a2, T(pref * ec * c1));
                for (int k = 0; k < 3; ++k) {
                    const double f = dedr * double(dl[3 * i + k]);
                    g1[1 + k] = -f;
                    atomicAdd(dpos + 3 * a2 + k, T(f));
                }
            }
        }
    }
    if (GRAD) {
        if (run_reduce<double, 4>(row, g1) && row >= 0) {
            atomicAdd(dq + row, T(g1[0]));
            for (int k = 0; k < 3; ++k) atomicAdd(dpos + 3 * row + k, T(g1[1 + k]));
        }
    }
    block_partial(e, partials);
}

// Excluded pairs' erf term, removed from the reciprocal-space sum (pme_cpu.cpp:137-162).
// One thread per atom a; a's own derivative terms are summed over its exclusions
// and added once.  Pair terms in fp64 as above.
template <typename T, bool GRAD>
__global__ void __launch_bounds__(kConvThreads) k_direct_excl(const T* __restrict__ pos, const T* __restrict__ q,
                                                              int64_t n, const int32_t* __restrict__ excl,
                                                              int max_excl, double alpha, double coulomb,
                                                              T* __restrict__ dpos, T* __restrict__ dq,
                                                              double* __restrict__ partials) {
    const int64_t a = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    double e = 0.0;
    if (a < n) {
        double ga[4] = {0, 0, 0, 0};
        for (int j = 0; j < max_excl; ++j) {
            const int b = excl[a * max_excl + j];
            if (!(b > a)) break;
            if (b >= n) continue;
            double dr[3];
            for (int k = 0; k < 3; ++k) dr[k] = double(pos[3 * a + k]) - double(pos[3 * int64_t(b) + k]);
            const double rr = sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
            const double inv = 1.0 / rr;
            const double ar = alpha * rr;
            const double ef = erf(ar);
            const double pref = coulomb * inv;
            const double c1 = double(q[a]), c2 = double(q[b]);
            e -= pref * ef * c1 * c2;
            if (GRAD) {
                const double ex = exp(-ar * ar);
                const double dedr = pref * c1 * c2 * (ef - ar * ex * M_2_SQRTPI) * inv * inv;
                ga[0] -= pref * ef * c2;
                atomicAdd(dq + b, T(-pref * ef * c1));
                for (int k = 0; k < 3; ++k) {
                    ga[1 + k] += dedr * dr[k];
                    atomicAdd(dpos + 3 * int64_t(b) + k, T(-dedr * dr[k]));
                }
            }
        }
        if (GRAD && max_excl > 0) {
            atomicAdd(dq + a, T(ga[0]));
            for (int k = 0; k < 3; ++k) atomicAdd(dpos + 3 * a + k, T(ga[1 + k]));
        }
    }
    block_partial(e, partials);
}

template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = T(0);
}

int check_grid(int gx, int gy, int gz, int order) {
    MNX_REQUIRE(gx > 0 && gy > 0 && gz > 0 && int64_t(gx) * gy * gz < (int64_t(1) << 31), "bad grid size");
    MNX_REQUIRE(order >= 3 && order <= kMaxOrder, "spline order %d not in [3, %d]", order, kMaxOrder);
    MNX_REQUIRE(gx >= order && gy >= order && gz >= order, "grid smaller than the spline order");
    return MNX_OK;
}

struct BrickWs {
    int32_t *counts, *ptr, *tiles, *brick, *rank, *slots;
    void* recs;  // SpreadRec<T>
};

BrickWs carve_bricks(void* base, int64_t n, int64_t nbricks, size_t* used) {
    Workspace ws{static_cast<char*>(base), 0};
    BrickWs w;
    w.counts = ws.take<int32_t>(nbricks + 1);
    w.ptr = ws.take<int32_t>(nbricks + 1);
    w.tiles = ws.take<int32_t>(scan_workspace_elems(nbricks + 1));
    w.brick = ws.take<int32_t>(n);
    w.rank = ws.take<int32_t>(n);
    w.slots = ws.take<int32_t>(n);
    w.recs = ws.take<SpreadRec<double>>(n);
    *used = ws.used;
    return w;
}

int64_t brick_count(int g) { return ceil_div(g, kBrick); }

size_t spread_ws(int64_t n, int gx, int gy, int gz) {
    size_t used = 0;
    carve_bricks(nullptr, n > 0 ? n : 0, brick_count(gx) * brick_count(gy) * brick_count(gz), &used);
    return used + 256;
}

template <typename T>
int spread(const T* pos, const T* q, const T* box, int64_t n, int gx, int gy, int gz, int order, double coulomb,
           T* grid, void* ws, size_t ws_bytes, hipStream_t s) {
    clear_error();
    int rc = check_grid(gx, gy, gz, order);
    if (rc) return rc;
    MNX_REQUIRE(n >= 0 && n < (int64_t(1) << 31), "atom count out of range");
    MNX_REQUIRE(grid && box && (n == 0 || (pos && q)), "null pointer argument");
    const int nbx = int(brick_count(gx)), nby = int(brick_count(gy)), nbz = int(brick_count(gz));
    const int64_t nbricks = int64_t(nbx) * nby * nbz;
    size_t need = 0;
    BrickWs w = carve_bricks(ws, n, nbricks, &need);
    if (!ws || ws_bytes < need) return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
    const int tb = 256;
    hipLaunchKernelGGL((k_fill<int32_t>), dim3(ceil_div(nbricks + 1, tb)), dim3(tb), 0, s, w.counts, nbricks + 1);
    MNX_CHECK_LAUNCH();
    if (n > 0) {
        hipLaunchKernelGGL((k_bin_count<T>), dim3(ceil_div(n, tb)), dim3(tb), 0, s, pos, box, n, gx, gy, gz, nby, nbz,
                           w.brick, w.rank, w.counts);
        MNX_CHECK_LAUNCH();
    }
    rc = exclusive_scan<int32_t, int32_t>(w.counts, nbricks + 1, w.ptr, w.tiles, (int32_t*)nullptr, s);
    if (rc) return rc;
    SpreadRec<T>* recs = static_cast<SpreadRec<T>*>(w.recs);
    if (n > 0) {
        hipLaunchKernelGGL(k_bin_place, dim3(ceil_div(n, tb)), dim3(tb), 0, s, w.brick, n, w.ptr, w.rank, w.slots);
        MNX_CHECK_LAUNCH();
        hipLaunchKernelGGL((k_bin_rank<T>), dim3(ceil_div(n, tb)), dim3(tb), 0, s, pos, q, box, gx, gy, gz,
                           T(sqrt(coulomb)), w.brick, w.ptr, w.slots, n, recs);
        MNX_CHECK_LAUNCH();
    }
    with_order(order, [&](auto o) {
        hipLaunchKernelGGL((k_spread_bricks<T, decltype(o)::value>), dim3(nbricks), dim3(kBrickThreads), 0, s, gx, gy, gz,
                           nbx, nby, nbz, w.ptr, recs, grid);
    });
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

int64_t conv_blocks(int gx, int gy, int gz) { return ceil_div(int64_t(gx) * gy * (gz / 2 + 1), kConvThreads); }

template <typename T>
int convolve(T* cgrid, const T* box, int gx, int gy, int gz, double alpha, const void* xm, const void* ym, const void* zm,
             bool mods64, double coulomb, const double* more, int64_t nmore, T* energy, void* ws, size_t ws_bytes,
             hipStream_t s) {
    clear_error();
    int rc = check_grid(gx, gy, gz, 3);
    MNX_REQUIRE(rc || nmore == 0 || more, "null pointer argument");
    if (rc) return rc;
    MNX_REQUIRE(cgrid && box && xm && ym && zm && energy, "null pointer argument");
    const int64_t nb = conv_blocks(gx, gy, gz);
    if (!ws || ws_bytes < size_t(nb) * sizeof(double))
        return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, size_t(nb) * sizeof(double));
    double* part = static_cast<double*>(ws);
    // the mesh holds charges times sqrt(coulomb) rounded to T: a factor common to all terms, so taken out
    // of the sum (energy error of 50k atoms in float32, six inputs: 0.8e-6..5.8e-6 -> 0.7e-6..4.7e-6)
    const double sk = double(T(sqrt(coulomb))), fix = sk > 0 ? coulomb / (sk * sk) : 1.0;
    hipLaunchKernelGGL((k_convolve<T>), dim3(nb), dim3(kConvThreads), 0, s, cgrid, box, gx, gy, gz, alpha, xm, ym,
                       zm, mods64, part);
    MNX_CHECK_LAUNCH();
    hipLaunchKernelGGL((k_sum_partials<T>), dim3(1), dim3(1024), 0, s, part, nb, 0.5 * fix, more, nmore, energy);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

template <typename T>
int gather(const T* pos, const T* q, const T* box, int64_t n, const T* grid, int gx, int gy, int gz, int order,
           double coulomb, const T* grad, const T* dpos_add, const T* dq_add, T* dpos, T* dq, hipStream_t s) {
    clear_error();
    int rc = check_grid(gx, gy, gz, order);
    if (rc) return rc;
    if (n == 0) return MNX_OK;
    MNX_REQUIRE(pos && q && box && grid && dpos && dq, "null pointer argument");
    MNX_REQUIRE((dpos_add == nullptr) == (dq_add == nullptr), "dpos_add and dq_add must both be given or both be null");
    with_order(order, [&](auto o) {
        constexpr int kOrder = decltype(o)::value, kAtoms = kGatherThreads / (kOrder <= 4 ? 16 : 32);
        hipLaunchKernelGGL((k_gather<T, kOrder>), dim3(ceil_div(n, kAtoms)), dim3(kGatherThreads), 0, s, pos, q, box, n,
                           grid, gx, gy, gz, T(sqrt(coulomb)), grad, dpos_add, dq_add, dpos, dq);
    });
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

size_t direct_ws(int64_t n, int64_t P) { return size_t(ceil_div(P > 0 ? P : 1, kConvThreads) + ceil_div(n > 0 ? n : 1, kConvThreads)) * sizeof(double); }

template <typename T, bool GRAD>
void launch_direct(const T* pos, const T* q, int64_t n, const int32_t* nb, int64_t P, const T* deltas, const T* dist,
                   const int32_t* excl, int max_excl, double alpha, double coulomb, T* dpos, T* dq, double* part,
                   int64_t b1, int64_t b2, hipStream_t s) {
    if (b1 > 0)
        hipLaunchKernelGGL((k_direct_pairs<T, GRAD>), dim3(b1), dim3(kConvThreads), 0, s, q, n, nb, P, deltas, dist,
                           excl, max_excl, alpha, coulomb, dpos, dq, part);
    if (b2 > 0)
        hipLaunchKernelGGL((k_direct_excl<T, GRAD>), dim3(b2), dim3(kConvThreads), 0, s, pos, q, n, excl, max_excl,
                           alpha, coulomb, dpos, dq, part + b1);
}

template <typename T>
int direct(const T* pos, const T* q, int64_t n, const int32_t* nb, int64_t P, const T* deltas, const T* dist,
           const int32_t* excl, int max_excl, double alpha, double coulomb, T* energy, T* dpos, T* dq, void* ws,
           size_t ws_bytes, hipStream_t s) {
    clear_error();
    MNX_REQUIRE(n >= 0 && P >= 0 && max_excl >= 0, "sizes out of range");
    MNX_REQUIRE(energy && (n == 0 || (pos && q)), "null pointer argument");
    MNX_REQUIRE((dpos == nullptr) == (dq == nullptr), "dpos and dq must both be given or both be null");
    MNX_REQUIRE(max_excl == 0 || excl, "exclusions pointer is null");
    MNX_REQUIRE(P == 0 || (nb && deltas && dist), "null pair-list pointer");
    if (!ws || ws_bytes < direct_ws(n, P)) return set_error(MNX_ERR_WORKSPACE, "workspace too small");
    double* part = static_cast<double*>(ws);
    const int64_t b1 = P > 0 ? ceil_div(P, kConvThreads) : 0;
    const int64_t b2 = (n > 0 && max_excl > 0) ? ceil_div(n, kConvThreads) : 0;
    const bool grad = dpos != nullptr;
    if (grad && n > 0) {
        hipLaunchKernelGGL((k_fill<T>), dim3(ceil_div(3 * n, 256)), dim3(256), 0, s, dpos, 3 * n);
        MNX_CHECK_LAUNCH();
        hipLaunchKernelGGL((k_fill<T>), dim3(ceil_div(n, 256)), dim3(256), 0, s, dq, n);
        MNX_CHECK_LAUNCH();
    }
    if (grad)
        launch_direct<T, true>(pos, q, n, nb, P, deltas, dist, excl, max_excl, alpha, coulomb, dpos, dq, part, b1, b2,
                               s);
    else
        launch_direct<T, false>(pos, q, n, nb, P, deltas, dist, excl, max_excl, alpha, coulomb, dpos, dq, part, b1,
                                b2, s);
    MNX_CHECK_LAUNCH();
    // every launched block wrote its partial; with no blocks the energy is 0
    hipLaunchKernelGGL((k_sum_partials<T>), dim3(1), dim3(1024), 0, s, part, b1 + b2, 1.0,
                       (const double*)nullptr, int64_t(0), energy);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

}  // namespace
}  // namespace mnx

using namespace mnx;

extern "C" {

size_t mnx_pme_spread_workspace_bytes(int64_t n, int32_t gx, int32_t gy, int32_t gz) {
    return spread_ws(n, gx > 0 ? gx : 1, gy > 0 ? gy : 1, gz > 0 ? gz : 1);
}
int mnx_pme_spread_f32(const float* pos, const float* q, const float* box, int64_t n, int32_t gx, int32_t gy,
                       int32_t gz, int32_t order, double coulomb, float* grid, void* ws, size_t ws_bytes,
                       mnx_stream_t s) {
    return spread<float>(pos, q, box, n, gx, gy, gz, order, coulomb, grid, ws, ws_bytes, (hipStream_t)s);
}
int mnx_pme_spread_f64(const double* pos, const double* q, const double* box, int64_t n, int32_t gx, int32_t gy,
                       int32_t gz, int32_t order, double coulomb, double* grid, void* ws, size_t ws_bytes,
                       mnx_stream_t s) {
    return spread<double>(pos, q, box, n, gx, gy, gz, order, coulomb, grid, ws, ws_bytes, (hipStream_t)s);
}
size_t mnx_pme_convolve_workspace_bytes(int32_t gx, int32_t gy, int32_t gz) {
    return size_t(conv_blocks(gx, gy, gz)) * sizeof(double) + 256;
}
int mnx_pme_convolve_f32(float* cgrid, const float* box, int32_t gx, int32_t gy, int32_t gz, double alpha,
                         const float* xm, const float* ym, const float* zm, float* energy, void* ws, size_t ws_bytes,
                         mnx_stream_t s) {
    return convolve<float>(cgrid, box, gx, gy, gz, alpha, xm, ym, zm, false, 1.0, nullptr, 0, energy, ws, ws_bytes, (hipStream_t)s);
}
int mnx_pme_convolve_f64(double* cgrid, const double* box, int32_t gx, int32_t gy, int32_t gz, double alpha,
                         const double* xm, const double* ym, const double* zm, double* energy, void* ws,
                         size_t ws_bytes, mnx_stream_t s) {
    return convolve<double>(cgrid, box, gx, gy, gz, alpha, xm, ym, zm, false, 1.0, nullptr, 0, energy, ws, ws_bytes, (hipStream_t)s);
}
int mnx_pme_gather_f32(const float* pos, const float* q, const float* box, int64_t n, const float* grid, int32_t gx,
                       int32_t gy, int32_t gz, int32_t order, double coulomb, float* dpos, float* dq, mnx_stream_t s) {
    return gather<float>(pos, q, box, n, grid, gx, gy, gz, order, coulomb, nullptr, nullptr, nullptr, dpos, dq, (hipStream_t)s);
}
int mnx_pme_gather_f64(const double* pos, const double* q, const double* box, int64_t n, const double* grid,
                       int32_t gx, int32_t gy, int32_t gz, int32_t order, double coulomb, double* dpos, double* dq,
                       mnx_stream_t s) {
    return gather<double>(pos, q, box, n, grid, gx, gy, gz, order, coulomb, nullptr, nullptr, nullptr, dpos, dq, (hipStream_t)s);
}
size_t mnx_pme_direct_workspace_bytes(int64_t n, int64_t num_pairs) { return direct_ws(n, num_pairs) + 256; }
int mnx_pme_direct_f32(const float* pos, const float* q, int64_t n, const int32_t* neighbors, int64_t num_pairs,
                       const float* deltas, const float* distances, const int32_t* exclusions, int32_t max_excl,
                       double alpha, double coulomb, float* energy, float* dpos, float* dq, void* ws,
                       size_t ws_bytes, mnx_stream_t s) {
    return direct<float>(pos, q, n, neighbors, num_pairs, deltas, distances, exclusions, max_excl, alpha, coulomb,
                         energy, dpos, dq, ws, ws_bytes, (hipStream_t)s);
}
int mnx_pme_direct_f64(const double* pos, const double* q, int64_t n, const int32_t* neighbors, int64_t num_pairs,
                       const double* deltas, const double* distances, const int32_t* exclusions, int32_t max_excl,
                       double alpha, double coulomb, double* energy, double* dpos, double* dq, void* ws,
                       size_t ws_bytes, mnx_stream_t s) {
    return direct<double>(pos, q, n, neighbors, num_pairs, deltas, distances, exclusions, max_excl, alpha, coulomb,
                          energy, dpos, dq, ws, ws_bytes, (hipStream_t)s);
}

int mnx_pme_convolve_add_f32(float* cgrid, const float* box, int32_t gx, int32_t gy, int32_t gz, double alpha,
                             const void* xm, const void* ym, const void* zm, int32_t mods64, double coulomb,
                             const double* more, int64_t nmore, float* energy, void* ws, size_t ws_bytes, mnx_stream_t s) {
    return convolve<float>(cgrid, box, gx, gy, gz, alpha, xm, ym, zm, mods64 != 0, coulomb, more, nmore, energy, ws, ws_bytes,
                           (hipStream_t)s);
}
int mnx_pme_gather_add_f32(const float* pos, const float* q, const float* box, int64_t n, const float* grid, int32_t gx,
                           int32_t gy, int32_t gz, int32_t order, double coulomb, const float* grad, const float* dpos_add,
                           const float* dq_add, float* dpos, float* dq, mnx_stream_t s) {
    return gather<float>(pos, q, box, n, grid, gx, gy, gz, order, coulomb, grad, dpos_add, dq_add, dpos, dq, (hipStream_t)s);
}
int mnx_pme_convolve_add_f64(double* cgrid, const double* box, int32_t gx, int32_t gy, int32_t gz, double alpha,
                             const void* xm, const void* ym, const void* zm, int32_t mods64, double coulomb,
                             const double* more, int64_t nmore, double* energy, void* ws, size_t ws_bytes, mnx_stream_t s) {
    return convolve<double>(cgrid, box, gx, gy, gz, alpha, xm, ym, zm, mods64 != 0, coulomb, more, nmore, energy, ws, ws_bytes,
                           (hipStream_t)s);
}
int mnx_pme_gather_add_f64(const double* pos, const double* q, const double* box, int64_t n, const double* grid, int32_t gx,
                           int32_t gy, int32_t gz, int32_t order, double coulomb, const double* grad, const double* dpos_add,
                           const double* dq_add, double* dpos, double* dq, mnx_stream_t s) {
    return gather<double>(pos, q, box, n, grid, gx, gy, gz, order, coulomb, grad, dpos_add, dq_add, dpos, dq, (hipStream_t)s);
}

}  // extern "C"
