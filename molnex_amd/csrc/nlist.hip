// Cell-list neighbor list for gfx950.
//
// Replaces the O(N^2) pair enumeration of torch.ops.molix.get_neighbor_pairs
// (reference CPU src/molix/op/src/neighbors/get_neighbor_pairs.cpp:28-77, CUDA
// get_neighbor_pairs.cu:29-79) with a cell list, while keeping the reference
// CPU path's pair predicate and geometry bit for bit:
//   d = pos[i] - pos[j]                                      (.cpp:44)
//   for k = 2, 1, 0: d -= rint(d[k] / box[k][k]) * box[k]   (.cpp:45-49; torch::round is
//                                                             round-half-even)
//   dist = sqrt(fma(d2, d2, fma(d1, d1, d0 * d0)))            (linalg_vector_norm, .cpp:50)
//   keep iff dist <= cutoff && dist > 0                       (.cpp:52)
// Output is sorted by (i, j) like the CPU enumeration order (.cpp:38-43), which
// the CUDA reference does not guarantee (atomicAdd slots, .cu:69).
//
// Layout of the work.  Up to kNlSmall atoms: one wavefront per atom tests all
// the others in id order and keeps the accept ballots, one workgroup scans the
// counts, and the emit expands the ballots, already in (i, j) order: three
// launches and the host's read of the count.
//
// Above that, a cell list.  Atoms are binned into cells whose slab widths exceed
// the cutoff (fractional coordinates for periodic cells); a cell's atoms take a
// run of the cell-ordered arrays in whatever order they arrive (no list depends
// on it; the real-space sum below, whose last bits would, takes them by id).  A workgroup takes a cell: its four wavefronts stage the
// atoms of the 27 neighbour cells in LDS (wrapped next to the cell), then each
// tests them against every fourth atom of the cell as a centre, whose position is
// wave-uniform (a screening distance on positions moved into the primary cell, the
// reference arithmetic near the cutoff), appends the accepted j to the centre's
// list in LDS, sorts it in registers (bitonic) and leaves it in the centre's row of
// kSlots entries in the workspace.  The emit then is a stream: half a wavefront per
// atom reads its sorted row and writes the pairs, the vectors through LDS so that
// every store is contiguous.  Atoms with more than kSlots neighbours, and grids
// with fewer than 3 cells along a periodic axis (all-pairs scan), are listed and
// sorted by the emit itself.  This translation unit is compiled with
// -ffp-contract=off.
//
// Bound by the candidate tests and launches, not by its 36 bytes per pair:
// 100k atoms, 5.24 M ordered pairs (189 MB written): 206 us in all, the count
// pass 88 us (1100 vector and as many scalar instructions per wavefront: the
// tests, the sort and each cell's set-up), the emit 53 us (3.6 TB/s; 67 us with the
// atoms in another order), five binning
// and scan launches and the host's read of the total the rest; 283 us with a
// sorting emit behind accept ballots (130 us), a second sort inside the cells and
// 18 launches.  96 atoms: 49 us (three launches of 3 us, the host's calls and its
// read of the total), 116 us through the cell list.

#include <math.h>

#include <algorithm>

#include "common.h"
#include "nlist_run.h"
#include "scan.h"

namespace mnx {
namespace {

constexpr int kNlSmall = 2048;  // atoms of the all-pairs path (its lists hold 16-bit ids; where both were
                                // timed the cell list passes it at about this size)
constexpr int kNlCap = MNX_NLIST_MAX_NEIGHBORS;  // of one atom
constexpr int kSlots = 128;    // sorted neighbours kept per atom by the count pass
constexpr int kMidCap = 1024;  // LDS list per wavefront of the emit for atoms with more
constexpr int kCand = 512;     // candidates staged in LDS at once (394 on average at liquid density, cells of 5 A)
constexpr int kCentres = 4;    // centres whose lists a wavefront holds in LDS at once
constexpr int kParts = 4;      // wavefronts per cell (each takes every 4th atom of it)
constexpr int64_t kNlBlocks = 8192;  // grid-stride launch of the count pass
constexpr float kCellMargin = 1.0001f;

struct NlGrid {
    int32_t brute;  // 1: all-pairs scan (periodic axis with < 3 cells)
    int32_t periodic;
    int32_t n[3];
    int32_t ncells;
    int32_t overflow;  // set when an atom has more than kNlCap neighbours
    int32_t nbig;      // atoms with more than kMidCap neighbours (listed from the end of NlWs::big)
    int32_t nmid;      // atoms with more than kSlots, at most kMidCap neighbours (from its front)
    int32_t filled;    // cell-ordered slots handed out
    uint64_t lo_key[3], hi_key[3];  // bounding box of an open system, as ordered integers
    double lo[3];
    double inv_w[3];
    double rinv[6];  // inverse of the lower-triangular cell: f_c = z*r5, ...
};

// Position moved into the primary cell, in cell order (screening test of the count pass);
// w carries nothing.
template <typename T>
struct alignas(4 * sizeof(T)) PosW {
    T x, y, z, w;
};

struct NlWs {
    NlGrid* grid;
    int32_t* cell_of;
    int32_t* rank;  // arrival number of the atom in its cell
    int32_t* cell_count;
    int32_t* cell_start;
    int32_t* atoms_sorted;
    int32_t* counts;
    int32_t* big;
    int32_t* ids;     // the real-space sum's: each cell's atoms in order of arrival
    int32_t* slots;   // [n][kSlots]: an atom's neighbours, ascending
    uint64_t* masks;  // small systems: [n][words] accept ballots
    void* posw;       // PosW<T> per cell-ordered slot
    int64_t* offsets;
    int64_t* tiles64;
    int64_t max_cells;
};

int64_t max_cells_for(int64_t n) { return 2 * n + 64; }

// The cell grid and the atoms in cell order.
void take_cells(Workspace& ws, int64_t n, size_t posw_bytes, NlWs& w) {
    w.max_cells = max_cells_for(n);
    w.grid = ws.take<NlGrid>(1);
    w.cell_of = ws.take<int32_t>(n);
    w.rank = ws.take<int32_t>(n);
    w.cell_count = ws.take<int32_t>(w.max_cells);
    w.cell_start = ws.take<int32_t>(w.max_cells);
    w.atoms_sorted = ws.take<int32_t>(n);
    w.posw = ws.take<char>(size_t(n) * posw_bytes);
}

NlWs carve(void* base, size_t bytes, int64_t n, size_t* used) {
    Workspace ws{static_cast<char*>(base), bytes};
    NlWs w{};
    w.offsets = ws.take<int64_t>(n + 1);
    w.counts = ws.take<int32_t>(n > 0 ? n : 1);
    if (n <= kNlSmall) {
        w.masks = ws.take<uint64_t>(size_t(n > 0 ? n : 1) * ((n + kWave - 1) / kWave + 1));
    } else {
        take_cells(ws, n, sizeof(PosW<double>), w);
        w.big = ws.take<int32_t>(n);
        w.slots = ws.take<int32_t>(size_t(n) * kSlots);
        w.tiles64 = ws.take<int64_t>(scan_workspace_elems(n));
    }
    *used = ws.used;
    return w;
}

// What the real-space sum needs of it: no rows, counts or offsets (48 bytes an atom, 64 in float64, instead
// of 588), and nothing for small systems.
NlWs carve_real(void* base, size_t bytes, int64_t n, size_t posw_bytes, size_t* used) {
    Workspace ws{static_cast<char*>(base), bytes};
    NlWs w{};
    if (n > kNlSmall) {
        take_cells(ws, n, posw_bytes, w);
        w.ids = ws.take<int32_t>(n);
    }
    *used = ws.used;
    return w;
}

// ---------------------------------------------------------------------------
// Exact reference geometry
// ---------------------------------------------------------------------------

template <typename T>
struct Geo {
    T d[3];
    T dist;
    T shift[3];
};

__device__ __forceinline__ float fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float rint_(float a) { return rintf(a); }
__device__ __forceinline__ double rint_(double a) { return rint(a); }
__device__ __forceinline__ float sqrt_(float a) { return sqrtf(a); }
__device__ __forceinline__ double sqrt_(double a) { return sqrt(a); }

// rint(d / b), with 1 / b approximately inv: the product decides it except within 1e-3 (and its own
// rounding) of a half-way point, where the quotient is formed.
__device__ __forceinline__ float fabs_(float a) { return fabsf(a); }
__device__ __forceinline__ double fabs_(double a) { return fabs(a); }
__device__ __forceinline__ float rcp_(float a) { return __builtin_amdgcn_rcpf(a); }
__device__ __forceinline__ double rcp_(double a) { return 1.0 / a; }
template <typename T>
__device__ __forceinline__ T rint_quotient(T d, T b, T inv) {
    const T t = d * inv;
    T s = rint_(t);
    if (!(fabs_(t - s) < T(0.499) - fabs_(t) * T(1e-6))) s = rint_(d / b);
    return s;
}

// Minimum image and distance of the difference vector d, the reference's arithmetic.
template <typename T>
__device__ __forceinline__ void geo_from_d(const T* __restrict__ box, T d0, T d1, T d2, bool periodic, bool want_shift,
                                           Geo<T>& g) {
    T s0 = 0, s1 = 0, s2 = 0;
    if (periodic) {
#pragma unroll
        for (int k = 2; k >= 0; --k) {
            const T dk = k == 2 ? d2 : (k == 1 ? d1 : d0);
            const T s = rint_quotient(dk, box[4 * k], rcp_(box[4 * k]));
            const T b0 = s * box[3 * k + 0], b1 = s * box[3 * k + 1], b2 = s * box[3 * k + 2];
            d0 = d0 - b0;
            d1 = d1 - b1;
            d2 = d2 - b2;
            if (want_shift) {
                s0 = s0 + b0;
                s1 = s1 + b1;
                s2 = s2 + b2;
            }
        }
    }
    g.d[0] = d0;
    g.d[1] = d1;
    g.d[2] = d2;
    g.dist = sqrt_(fma_(d2, d2, fma_(d1, d1, d0 * d0)));
    g.shift[0] = s0;
    g.shift[1] = s1;
    g.shift[2] = s2;
}

// Geometry of the pair (hi, lo) with hi > lo, in the reference's orientation.
template <typename T>
__device__ __forceinline__ void pair_geo(const T* __restrict__ pos, const T* __restrict__ box, int hi, int lo,
                                         bool periodic, bool want_shift, Geo<T>& g) {
    geo_from_d<T>(box, pos[3 * hi + 0] - pos[3 * lo + 0], pos[3 * hi + 1] - pos[3 * lo + 1],
                  pos[3 * hi + 2] - pos[3 * lo + 2], periodic, want_shift, g);
}

// Acceptance of a candidate pair, decided as the reference decides it.  A cheap test
// (minimum image through the reciprocal box diagonal, squared distance without the fma
// chain) settles every candidate whose squared distance is clear of cutoff^2 by a relative
// 1e-4 -- far more than the rounding difference between the two evaluations -- and the
// exact reference arithmetic decides the rest (the band around the cutoff and zero
// distance).  The two image choices can differ only where a fractional coordinate is
// within rounding of 1/2, i.e. at about half a cell height of the box, which the cell list
// keeps above the cutoff (>= 3 cells of width >= cutoff along every periodic axis).
template <typename T>
struct AcceptTest {
    T inv[3];
    T c2lo, c2hi, c2tiny;
    T b[9];  // the box, held in registers for the cheap test
};

// The all-pairs fallback (a periodic axis with < 3 cells) gets no cheap test: there the
// half-box distance can be within the cutoff.
template <typename T>
__device__ __forceinline__ AcceptTest<T> accept_test(const T* box, bool periodic, bool brute, T cutoff) {
    AcceptTest<T> a;
    for (int k = 0; k < 3; ++k) a.inv[k] = periodic ? T(1) / box[4 * k] : T(0);
    const T c2 = cutoff * cutoff;
    a.c2lo = brute ? T(0) : c2 * T(0.9999);
    a.c2hi = brute ? T(INFINITY) : c2 * T(1.0001);
    a.c2tiny = c2 * T(1e-20);
    for (int k = 0; k < 9; ++k) a.b[k] = periodic ? box[k] : T(0);
    return a;
}

// Value of lane (lane ^ s) for a power of two s < 64: DPP for 1, 2 (quad permutes) and 8
// (rotation by 8 within a row of 16), the LDS crossbar without memory (ds_swizzle, xor
// within 32 lanes) for 4 and 16, ds_bpermute for 32.
__device__ __forceinline__ int lane_xor(int v, int s) {
    switch (s) {
        case 1: return __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
        case 2: return __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
        case 8: return __builtin_amdgcn_update_dpp(v, v, 0x128, 0xF, 0xF, false);  // row_ror:8
        case 4: return __builtin_amdgcn_ds_swizzle(v, 0x101F);                     // and 31, xor 4
        case 16: return __builtin_amdgcn_ds_swizzle(v, 0x401F);                    // and 31, xor 16
        default: return __shfl_xor(v, s, kWave);
    }
}

// Decision for the pair at positions a, b.  It does not depend on the order: a - b is the
// exact negation of b - a, and the minimum image and the norm are symmetric in sign.
template <typename T>
__device__ __forceinline__ bool accept_xyz(const T* box, T ax, T ay, T az, T bx, T by, T bz, bool periodic, T cutoff,
                                           const AcceptTest<T>& at) {
    T d0 = ax - bx, d1 = ay - by, d2 = az - bz;
    const T e0 = d0, e1 = d1, e2 = d2;
    if (periodic) {
#pragma unroll
        for (int k = 2; k >= 0; --k) {
            const T dk = k == 2 ? d2 : (k == 1 ? d1 : d0);
            const T s = rint_(dk * at.inv[k]);
            d0 = d0 - s * at.b[3 * k + 0];
            d1 = d1 - s * at.b[3 * k + 1];
            d2 = d2 - s * at.b[3 * k + 2];
        }
    }
    const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
    if (r2 > at.c2hi) return false;
    if (r2 < at.c2lo && r2 > at.c2tiny) return true;
    Geo<T> g;
    geo_from_d<T>(box, e0, e1, e2, periodic, false, g);
    return g.dist <= cutoff && g.dist > T(0);
}

template <typename T>
__device__ __forceinline__ bool accept(const T* pos, const T* box, int i, int j, bool periodic, T cutoff,
                                       const AcceptTest<T>& at) {
    return accept_xyz<T>(box, pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], pos[3 * j], pos[3 * j + 1], pos[3 * j + 2],
                         periodic, cutoff, at);
}

// ---------------------------------------------------------------------------
// Grid set-up and binning
// ---------------------------------------------------------------------------

// Ordered integers of doubles (bounding box by integer atomics).
__device__ __forceinline__ uint64_t to_key(double v) {
    const uint64_t b = uint64_t(__double_as_longlong(v));
    return b >> 63 ? ~b : b | (uint64_t(1) << 63);
}
__device__ __forceinline__ double from_key(uint64_t k) {
    return __longlong_as_double((long long)(k >> 63 ? k & ~(uint64_t(1) << 63) : ~k));
}

// The cell grid of box (or of an open system's bounding box, from gp).
template <typename T>
__device__ NlGrid make_grid(int64_t n, const T* __restrict__ box, double cutoff, int64_t max_cells,
                            const NlGrid* __restrict__ gp) {
    NlGrid g{};
    const double cw = cutoff * double(kCellMargin) + 1e-12;
    if (box) {
        const double ax = box[0], bx = box[3], by = box[4], cx = box[6], cy = box[7], cz = box[8];
        // perpendicular slab widths of the lower-triangular cell
        const double vol = fabs(ax * by * cz);
        const double bxc = sqrt((by * cz) * (by * cz) + (bx * cz) * (bx * cz) + (bx * cy - by * cx) * (bx * cy - by * cx));
        const double axc = sqrt((ax * cz) * (ax * cz) + (ax * cy) * (ax * cy));
        const double h[3] = {vol / bxc, vol / axc, fabs(cz)};
        g.periodic = 1;
        for (int k = 0; k < 3; ++k) {
            double m = floor(h[k] / cw);
            g.n[k] = m < 1 ? 1 : (m > 1024 ? 1024 : int(m));
        }
        g.rinv[0] = 1.0 / ax;
        g.rinv[1] = bx;
        g.rinv[2] = 1.0 / by;
        g.rinv[3] = cx;
        g.rinv[4] = cy;
        g.rinv[5] = 1.0 / cz;
        while (int64_t(g.n[0]) * g.n[1] * g.n[2] > max_cells) {
            int kmax = g.n[0] >= g.n[1] ? (g.n[0] >= g.n[2] ? 0 : 2) : (g.n[1] >= g.n[2] ? 1 : 2);
            g.n[kmax] = (g.n[kmax] + 1) / 2;
        }
        g.brute = (g.n[0] < 3 || g.n[1] < 3 || g.n[2] < 3) ? 1 : 0;
    } else {
        g.periodic = 0;
        for (int k = 0; k < 3; ++k) {
            double lo = n > 0 ? from_key(gp->lo_key[k]) : 0.0, hi = n > 0 ? from_key(gp->hi_key[k]) : 0.0;
            double ext = hi - lo;
            double m = floor(ext / cw);
            g.n[k] = m < 1 ? 1 : (m > 1024 ? 1024 : int(m));
            g.lo[k] = lo;
        }
        while (int64_t(g.n[0]) * g.n[1] * g.n[2] > max_cells) {
            int kmax = g.n[0] >= g.n[1] ? (g.n[0] >= g.n[2] ? 0 : 2) : (g.n[1] >= g.n[2] ? 1 : 2);
            g.n[kmax] = (g.n[kmax] + 1) / 2;
        }
        for (int k = 0; k < 3; ++k) {
            double ext = (n > 0 ? from_key(gp->hi_key[k]) : 0.0) - g.lo[k];
            g.inv_w[k] = ext > 0 ? double(g.n[k]) / ext : 0.0;
        }
        g.brute = 0;
    }
    g.ncells = g.brute ? 1 : g.n[0] * g.n[1] * g.n[2];
    return g;
}


// Zeroes the cell counters (and the caller's flag); the first thread sets up the grid of a periodic system (an open one
// waits for its bounding box).
template <typename T>
__global__ void __launch_bounds__(256) k_nl_clear(int32_t* __restrict__ cell_count, int64_t n, const T* __restrict__ box,
                                                  double cutoff, int64_t max_cells, NlGrid* __restrict__ gp,
                                                  int32_t* __restrict__ flag) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < max_cells) cell_count[i] = 0;
    if (i) return;
    if (flag) *flag = 0;
    if (box) {
        *gp = make_grid<T>(n, box, cutoff, max_cells, nullptr);
    } else {
        NlGrid g{};
        for (int k = 0; k < 3; ++k) {
            g.lo_key[k] = to_key(1e300);
            g.hi_key[k] = to_key(-1e300);
        }
        *gp = g;
    }
}

// Bounding box of an open system (NaN coordinates left out).
template <typename T>
__global__ void __launch_bounds__(256) k_nl_bounds(const T* __restrict__ pos, int64_t n, NlGrid* __restrict__ gp) {
    double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        for (int k = 0; k < 3; ++k) {
            const double v = double(pos[3 * i + k]);
            mn[k] = fmin(mn[k], v);
            mx[k] = fmax(mx[k], v);
        }
    for (int k = 0; k < 3; ++k) {
        for (int o = 32; o > 0; o >>= 1) {
            mn[k] = fmin(mn[k], __shfl_xor(mn[k], o, kWave));
            mx[k] = fmax(mx[k], __shfl_xor(mx[k], o, kWave));
        }
        if ((threadIdx.x & (kWave - 1)) == 0) {
            atomicMin(reinterpret_cast<unsigned long long*>(&gp->lo_key[k]), (unsigned long long)to_key(mn[k]));
            atomicMax(reinterpret_cast<unsigned long long*>(&gp->hi_key[k]), (unsigned long long)to_key(mx[k]));
        }
    }
}

template <typename T>
__global__ void k_nl_open_grid(int64_t n, double cutoff, int64_t max_cells, NlGrid* __restrict__ gp) {
    const NlGrid g = make_grid<T>(n, nullptr, cutoff, max_cells, gp);
    *gp = g;
}

template <typename T>
__device__ __forceinline__ void cell_coords(const T* pos, int64_t i, const NlGrid& g, int c[3]) {
    const double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2];
    if (g.periodic) {
        double f[3];
        f[2] = z * g.rinv[5];
        f[1] = (y - f[2] * g.rinv[4]) * g.rinv[2];
        f[0] = (x - f[1] * g.rinv[1] - f[2] * g.rinv[3]) * g.rinv[0];
        for (int k = 0; k < 3; ++k) {
            double fk = f[k] - floor(f[k]);
            int ck = int(fk * g.n[k]);
            c[k] = ck < 0 ? 0 : (ck >= g.n[k] ? g.n[k] - 1 : ck);
        }
    } else {
        const double v[3] = {x, y, z};
        for (int k = 0; k < 3; ++k) {
            int ck = int((v[k] - g.lo[k]) * g.inv_w[k]);
            c[k] = ck < 0 ? 0 : (ck >= g.n[k] ? g.n[k] - 1 : ck);
        }
    }
}

template <typename T>
__global__ void k_bin(const T* __restrict__ pos, int64_t n, const NlGrid* __restrict__ gp, int32_t* __restrict__ cell_of,
                      int32_t* __restrict__ rank, int32_t* __restrict__ cell_count) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const NlGrid g = *gp;
    if (g.brute) return;  // no cells
    int c[3];
    cell_coords<T>(pos, i, g, c);
    const int cid = (c[2] * g.n[1] + c[1]) * g.n[0] + c[0];
    cell_of[i] = cid;
    rank[i] = atomicAdd(&cell_count[cid], 1);
}

// Each cell's run of the cell-ordered arrays: contiguous in cell order within a workgroup's 2048
// cells, the workgroups' runs in the order they arrive.
__global__ void __launch_bounds__(kScanThreads) k_cell_runs(NlGrid* __restrict__ gp,
                                                            const int32_t* __restrict__ cell_count,
                                                            int32_t* __restrict__ cell_start) {
    __shared__ int32_t sh[kScanThreads];
    __shared__ int32_t s_base;
    const int ncells = gp->brute ? 0 : gp->ncells;
    const int base = int(blockIdx.x) * kScanTile + int(threadIdx.x) * kScanItems;
    if (int(blockIdx.x) * kScanTile >= ncells) return;
    int32_t v[kScanItems], sum = 0, total;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < ncells ? cell_count[base + k] : 0;
        sum += v[k];
    }
    int32_t run = block_exclusive_scan<int32_t>(sum, sh, &total);
    if (threadIdx.x == 0) s_base = atomicAdd(&gp->filled, total);
    __syncthreads();
    run += s_base;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < ncells) cell_start[base + k] = run;
        run += v[k];
    }
}

// The slots of each cell's atoms in order of arrival, their ids alone.
__global__ void __launch_bounds__(256) k_place_ids(int64_t n, const NlGrid* __restrict__ gp,
                                                   const int32_t* __restrict__ cell_of,
                                                   const int32_t* __restrict__ rank,
                                                   const int32_t* __restrict__ cell_start, int32_t* __restrict__ ids) {
    const int64_t a = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (a >= n || gp->brute) return;
    ids[cell_start[cell_of[a]] + rank[a]] = int32_t(a);
}

// Each atom into its slot of the cell order, with its position moved into the primary cell (by
// whole box vectors, from the fractional coordinates that binned it), which the count pass's
// screening test reads.  Within a cell the atoms take their slots as they arrived (rank) or, ORDERED,
// by id: a thread per slot of `ids` counts the smaller ids of its cell.
template <typename T, bool ORDERED>
__global__ void __launch_bounds__(256) k_place(int64_t n, const T* __restrict__ pos, const T* __restrict__ box,
                                               const NlGrid* __restrict__ gp, const int32_t* __restrict__ cell_of,
                                               const int32_t* __restrict__ rank,
                                               const int32_t* __restrict__ cell_start,
                                               const int32_t* __restrict__ cell_count, const int32_t* __restrict__ ids,
                                               int32_t* __restrict__ atoms_sorted, PosW<T>* __restrict__ posw) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n || gp->brute) return;
    const int64_t a = ORDERED ? ids[t] : t;
    const int c = cell_of[a], first = cell_start[c];
    int r = 0;
    if (ORDERED) {
        const int m = cell_count[c];
        for (int k = 0; k < m; ++k) r += ids[first + k] < a;
    } else {
        r = rank[a];
    }
    const int slot = first + r;
    atoms_sorted[slot] = int32_t(a);
    const double x = pos[3 * a], y = pos[3 * a + 1], z = pos[3 * a + 2];
    PosW<T> p;
    if (gp->periodic) {
        // the fractional coordinates of cell_coords; box rows (ax,0,0), (bx,by,0), (cx,cy,cz)
        const NlGrid& g = *gp;
        const double f2 = z * g.rinv[5];
        const double f1 = (y - f2 * g.rinv[4]) * g.rinv[2];
        const double f0 = (x - f1 * g.rinv[1] - f2 * g.rinv[3]) * g.rinv[0];
        const double n0 = floor(f0), n1 = floor(f1), n2 = floor(f2);
        p.x = T(x - n0 * double(box[0]) - n1 * double(box[3]) - n2 * double(box[6]));
        p.y = T(y - n1 * double(box[4]) - n2 * double(box[7]));
        p.z = T(z - n2 * double(box[8]));
    } else {
        p.x = T(x);
        p.y = T(y);
        p.z = T(z);
    }
    p.w = T(0);
    posw[slot] = p;
}

// ---------------------------------------------------------------------------
// Candidate scan: one wavefront per atom
// ---------------------------------------------------------------------------

// Atom ranges of the 27 neighbour cells of cell (cx, cy, cz), flattened: lanes 0..26 hold
// (begin, length) of neighbour cell (dz, dy, dx) = lane in base 3, fetched in one round trip,
// and `incl` is the inclusive prefix sum of the lengths over lanes; `total` candidates in all.
struct CellRanges {
    int rb, rlen, incl, total;
};

__device__ __forceinline__ CellRanges cell_ranges(const NlGrid& g, int cx, int cy, int cz,
                                                  const int32_t* __restrict__ cell_start,
                                                  const int32_t* __restrict__ cell_count, int lane) {
    CellRanges cr{0, 0, 0, 0};
    if (lane < 27) {
        int z = cz + lane / 9 - 1, y = cy + (lane / 3) % 3 - 1, x = cx + lane % 3 - 1;
        bool in = true;
        if (g.periodic) {
            // one step outside at most
            z += z < 0 ? g.n[2] : (z >= g.n[2] ? -g.n[2] : 0);
            y += y < 0 ? g.n[1] : (y >= g.n[1] ? -g.n[1] : 0);
            x += x < 0 ? g.n[0] : (x >= g.n[0] ? -g.n[0] : 0);
        } else {
            in = z >= 0 && z < g.n[2] && y >= 0 && y < g.n[1] && x >= 0 && x < g.n[0];
        }
        if (in) {
            const int cid = (z * g.n[1] + y) * g.n[0] + x;
            cr.rb = cell_start[cid];
            cr.rlen = cell_count[cid];
        }
    }
    int incl = cr.rlen;  // lanes >= 27 add 0
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += v;
    }
    cr.incl = incl;
    cr.total = __shfl(incl, 26, kWave);
    return cr;
}

// Candidate number k of the flattened ranges (-1 past the end); every lane must call it.
__device__ __forceinline__ int cell_candidate(const CellRanges& cr, int k, const int32_t* __restrict__ atoms_sorted) {
    int r = 0;  // number of ranges that end at or before k (branch-free search over 27 entries)
#pragma unroll
    for (int step = 16; step > 0; step >>= 1) {
        const int probe = __shfl(cr.incl, r + step - 1, kWave);
        if (r + step <= 26 && probe <= k) r += step;
    }
    const int start = __shfl(cr.rb, r, kWave);
    const int first = __shfl(cr.incl - cr.rlen, r, kWave);
    return k < cr.total ? atoms_sorted[start + (k - first)] : -1;
}

// Calls f(j) for every candidate j of atom i (each j at most once), lanes in parallel; of the chunks of
// one wavefront's width, every `waves`-th from number `wave` on.
template <typename T, typename F>
__device__ __forceinline__ void for_candidates(const T* pos, int i, int64_t n, const NlGrid& g,
                                               const int32_t* __restrict__ cell_start,
                                               const int32_t* __restrict__ cell_count,
                                               const int32_t* __restrict__ atoms_sorted, int mode, F&& f, int wave = 0,
                                               int waves = 1) {
    const int lane = threadIdx.x & (kWave - 1);
    if (g.brute) {
        const int64_t end = mode == MNX_NLIST_HALF ? i : n;
        for (int64_t base = wave * kWave; base < end; base += waves * kWave) {
            const int64_t j = base + lane;
            f(j < end && j != i ? int(j) : -1);
        }
        return;
    }
    int c[3];
    cell_coords<T>(pos, i, g, c);
    const CellRanges cr = cell_ranges(g, c[0], c[1], c[2], cell_start, cell_count, lane);
    for (int base = wave * kWave; base < cr.total; base += waves * kWave) {
        int j = cell_candidate(cr, base + lane, atoms_sorted);
        if (mode == MNX_NLIST_HALF ? j >= i : j == i) j = -1;
        f(j);
    }
}

// All-pairs fallback (a periodic axis with fewer than 3 cells): one wavefront per atom, grid-stride.
template <typename T>
__device__ __forceinline__ void count_all_pairs(const T* __restrict__ pos, int64_t n, const T* __restrict__ box,
                                                T cutoff, int mode, NlGrid* __restrict__ gp, const NlGrid& g,
                                                int32_t* __restrict__ counts) {
    const bool periodic = g.periodic;
    const AcceptTest<T> at = accept_test<T>(box, periodic, true, cutoff);
    const int lane = threadIdx.x & (kWave - 1);
    for (int64_t i = int64_t(blockIdx.x) * kParts + (threadIdx.x >> 6); i < n; i += int64_t(gridDim.x) * kParts) {
        int count = 0;
        for_candidates<T>(pos, int(i), n, g, nullptr, nullptr, nullptr, mode, [&](int j) {
            const bool ok = j >= 0 && accept<T>(pos, box, int(i), j, periodic, cutoff, at);
            count += __popcll(__ballot(ok));
        });
        if (lane == 0) {
            counts[i] = count;
            if (count > kNlCap) atomicExch(&gp->overflow, 1);
        }
    }
}

// Orders this wavefront's LDS writes before its reads (LDS operations of one wavefront complete in
// order; the compiler must not move them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bitonic sort of `len` ints in LDS, ascending, by one wavefront or (GROUP) the whole workgroup of four;
// buf has room for the next power of two of len (padded with INT_MAX).
template <bool GROUP>
__device__ void lds_sort(int32_t* buf, int len) {
    int m = 1;
    while (m < len) m <<= 1;
    constexpr int kStep = GROUP ? 4 * kWave : kWave;
    const int first = threadIdx.x & (kStep - 1);
    auto fence = [] {
        if (GROUP) __syncthreads();
        else wave_lds_fence();
    };
    for (int k = len + first; k < m; k += kStep) buf[k] = 0x7fffffff;
    fence();
    for (int size = 2; size <= m; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = first; t < (m >> 1); t += kStep) {
                const int lo = 2 * t - (t & (stride - 1));
                const int hi = lo + stride;
                const bool up = (lo & size) == 0;
                const int a = buf[lo], b = buf[hi];
                if ((a > b) == up) {
                    buf[lo] = b;
                    buf[hi] = a;
                }
            }
            fence();
        }
    }
}

// One compare-exchange step of a bitonic sort over the lanes' values: the smaller of a pair stays in
// the lane where `keep_low`.  The median of the two and an extreme value is their minimum or maximum.
__device__ __forceinline__ int bitonic_step(int v, int stride, bool keep_low) {
    const int other = lane_xor(v, stride);
    const int bound = keep_low ? INT32_MIN : INT32_MAX;
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(other), "v"(bound));
    return r;
}

// The lanes' values sorted over the wavefront, ascending or descending.
__device__ __forceinline__ int wave_sort(int v, bool ascending, int lane) {
#pragma unroll
    for (int size = 2; size <= kWave; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1)
            v = bitonic_step(v, stride, ((size == kWave || (lane & size) == 0) == ascending) == ((lane & stride) == 0));
    }
    return v;
}

// Writes pair (i, j) at `slot` with the reference geometry (row = the larger index).
template <typename T>
__device__ __forceinline__ void write_pair(const T* __restrict__ pos, const T* __restrict__ box, bool periodic, int i,
                                           int j, int64_t slot, int32_t* __restrict__ idx_i,
                                           int32_t* __restrict__ idx_j, T* __restrict__ deltas,
                                           T* __restrict__ dist, T* __restrict__ shifts) {
    Geo<T> gg;
    const bool flip = i < j;
    pair_geo<T>(pos, box, flip ? j : i, flip ? i : j, periodic, shifts != nullptr, gg);
    if (idx_i) idx_i[slot] = i;
    if (idx_j) idx_j[slot] = j;
    if (deltas) {
        deltas[3 * slot + 0] = flip ? -gg.d[0] : gg.d[0];
        deltas[3 * slot + 1] = flip ? -gg.d[1] : gg.d[1];
        deltas[3 * slot + 2] = flip ? -gg.d[2] : gg.d[2];
    }
    if (dist) dist[slot] = gg.dist;
    if (shifts) {
        shifts[3 * slot + 0] = flip ? -gg.shift[0] : gg.shift[0];
        shifts[3 * slot + 1] = flip ? -gg.shift[1] : gg.shift[1];
        shifts[3 * slot + 2] = flip ? -gg.shift[2] : gg.shift[2];
    }
}

// What the emit's stream leaves: atoms with more than kSlots neighbours (listed by the count pass),
// and every atom of an all-pairs grid.  Candidates are tested again, collected in LDS and sorted: a
// wavefront each with a list of kMidCap for the former, then the whole workgroup, with the whole
// buffer, for each atom with still more and of all-pairs grids (one wavefront of the four left it idle:
// 6000 atoms with 1150 neighbours 1459 us, with all four 567; an all-pairs grid of 8000 atoms 728, 387).
// Called by whole workgroups.
template <typename T>
__device__ void emit_rest(int32_t* buf, const T* __restrict__ pos, int64_t n, const T* __restrict__ box, T cutoff,
                          int mode, int layout, const NlGrid& g, const int32_t* __restrict__ cell_start,
                          const int32_t* __restrict__ cell_count, const int32_t* __restrict__ atoms_sorted,
                          const int32_t* __restrict__ big, const int64_t* __restrict__ offsets, int64_t capacity,
                          int32_t* __restrict__ idx_i, int32_t* __restrict__ idx_j, T* __restrict__ deltas,
                          T* __restrict__ dist, T* __restrict__ shifts) {
    static_assert(kNlCap == 4 * kMidCap, "one list per wavefront");
    __shared__ int s_found;
    const bool periodic = g.periodic;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    const AcceptTest<T> at = accept_test<T>(box, periodic, true, cutoff);
    // the sorted list's pairs, by `step` threads from number `first` on
    auto write = [&](int i, const int32_t* list, int count, int first, int step) {
        const int64_t base = layout == MNX_NLIST_TRIANGULAR ? 0 : offsets[i];
        for (int k = first; k < count; k += step) {
            const int j = list[k];
            const int64_t slot = layout == MNX_NLIST_TRIANGULAR ? int64_t(i) * (i - 1) / 2 + j : base + k;
            if (slot < capacity) write_pair<T>(pos, box, periodic, i, j, slot, idx_i, idx_j, deltas, dist, shifts);
        }
    };
    __syncthreads();  // the caller's use of the buffer is over
    if (!g.brute)
        for (int64_t t = int64_t(blockIdx.x) * 4 + wave; t < g.nmid; t += int64_t(gridDim.x) * 4) {
            const int i = big[t];
            int32_t* list = buf + wave * kMidCap;
            int count = 0;
            wave_lds_fence();  // the list is reused across atoms
            for_candidates<T>(pos, i, n, g, cell_start, cell_count, atoms_sorted, mode, [&](int j) {
                const bool ok = j >= 0 && accept<T>(pos, box, i, j, periodic, cutoff, at);
                const uint64_t m = __ballot(ok);
                const int to = count + __popcll(m & below);
                if (ok && to < kMidCap) list[to] = j;
                count += __popcll(m);
            });
            count = min(count, kMidCap);
            lds_sort<false>(list, count);
            write(i, list, count, lane, kWave);
        }
    for (int64_t t = blockIdx.x; t < (g.brute ? n : g.nbig); t += gridDim.x) {
        const int i = g.brute ? int(t) : big[n - 1 - t];
        __syncthreads();
        if (threadIdx.x == 0) s_found = 0;
        __syncthreads();
        for_candidates<T>(
            pos, i, n, g, cell_start, cell_count, atoms_sorted, mode,
            [&](int j) {
                const bool ok = j >= 0 && accept<T>(pos, box, i, j, periodic, cutoff, at);
                const uint64_t m = __ballot(ok);
                if (m == 0) return;
                int to = 0;
                if (lane == 0) to = atomicAdd(&s_found, __popcll(m));
                to = __builtin_amdgcn_readfirstlane(to) + __popcll(m & below);
                if (ok && to < kNlCap) buf[to] = j;
            },
            wave, 4);
        __syncthreads();
        const int count = min(s_found, kNlCap);  // more: flagged by the count pass; the host reports the error
        lds_sort<true>(buf, count);
        write(i, buf, count, threadIdx.x, 4 * kWave);
    }
}

// ---------------------------------------------------------------------------
// Small systems: all pairs, one wavefront per atom, candidates in id order.
// ---------------------------------------------------------------------------

// Whether the cheap test of AcceptTest applies: every box height at least 3 cutoffs (the cell
// grid's condition), or an open system.
template <typename T>
__device__ __forceinline__ bool wide_box(const T* __restrict__ box, double cutoff) {
    if (!box) return true;
    const double ax = box[0], bx = box[3], by = box[4], cx = box[6], cy = box[7], cz = box[8];
    const double vol = fabs(ax * by * cz), cw = cutoff * double(kCellMargin) + 1e-12;
    const double bxc = sqrt((by * cz) * (by * cz) + (bx * cz) * (bx * cz) + (bx * cy - by * cx) * (bx * cy - by * cx));
    const double axc = sqrt((ax * cz) * (ax * cz) + (ax * cy) * (ax * cy));
    return vol >= 3 * cw * bxc && vol >= 3 * cw * axc && fabs(cz) >= 3 * cw;
}

template <typename T>
__global__ void __launch_bounds__(256) k_small_count(const T* __restrict__ pos, int n, const T* __restrict__ box,
                                                     T cutoff, int mode, int words, int32_t* __restrict__ counts,
                                                     uint64_t* __restrict__ masks) {
    const int lane = threadIdx.x & (kWave - 1);
    const int i = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * 4 + (threadIdx.x >> 6));
    if (i >= n) return;
    const bool periodic = box != nullptr;
    const AcceptTest<T> at = accept_test<T>(box, periodic, !wide_box<T>(box, double(cutoff)), cutoff);
    const T ax = pos[3 * i], ay = pos[3 * i + 1], az = pos[3 * i + 2];
    const int end = mode == MNX_NLIST_HALF ? i : n;
    int count = 0;
    for (int base = 0; base < end; base += kWave) {
        const int j = base + lane;
        bool ok = j < end && j != i;
        if (ok) ok = accept_xyz<T>(box, ax, ay, az, pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], periodic, cutoff, at);
        const uint64_t m = __ballot(ok);
        if (lane == 0) masks[int64_t(i) * words + base / kWave] = m;
        count += __popcll(m);
    }
    if (lane == 0) counts[i] = count;
}

// Offsets of up to kNlSmall counts and their total, one workgroup.
__global__ void __launch_bounds__(kScanThreads) k_small_scan(const int32_t* __restrict__ counts, int n,
                                                             int64_t* __restrict__ offsets,
                                                             int64_t* __restrict__ d_total) {
    static_assert(kNlSmall <= kScanTile, "one tile");
    __shared__ int32_t sh[kScanThreads];
    const int base = int(threadIdx.x) * kScanItems;
    int32_t v[kScanItems], sum = 0, total;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? counts[base + k] : 0;
        sum += v[k];
    }
    int32_t run = block_exclusive_scan<int32_t>(sum, sh, &total);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < n) offsets[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 0) {
        offsets[n] = total;
        if (d_total) *d_total = total;
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_small_emit(const T* __restrict__ pos, int n, const T* __restrict__ box,
                                                    int mode, int layout, int words,
                                                    const uint64_t* __restrict__ masks,
                                                    const int64_t* __restrict__ offsets, int64_t capacity,
                                                    int32_t* __restrict__ idx_i, int32_t* __restrict__ idx_j,
                                                    T* __restrict__ deltas, T* __restrict__ dist,
                                                    T* __restrict__ shifts) {
    __shared__ uint16_t lists[4][kNlSmall];
    static_assert(kNlSmall <= 65536, "16-bit ids");
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int i = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * 4 + wave);
    if (i >= n) return;
    uint16_t* list = lists[wave];
    const int end = mode == MNX_NLIST_HALF ? i : n;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    int count = 0;
    for (int base = 0; base < end; base += kWave) {
        const uint64_t m = masks[int64_t(i) * words + base / kWave];
        if ((m >> lane) & 1) list[count + __popcll(m & below)] = uint16_t(base + lane);
        count += __popcll(m);
    }
    wave_lds_fence();
    const int64_t off = layout == MNX_NLIST_TRIANGULAR ? 0 : offsets[i];
    for (int k = lane; k < count; k += kWave) {
        const int j = list[k];
        const int64_t slot = layout == MNX_NLIST_TRIANGULAR ? int64_t(i) * (i - 1) / 2 + j : off + k;
        if (slot < capacity) write_pair<T>(pos, box, box != nullptr, i, j, slot, idx_i, idx_j, deltas, dist, shifts);
    }
}

// ---------------------------------------------------------------------------
// Cell grids: a workgroup per cell, grid-stride.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void cell_coords_of(uint32_t c, const NlGrid& g, int* cx, int* cy, int* cz) {
    const uint32_t t = c / uint32_t(g.n[0]);
    *cx = int(c - t * uint32_t(g.n[0]));
    const uint32_t z = t / uint32_t(g.n[1]);
    *cy = int(t - z * uint32_t(g.n[1]));
    *cz = int(z);
}

// Slot (index into the cell-ordered arrays) of candidate number k of the flattened ranges,
// -1 past the end, and in *cell the neighbour-cell lane (0..26) it comes from; every lane must
// call it.
__device__ __forceinline__ int cell_candidate_slot(const CellRanges& cr, int k, int* cell) {
    int r = 0;
#pragma unroll
    for (int step = 16; step > 0; step >>= 1) {
        const int probe = __shfl(cr.incl, r + step - 1, kWave);
        if (r + step <= 26 && probe <= k) r += step;
    }
    const int start = __shfl(cr.rb, r, kWave);
    const int first = __shfl(cr.incl - cr.rlen, r, kWave);
    *cell = r;
    return k < cr.total ? start + (k - first) : -1;
}

// The count pass screens each (centre, candidate) pair by the squared distance between the
// centre's position in the primary cell and the candidate's, moved by the box vectors that
// wrap its neighbour cell next to the centre's cell.  With >= 3 cells of width >= the cutoff
// along every periodic axis this is the minimum image for every pair within the cutoff (any
// other image is more than twice the cutoff away).  Pairs clear of cutoff^2 by a relative
// 1e-3 are settled by it -- the rounding of the wrapped positions is orders of magnitude
// smaller -- and the reference arithmetic on the original positions decides the band and
// zero distances, so the accepted set is the reference's.
//
// Sink: what becomes of a centre's accepted j.  A collecting sink (kStream false) gets the list at
// the end, its first kSlots entries; a streaming one gets 64 at a time as they arrive, then the rest.
template <typename T, bool HALF, typename Sink>
__device__ __forceinline__ void scan_cells(const T* __restrict__ pos, const T* __restrict__ box, T cutoff, const NlGrid& g,
                                           const int32_t* __restrict__ cell_start,
                                           const int32_t* __restrict__ cell_count,
                                           const int32_t* __restrict__ atoms_sorted,
                                           const PosW<T>* __restrict__ posw, Sink& sink) {
    __shared__ T s_x[kCand], s_y[kCand], s_z[kCand];
    __shared__ int32_t s_id[kCand];
    __shared__ int32_t s_list[kParts][kCentres][kSlots];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool periodic = g.periodic;
    const T c2 = cutoff * cutoff;
    const T c2lo = c2 * T(0.999), c2hi = c2 * T(1.001), c2tiny = c2 * T(1e-20);
    for (int c = blockIdx.x; c < g.ncells; c += gridDim.x) {
        const int cb = cell_start[c], ncell = cell_count[c];
        int cx, cy, cz;
        cell_coords_of(uint32_t(c), g, &cx, &cy, &cz);
        const CellRanges cr = cell_ranges(g, cx, cy, cz, cell_start, cell_count, lane);
        if (ncell == 0) continue;
        // lanes 0..26: the box vectors that bring neighbour cell `lane` next to this cell
        T shx = T(0), shy = T(0), shz = T(0);
        if (periodic && lane < 27) {
            const int z = cz + lane / 9 - 1, y = cy + (lane / 3) % 3 - 1, x = cx + lane % 3 - 1;
            const int wz = z < 0 ? -1 : (z >= g.n[2] ? 1 : 0), wy = y < 0 ? -1 : (y >= g.n[1] ? 1 : 0),
                      wx = x < 0 ? -1 : (x >= g.n[0] ? 1 : 0);
            shx = T(wx) * box[0] + T(wy) * box[3] + T(wz) * box[6];
            shy = T(wy) * box[4] + T(wz) * box[7];
            shz = T(wz) * box[8];
        }
        int staged = -1;  // first candidate of those in LDS
        for (int q0 = 0; q0 < ncell; q0 += kParts * kCentres) {
            // this wavefront's centres q0 + wave, q0 + wave + 4, ...
            const int left = ncell - q0 - wave;
            const int nq = left <= 0 ? 0 : min((left + kParts - 1) / kParts, kCentres);
            int ci[kCentres], cnt[kCentres], held[kCentres];  // accepted, of them in the list
            T px[kCentres], py[kCentres], pz[kCentres];
#pragma unroll
            for (int q = 0; q < kCentres; ++q) {
                const int slot = cb + (q < nq ? q0 + wave + q * kParts : 0);
                ci[q] = atoms_sorted[slot];
                const PosW<T> p = posw[slot];
                px[q] = p.x;
                py[q] = p.y;
                pz[q] = p.z;
                cnt[q] = held[q] = 0;
                sink.begin(q, ci[q]);
            }
            for (int b0 = 0; b0 < cr.total; b0 += kCand) {
                const int nb = min(kCand, cr.total - b0);
                if (staged != b0) {  // (a cell's only batch is kept for its further centres)
                    __syncthreads();
                    for (int base = wave * kWave; base < nb; base += kParts * kWave) {
                        int r;
                        const int slot = cell_candidate_slot(cr, b0 + base + lane, &r);
                        const T sx = __shfl(shx, r, kWave), sy = __shfl(shy, r, kWave), sz = __shfl(shz, r, kWave);
                        if (slot >= 0) {
                            const PosW<T> p = posw[slot];
                            s_x[base + lane] = p.x + sx;
                            s_y[base + lane] = p.y + sy;
                            s_z[base + lane] = p.z + sz;
                            s_id[base + lane] = atoms_sorted[slot];
                        } else {  // past the end (of the last 64): NaN passes no test, whatever the cutoff
                            s_x[base + lane] = s_y[base + lane] = s_z[base + lane] = T(__builtin_nan(""));
                            s_id[base + lane] = INT32_MAX;
                        }
                    }
                    __syncthreads();
                    staged = b0;
                }
                if (nq == 0) continue;
                for (int base = 0; base < nb; base += kWave) {
                    const T jx = s_x[base + lane], jy = s_y[base + lane], jz = s_z[base + lane];
                    const int j = s_id[base + lane];
#pragma unroll
                    for (int q = 0; q < kCentres; ++q) {
                        if (q >= nq) break;
                        const T dx = px[q] - jx, dy = py[q] - jy, dz = pz[q] - jz;
                        const T r2 = dx * dx + dy * dy + dz * dz;
                        bool ok = r2 <= c2hi && (HALF ? j < ci[q] : j != ci[q]);
                        // the band around the cutoff and (near-)zero distances: reference arithmetic
                        const bool band = ok && !(r2 < c2lo && r2 > c2tiny);
                        if (__ballot(band)) {
                            if (band) {
                                Geo<T> gg;
                                pair_geo<T>(pos, box, ci[q], j, periodic, false, gg);
                                ok = gg.dist <= cutoff && gg.dist > T(0);
                            }
                        }
                        const uint64_t m = __ballot(ok);
                        const int at = held[q] + __popcll(m & ((uint64_t(1) << lane) - 1));
                        if (ok && at < kSlots) s_list[wave][q][at] = j;
                        cnt[q] += __popcll(m);
                        held[q] += __popcll(m);
                        if constexpr (Sink::kStream) {
                            if (held[q] >= kWave) {
                                int32_t* list = s_list[wave][q];
                                wave_lds_fence();
                                sink.take(q, ci[q], list, kWave);
                                held[q] -= kWave;
                                const int rest = list[kWave + lane];
                                if (lane < held[q]) list[lane] = rest;
                            }
                        }
                    }
                }
            }
            wave_lds_fence();
#pragma unroll
            for (int q = 0; q < kCentres; ++q) {
                if (q >= nq) break;
                sink.finish(q, ci[q], s_list[wave][q], cnt[q], held[q]);
            }
            wave_lds_fence();  // the lists are reused
        }
    }
}

// Collects the rows of the neighbor list.
template <typename T>
struct RowSink {
    static constexpr bool kStream = false;
    int64_t n;
    NlGrid* gp;
    int32_t *counts, *big, *slots;
    __device__ __forceinline__ void begin(int, int) {}
    __device__ __forceinline__ void take(int, int, const int32_t*, int) {}
    // the list in ascending order into the centre's row
    __device__ __forceinline__ void finish(int, int i, const int32_t* list, int count, int) {
        const int lane = threadIdx.x & (kWave - 1);
        if (lane == 0) {
            counts[i] = count;
            if (count > kNlCap) atomicExch(&gp->overflow, 1);
            if (count > kMidCap) big[n - 1 - atomicAdd(&gp->nbig, 1)] = i;
            else if (count > kSlots) big[atomicAdd(&gp->nmid, 1)] = i;
        }
        if (count > kSlots) return;
        int32_t* row = slots + int64_t(i) * kSlots;
        int a = lane < count ? list[lane] : INT32_MAX;
        a = wave_sort(a, true, lane);
        if (count > kWave) {
            // two runs, the second descending: one bitonic sequence of 128, merged
            int b = kWave + lane < count ? list[kWave + lane] : INT32_MAX;
            b = wave_sort(b, false, lane);
            const int lo = min(a, b);
            b = max(a, b);
            a = lo;
#pragma unroll
            for (int stride = kWave / 2; stride > 0; stride >>= 1) {
                a = bitonic_step(a, stride, (lane & stride) == 0);
                b = bitonic_step(b, stride, (lane & stride) == 0);
            }
            if (kWave + lane < count) row[kWave + lane] = b;
        }
        if (lane < count) row[lane] = a;
    }
};

template <typename T, bool HALF>
__global__ void __launch_bounds__(256) k_count_cells(const T* __restrict__ pos, int64_t n, const T* __restrict__ box,
                                                     T cutoff, NlGrid* __restrict__ gp,
                                                     const int32_t* __restrict__ cell_start,
                                                     const int32_t* __restrict__ cell_count,
                                                     const int32_t* __restrict__ atoms_sorted,
                                                     const PosW<T>* __restrict__ posw,
                                                     int32_t* __restrict__ counts, int32_t* __restrict__ big,
                                                     int32_t* __restrict__ slots) {
    const NlGrid g = *gp;
    if (g.brute) {
        count_all_pairs<T>(pos, n, box, cutoff, HALF ? MNX_NLIST_HALF : MNX_NLIST_FULL, gp, g, counts);
        return;
    }
    RowSink<T> sink{n, gp, counts, big, slots};
    scan_cells<T, HALF>(pos, box, cutoff, g, cell_start, cell_count, atoms_sorted, posw, sink);
}

// The pairs of every atom with at most kSlots neighbours, from its sorted row: half a wavefront per
// atom (52 neighbours of a full list at liquid density fill two passes of 32 lanes, 26 of a half
// list one); then what needs its own search.
template <typename T>
__global__ void __launch_bounds__(256) k_emit_slots(const T* __restrict__ pos, int64_t n, const T* __restrict__ box,
                                                    T cutoff, int mode, int layout, const NlGrid* __restrict__ gp,
                                                    const int32_t* __restrict__ cell_start,
                                                    const int32_t* __restrict__ cell_count,
                                                    const int32_t* __restrict__ atoms_sorted,
                                                    const int32_t* __restrict__ counts,
                                                    const int32_t* __restrict__ slots, const int32_t* __restrict__ big,
                                                    const int64_t* __restrict__ offsets, int64_t capacity,
                                                    int32_t* __restrict__ idx_i, int32_t* __restrict__ idx_j,
                                                    T* __restrict__ deltas, T* __restrict__ dist,
                                                    T* __restrict__ shifts) {
    __shared__ int32_t buf[kNlCap];
    static_assert(sizeof(buf) >= 8 * 2 * 96 * sizeof(double), "the vectors of 32 pairs per half wavefront");
    const int64_t i = int64_t(blockIdx.x) * 8 + (threadIdx.x >> 5);
    const int l = threadIdx.x & 31;
    if (!gp->brute && i < n) {
        T* vec = reinterpret_cast<T*>(buf) + (threadIdx.x >> 5) * 192;  // [delta | shift] of 32 pairs
        // the row's first 64 entries with the count and the offset (entries past the count are in the
        // row too), then the positions of both halves together: two round trips
        const int32_t* row = slots + i * kSlots;
        int jn[2] = {row[l], row[32 + l]};
        const int cnt = counts[i] > kSlots ? 0 : counts[i];
        const int64_t off = layout == MNX_NLIST_TRIANGULAR ? 0 : offsets[i];
        const T xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
        for (int k0 = 0; k0 < cnt; k0 += 64) {
            const int j[2] = {k0 + l < cnt ? jn[0] : -1, k0 + 32 + l < cnt ? jn[1] : -1};
            T px[2], py[2], pz[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int64_t a = j[h] < 0 ? i : j[h];
                px[h] = pos[3 * a];
                py[h] = pos[3 * a + 1];
                pz[h] = pos[3 * a + 2];
            }
            if (k0 + 64 < cnt) {
                jn[0] = row[k0 + 64 + l];
                jn[1] = row[k0 + 96 + l];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int first_k = k0 + 32 * h;
                if (first_k >= cnt) break;
                Geo<T> gg;
                const bool flip = i < j[h];  // the reference's orientation: larger index first
                geo_from_d<T>(box, flip ? px[h] - xi : xi - px[h], flip ? py[h] - yi : yi - py[h],
                              flip ? pz[h] - zi : zi - pz[h], box != nullptr, shifts != nullptr, gg);
                const int64_t slot = layout == MNX_NLIST_TRIANGULAR ? i * (i - 1) / 2 + j[h] : off + first_k + l;
                const bool in = j[h] >= 0 && slot < capacity;
                if (in) {
                    if (idx_i) idx_i[slot] = int32_t(i);
                    if (idx_j) idx_j[slot] = j[h];
                    if (dist) dist[slot] = gg.dist;
                }
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    gg.d[x] = flip ? -gg.d[x] : gg.d[x];
                    gg.shift[x] = flip ? -gg.shift[x] : gg.shift[x];
                }
                if (layout == MNX_NLIST_TRIANGULAR) {
                    for (int x = 0; in && x < 3; ++x) {
                        if (deltas) deltas[3 * slot + x] = gg.d[x];
                        if (shifts) shifts[3 * slot + x] = gg.shift[x];
                    }
                    continue;
                }
                wave_lds_fence();  // the vectors of the pass before are read
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    vec[3 * l + x] = gg.d[x];
                    vec[96 + 3 * l + x] = gg.shift[x];
                }
                wave_lds_fence();
                const int64_t first = 3 * (off + first_k);
                const int here = run_components(off + first_k, min(32, cnt - first_k), capacity);
#pragma unroll
                for (int x = l; x < 96; x += 32) {
                    if (x < here) {
                        if (deltas) deltas[first + x] = vec[x];
                        if (shifts) shifts[first + x] = vec[96 + x];
                    }
                }
            }
        }
    }
    if (!gp->brute && gp->nmid == 0 && gp->nbig == 0) return;
    const NlGrid g = *gp;
    emit_rest<T>(buf, pos, n, box, cutoff, mode, layout, g, cell_start, cell_count, atoms_sorted, big, offsets,
                 capacity, idx_i, idx_j, deltas, dist, shifts);
}

// Reference padding (-1 / NaN) for slots [from, capacity); `from` read from device when from_dev != null.
template <typename T>
__global__ void k_pad(int64_t from_host, const int64_t* __restrict__ from_dev, int64_t capacity,
                      int32_t* __restrict__ idx_i, int32_t* __restrict__ idx_j, T* __restrict__ deltas,
                      T* __restrict__ dist, T* __restrict__ shifts) {
    const int64_t from = from_dev ? *from_dev : from_host;
    const T nan = T(NAN);
    for (int64_t s = from + int64_t(blockIdx.x) * blockDim.x + threadIdx.x; s < capacity;
         s += int64_t(gridDim.x) * blockDim.x) {
        if (s < 0) continue;
        if (idx_i) idx_i[s] = -1;
        if (idx_j) idx_j[s] = -1;
        if (deltas) deltas[3 * s] = deltas[3 * s + 1] = deltas[3 * s + 2] = nan;
        if (dist) dist[s] = nan;
        if (shifts) shifts[3 * s] = shifts[3 * s + 1] = shifts[3 * s + 2] = nan;
    }
}

// offsets = exclusive scan of the counts (tile sums in `tiles`), offsets[n] and *d_total their sum;
// *d_total = -1 when some atom exceeded kNlCap neighbours.
__global__ void __launch_bounds__(kScanThreads) k_nl_offsets(const int32_t* __restrict__ counts, int64_t n,
                                                             const int64_t* __restrict__ tiles,
                                                             const NlGrid* __restrict__ gp,
                                                             int64_t* __restrict__ offsets,
                                                             int64_t* __restrict__ d_total) {
    __shared__ int64_t sh[kScanThreads];
    // the tiles before this one
    int64_t before = 0;
    for (int64_t t = threadIdx.x; t < blockIdx.x; t += kScanThreads) before += tiles[t];
    int64_t head;
    block_exclusive_scan<int64_t>(before, sh, &head);
    const int64_t base = int64_t(blockIdx.x) * kScanTile + int64_t(threadIdx.x) * kScanItems;
    int64_t v[kScanItems], sum = 0, total;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? counts[base + k] : 0;
        sum += v[k];
    }
    int64_t run = head + block_exclusive_scan<int64_t>(sum, sh, &total);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < n) offsets[base + k] = run;
        run += v[k];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        offsets[n] = head + total;
        if (d_total) *d_total = gp->overflow ? int64_t(-1) : head + total;
    }
}

// Cell grid and cell-ordered atoms of a system of more than kNlSmall atoms; ORDERED: by id within a
// cell (w.ids), for a scan that sums in the order of its candidates.
template <typename T, bool ORDERED>
int bin_atoms(const T* pos, int64_t n, double cutoff, const T* box, const NlWs& w, hipStream_t stream,
              int32_t* flag = nullptr) {
    const int tb = 256;
    MNX_REQUIRE(w.max_cells < (int64_t(1) << 31), "too many atoms");
    // cleared by a kernel rather than hipMemsetAsync, so the sequence can sit in a captured HIP graph
    hipLaunchKernelGGL((k_nl_clear<T>), dim3(ceil_div(w.max_cells, tb)), dim3(tb), 0, stream, w.cell_count, n, box,
                       cutoff, w.max_cells, w.grid, flag);
    MNX_CHECK_LAUNCH();
    if (!box) {
        hipLaunchKernelGGL((k_nl_bounds<T>), dim3(std::min<int64_t>(ceil_div(n, tb), 256)), dim3(tb), 0, stream, pos, n,
                           w.grid);
        MNX_CHECK_LAUNCH();
        hipLaunchKernelGGL((k_nl_open_grid<T>), dim3(1), dim3(1), 0, stream, n, cutoff, w.max_cells, w.grid);
        MNX_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL((k_bin<T>), dim3(ceil_div(n, tb)), dim3(tb), 0, stream, pos, n, w.grid, w.cell_of, w.rank,
                       w.cell_count);
    MNX_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_cell_runs, dim3(ceil_div(w.max_cells, kScanTile)), dim3(kScanThreads), 0, stream, w.grid,
                       w.cell_count, w.cell_start);
    MNX_CHECK_LAUNCH();
    if (ORDERED) {
        hipLaunchKernelGGL(k_place_ids, dim3(ceil_div(n, tb)), dim3(tb), 0, stream, n, w.grid, w.cell_of, w.rank,
                           w.cell_start, w.ids);
        MNX_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL((k_place<T, ORDERED>), dim3(ceil_div(n, tb)), dim3(tb), 0, stream, n, pos, box, w.grid,
                       w.cell_of, w.rank, w.cell_start, w.cell_count, w.ids, w.atoms_sorted,
                       static_cast<PosW<T>*>(w.posw));
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

template <typename T>
int nlist_count(const T* pos, int64_t n, double cutoff, const T* box, int mode, void* ws, size_t ws_bytes,
                int64_t* d_total, hipStream_t stream) {
    clear_error();
    MNX_REQUIRE(n >= 0 && n < (int64_t(1) << 31), "num_atoms out of range: %lld", (long long)n);
    MNX_REQUIRE(mode == MNX_NLIST_HALF || mode == MNX_NLIST_FULL, "bad mode %d", mode);
    MNX_REQUIRE(n == 0 || pos, "positions is null");
    MNX_REQUIRE(cutoff > 0, "cutoff must be positive");
    size_t need = 0;
    NlWs w = carve(ws, ws_bytes, n, &need);
    if (ws_bytes < need || !ws) return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
    const int tb = 256;
    if (n <= kNlSmall) {
        if (n > 0) {
            hipLaunchKernelGGL((k_small_count<T>), dim3(ceil_div(n, 4)), dim3(tb), 0, stream, pos, int(n), box,
                               T(cutoff), mode, int(ceil_div(n, kWave)), w.counts, w.masks);
            MNX_CHECK_LAUNCH();
        }
        hipLaunchKernelGGL(k_small_scan, dim3(1), dim3(kScanThreads), 0, stream, w.counts, int(n), w.offsets, d_total);
        MNX_CHECK_LAUNCH();
        return MNX_OK;
    }
    int rc = bin_atoms<T, false>(pos, n, cutoff, box, w, stream);
    if (rc) return rc;
    const PosW<T>* posw = static_cast<const PosW<T>*>(w.posw);
    const unsigned blocks = unsigned(std::min<int64_t>(w.max_cells, kNlBlocks));
    if (mode == MNX_NLIST_HALF)
        hipLaunchKernelGGL((k_count_cells<T, true>), dim3(blocks), dim3(tb), 0, stream, pos, n, box, T(cutoff),
                           w.grid, w.cell_start, w.cell_count, w.atoms_sorted, posw, w.counts, w.big, w.slots);
    else
        hipLaunchKernelGGL((k_count_cells<T, false>), dim3(blocks), dim3(tb), 0, stream, pos, n, box, T(cutoff),
                           w.grid, w.cell_start, w.cell_count, w.atoms_sorted, posw, w.counts, w.big, w.slots);
    MNX_CHECK_LAUNCH();
    const unsigned tiles = unsigned(ceil_div(n, kScanTile));
    hipLaunchKernelGGL((k_scan_tile_sums<int32_t, int64_t>), dim3(tiles), dim3(kScanThreads), 0, stream, w.counts, n,
                       w.tiles64);
    MNX_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_nl_offsets, dim3(tiles), dim3(kScanThreads), 0, stream, w.counts, n, w.tiles64, w.grid,
                       w.offsets, d_total);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

template <typename T>
int nlist_emit(const T* pos, int64_t n, double cutoff, const T* box, int mode, int layout, const void* ws,
               size_t ws_bytes, int64_t capacity, int32_t* idx_i, int32_t* idx_j, T* deltas, T* dist, T* shifts,
               hipStream_t stream) {
    clear_error();
    MNX_REQUIRE(capacity >= 0, "capacity must be >= 0");
    MNX_REQUIRE(layout == MNX_NLIST_COMPACT || layout == MNX_NLIST_EXACT ||
                    (layout == MNX_NLIST_TRIANGULAR && mode == MNX_NLIST_HALF),
                "triangular layout needs the half list");
    size_t need = 0;
    NlWs w = carve(const_cast<void*>(ws), ws_bytes, n, &need);
    if (ws_bytes < need || !ws) return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
    if (capacity == 0) return MNX_OK;
    const int tb = 256;
    if (layout != MNX_NLIST_EXACT) {
        const int64_t pad_blocks = std::min<int64_t>(ceil_div(capacity, tb), 65536);
        const int64_t* from = layout == MNX_NLIST_TRIANGULAR ? nullptr : w.offsets + n;  // the pair count
        hipLaunchKernelGGL((k_pad<T>), dim3(pad_blocks), dim3(tb), 0, stream, int64_t(0), from, capacity, idx_i, idx_j,
                           deltas, dist, shifts);
        MNX_CHECK_LAUNCH();
    }
    if (n == 0) return MNX_OK;
    if (n <= kNlSmall) {
        hipLaunchKernelGGL((k_small_emit<T>), dim3(ceil_div(n, 4)), dim3(tb), 0, stream, pos, int(n), box, mode, layout,
                           int(ceil_div(n, kWave)), w.masks, w.offsets, capacity, idx_i, idx_j, deltas, dist, shifts);
        MNX_CHECK_LAUNCH();
        return MNX_OK;
    }
    hipLaunchKernelGGL((k_emit_slots<T>), dim3(ceil_div(n, 8)), dim3(tb), 0, stream, pos, n, box, T(cutoff), mode,
                       layout, w.grid, w.cell_start, w.cell_count, w.atoms_sorted, w.counts, w.slots, w.big, w.offsets,
                       capacity, idx_i, idx_j, deltas, dist, shifts);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

template <typename T>
__global__ void k_nl_backward(const int32_t* __restrict__ ii, const int32_t* __restrict__ jj,
                              const T* __restrict__ d, const T* __restrict__ dist, const T* __restrict__ gd,
                              const T* __restrict__ gdist, int64_t slots, T* __restrict__ gpos) {
    const int64_t s = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= slots) return;
    const int i = ii[s], j = jj[s];
    if (i < 0 || j < 0) return;
    const T inv = T(1) / dist[s];
    const T gds = gdist ? gdist[s] : T(0);
    for (int k = 0; k < 3; ++k) {
        T g = (gd ? gd[3 * s + k] : T(0)) + d[3 * s + k] * inv * gds;
        atomicAdd(&gpos[3 * i + k], g);
        atomicAdd(&gpos[3 * j + k], -g);
    }
}

// ---------------------------------------------------------------------------
// Real-space Ewald sum over the pairs within the cutoff (the reference's direct
// term, src/molix/op/src/pme/pme_cpu.cpp:95-135,195-215, and the self term):
//   E = 1/2 sum_i sum_{j != i} k q_i q_j erfc(alpha r) / r - k alpha / sqrt(pi) sum_i q_i^2
// with dE/dpos and dE/dq, straight from the cell scan: every atom meets all of its
// neighbours (each pair twice), so its derivatives stay in registers and are stored
// once -- no pair list in memory, no atomics and no read of a pair count on the host.
// The pairs and their geometry are the neighbor list's, bit for bit; their terms are
// evaluated and summed in fp64 whatever the storage type.
// The cells' atoms are ordered by id, so the sums have a fixed order and the results the same bits every time
// (one launch and 5 to 10 us of a 420 us term at 50k atoms; by arrival, 4 energies in 8 float64 runs).
// Measured, 50k atoms (1.3 M pairs): 123 us and six launches, bound by the fp64 erfc and exp of both
// ends; the list (150 us), the energy over it (12) and its derivatives with scattered atomics (147)
// took over 300 us and 30 launches.
// ---------------------------------------------------------------------------
template <typename T>
struct RealArgs {
    const T* q;
    double alpha, coulomb;
    T *dpos, *dq;  // both or neither
    double* partials;
    int32_t* overflow;
};

template <typename T>
struct RealSink {
    static constexpr bool kStream = true;
    const T* pos;
    const T* box;
    RealArgs<T> a;
    double energy = 0.0;  // this lane's share over all centres
    double c1[kCentres], dq[kCentres], g[kCentres][3];
    int lower[kCentres];  // neighbours of lower index: the half list's count, which is what is limited

    __device__ __forceinline__ void begin(int q, int i) {
        c1[q] = double(a.q[i]);
        lower[q] = 0;
        dq[q] = g[q][0] = g[q][1] = g[q][2] = 0.0;
    }
    __device__ __forceinline__ void take(int q, int i, const int32_t* list, int count) {
        const int lane = threadIdx.x & (kWave - 1);
        const int j = list[lane];
        lower[q] += __popcll(__ballot(lane < count && j < i));
        if (lane >= count) return;
        Geo<T> gg;
        const bool flip = i < j;
        pair_geo<T>(pos, box, flip ? j : i, flip ? i : j, box != nullptr, false, gg);
        const double rr = double(gg.dist);
        const double inv = 1.0 / rr;
        const double ar = a.alpha * rr;
        const double ec = erfc(ar);
        const double pref = a.coulomb * inv;
        const double c2 = double(a.q[j]);
        energy += 0.5 * pref * ec * c1[q] * c2;
        if (a.dpos) {
            const double ex = exp(-ar * ar);
            const double dedr = pref * c1[q] * c2 * (ec + ar * ex * M_2_SQRTPI) * inv * inv;
            dq[q] += pref * ec * c2;
            const double f = flip ? dedr : -dedr;
            for (int k = 0; k < 3; ++k) g[q][k] += f * double(gg.d[k]);
        }
    }
    __device__ __forceinline__ void finish(int q, int i, const int32_t* list, int, int held) {
        const int lane = threadIdx.x & (kWave - 1);
        take(q, i, list, held);
        const double self = a.coulomb * a.alpha * (0.5 * M_2_SQRTPI);
        if (lane == 0) {
            energy -= self * c1[q] * c1[q];
            if (lower[q] > kNlCap) atomicExch(a.overflow, 1);
        }
        if (!a.dpos) return;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) {
            dq[q] += __shfl_xor(dq[q], o, kWave);
            for (int k = 0; k < 3; ++k) g[q][k] += __shfl_xor(g[q][k], o, kWave);
        }
        if (lane == 0) {
            a.dq[i] = T(dq[q] - 2.0 * self * c1[q]);
            for (int k = 0; k < 3; ++k) a.dpos[3 * int64_t(i) + k] = T(g[q][k]);
        }
    }
};

// Sum of one value per thread of a workgroup of four wavefronts into *out.
__device__ __forceinline__ void block_energy(double e, double* __restrict__ out) {
    __shared__ double red[kParts];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) e += __shfl_xor(e, o, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) *out = (red[0] + red[1]) + (red[2] + red[3]);
}

// Every candidate of atom i in id order through the sink (all pairs).
template <typename T>
__device__ __forceinline__ void real_all_pairs(const T* __restrict__ pos, int i, int64_t n, const T* __restrict__ box,
                                               T cutoff, const AcceptTest<T>& at, int32_t* list, RealSink<T>& sink) {
    const int lane = threadIdx.x & (kWave - 1);
    const T ax = pos[3 * int64_t(i)], ay = pos[3 * int64_t(i) + 1], az = pos[3 * int64_t(i) + 2];
    int count = 0, held = 0;
    sink.begin(0, i);
    for (int64_t base = 0; base < n; base += kWave) {
        const int64_t j = base + lane;
        bool ok = j < n && j != i;
        if (ok)
            ok = accept_xyz<T>(box, ax, ay, az, pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], box != nullptr, cutoff, at);
        const uint64_t m = __ballot(ok);
        if (ok) list[held + __popcll(m & ((uint64_t(1) << lane) - 1))] = int32_t(j);
        count += __popcll(m);
        held += __popcll(m);
        if (held >= kWave) {
            wave_lds_fence();
            sink.take(0, i, list, kWave);
            held -= kWave;
            const int rest = list[kWave + lane];
            if (lane < held) list[lane] = rest;
        }
    }
    wave_lds_fence();
    sink.finish(0, i, list, count, held);
    wave_lds_fence();
}

template <typename T>
__global__ void __launch_bounds__(256) k_real_small(const T* __restrict__ pos, int n, const T* __restrict__ box, T cutoff,
                                                    RealArgs<T> a) {
    __shared__ int32_t lists[kParts][2 * kWave];
    const int wave = threadIdx.x >> 6;
    const int i = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * kParts + wave);
    RealSink<T> sink{pos, box, a};
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.overflow = 0;
    if (i < n) {
        const AcceptTest<T> at = accept_test<T>(box, box != nullptr, !wide_box<T>(box, double(cutoff)), cutoff);
        real_all_pairs<T>(pos, i, n, box, cutoff, at, lists[wave], sink);
    }
    block_energy(sink.energy, a.partials + blockIdx.x);
}

template <typename T>
__global__ void __launch_bounds__(256) k_real_cells(const T* __restrict__ pos, int64_t n, const T* __restrict__ box,
                                                    T cutoff, const NlGrid* __restrict__ gp,
                                                    const int32_t* __restrict__ cell_start,
                                                    const int32_t* __restrict__ cell_count,
                                                    const int32_t* __restrict__ atoms_sorted,
                                                    const PosW<T>* __restrict__ posw, RealArgs<T> a) {
    __shared__ int32_t lists[kParts][2 * kWave];
    const NlGrid g = *gp;
    const int wave = threadIdx.x >> 6;
    RealSink<T> sink{pos, box, a};
    if (g.brute) {
        const AcceptTest<T> at = accept_test<T>(box, true, true, cutoff);
        for (int64_t i = int64_t(blockIdx.x) * kParts + wave; i < n; i += int64_t(gridDim.x) * kParts)
            real_all_pairs<T>(pos, int(i), n, box, cutoff, at, lists[wave], sink);
    } else {
        scan_cells<T, false>(pos, box, cutoff, g, cell_start, cell_count, atoms_sorted, posw, sink);
    }
    block_energy(sink.energy, a.partials + blockIdx.x);
}

// Workgroups (energy partial sums) of the real-space sum.
int64_t real_blocks(int64_t n) {
    return n <= kNlSmall ? ceil_div(n, kParts) : std::min<int64_t>(max_cells_for(n), kNlBlocks);
}

template <typename T>
int pme_real(const T* pos, const T* q, int64_t n, const T* box, double cutoff, double alpha, double coulomb, T* dpos,
             T* dq, double* partials, int32_t* overflow, void* ws, size_t ws_bytes, hipStream_t stream) {
    clear_error();
    MNX_REQUIRE(n >= 0 && n < (int64_t(1) << 30), "num_atoms out of range: %lld", (long long)n);
    MNX_REQUIRE(cutoff > 0, "cutoff must be positive");
    if (n == 0) return MNX_OK;
    MNX_REQUIRE(pos && q && box && partials && overflow, "null pointer argument");
    MNX_REQUIRE((dpos == nullptr) == (dq == nullptr), "dpos and dq must both be given or both be null");
    size_t need = 0;
    NlWs w = carve_real(ws, ws_bytes, n, sizeof(PosW<T>), &need);
    if (need && (ws_bytes < need || !ws))
        return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
    const RealArgs<T> a{q, alpha, coulomb, dpos, dq, partials, overflow};
    const unsigned blocks = unsigned(real_blocks(n));
    static_assert(kNlSmall <= kNlCap, "a small system cannot exceed the limit");
    if (n <= kNlSmall) {
        hipLaunchKernelGGL((k_real_small<T>), dim3(blocks), dim3(256), 0, stream, pos, int(n), box, T(cutoff), a);
        MNX_CHECK_LAUNCH();
        return MNX_OK;
    }
    int rc = bin_atoms<T, true>(pos, n, cutoff, box, w, stream, overflow);
    if (rc) return rc;
    hipLaunchKernelGGL((k_real_cells<T>), dim3(blocks), dim3(256), 0, stream, pos, n, box, T(cutoff), w.grid,
                       w.cell_start, w.cell_count, w.atoms_sorted, static_cast<const PosW<T>*>(w.posw), a);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

}  // namespace
}  // namespace mnx

using namespace mnx;

extern "C" {

size_t mnx_nlist_workspace_bytes(int64_t num_atoms) {
    size_t used = 0;
    carve(nullptr, 0, num_atoms < 0 ? 0 : num_atoms, &used);
    return used + 256;
}

int mnx_nlist_count_f32(const float* pos, int64_t n, double cutoff, const float* box, int32_t mode, void* ws,
                        size_t ws_bytes, int64_t* d_total, mnx_stream_t stream) {
    return nlist_count<float>(pos, n, cutoff, box, mode, ws, ws_bytes, d_total, (hipStream_t)stream);
}
int mnx_nlist_count_f64(const double* pos, int64_t n, double cutoff, const double* box, int32_t mode, void* ws,
                        size_t ws_bytes, int64_t* d_total, mnx_stream_t stream) {
    return nlist_count<double>(pos, n, cutoff, box, mode, ws, ws_bytes, d_total, (hipStream_t)stream);
}
int mnx_nlist_emit_f32(const float* pos, int64_t n, double cutoff, const float* box, int32_t mode, int32_t layout,
                       const void* ws, size_t ws_bytes, int64_t capacity, int32_t* idx_i, int32_t* idx_j,
                       float* deltas, float* distances, float* shifts, mnx_stream_t stream) {
    return nlist_emit<float>(pos, n, cutoff, box, mode, layout, ws, ws_bytes, capacity, idx_i, idx_j, deltas,
                             distances, shifts, (hipStream_t)stream);
}
int mnx_nlist_emit_f64(const double* pos, int64_t n, double cutoff, const double* box, int32_t mode,
                       int32_t layout, const void* ws, size_t ws_bytes, int64_t capacity, int32_t* idx_i,
                       int32_t* idx_j, double* deltas, double* distances, double* shifts, mnx_stream_t stream) {
    return nlist_emit<double>(pos, n, cutoff, box, mode, layout, ws, ws_bytes, capacity, idx_i, idx_j, deltas,
                              distances, shifts, (hipStream_t)stream);
}

int mnx_nlist_backward_f32(const int32_t* idx_i, const int32_t* idx_j, const float* deltas, const float* distances,
                           const float* grad_deltas, const float* grad_distances, int64_t num_slots,
                           int64_t num_atoms, float* grad_pos, mnx_stream_t stream) {
    clear_error();
    (void)num_atoms;
    if (num_slots <= 0) return MNX_OK;
    const int tb = 256;
    hipLaunchKernelGGL((k_nl_backward<float>), dim3(ceil_div(num_slots, tb)), dim3(tb), 0, (hipStream_t)stream,
                       idx_i, idx_j, deltas, distances, grad_deltas, grad_distances, num_slots, grad_pos);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

int mnx_nlist_backward_f64(const int32_t* idx_i, const int32_t* idx_j, const double* deltas, const double* distances,
                           const double* grad_deltas, const double* grad_distances, int64_t num_slots,
                           int64_t num_atoms, double* grad_pos, mnx_stream_t stream) {
    clear_error();
    (void)num_atoms;
    if (num_slots <= 0) return MNX_OK;
    const int tb = 256;
    hipLaunchKernelGGL((k_nl_backward<double>), dim3(ceil_div(num_slots, tb)), dim3(tb), 0, (hipStream_t)stream,
                       idx_i, idx_j, deltas, distances, grad_deltas, grad_distances, num_slots, grad_pos);
    MNX_CHECK_LAUNCH();
    return MNX_OK;
}

size_t mnx_pme_real_workspace_bytes(int64_t num_atoms, int32_t f64) {
    size_t used = 0;
    carve_real(nullptr, 0, num_atoms, f64 ? sizeof(PosW<double>) : sizeof(PosW<float>), &used);
    return used + 256;
}
int64_t mnx_pme_real_partials(int64_t num_atoms) { return num_atoms > 0 ? real_blocks(num_atoms) : 0; }

int mnx_pme_real_f32(const float* pos, const float* q, int64_t n, const float* box, double cutoff, double alpha,
                     double coulomb, float* dpos, float* dq, double* partials, int32_t* overflow, void* ws,
                     size_t ws_bytes, mnx_stream_t stream) {
    return pme_real<float>(pos, q, n, box, cutoff, alpha, coulomb, dpos, dq, partials, overflow, ws, ws_bytes,
                           (hipStream_t)stream);
}
int mnx_pme_real_f64(const double* pos, const double* q, int64_t n, const double* box, double cutoff, double alpha,
                     double coulomb, double* dpos, double* dq, double* partials, int32_t* overflow, void* ws,
                     size_t ws_bytes, mnx_stream_t stream) {
    return pme_real<double>(pos, q, n, box, cutoff, alpha, coulomb, dpos, dq, partials, overflow, ws, ws_bytes,
                            (hipStream_t)stream);
}

}  // extern "C"
