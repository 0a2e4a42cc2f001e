// Equivariant (ir_mul) block linear on MFMA: one output irrep block
//   out[n][off + i*N + p] = sum_k A[(n, i)][k] * W[k][p]
// where row (n, i) of A (node n, irrep component i < d) concatenates
// segments of the input rows: segment s contributes len_s values starting at
// a[n*stride + col_s + i*comp_s].  This is cuet.Linear / e3nn Linear in ir_mul
// layout (src/molrep/interaction/linear.py:43-105): for an output block
// mul_o x ir the segments are the input blocks of the same irrep and W their
// stacked (mul_in x mul_o) weights, scaled by 1/sqrt(fan_in).  The gradient
// with respect to an input block is the same product with the output-gradient
// blocks as segments and the transposed weights.
//
// All blocks of a linear go in one launch.  A workgroup of four wavefronts takes
// 32 WR rows and up to 128 output columns (NT tiles of 32) of one block; each
// wavefront one 32-row tile (M side of v_mfma_f32_32x32x16_bf16) and NT WR / 4
// column tiles.  Blocks that read the same input columns with the same rows (the
// transposed product of several input blocks against one output irrep), and the
// column groups of one block, are dealt side by side to one XCD, whose L2 serves
// the shared rows.
//
// A is read straight from the strided input (32 bytes per lane and k-step, no
// gather copy) one chunk of 32 k ahead of its products.  W is read as the caller
// keeps it (rows of the parameter, its transpose, or the fragment order of
// mnx_block_linear_f32), scaled, split into its three bf16 planes and put into
// LDS in operand order by the whole workgroup, double-buffered with one barrier
// per chunk.  A 48 KB buffer pair and 160 registers let three workgroups share a
// CU, so that one's staging runs under the others' products; the two kernels
// that this one replaces (weights staged behind two barriers by eight wavefronts,
// or resident in 96 KB) held one workgroup per CU.
//
// WR (4, 2 or 1) is the largest that still gives two workgroups per CU over all
// blocks together: small systems spread a block's column tiles over the
// wavefronts instead of more rows.
//
// Bound by the six matrix-core products per value where K is a few hundred (the
// linear after a 128-channel 0e+1o convolution, 20k nodes, K 256 to 384: 271 us =
// 580 TFLOP/s of bf16 products, 288 us over four launches before), and by reading
// and writing the rows where it is 128 (its transpose, ten input blocks: 263 us
// against 362 us; the 0e+1o mixing of 50k nodes, 205 MB: 78 us = 2.6 TB/s, 80 us
// before).  The launches saved are the rest: one instead of one per block, and no
// gather of the weights into an operand order first (two more): the whole linear
// forward, backward and weight gradient takes 4 launches instead of 48.
//
// Arithmetic: fp32-accurate products on the bf16 matrix cores.  Each fp32
// operand x is split into x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 -
// x1); the six partial products x_i y_j with i + j <= 2 are accumulated in fp32,
// smallest first (the dropped terms are below 2^-25 |x y|), at 3/8 of the
// matrix-core cycles of fp32 MFMAs.  The D tiles are stored 128 contiguous bytes
// per row.
//
// Indexed mode (cuet.Linear(weight_classes=S, method="indexed_linear"),
// src/molrep/interaction/element_update.py:101-109,147-158): every node has a
// class (element) and its own weight set.  The caller groups the nodes by class
// (`order`, ascending class, rows of an out-of-range class last) and passes the
// class boundaries; workgroup b finds its class from those boundaries (each
// class owns ceil(count * d / (32 WR)) consecutive row groups), reads its rows
// through `order` and uses the weights of its class.  The out-of-range class
// writes zeros.  No host synchronisation: the grid is sized for the worst case
// (one partial workgroup per class) and surplus workgroups exit at once.

#include <algorithm>

#include "bf16_split.h"
#include "common.h"

namespace mnx {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kLinThreads = 256;
constexpr int kLinKC = 32;      // rows of W staged per chunk
constexpr int kLinMaxSeg = 8;   // input segments of a block
constexpr int kLinMaxBlock = 24, kLinMaxSegs = 72;  // per launch (kernel arguments below 4 KB)
constexpr int kLinFillWgs = 512;  // two workgroups per CU

// how the weights of a segment are stored: W[k][n] = w[woff + (k - k0) ld + n] (the parameter's
// rows), w[woff + n ld + k - k0] (its transpose), or MFMA fragment order (mnx_block_linear_f32)
enum { kLinRows = 0, kLinTransposed = 1, kLinFragments = 2 };

struct LinSeg {
    int32_t col;   // column of component 0
    int32_t comp;  // column step between components
    int32_t k0;    // first contraction index of the segment
    int32_t woff, ld;
    float scale;
};

struct LinBlock {
    int32_t seg0, nseg, K, N, d;
    uint32_t magic;  // ceil(2^32 / d)
    int32_t out_off, out_comp;
    // workgroups [wg0, ..) of the block's group, (row group, member) with members = (block, column
    // group); this block's members start at mem0
    int32_t wg0, members, mem0;
};

struct LinArgs {
    LinBlock blk[kLinMaxBlock];
    LinSeg seg[kLinMaxSegs];
    int32_t nblk, wgs;
    const float* a;
    int64_t a_stride;
    const float* w;
    float* out;
    int64_t out_stride;
    int64_t R;
    // indexed mode
    const int32_t* order;        // [R] node ids grouped by class
    const int32_t* class_start;  // [S + 2] first position in order of classes 0..S (S = out of range)
    int32_t S;
    int64_t w_class_stride;  // floats between the weight sets of consecutive classes
};

__device__ __forceinline__ f32x16 mfma_bf16(const bf16x8_t& a, const bf16x8_t& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <int NT, int WR, int WL, bool IDX>
__global__ void __launch_bounds__(kLinThreads, 3) k_block_linear(LinArgs p) {
    constexpr int NTW = NT * WR / 4;  // column tiles per wavefront
    static_assert(NTW * 4 == NT * WR, "the column tiles divide over the wavefronts");
    constexpr int COLS = 32 * NT;
    constexpr int ITEMS = (kLinKC / 8) * COLS;  // 8-value operands of a chunk
    constexpr int PER = (ITEMS + kLinThreads - 1) / kLinThreads;
    __shared__ bf16x8_t sw[2][3][kLinKC / 8][COLS];
    const int tid = threadIdx.x;
    const int lane = tid & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % WR, wc = wave / WR;
    const int per = (p.wgs + 7) / 8;
    const int wg = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
    if (wg >= p.wgs) return;
    int t = 0;
    while (t + 1 < p.nblk && wg >= p.blk[t + 1].wg0) ++t;  // the group's last block
    const int u = wg - p.blk[t].wg0;
    const int rg = u / p.blk[t].members, mem = u - rg * p.blk[t].members;
    while (mem < p.blk[t].mem0) --t;
    const LinBlock& B = p.blk[t];
    const LinSeg* seg = p.seg + B.seg0;
    const int col0 = (mem - B.mem0) * COLS;
    const int d = B.d;
    int K = B.K;
    int64_t row0, rows;
    const float* w = p.w;
    if (IDX) {
        // this workgroup's class: classes 0..S (S = out of range, zeros) own consecutive runs of
        // row groups
        int64_t first = 0;
        int cls = 0;
        for (; cls <= p.S; ++cls) {
            const int64_t cnt = int64_t(p.class_start[cls + 1] - p.class_start[cls]) * d;
            const int64_t nb = (cnt + 32 * WR - 1) / (32 * WR);
            if (rg < first + nb) break;
            first += nb;
        }
        if (cls > p.S) return;  // surplus workgroup (the grid is sized for the worst case)
        row0 = int64_t(p.class_start[cls]) * d + (rg - first) * (32 * WR) + wr * 32;
        rows = int64_t(p.class_start[cls + 1]) * d;
        if (cls == p.S) K = 0;  // out-of-range class: zero output
        else w += int64_t(cls) * p.w_class_stride;
    } else {
        row0 = int64_t(rg) * (32 * WR) + wr * 32;
        rows = p.R * d;
    }
    // (node, component) of row0 once; rows within the tile follow in 32-bit arithmetic
    auto over_d = [&](uint32_t v) { return d == 1 ? v : __umulhi(v, B.magic); };
    const int64_t n0 = row0 / d;
    const uint32_t c0 = uint32_t(row0 - n0 * d);
    // rows past the end read the last one; their products are never stored
    const int64_t last = rows - 1 - row0;  // may be negative: the whole tile is past the end
    const int rl = last < 0 ? 0 : (l32 < last ? l32 : int(last));
    const uint32_t q = over_d(c0 + rl);
    const int ci = int(c0 + rl - q * d);
    int64_t node = last < 0 ? 0 : n0 + q;
    if (IDX) node = last < 0 ? 0 : p.order[node];
    const float* arow = p.a + node * p.a_stride;
    // per segment, this lane's offset of contraction index k is base[s] + k (row-relative)
    int32_t base[kLinMaxSeg];
#pragma unroll
    for (int s = 0; s < kLinMaxSeg; ++s) base[s] = s < B.nseg ? seg[s].col + ci * seg[s].comp - seg[s].k0 : 0;

    f32x16 acc[NTW];
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;

    // k of a group past K is moved to the last group (in bounds) and its values zeroed at the split
    float av[2][8], wv[PER][8];
    auto load_a = [&](int k0) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int k = min(k0 + 16 * s + 8 * half, K - 8);
            int32_t off = base[0];
#pragma unroll
            for (int g = 1; g < kLinMaxSeg; ++g)
                if (g < B.nseg && k >= seg[g].k0) off = base[g];
            const f32x4 lo = *reinterpret_cast<const f32x4*>(arow + off + k);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(arow + off + k + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                av[s][j] = lo[j];
                av[s][4 + j] = hi[j];
            }
        }
    };
    // operand (k8, column) of this thread's i-th item; consecutive threads read consecutive memory
    auto item = [&](int i, int& k8, int& c) {
        const int it = min(tid + i * kLinThreads, ITEMS - 1);
        if (WL == kLinTransposed) {
            k8 = it & 3;
            c = it >> 2;
        } else {
            k8 = it / COLS;
            c = it % COLS;
        }
    };
    auto load_w = [&](int k0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int k8, c;
            item(i, k8, c);
            const int k = min(k0 + 8 * k8, K - 8), n = min(col0 + c, B.N - 1);
            if constexpr (WL == kLinFragments) {
                const int nch = (K + 63) / 64;
                const int64_t f = ((int64_t(col0 / COLS) * nch * 4 + (k >> 4)) * NT + (c >> 5)) * 64 + 32 * ((k >> 3) & 1) + (c & 31);
                const float* src = w + seg[0].woff + f * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) wv[i][j] = src[j];
            } else {
                int g = 0;
#pragma unroll
                for (int s = 1; s < kLinMaxSeg; ++s)
                    if (s < B.nseg && k >= seg[s].k0) g = s;
                const int kk = k - seg[g].k0;
                if constexpr (WL == kLinRows) {
                    const float* src = w + seg[g].woff + int64_t(kk) * seg[g].ld + n;
#pragma unroll
                    for (int j = 0; j < 8; ++j) wv[i][j] = src[int64_t(j) * seg[g].ld];
                } else {
                    const f32x4* src = reinterpret_cast<const f32x4*>(w + seg[g].woff + int64_t(n) * seg[g].ld + kk);
                    const f32x4 lo = src[0], hi = src[1];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        wv[i][j] = lo[j];
                        wv[i][4 + j] = hi[j];
                    }
                }
            }
        }
    };
    auto put_w = [&](int k0, int buf) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int k8, c;
            item(i, k8, c);
            const int k = k0 + 8 * k8;
            if constexpr (WL != kLinFragments) {
                int g = 0;
#pragma unroll
                for (int s = 1; s < kLinMaxSeg; ++s)
                    if (s < B.nseg && k >= seg[s].k0) g = s;
                const float sc = seg[g].scale;
#pragma unroll
                for (int j = 0; j < 8; ++j) wv[i][j] *= sc;
            }
            if (k >= K) {
#pragma unroll
                for (int j = 0; j < 8; ++j) wv[i][j] = 0.f;
            }
            bf16x8_t b0, b1, b2;
            bf16_split8(wv[i], b0, b1, b2);
            if (ITEMS % kLinThreads == 0 || tid + i * kLinThreads < ITEMS) {
                sw[buf][0][k8][c] = b0;
                sw[buf][1][k8][c] = b1;
                sw[buf][2][k8][c] = b2;
            }
        }
    };
    if (K > 0) {
        load_w(0);
        load_a(0);
        put_w(0, 0);
    }
    __syncthreads();
    for (int k0 = 0, c = 0; k0 < K; k0 += kLinKC, ++c) {
        // the last chunk reloads itself: no branch around the loads in flight
        const int next = k0 + kLinKC < K ? k0 + kLinKC : k0;
        load_w(next);
        bf16x8_t a[2][3];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (k0 + 16 * s + 8 * half >= K) {
#pragma unroll
                for (int j = 0; j < 8; ++j) av[s][j] = 0.f;
            }
            bf16_split8(av[s], a[s][0], a[s][1], a[s][2]);
        }
        load_a(next);
        constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int z = 0; z < 6; ++z)
#pragma unroll
                for (int i = 0; i < NTW; ++i)
                    acc[i] = mfma_bf16(a[s][PA[z]], sw[c & 1][PB[z]][2 * s + half][32 * (wc * NTW + i) + l32], acc[i]);
        if (next != k0) put_w(next, (c + 1) & 1);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int o = 8 * (r / 4) + 4 * half + r % 4;
        if (o > last) continue;
        const uint32_t qq = over_d(c0 + o);
        int64_t nn = n0 + qq;
        if (IDX) nn = p.order[nn];
        float* ob = p.out + nn * p.out_stride + B.out_off + int64_t(c0 + o - qq * d) * B.out_comp;
#pragma unroll
        for (int i = 0; i < NTW; ++i) {
            const int c = col0 + 32 * (wc * NTW + i) + l32;
            if (c < B.N) ob[c] = acc[i][r];
        }
    }
}

// output tiles of 32 columns per workgroup for N columns (the column-group width is 32 * this)
int lin_tiles(int N) { return N >= 128 ? 4 : int(ceil_div(N, 32)); }

template <int NT, int WR>
void launch_linear(int wl, bool idx, hipStream_t s, const LinArgs& p) {
    const dim3 grid(unsigned(8 * ceil_div(p.wgs, 8)));
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kLinThreads), 0, s, p); };
    if (wl == kLinRows) idx ? go(k_block_linear<NT, WR, kLinRows, true>) : go(k_block_linear<NT, WR, kLinRows, false>);
    else if (wl == kLinTransposed)
        idx ? go(k_block_linear<NT, WR, kLinTransposed, true>) : go(k_block_linear<NT, WR, kLinTransposed, false>);
    else idx ? go(k_block_linear<NT, WR, kLinFragments, true>) : go(k_block_linear<NT, WR, kLinFragments, false>);
}

struct LinCall {
    const float* a;
    int64_t a_stride, R;
    const float* w;
    int wl;
    int64_t w_class_stride;
    const int32_t* order;
    const int32_t* class_start;
    int32_t S;
    float* out;
    int64_t out_stride;
    hipStream_t stream;
};

// One output block as the entry points describe it.
struct LinDesc {
    int64_t out_off, out_comp, N, d;
    int nseg;
    const int64_t* seg;  // per segment: col, comp, len, woff, ld
    const float* scale;  // per segment (null: 1)
};

int check_desc(const LinCall& c, const LinDesc& b) {
    MNX_REQUIRE(b.nseg >= 0 && b.nseg <= kLinMaxSeg, "segment count %d not in [0, %d]", b.nseg, kLinMaxSeg);
    MNX_REQUIRE(b.d >= 1 && b.d < (1 << 16) && b.N >= 1 && b.N < (1 << 24) && c.R * b.d < (int64_t(1) << 36),
                "sizes out of range");
    MNX_REQUIRE(b.out_off >= 0 && b.out_comp >= 0 && b.out_off < (int64_t(1) << 31) && b.out_comp < (int64_t(1) << 31),
                "output block out of range");
    int64_t k = 0;
    for (int s = 0; s < b.nseg; ++s) {
        const int64_t* e = b.seg + 5 * s;
        MNX_REQUIRE(e[0] >= 0 && e[1] >= 0 && e[2] > 0 && e[2] % 8 == 0 && e[1] % 4 == 0 && e[0] % 4 == 0,
                    "segment %d: length must be a positive multiple of 8, offsets multiples of 4", s);
        MNX_REQUIRE(e[0] + (b.d - 1) * e[1] + e[2] < (int64_t(1) << 31), "segment %d exceeds 2^31 columns", s);
        MNX_REQUIRE(e[3] >= 0 && e[4] >= 0 && e[3] % 4 == 0 && (c.wl != kLinTransposed || e[4] % 4 == 0) &&
                        e[3] < (int64_t(1) << 31) && e[4] < (int64_t(1) << 31),
                    "segment %d: bad weight offsets", s);
        k += e[2];
    }
    MNX_REQUIRE(k < (int64_t(1) << 31), "too many contraction indices");
    return MNX_OK;
}

int run_linear(const LinCall& c, const LinDesc* desc, int ndesc) {
    MNX_REQUIRE(c.R >= 0 && c.a_stride >= 0 && c.out_stride >= 0, "sizes out of range");
    bool any = false;
    for (int i = 0; i < ndesc; ++i) {
        int rc = check_desc(c, desc[i]);
        if (rc) return rc;
        any = any || desc[i].nseg > 0;
    }
    if (c.R == 0 || ndesc == 0) return MNX_OK;
    MNX_REQUIRE(c.out && (!any || (c.a && c.w)), "null pointer argument");
    const bool idx = c.order != nullptr;
    MNX_REQUIRE(!idx || (c.class_start && c.S >= 1 && c.S <= 4096 && c.w_class_stride >= 0 && c.w_class_stride % 4 == 0),
                "indexed linear: bad class arguments");
    MNX_REQUIRE(!any || (c.a_stride % 4 == 0 && (uintptr_t)c.a % 16 == 0), "input rows must be 16-byte aligned");
    MNX_REQUIRE(!any || (uintptr_t)c.w % 16 == 0, "weights must be 16-byte aligned");
    auto fits = [](const LinDesc& x, const LinDesc& y) {  // the same input columns and rows
        if (x.d != y.d || x.nseg != y.nseg || x.nseg == 0) return false;
        for (int s = 0; s < x.nseg; ++s)
            for (int k = 0; k < 3; ++k)
                if (x.seg[5 * s + k] != y.seg[5 * s + k]) return false;
        return true;
    };
    for (int nt = 1; nt <= 4; ++nt) {
        // workgroups of 128 rows over the blocks of this width
        int64_t wgs4 = 0;
        for (int i = 0; i < ndesc; ++i)
            if (lin_tiles(int(desc[i].N)) == nt) wgs4 += ceil_div(c.R * desc[i].d, 128) * ceil_div(desc[i].N, 32 * nt);
        if (wgs4 == 0) continue;
        const int wr = wgs4 >= kLinFillWgs || nt == 1 || nt == 3 ? 4 : (2 * wgs4 >= kLinFillWgs || nt == 2 ? 2 : 1);
        for (int i = 0; i < ndesc;) {
            LinArgs p{};
            int segs = 0;
            int64_t wgs = 0;
            int lead = -1;  // descriptor of the current group's first block
            for (; i < ndesc && p.nblk < kLinMaxBlock; ++i) {
                const LinDesc& b = desc[i];
                if (lin_tiles(int(b.N)) != nt) continue;
                const int64_t rowg = ceil_div(c.R * b.d, 32 * wr) + (idx ? c.S + 1 : 0);
                const int64_t more = rowg * ceil_div(b.N, 32 * nt);
                MNX_REQUIRE(more < (int64_t(1) << 30), "too many rows");
                if (segs + b.nseg > kLinMaxSegs || wgs + more >= (int64_t(1) << 30)) break;
                LinBlock& q = p.blk[p.nblk];
                q.seg0 = segs;
                q.nseg = b.nseg;
                q.N = int32_t(b.N);
                q.d = int32_t(b.d);
                q.magic = uint32_t(((uint64_t(1) << 32) + b.d - 1) / b.d);
                q.out_off = int32_t(b.out_off);
                q.out_comp = int32_t(b.out_comp);
                for (int s = 0; s < b.nseg; ++s) {
                    const int64_t* e = b.seg + 5 * s;
                    p.seg[segs++] = LinSeg{int32_t(e[0]), int32_t(e[1]), q.K, int32_t(e[3]), int32_t(e[4]),
                                           b.scale ? b.scale[s] : 1.f};
                    q.K += int32_t(e[2]);
                }
                const int cols = int(ceil_div(b.N, 32 * nt));
                if (lead >= 0 && fits(desc[lead], b)) {  // joins the group of the block before
                    const LinBlock& f = p.blk[p.nblk - 1];
                    q.wg0 = f.wg0;
                    q.mem0 = f.members;
                    q.members = f.members + cols;
                    for (int k = p.nblk - 1; k >= 0 && p.blk[k].wg0 == q.wg0; --k) p.blk[k].members = q.members;
                } else {
                    q.wg0 = int32_t(wgs);
                    q.mem0 = 0;
                    q.members = cols;
                    lead = i;
                }
                wgs += more;
                ++p.nblk;
            }
            if (p.nblk == 0) continue;  // the rest of the list has other widths
            p.wgs = int32_t(wgs);
            p.a = c.a;
            p.a_stride = c.a_stride;
            p.w = c.w;
            p.out = c.out;
            p.out_stride = c.out_stride;
            p.R = c.R;
            p.order = c.order;
            p.class_start = c.class_start;
            p.S = c.S;
            p.w_class_stride = c.w_class_stride;
            if (nt == 1) launch_linear<1, 4>(c.wl, idx, c.stream, p);
            else if (nt == 2) wr == 4 ? launch_linear<2, 4>(c.wl, idx, c.stream, p) : launch_linear<2, 2>(c.wl, idx, c.stream, p);
            else if (nt == 3) launch_linear<3, 4>(c.wl, idx, c.stream, p);
            else if (wr == 4) launch_linear<4, 4>(c.wl, idx, c.stream, p);
            else if (wr == 2) launch_linear<4, 2>(c.wl, idx, c.stream, p);
            else launch_linear<4, 1>(c.wl, idx, c.stream, p);
            MNX_CHECK_LAUNCH();
        }
    }
    return MNX_OK;
}

// The entry points with fragment-ordered weights: one block.
int frag_linear(const float* a, int64_t a_stride, int32_t nseg, const int64_t* seg_col, const int32_t* seg_comp,
                const int32_t* seg_len, const float* w, int32_t N, int64_t R, int32_t d, float* out,
                int64_t out_stride, int64_t out_off, int32_t out_comp, const int32_t* order,
                const int32_t* class_start, int32_t S, int64_t w_class_stride, hipStream_t stream) {
    MNX_REQUIRE(nseg >= 0 && nseg <= kLinMaxSeg, "segment count %d not in [0, %d]", nseg, kLinMaxSeg);
    MNX_REQUIRE(nseg == 0 || (seg_col && seg_comp && seg_len), "null pointer argument");
    int64_t seg[5 * kLinMaxSeg];
    for (int s = 0; s < nseg; ++s) {
        const int64_t e[5] = {seg_col[s], seg_comp[s], seg_len[s], 0, 0};
        std::copy(e, e + 5, seg + 5 * s);
    }
    const LinCall c{a, a_stride, R, w, kLinFragments, w_class_stride, order, class_start, S, out, out_stride, stream};
    const LinDesc b{out_off, out_comp, N, d, nseg, seg, nullptr};
    return run_linear(c, &b, 1);
}

}  // namespace
}  // namespace mnx

using namespace mnx;

extern "C" {

int64_t mnx_block_linear_frag_floats(int32_t K, int32_t N) {
    if (K < 0 || N < 1) return -1;
    const int nt = lin_tiles(N);
    return ceil_div(N, nt * 32) * ceil_div(K, 64) * int64_t(4) * nt * kWave * 8;
}

int mnx_block_linear_f32(const float* a, int64_t a_stride, int32_t nseg, const int64_t* seg_col,
                         const int32_t* seg_comp, const int32_t* seg_len, const float* w, int32_t N, int64_t R,
                         int32_t d, float* out, int64_t out_stride, int64_t out_off, int32_t out_comp,
                         mnx_stream_t stream) {
    clear_error();
    return frag_linear(a, a_stride, nseg, seg_col, seg_comp, seg_len, w, N, R, d, out, out_stride, out_off, out_comp,
                       nullptr, nullptr, 0, 0, (hipStream_t)stream);
}

int mnx_indexed_block_linear_f32(const float* a, int64_t a_stride, int32_t nseg, const int64_t* seg_col,
                                 const int32_t* seg_comp, const int32_t* seg_len, const float* w,
                                 int64_t w_class_stride, int32_t num_classes, const int32_t* order,
                                 const int32_t* class_start, int32_t N, int64_t R, int32_t d, float* out,
                                 int64_t out_stride, int64_t out_off, int32_t out_comp, mnx_stream_t stream) {
    clear_error();
    MNX_REQUIRE(order && class_start, "indexed linear: order and class_start are required");
    return frag_linear(a, a_stride, nseg, seg_col, seg_comp, seg_len, w, N, R, d, out, out_stride, out_off, out_comp,
                       order, class_start, num_classes, w_class_stride, (hipStream_t)stream);
}

int mnx_linear_blocks_f32(const float* a, int64_t a_stride, int64_t R, const float* w, int32_t transposed,
                          int64_t w_class_stride, int32_t num_classes, const int32_t* order,
                          const int32_t* class_start, int32_t nblocks, const int64_t* desc, const float* scale,
                          float* out, int64_t out_stride, mnx_stream_t stream) {
    clear_error();
    MNX_REQUIRE(nblocks >= 0 && nblocks <= 4096 && (nblocks == 0 || desc), "linear blocks: bad block list");
    MNX_REQUIRE((order == nullptr) == (class_start == nullptr), "linear blocks: order and class_start go together");
    LinDesc b[64];
    const LinCall c{a, a_stride, R, w, transposed ? kLinTransposed : kLinRows, w_class_stride, order, class_start,
                    num_classes, out, out_stride, (hipStream_t)stream};
    int n = 0;
    for (int i = 0; i < nblocks; ++i) {
        MNX_REQUIRE(desc[4] >= 0 && desc[4] <= kLinMaxSeg, "segment count %lld not in [0, %d]", (long long)desc[4],
                    kLinMaxSeg);
        MNX_REQUIRE(desc[4] == 0 || scale, "null pointer argument");
        b[n++] = LinDesc{desc[0], desc[1], desc[2], desc[3], int(desc[4]), desc + 5, scale};
        scale = scale ? scale + desc[4] : nullptr;
        desc += 5 + 5 * desc[4];
        if (n == 64 || i + 1 == nblocks) {
            const int rc = run_linear(c, b, n);
            if (rc) return rc;
            n = 0;
        }
    }
    return MNX_OK;
}

}  // extern "C"
