// Weight gradient of the equivariant (ir_mul) block linear (csrc/linear.hip;
// src/molrep/interaction/linear.py:43-105): for every (input block, output
// block) pair of one irrep
//   gw[wo + c * N + p] = scale * sum_{n < R, i < d} x[n][xcol + i xcomp + c]
//                                                 * g[n][gcol + i gcomp + p]
// i.e. A^T B over the rows (node n, component i), A and B read in place from
// the ir_mul rows.
//
// fp32-accurate products on the bf16 matrix cores, as in the block linear (three
// bf16 parts per operand value, the six partial products i + j <= 2, smallest
// first, v_mfma_f32_32x32x16_bf16).  A lane of that instruction holds 8 rows of
// one channel, and which rows is free as long as both operands agree: the lower
// half wavefront takes rows of the first half of a slab, the upper half the same
// rows of the second, so every load is 32 consecutive lanes of one row, its row
// offset is wave-uniform (scalar registers) and the operands go from global
// memory straight to registers: no LDS, no barrier, no transposed copy.  A
// wavefront owns a 32T x 32T tile of one pair's gradient over one slab of rows.
// T = 2 where every block is a multiple of 64 channels wide (one 8-byte load a
// lane, columns 2l and 2l + 1 in the two tiles; each value is split once for two
// products; the four tiles of a 128 x 128 block share their rows through the
// CU's L1), T = 1 otherwise.  Pairs with the same output block walk the same
// slabs side by side on one XCD, so that its L2 serves the gradient rows to all
// but the first.  Slabs are sized for two wavefronts per SIMD over all pairs
// together (one launch for the whole linear), at least 128 rows; their partial
// tiles are written in accumulator order and summed in a fixed order by a second
// kernel (deterministic, no atomics).
//
// Bound by reading x and g through two wavefronts' loads per SIMD: the linear
// after a 128-channel 0e+1o convolution (20k nodes, ten pairs, 574 MB) takes
// 200 us = 2.9 TB/s, the two pairs of a 0e+1o mixing (50k nodes, 205 MB) 67 us =
// 3.1 TB/s, both kernels together (profiles/timed_cases_kernel_stats.md).  More, shorter
// slabs cost partial tiles (in another session, against 217 and 55 us): 2950 wavefronts
// 229 / 71 us, 5900 247 / 91 us.  fp32 MFMAs instead of the
// split took 473 us, per-pair slabs (the gradient rows re-read from HBM) 268 us.
// The form before, torch gathers of every pair's rows into GEMM operands and a
// batched library GEMM each, took about 700 us over 30 launches.

#include <type_traits>

#include "bf16_split.h"
#include "common.h"

namespace mnx {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWgThreads = 256;
constexpr int kWgMaxTask = 40;  // pairs per launch (kernel arguments stay below 4 KB)
constexpr int kWgTargetWaves = 1980;
constexpr int kWgMinRows = 128;  // rows of a slab

// One pair.  Pairs of one output block (the same gradient columns) form a group: they share the
// group's slabs, and a slab's tiles of all of them are consecutive wavefronts.
struct WgTask {
    int32_t xcol, xcomp, M, gcol, gcomp, N, d, wo;
    float scale;
    int32_t mt, ntile;     // tiles along M, tiles in all
    int32_t tile0, gtiles; // first tile within the group, tiles of the group
    int32_t slabs;
    int32_t unit0;         // first wavefront of the group
    int32_t elem0;         // first output tile of the pair
};

struct WgArgs {
    WgTask task[kWgMaxTask];
    int32_t ntask, units, tiles;
};

template <int T>
__global__ void __launch_bounds__(kWgThreads) k_linear_wgrad(WgArgs p, const float* __restrict__ x, int64_t sx,
                                                             const float* __restrict__ g, int64_t sg, int64_t R,
                                                             float* __restrict__ part) {
    const int lane = threadIdx.x & (kWave - 1);
    const int half = lane >> 5, l32 = lane & 31;
    // Workgroups are dealt round-robin over the 8 XCDs: XCD b mod 8 takes a contiguous range of
    // them, so that a slab's pairs run side by side and read its gradient rows through one L2.
    const int blocks = (p.units + kWgThreads / kWave - 1) / (kWgThreads / kWave), per = (blocks + 7) / 8;
    const int block = int(blockIdx.x & 7) * per + int(blockIdx.x >> 3);
    const int unit = block * (kWgThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (block >= blocks || unit >= p.units) return;
    int t = 0;
    while (t + 1 < p.ntask && unit >= p.task[t + 1].unit0) ++t;  // the group's last pair
    const int u = unit - p.task[t].unit0;
    const int slab = u / p.task[t].gtiles, gt = u - slab * p.task[t].gtiles;
    while (gt < p.task[t].tile0) --t;
    const WgTask& k = p.task[t];
    const int tile = gt - k.tile0;
    const int tn = tile / k.mt, tm = tile - tn * k.mt;
    // the slab's nodes, split evenly over the slabs; the lower half wavefront takes the first hn of them
    const int64_t n0 = slab * R / k.slabs;
    const int nodes = int((slab + 1) * R / k.slabs - n0);
    const int d = k.d, hn = (nodes + 1) / 2, H = hn * d;
    const int n = nodes * d;  // rows
    const float* xb = x + n0 * sx + k.xcol;
    const float* gb = g + n0 * sg + k.gcol;
    // the host keeps a slab's byte offsets below 2^31
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)xb, (short)0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void*)gb, (short)0, 0x7fffffff, 0x00020000);
    // lane offsets (bytes): its half of the slab and its columns; columns past the block read its
    // last ones, and their products are never stored
    const int va = 4 * (half * hn * int(sx) + min(32 * T * tm + T * l32, k.M - T));
    const int vb = 4 * (half * hn * int(sg) + min(32 * T * tn + T * l32, k.N - T));
    const int mine = half ? n - H : H;  // rows of this lane's half
    // the next row's scalar offsets (bytes), common to both halves
    int comp = 0, oa = 0, og = 0;
    const int wa = 4 * (int(sx) - d * k.xcomp), wg = 4 * (int(sg) - d * k.gcomp);

    // rows [r, r + 8) of either half; TAIL: only those that exist, the rest zero
    auto load = [&](auto tail, int r, float (&a)[T][8], float (&b)[T][8]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if constexpr (decltype(tail)::value) {
#pragma unroll
                for (int i = 0; i < T; ++i) a[i][j] = b[i][j] = 0.f;
            }
            if (!decltype(tail)::value || r + j < mine) {
                if constexpr (T == 2) {
                    const auto u = __builtin_amdgcn_raw_buffer_load_b64(rx, va, oa, 0);
                    const auto v = __builtin_amdgcn_raw_buffer_load_b64(rg, vb, og, 0);
                    a[0][j] = __uint_as_float(u[0]);
                    a[1][j] = __uint_as_float(u[1]);
                    b[0][j] = __uint_as_float(v[0]);
                    b[1][j] = __uint_as_float(v[1]);
                } else {
                    a[0][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, va, oa, 0));
                    b[0][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rg, vb, og, 0));
                }
            }
            oa += 4 * k.xcomp;
            og += 4 * k.gcomp;
            if (++comp == d) {
                comp = 0;
                oa += wa;
                og += wg;
            }
        }
    };
    f32x16 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    struct Planes {
        bf16x8_t a[T][3], b[T][3];
    };
    auto split = [&](const float (&a)[T][8], const float (&b)[T][8], Planes& p_) {
#pragma unroll
        for (int i = 0; i < T; ++i) {
            bf16_split8(a[i], p_.a[i][0], p_.a[i][1], p_.a[i][2]);
            bf16_split8(b[i], p_.b[i][0], p_.b[i][1], p_.b[i][2]);
        }
    };
    auto products = [&](const Planes& p_) {
        constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
                    acc[i][j] =
                        __builtin_amdgcn_mfma_f32_32x32x16_bf16(p_.a[i][PA[q]], p_.b[j][PB[q]], acc[i][j], 0, 0, 0);
    };
    // Stages that both halves have whole run one load ahead (the last one's look-ahead is peeled);
    // the remaining d + 7 rows at most follow stage by stage.
    const int full = (n - H) / 8 * 8;
    constexpr auto kFull = std::integral_constant<bool, false>{};
    constexpr auto kTail = std::integral_constant<bool, true>{};
    float a[T][8], b[T][8];
    Planes pl;
    if (full > 0) {
        load(kFull, 0, a, b);
        for (int r = 8; r < full; r += 8) {
            split(a, b, pl);
            load(kFull, r, a, b);
            products(pl);
        }
        split(a, b, pl);
        products(pl);
    }
    for (int r = full; r < H; r += 8) {
        load(kTail, r, a, b);
        split(a, b, pl);
        products(pl);
    }
    // The parts of a value that bf16 cannot hold (infinite, or above its largest, 3.39e38) are not
    // finite, and their products are NaN: such a tile is formed again by fp32 products, whose infinities
    // and finite results are those of the sum.  The test is once per slab (a linear of 20k nodes, 128
    // channels, with its gradients: 659.2 us without, 660.6 with; runs differ by 0.6 %).
    float odd = 0.f;
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) odd = fmaf(acc[i][j][r], 0.f, odd);  // 0, or NaN of any infinity or NaN
    if (__ballot(odd != 0.f)) {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        comp = oa = og = 0;
        for (int r = 0; r < H; r += 8) {
            load(kTail, r, a, b);
#pragma unroll
            for (int z = 0; z < 8; ++z)
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int j = 0; j < T; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][z], b[j][z], acc[i][j], 0, 0, 0);
        }
    }
    float* dst = part + int64_t(unit) * (1024 * T * T) + lane;
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) dst[((i * T + j) * 16 + r) * kWave] = acc[i][j][r];
}

// gw = scale * (sum of the slabs' partial tiles).  A workgroup takes 64 elements (one accumulator
// register of one tile) with its four wavefronts summing every fourth slab, four loads in flight,
// and adds the four sums in order.
template <int T>
__global__ void __launch_bounds__(256) k_linear_wgrad_sum(WgArgs p, const float* __restrict__ part,
                                                          float* __restrict__ gw) {
    __shared__ float red[4][kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x >> 6;
    const int tl = blockIdx.x / (16 * T * T), reg = blockIdx.x - tl * (16 * T * T);
    int t = 0;
    while (t + 1 < p.ntask && tl >= p.task[t + 1].elem0) ++t;
    const WgTask& k = p.task[t];
    const int tile = tl - k.elem0;
    const int64_t step = int64_t(k.gtiles) * (1024 * T * T);
    const float* src = part + (int64_t(k.unit0) + k.tile0 + tile) * (1024 * T * T) + reg * kWave + lane;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    int z = w;
    for (; z + 12 < k.slabs; z += 16) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = src[(z + 4 * j) * step];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] += v[j];
    }
    for (int j = 0; z < k.slabs; z += 4, ++j) s[j] += src[z * step];
    red[w][lane] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (w) return;
    const float v = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
    // accumulator layout: register r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
    const int r = reg & 15, ij = reg >> 4, i = ij / T, j = ij - i * T;
    const int tn = tile / k.mt, tm = tile - tn * k.mt;
    // of tile (i, j), whose row / column q is channel T q + i / T q + j of the 32T-wide tile
    const int m = 32 * T * tm + T * (8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) + i;
    const int c = 32 * T * tn + T * (lane & 31) + j;
    if (m < k.M && c < k.N) gw[k.wo + int64_t(m) * k.N + c] = k.scale * v;
}

struct WgPlan {
    WgArgs args;
    int T;
};

// desc: 8 integers per pair (xcol, xcomp, M, gcol, gcomp, N, d, wo), pairs [first, last)
WgPlan wgrad_plan(const int64_t* desc, const float* scale, int first, int last, int64_t sx, int64_t sg, int64_t R) {
    WgPlan pl{};
    pl.T = 2;
    for (int i = first; i < last; ++i)
        if (desc[8 * i + 2] % 64 || desc[8 * i + 5] % 64) pl.T = 1;
    const int64_t w = 32 * pl.T;
    int64_t work = 0;  // tile rows
    for (int i = first; i < last; ++i)
        work += ceil_div(desc[8 * i + 2], w) * ceil_div(desc[8 * i + 5], w) * R * desc[8 * i + 6];
    const int64_t want = std::max<int64_t>(ceil_div(work, kWgTargetWaves), kWgMinRows);  // rows of a slab
    // byte offsets within a slab stay below 2^31
    const int64_t most = std::max<int64_t>((int64_t(1) << 29) / std::max(sx, sg) - 2, 1);
    int64_t units = 0, tiles = 0;
    for (int i = first; i < last;) {
        // the group of pairs with this output block
        const int64_t* e = desc + 8 * i;
        int j = i;
        int64_t gtiles = 0;
        for (; j < last && desc[8 * j + 3] == e[3] && desc[8 * j + 4] == e[4] && desc[8 * j + 5] == e[5] &&
               desc[8 * j + 6] == e[6]; ++j)
            gtiles += ceil_div(desc[8 * j + 2], w) * ceil_div(e[5], w);
        const int64_t nodes = std::min(most, ceil_div(want, e[6]));
        const int64_t slabs = ceil_div(R, nodes);
        int64_t tile0 = 0;
        for (; i < j; ++i) {
            e = desc + 8 * i;
            WgTask k;
            k.xcol = int32_t(e[0]);
            k.xcomp = int32_t(e[1]);
            k.M = int32_t(e[2]);
            k.gcol = int32_t(e[3]);
            k.gcomp = int32_t(e[4]);
            k.N = int32_t(e[5]);
            k.d = int32_t(e[6]);
            k.wo = int32_t(e[7]);
            k.scale = scale ? scale[i] : 1.f;
            k.mt = int32_t(ceil_div(e[2], w));
            k.ntile = int32_t(k.mt * ceil_div(e[5], w));
            k.tile0 = int32_t(tile0);
            k.gtiles = int32_t(gtiles);
            k.slabs = int32_t(slabs);
            k.unit0 = int32_t(units);
            k.elem0 = int32_t(tiles);
            tile0 += k.ntile;
            tiles += k.ntile;
            pl.args.task[i - first] = k;
        }
        units += slabs * gtiles;
    }
    pl.args.ntask = last - first;
    pl.args.units = int32_t(units);
    pl.args.tiles = int32_t(tiles);
    return pl;
}

int wgrad_check(const int64_t* desc, const float* scale, int32_t npair, int64_t sx, int64_t sg, int64_t R) {
    MNX_REQUIRE(npair >= 0 && (npair == 0 || (desc && scale)), "linear weight gradient: bad pair list");
    MNX_REQUIRE(R >= 0 && R < (int64_t(1) << 31) && sx >= 0 && sg >= 0 && sx < (int64_t(1) << 24) &&
                    sg < (int64_t(1) << 24), "linear weight gradient: sizes out of range");
    for (int i = 0; i < npair; ++i) {
        const int64_t* e = desc + 8 * i;
        MNX_REQUIRE(e[2] > 0 && e[5] > 0 && e[6] > 0 && e[0] >= 0 && e[1] >= 0 && e[3] >= 0 && e[4] >= 0 && e[7] >= 0 &&
                        e[2] <= 65536 && e[5] <= 65536 && e[6] <= 1024,
                    "linear weight gradient: bad pair %d", i);
        MNX_REQUIRE((e[0] | e[1] | e[2] | e[3] | e[4] | e[5] | sx | sg) % 2 == 0,
                    "linear weight gradient: pair %d: widths, offsets and strides must be even", i);
        MNX_REQUIRE(e[0] + (e[6] - 1) * e[1] + e[2] <= sx && e[3] + (e[6] - 1) * e[4] + e[5] <= sg,
                    "linear weight gradient: pair %d outside the rows", i);
        MNX_REQUIRE(e[7] + e[2] * e[5] < (int64_t(1) << 31), "linear weight gradient: pair %d outside the weights", i);
    }
    return MNX_OK;
}

}  // namespace
}  // namespace mnx

using namespace mnx;

extern "C" {

size_t mnx_block_linear_wgrad_workspace_bytes(const int64_t* desc, int32_t npair, int64_t x_stride, int64_t g_stride,
                                              int64_t R) {
    if (npair <= 0 || R <= 0 || !desc) return 0;
    size_t most = 0;
    for (int a = 0; a < npair; a += kWgMaxTask) {
        const int b = std::min(npair, a + kWgMaxTask);
        const WgPlan p = wgrad_plan(desc, nullptr, a, b, x_stride, g_stride, R);
        most = std::max(most, size_t(p.args.units) * 1024 * p.T * p.T * sizeof(float));
    }
    return most;
}

int mnx_block_linear_wgrad_f32(const float* x, int64_t x_stride, const float* g, int64_t g_stride, int64_t R,
                               int32_t npair, const int64_t* desc, const float* scale, float* gw, void* ws,
                               size_t ws_bytes, mnx_stream_t stream_) {
    clear_error();
    hipStream_t stream = (hipStream_t)stream_;
    int rc = wgrad_check(desc, scale, npair, x_stride, g_stride, R);
    if (rc) return rc;
    if (npair == 0) return MNX_OK;
    MNX_REQUIRE(gw && (R == 0 || (x && g)), "linear weight gradient: null pointer argument");
    MNX_REQUIRE((uintptr_t(x) | uintptr_t(g)) % 8 == 0, "linear weight gradient: rows must be 8-byte aligned");
    float* part = static_cast<float*>(ws);
    for (int a = 0; a < npair; a += kWgMaxTask) {
        const int b = std::min(npair, a + kWgMaxTask);
        const WgPlan p = wgrad_plan(desc, scale, a, b, x_stride, g_stride, R);
        const size_t need = size_t(p.args.units) * 1024 * p.T * p.T * sizeof(float);
        if (need && (!ws || ws_bytes < need))
            return set_error(MNX_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
        if (p.args.units > 0) {
            const dim3 grid(unsigned(8 * ceil_div(ceil_div(p.args.units, kWgThreads / kWave), 8)));
            if (p.T == 2)
                hipLaunchKernelGGL((k_linear_wgrad<2>), grid, dim3(kWgThreads), 0, stream, p.args, x, x_stride, g,
                                   g_stride, R, part);
            else
                hipLaunchKernelGGL((k_linear_wgrad<1>), grid, dim3(kWgThreads), 0, stream, p.args, x, x_stride, g,
                                   g_stride, R, part);
            MNX_CHECK_LAUNCH();
        }
        const dim3 sgrid(unsigned(p.args.tiles * 16 * p.T * p.T));
        if (p.T == 2)
            hipLaunchKernelGGL((k_linear_wgrad_sum<2>), sgrid, dim3(256), 0, stream, p.args, part, gw);
        else
            hipLaunchKernelGGL((k_linear_wgrad_sum<1>), sgrid, dim3(256), 0, stream, p.args, part, gw);
        MNX_CHECK_LAUNCH();
    }
    return MNX_OK;
}

}  // extern "C"
