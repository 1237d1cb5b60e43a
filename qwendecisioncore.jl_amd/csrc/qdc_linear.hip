// qdc_linear.hip -- bf16 projections back into the residual stream, for row counts
// at which their output has too few tiles to fill the chip.
//
// The output and MLP down projections of a layer are [rows, hidden]: at 1200 rows
// and 1024 columns, 80 tiles of 128 x 128 for 256 compute units, each with an inner
// dimension of up to 7168 to walk alone.  Here the inner dimension is cut into
// `parts` as well, every tile of every part a workgroup of its own that leaves fp32
// sums, and the pass that follows anyway -- the residual add and the next RMSNorm --
// adds the parts in order as it reads them.  A step of 64 values (16 products a
// wavefront, 512 cycles) takes about 1450 where a workgroup has its unit alone: its
// LDS writes, reads and products follow each other, so two workgroups a unit gain
// most.  Product + residual norm, library / here, us: 3584 split columns to 1024 at
// 64, 300, 600, 1200, 1800 rows 36 / 17, 35 / 21, 48 / 28, 67 / 43, 64 / 48; 3584 bf16
// 22 / 14, 22 / 19, 26 / 21, 39 / 31, 36 / 34; 6144 split to 2048 at 600 rows 106 / 61.
//
// Operands: a [rows, inner], w [cols, inner] as a checkpoint stores it, both with
// the inner dimension contiguous.  A split `a` (each group of 4 values as [4 hi |
// 4 lo]) multiplies each group of 4 weights twice: the lane that holds such a group
// repeats its 8 bytes of w in registers, so w is stored, loaded and staged once.
#include "qdc_common.hpp"
#include "qdc_hip_workspace.h"

namespace qdc {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kTile = 128;  // rows and columns of a tile; 4 wavefronts of 64 x 64
constexpr int kSlots = 64;  // bf16 values of a row of `a` per step

struct Linear {
    const bf16_t *a, *w;
    float *parts;            // [parts][rows][cols]
    int64_t ld_a, ld_w;
    int rows, cols, steps;   // steps of kSlots
};

template <bool SPLIT> __global__ __launch_bounds__(kBlock, 2) void linear_parts(Linear p) {
    constexpr int WK = SPLIT ? kSlots / 2 : kSlots;  // weights per step and column
    constexpr int ALD = kSlots + 8;                  // LDS row strides: 4 and 18 banks, so the
    constexpr int WLD = SPLIT ? WK + 4 : WK + 8;     // rows of a read fall on different banks
    constexpr int AN = kTile * kSlots / 8 / kBlock, WN = kTile * WK / 8 / kBlock;
    __shared__ __align__(16) bf16_t sa[2][kTile * ALD], sw[2][kTile * WLD];
    const int tid = threadIdx.x, l = tid % kWave, wv = tid / kWave;
    const int lq = l % 32, lh = l / 32;
    const int n0 = blockIdx.x * kTile, m0 = blockIdx.y * kTile;
    const int first = (int)((int64_t)p.steps * blockIdx.z / gridDim.z);
    const int last = (int)((int64_t)p.steps * (blockIdx.z + 1) / gridDim.z);
    const int mw = 64 * (wv / 2), nw = 64 * (wv % 2);  // this wavefront's corner

    // two steps' values on their way: memory is further away than one step's products
    u32x4 xa[2][AN], xw[2][WN];
    uint32_t oa[AN], ow[WN];  // byte offsets of this thread's pieces, from a uniform base
#pragma unroll
    for (int n = 0; n < AN; ++n) {
        const int i = tid + n * kBlock, r = min(m0 + i / (kSlots / 8), p.rows - 1);
        oa[n] = 2u * ((uint32_t)r * (uint32_t)p.ld_a + 8u * (i % (kSlots / 8)));
    }
#pragma unroll
    for (int n = 0; n < WN; ++n) {
        const int i = tid + n * kBlock, r = n0 + i / (WK / 8);
        ow[n] = 2u * ((uint32_t)r * (uint32_t)p.ld_w + 8u * (i % (WK / 8)));
    }
    auto load = [&](int s, int set) {
        const int t = min(s, last - 1);  // past the end: loaded, not used
        const char *ab = reinterpret_cast<const char *>(p.a + (int64_t)t * kSlots);
        const char *wb = reinterpret_cast<const char *>(p.w + (int64_t)t * WK);
#pragma unroll
        for (int n = 0; n < AN; ++n) xa[set][n] = load_raw(ab + oa[n]);
#pragma unroll
        for (int n = 0; n < WN; ++n) xw[set][n] = load_raw(wb + ow[n]);
    };
    auto stage = [&](int buf, int set) {
#pragma unroll
        for (int n = 0; n < AN; ++n) {
            const int i = tid + n * kBlock;
            *reinterpret_cast<u32x4 *>(
                &sa[buf][i / (kSlots / 8) * ALD + 8 * (i % (kSlots / 8))]) = xa[set][n];
        }
#pragma unroll
        for (int n = 0; n < WN; ++n) {
            const int i = tid + n * kBlock;
            bf16_t *dst = &sw[buf][i / (WK / 8) * WLD + 8 * (i % (WK / 8))];
            if constexpr (SPLIT) {  // rows of 72 bytes
                *reinterpret_cast<u32x2 *>(dst) = u32x2{xw[set][n][0], xw[set][n][1]};
                *reinterpret_cast<u32x2 *>(dst + 4) = u32x2{xw[set][n][2], xw[set][n][3]};
            } else {
                *reinterpret_cast<u32x4 *>(dst) = xw[set][n];
            }
        }
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // (all of a step's operands read before its first product measured 6% slower)
    auto products = [&](int buf) {
#pragma unroll
        for (int k = 0; k < kSlots / 16; ++k) {
            bf16x8 af[2], wf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                af[i] = *reinterpret_cast<const bf16x8 *>(
                    &sa[buf][(mw + 32 * i + lq) * ALD + 16 * k + 8 * lh]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const bf16_t *src = &sw[buf][(nw + 32 * j + lq) * WLD];
                if constexpr (SPLIT) {
                    const u32x2 g = *reinterpret_cast<const u32x2 *>(src + 8 * k + 4 * lh);
                    wf[j] = __builtin_bit_cast(bf16x8, u32x4{g[0], g[1], g[0], g[1]});
                } else {
                    wf[j] = *reinterpret_cast<const bf16x8 *>(src + 16 * k + 8 * lh);
                }
            }
            // transposed: a lane holds one row of the output, 4 consecutive columns
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], af[i], acc[i][j],
                                                                        0, 0, 0);
        }
    };
    load(first, 0);
    load(first + 1, 1);
    stage(0, 0);
    __syncthreads();
    for (int s = first; s < last; s += 2)
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // step s + h: buffer h, set h free for s + h + 2
            if (s + h >= last) break;  // uniform
            load(s + h + 2, h);
            __builtin_amdgcn_sched_barrier(0);  // the loads leave before the products
            products(h);
            stage(h ^ 1, h ^ 1);  // that buffer was read a step ago, a barrier back
            __syncthreads();
        }
    float *out = p.parts + (int64_t)blockIdx.z * p.rows * p.cols;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = m0 + mw + 32 * i + lq;
        if (row >= p.rows) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<f32x4 *>(out + (int64_t)row * p.cols + n0 + nw + 32 * j + 8 * r +
                                           4 * lh) =
                    f32x4{acc[i][j][4 * r], acc[i][j][4 * r + 1], acc[i][j][4 * r + 2],
                          acc[i][j][4 * r + 3]};
    }
}

struct Merge {
    float *residual;
    void *normed;
    const float *x, *parts;
    const void *norm;
    const int32_t *mask;
    int64_t stride;  // elements between parts
    int rows, width, n;
    float eps;
};

// residual = x + sum of the parts, normed = rms(residual) * (1 + norm) * mask: a
// wavefront per row, 4 columns per lane and chunk.
template <int CPL, typename TO> __global__ __launch_bounds__(kBlock) void merge_parts(Merge m) {
    typedef Aux<TO> TW;
    const int l = threadIdx.x % kWave;
    const int row = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= m.rows) return;
    const int64_t base = (int64_t)row * m.width + 4 * l;
    f32x4 v[CPL], x[CPL];
    Frag<TW, 4> w[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int64_t o = base + 4 * kWave * c;
        x[c] = __builtin_bit_cast(f32x4, load_raw(m.x + o));
        v[c] = __builtin_bit_cast(f32x4, load_raw(m.parts + o));
        w[c] = load_frag<TW, 4>(reinterpret_cast<const TW *>(m.norm) + 4 * l + 4 * kWave * c);
    }
    for (int n = 1; n < m.n; ++n)
#pragma unroll
        for (int c = 0; c < CPL; ++c)
            v[c] += __builtin_bit_cast(f32x4,
                                       load_raw(m.parts + n * m.stride + base + 4 * kWave * c));
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        v[c] += x[c];
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = __builtin_fmaf(v[c][j], v[c][j], ss);
    }
    const float s = rms_scale(group_sum<kWave>(ss), (float)m.width, m.eps);
    const float keep = m.mask ? (float)m.mask[row] : 1.0f;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int64_t o = base + 4 * kWave * c;
        float g[4], y[4], r[4];
        unpack(w[c], g);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r[j] = v[c][j];
            y[j] = (v[c][j] * s) * (1.0f + g[j]) * keep;
        }
        store_frag<4>(m.residual + o, r);
        store_frag<4>(reinterpret_cast<TO *>(m.normed) + o, y);
    }
}

}  // namespace
}  // namespace qdc

using namespace qdc;

extern "C" int32_t qdc_linear_parts(float *out, const void *a, const void *w, int64_t rows,
                                    int64_t inner, int64_t cols, int64_t ld_a, int64_t ld_w,
                                    int64_t parts, int32_t a_dtype, hipStream_t stream) {
    const bool split = a_dtype == QDC_BF16X2;
    if (a_dtype != QDC_BF16 && !split) return QDC_ERR_DTYPE;
    const int64_t lim = (int64_t)1 << 24, slots = split ? 2 * inner : inner;
    if (rows < 0 || inner <= 0 || cols <= 0 || rows >= lim || inner >= lim || cols >= lim ||
        parts <= 0 || parts > 64)
        return QDC_ERR_SHAPE;
    if (slots % kSlots || cols % kTile || parts > slots / kSlots || ld_a < slots || ld_w < inner ||
        ld_a % 8 || ld_w % 8)
        return QDC_ERR_SHAPE;
    if (rows == 0) return QDC_OK;
    const int64_t row_tiles = ceil_div(rows, (int64_t)kTile);
    // byte offsets into a and w are 32 bits wide
    const int64_t lim32 = (int64_t)1 << 31;
    if (row_tiles > 65535 || rows * ld_a >= lim32 || cols * ld_w >= lim32) return QDC_ERR_SHAPE;
    if (!out || !a || !w) return QDC_ERR_NULL;
    if (!aligned16(out) || !aligned16(a) || !aligned16(w)) return QDC_ERR_SHAPE;
    const int64_t bytes = parts * rows * cols * 4;
    if (overlaps(out, bytes, a, ((rows - 1) * ld_a + slots) * 2) ||
        overlaps(out, bytes, w, ((cols - 1) * ld_w + inner) * 2))
        return QDC_ERR_ALIAS;
    Linear p{};
    p.a = reinterpret_cast<const bf16_t *>(a);
    p.w = reinterpret_cast<const bf16_t *>(w);
    p.parts = out;
    p.ld_a = ld_a;
    p.ld_w = ld_w;
    p.rows = (int)rows;
    p.cols = (int)cols;
    p.steps = (int)(slots / kSlots);
    const dim3 grid((uint32_t)(cols / kTile), (uint32_t)row_tiles, (uint32_t)parts);
    if (split) hipLaunchKernelGGL((linear_parts<true>), grid, dim3(kBlock), 0, stream, p);
    else hipLaunchKernelGGL((linear_parts<false>), grid, dim3(kBlock), 0, stream, p);
    return launch_status();
}

extern "C" int32_t qdc_residual_rms_parts(float *residual, void *normed, const float *x,
                                          const float *sums, int64_t parts, const void *norm,
                                          const int32_t *mask, int64_t rows, int64_t width,
                                          float eps, int32_t out_dtype, hipStream_t stream) {
    const bool split = out_dtype == QDC_BF16X2;
    if (!valid_dtype(out_dtype) && !split) return QDC_ERR_DTYPE;
    if (rows < 0 || rows >= ((int64_t)1 << 24) || parts <= 0 || parts > 64) return QDC_ERR_SHAPE;
    if (width != 256 && width != 512 && width != 1024 && width != 2048) return QDC_ERR_SHAPE;
    if (rows == 0) return QDC_OK;
    if (!residual || !normed || !x || !sums || !norm) return QDC_ERR_NULL;
    if (!aligned16(residual) || !aligned16(normed) || !aligned16(x) || !aligned16(sums) ||
        !aligned16(norm) || ((uintptr_t)mask & 3u))
        return QDC_ERR_SHAPE;
    const int64_t bytes = rows * width * 4, nbytes = rows * width * elem_size(out_dtype);
    const int64_t wbytes = width * (out_dtype == QDC_F32 ? 4 : 2);
    if (overlaps(residual, bytes, normed, nbytes) || overlaps(residual, bytes, sums, parts * bytes) ||
        overlaps(normed, nbytes, sums, parts * bytes) || overlaps(normed, nbytes, x, bytes) ||
        (residual != x && overlaps(residual, bytes, x, bytes)) ||
        overlaps(residual, bytes, norm, wbytes) || overlaps(normed, nbytes, norm, wbytes) ||
        (mask && (overlaps(residual, bytes, mask, rows * 4) ||
                  overlaps(normed, nbytes, mask, rows * 4))))
        return QDC_ERR_ALIAS;
    Merge m{};
    m.residual = residual;
    m.normed = normed;
    m.x = x;
    m.parts = sums;
    m.norm = norm;
    m.mask = mask;
    m.stride = rows * width;
    m.rows = (int)rows;
    m.width = (int)width;
    m.n = (int)parts;
    m.eps = eps;
    const dim3 grid((uint32_t)ceil_div(rows, (int64_t)(kBlock / kWave)));
#define QDC_MERGE(CPL, TO)                                                                 \
    hipLaunchKernelGGL((merge_parts<CPL, TO>), grid, dim3(kBlock), 0, stream, m);          \
    return launch_status();
#define QDC_MERGE_W(CPL)                                                                   \
    if (width == CPL * 4 * kWave) {                                                        \
        if (split) { QDC_MERGE(CPL, split_t) }                                             \
        if (out_dtype == QDC_BF16) { QDC_MERGE(CPL, bf16_t) }                              \
        QDC_MERGE(CPL, float)                                                              \
    }
    QDC_MERGE_W(1)
    QDC_MERGE_W(2)
    QDC_MERGE_W(4)
    QDC_MERGE_W(8)
#undef QDC_MERGE_W
#undef QDC_MERGE
    return QDC_ERR_SHAPE;
}
