// qdc_linear_f32.hip -- the fp32 projections of a small model with the row work
// around them: the norm that makes the projection's input, and SwiGLU after it.
//
// A decision model's projections (16 to 512 tokens, an inner dimension of 256 or 512)
// hold about a microsecond of matrix work; with each norm and SwiGLU a launch of its
// own, a forward is 45 launches of 3 to 8 us each, most of it first loads and chains
// too short to hide them.  Here a tile is 16 rows by 64 or 32 columns, four wavefronts
// share its inner dimension in blocks of 16, and the workgroup forms its 16 input
// rows itself, in LDS: residual add and RMSNorm, or the gated per-head norm.  Every
// column tile repeats that row work; it is 16 KB a tile from L2, next to the weight
// loads that are in flight meanwhile.
//
// Bound by latency: first loads, one norm chain, at most 8 blocks of products.  At 64
// rows, medians of a launch (the library's product and the row kernels in brackets):
//   norm, [256 x 1792]         4.7 us  (4.8 + 4.4)
//   norm, [256 x 2 512], GLU   4.9     (4.8 + 4.3 + 1.6)
//   [512 x 256]                4.7     (6.9)
//   gated norm, [512 x 256]    6.2     (4.8 + 6.9)
// An fp32 decision forward (4 layers, hidden 256, inner 512), wall time:
//   tokens    16   64  128  200  256  300  411  512
//   before   218  232  251  273  285  315  343  384 us
//   with     182  200  228  249  259  289  320  332 us
// and its error against 64 bits, relative, over those sizes and 8 seeds each: 1.02e-7
// to 1.14e-7 before and 0.98e-7 to 1.14e-7 with it, larger at no size.
//
// Products: (i, j) of a block contracts the columns 16 i + 4 s + j of A (s the k-slot,
// lane / 16), so a lane's A operands of a block are 16 consecutive bytes; tile column
// 4 (lane % 16) + c belongs to accumulator c, so its weights are too and a wavefront
// reads whole 256-byte rows (2 and 128 in the narrow tiles).
#include "qdc_common.hpp"
#include "qdc_hip_workspace.h"

namespace qdc {
namespace {

constexpr int kParts = kBlock / kWave;  // wavefronts the inner dimension is dealt to
constexpr int kTileRows = 16;

enum class Input { kRows, kResidualNorm, kGatedNorm };

struct Linear {
    const float *a;            // rows, ld_a apart: the input, the stream x, or the core output
    const float *b;            // residual form: added to x; gated form: z, rows ld_b apart
    const float *norm;         // the norm's weight: [inner], or [head_dim]
    const int32_t *mask;       // residual form: per row, or null
    float *residual;           // residual form: x + b
    const float *w;            // [inner, cols], or with GLU [inner, gate | up]
    float *out;
    int64_t ld_a, ld_b, ld_w, ld_out;
    int rows, inner, cols, head_dim;
    float eps;
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 load4(const float *p) {
    return *reinterpret_cast<const f32x4 *>(p);
}

// CHUNKS: inner / 64 (the input rows are formed by 16 lanes of 4 columns a chunk).
// NC: columns per lane, 16 NC per tile.
template <int NC> struct Cols {
    typedef float type __attribute__((ext_vector_type(NC)));
};
template <Input IN, bool GLU, int CHUNKS, int NC>
__global__ __launch_bounds__(kBlock) void linear_f32(Linear p) {
    constexpr int B = GLU ? 2 : 1;
    constexpr int INNER = 64 * CHUNKS, ALD = INNER + 4;
    constexpr int STEPS = INNER / 16 / kParts;  // blocks of the inner dimension per wavefront
    __shared__ __align__(16) float sa[kTileRows * ALD];
    typedef typename Cols<NC>::type Vec;
    __shared__ Vec part[kParts][B][4][kWave];
    const int tid = threadIdx.x, l = tid % kWave, lr = l % 16, lg = l / 16;
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r0 = blockIdx.y * kTileRows, n0 = blockIdx.x * (16 * NC) + NC * lr;

    // the weights of the first blocks leave before the rows are formed
    constexpr int AHEAD = STEPS < 4 ? STEPS : 4;
    Vec wf[STEPS][B][4];
    auto fetch = [&](int i) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                wf[i][b][j] = *reinterpret_cast<const Vec *>(
                    p.w + (int64_t)(16 * (wv + kParts * i) + 4 * lg + j) * p.ld_w + n0 +
                    b * p.cols);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i);

    {   // row tid / 16, columns 64 c + 4 (tid % 16) .. + 3
        const int r = tid / 16, col = 4 * (tid % 16);
        const int64_t row = min(r0 + r, p.rows - 1);
        f32x4 v[CHUNKS], u[CHUNKS], g[CHUNKS];
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            v[c] = load4(p.a + row * p.ld_a + 64 * c + col);
            if constexpr (IN != Input::kRows) u[c] = load4(p.b + row * p.ld_b + 64 * c + col);
            if constexpr (IN == Input::kResidualNorm) g[c] = load4(p.norm + 64 * c + col);
            if constexpr (IN == Input::kGatedNorm)
                g[c] = load4(p.norm + (64 * c) % p.head_dim + col);
        }
        if constexpr (IN == Input::kResidualNorm) {
            const float keep = p.mask ? (float)p.mask[row] : 1.0f;
            float ss = 0.0f;
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c) {
                v[c] += u[c];
#pragma unroll
                for (int j = 0; j < 4; ++j) ss = __builtin_fmaf(v[c][j], v[c][j], ss);
                if (blockIdx.x == 0 && r0 + r < p.rows)
                    *reinterpret_cast<f32x4 *>(p.residual + row * INNER + 64 * c + col) = v[c];
            }
            const float s = rms_scale(group_sum<16>(ss), (float)INNER, p.eps);
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[c][j] = (v[c][j] * s) * (1.0f + g[c][j]) * keep;
        }
        if constexpr (IN == Input::kGatedNorm) {
            const int per = p.head_dim / 64;  // chunks of a head (uniform)
            float ss[CHUNKS];
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c) {
                ss[c] = 0.0f;
#pragma unroll
                for (int j = 0; j < 4; ++j) ss[c] = __builtin_fmaf(v[c][j], v[c][j], ss[c]);
                ss[c] = group_sum<16>(ss[c]);
            }
#pragma unroll
            for (int c = 0; c < CHUNKS; ++c) {
                float head = 0.0f;  // of the head that chunk c belongs to
#pragma unroll
                for (int e = 0; e < CHUNKS; ++e) head += e / per == c / per ? ss[e] : 0.0f;
                const float s = rms_scale(head, (float)p.head_dim, p.eps);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[c][j] = (v[c][j] * s) * g[c][j] * silu(u[c][j]);
            }
        }
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c)
            *reinterpret_cast<f32x4 *>(&sa[r * ALD + 64 * c + col]) = v[c];
    }
    __syncthreads();

    f32x4 acc[B][NC];
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[b][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        if (i + AHEAD < STEPS) fetch(i + AHEAD);
        const f32x4 af = load4(&sa[lr * ALD + 16 * (wv + kParts * i) + 4 * lg]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    acc[b][c] = mfma4(af[j], wf[i][b][j][c], acc[b][c]);
    }
    // the four sums meet: this wavefront ends with rows 4 (l / 16) + wv
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            Vec v;
#pragma unroll
            for (int c = 0; c < NC; ++c) v[c] = acc[b][c][j];
            part[wv][b][j][l] = v;
        }
    __syncthreads();
    Vec sum[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        sum[b] = part[0][b][wv][l];
#pragma unroll
        for (int s = 1; s < kParts; ++s) sum[b] += part[s][b][wv][l];
    }
    const int row = r0 + 4 * lg + wv;
    if (row >= p.rows) return;
    Vec o = sum[0];
    if constexpr (GLU) {
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c] = silu(sum[0][c]) * sum[B - 1][c];
    }
    *reinterpret_cast<Vec *>(p.out + (int64_t)row * p.ld_out + n0) = o;
}

}  // namespace
}  // namespace qdc

using namespace qdc;

extern "C" int32_t qdc_linear_f32(float *out, float *residual, const float *a, const float *b,
                                  const float *norm, const int32_t *mask, const float *w,
                                  int64_t rows, int64_t inner, int64_t cols, int64_t head_dim,
                                  int64_t ld_a, int64_t ld_b, int64_t ld_w, int64_t ld_out,
                                  float eps, int32_t input, int32_t swiglu, hipStream_t stream) {
    if (input < 0 || input > 2) return QDC_ERR_RANGE;
    const int64_t lim = (int64_t)1 << 20, wcols = swiglu ? 2 * cols : cols;
    if (rows < 0 || rows >= lim || cols <= 0 || cols >= lim || cols % 64) return QDC_ERR_SHAPE;
    if (inner != 128 && inner != 256 && inner != 512) return QDC_ERR_SHAPE;
    if (input == 2 && (head_dim <= 0 || head_dim % 64 || inner % head_dim || swiglu))
        return QDC_ERR_SHAPE;
    if (ld_a < inner || ld_w < wcols || ld_out < cols || ld_a % 4 || ld_w % 4 || ld_out % 4)
        return QDC_ERR_SHAPE;
    if (input != 0 && (ld_b < inner || ld_b % 4)) return QDC_ERR_SHAPE;
    if (rows == 0) return QDC_OK;
    const int64_t row_tiles = ceil_div(rows, (int64_t)kTileRows);
    if (row_tiles > 65535) return QDC_ERR_SHAPE;
    if (!out || !a || !w || (input != 0 && (!b || !norm)) || (input == 1 && !residual))
        return QDC_ERR_NULL;
    if (!aligned16(out) || !aligned16(a) || !aligned16(w) ||
        (input != 0 && (!aligned16(b) || !aligned16(norm))) ||
        (input == 1 && (!aligned16(residual) || ((uintptr_t)mask & 3u))))
        return QDC_ERR_SHAPE;
    const int64_t out_bytes = ((rows - 1) * ld_out + cols) * 4, res_bytes = rows * inner * 4;
    const int64_t a_bytes = ((rows - 1) * ld_a + inner) * 4, b_bytes = ((rows - 1) * ld_b + inner) * 4;
    const int64_t w_bytes = ((inner - 1) * ld_w + wcols) * 4, n_bytes = (input == 2 ? head_dim : inner) * 4;
    float *const outs[2] = {out, input == 1 ? residual : nullptr};
    const int64_t sizes[2] = {out_bytes, res_bytes};
    if (outs[1] && overlaps(out, out_bytes, residual, res_bytes)) return QDC_ERR_ALIAS;
    for (int i = 0; i < 2; ++i)  // every column tile reads the inputs: no output in place
        if (outs[i] && (overlaps(outs[i], sizes[i], a, a_bytes) ||
                        overlaps(outs[i], sizes[i], w, w_bytes) ||
                        (input != 0 && (overlaps(outs[i], sizes[i], b, b_bytes) ||
                                        overlaps(outs[i], sizes[i], norm, n_bytes))) ||
                        (input == 1 && mask && overlaps(outs[i], sizes[i], mask, rows * 4))))
            return QDC_ERR_ALIAS;
    Linear p{};
    p.a = a;
    p.b = b;
    p.norm = norm;
    p.mask = mask;
    p.residual = residual;
    p.w = w;
    p.out = out;
    p.ld_a = ld_a;
    p.ld_b = ld_b;
    p.ld_w = ld_w;
    p.ld_out = ld_out;
    p.rows = (int)rows;
    p.inner = (int)inner;
    p.cols = (int)cols;
    p.head_dim = (int)head_dim;
    p.eps = eps;
    // Half as wide tiles while those of 64 columns leave compute units idle: a tile's
    // products are 4096 cycles of its unit at inner 512.  Against the forward
    // without this file: 1.18x with them and 1.03x without at 64 tokens, 1.09x and 1.04x
    // at 300.
    const bool narrow = cols / 64 * row_tiles <= 192;
    const dim3 grid((uint32_t)(cols / (narrow ? 32 : 64)), (uint32_t)row_tiles);
#define QDC_LINEAR(IN, GLU, C)                                                                 \
    if (inner == 64 * C) {                                                                     \
        if (narrow)                                                                            \
            hipLaunchKernelGGL((linear_f32<IN, GLU, C, 2>), grid, dim3(kBlock), 0, stream, p); \
        else                                                                                   \
            hipLaunchKernelGGL((linear_f32<IN, GLU, C, 4>), grid, dim3(kBlock), 0, stream, p); \
        return launch_status();                                                                \
    }
#define QDC_LINEAR_C(IN, GLU) QDC_LINEAR(IN, GLU, 2) QDC_LINEAR(IN, GLU, 4) QDC_LINEAR(IN, GLU, 8)
    if (input == 0 && !swiglu) { QDC_LINEAR_C(Input::kRows, false) }
    if (input == 0) { QDC_LINEAR_C(Input::kRows, true) }
    if (input == 1 && !swiglu) { QDC_LINEAR_C(Input::kResidualNorm, false) }
    if (input == 1) { QDC_LINEAR_C(Input::kResidualNorm, true) }
    QDC_LINEAR_C(Input::kGatedNorm, false)
#undef QDC_LINEAR_C
#undef QDC_LINEAR
    return QDC_ERR_SHAPE;
}
