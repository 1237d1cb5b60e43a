// qdc_attention_fused.hip -- causal attention of prepared heads in one pass:
// scores, masked softmax, the product with V and the sigmoid output gate, with
// no score matrix in memory.
//
// The same result as qdc_attention_softmax and qdc_attention_gate around two
// batched products (attention_softmax_kernel!, merge_gate_kernel!,
// ext/amdgpu_attention.jl:61-106): query i sees the keys j <= i whose mask is not
// zero; a query that sees none spreads evenly over every key of its sequence.
// Scores, exponentials, row sums and outputs are fp32; the exponentials enter the
// product with V in the storage type.
//
// A wavefront owns 32 queries of one head.  Scores are computed transposed,
// S^T = K Q^T, so a lane holds one query's column (query l%32, its keys split over
// the two half-wavefronts): row maxima and sums are in-lane reductions and one
// lane swap, and the exponentials are already the B operand of O^T = V^T P^T, whose
// accumulators again hold one query per lane, so rescaling is a multiply by a
// lane's own factor.  The four wavefronts of a workgroup take four (head, query
// block) units of one KV head and share its K and V tiles of 32 keys.
//
// What the score matrix cost was memory: at 8 x 2048 tokens, 8 heads over 2 of 256,
// 1.07 GB of scores written, read and rewritten around the softmax, at odd lengths
// with unaligned rows.  Kernel times in a trace that alternates the two, medians, us, the
// two products, softmax and gate merge / this kernel: bf16 8 x 2048 850 / 298, 1 x 6001
// 1346 / 266, 4 x 300 48 / 28; fp32 8 x 2048 2480 / 1490, 1 x 6001 3005 / 1310, 3 x 777
// 227 / 115.  Inside a forward of 8 x 2048 tokens 266 a layer.  Bound by the matrix
// products and what a wavefront issues beside them: bf16 137 GFLOP in 266 us is 515
// TFLOP/s, fp32 92 to 100 TFLOP/s of the 157 of the fp32 matrix cores.  The exact sigmoid
// of the gate, 26 instructions a value in an epilogue that has its SIMD to itself, is
// 20 to 25 us of the 298 and 4 of the 28; the same bits with a shorter reciprocal were no
// faster (a branch a value 1034 us a layer, one for eight values 1010, this 987).
#include <cfloat>

#include "qdc_common.hpp"
#include "qdc_hip_workspace.h"

namespace qdc {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

constexpr int kQ = 32;     // queries per wavefront
constexpr int kKeys = 32;  // keys per tile

struct Attention {
    void *out;
    const void *q, *k, *v, *gate;
    const int32_t *mask;  // [batch, S] or null
    int64_t q_tok, q_head, k_tok, k_head, v_tok, v_head, gate_tok, gate_head, out_tok;
    int S, KV, G;
    int units;            // G * query blocks, per KV head
    float scale_log2;     // scale * log2(e)
};

__device__ __forceinline__ float swap_max32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// bf16 heads.  The LDS rows of K and V are padded by 16 and 32 bytes: the 8 rows
// read together at one column of K, and the 4 rows of 32 bytes of a transposing
// read of V, then fall on different banks, at addresses that are a lane's own plus
// a constant.  A step covers SUBS tiles of 32 keys between two barriers.
template <int HD, typename TO>
__global__ __launch_bounds__(kBlock, HD > 128 ? 1 : 2) void attention_fused_bf16(Attention a) {
    constexpr int SUBS = 2, KEYS = SUBS * kKeys;
    constexpr int CPR = HD / 8;                       // 16-byte pieces per row
    constexpr int KLD = HD + 8, VLD = HD + 16;        // LDS row strides
    constexpr int RPI = kWave / CPR;                  // rows per wavefront load
    constexpr int LOADS = KEYS / RPI / 4;             // loads per lane of one step's K or V
    constexpr int STEPS = HD / 16, TILES = HD / 32;   // STEPS == 2 TILES
    static_assert(CPR <= kWave && RPI * CPR == kWave && LOADS >= 1, "tile shape");
    __shared__ __align__(16) bf16_t sk[2][KEYS * KLD], sv[2][KEYS * VLD];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), l = threadIdx.x % kWave;
    const int lq = l % 32, lh = l / 32;
    const int b = blockIdx.x / a.KV, kv = blockIdx.x - b * a.KV;
    const int S = a.S;
    // the longest key ranges first
    const int first = 4 * (int)(gridDim.y - 1 - blockIdx.y);
    const int unit = first + wv;
    const bool live = unit < a.units;
    const int head = kv * a.G + unit % a.G, qb = unit / a.G;
    const int query = qb * kQ + lq;
    const int last = min(first + 3, a.units - 1) / a.G;  // last query block of the workgroup
    const int nsteps = last / SUBS + 1;                  // kQ == kKeys
    const int mine = live ? qb / SUBS + 1 : 0;           // steps this wavefront needs
    const int64_t row0 = (int64_t)b * S;
    const bf16_t *kp = reinterpret_cast<const bf16_t *>(a.k) + row0 * a.k_tok + kv * a.k_head;
    const bf16_t *vp = reinterpret_cast<const bf16_t *>(a.v) + row0 * a.v_tok + kv * a.v_head;
    const int32_t *mp = a.mask ? a.mask + row0 : nullptr;

    // one step's rows, 16 bytes per lane and load: global to registers, then to LDS
    const int lrow = wv * RPI + l / CPR, lpiece = l % CPR;
    auto load_rows = [&](const bf16_t *src, int64_t tok, int t, u32x4 (&x)[LOADS]) {
#pragma unroll
        for (int n = 0; n < LOADS; ++n) {
            const int key = min(t * KEYS + lrow + 4 * RPI * n, S - 1);  // past the end: unweighted
            x[n] = load_raw(src + (int64_t)key * tok + 8 * lpiece);
        }
    };
    auto stage_rows = [&](const u32x4 (&x)[LOADS], bf16_t *dst, int ld) {
#pragma unroll
        for (int n = 0; n < LOADS; ++n)
            *reinterpret_cast<u32x4 *>(dst + (lrow + 4 * RPI * n) * ld + 8 * lpiece) = x[n];
    };

    u32x4 xk[LOADS], xv[LOADS];
    load_rows(kp, a.k_tok, 0, xk);
    bf16x8 qf[STEPS];
    {
        const bf16_t *qp = reinterpret_cast<const bf16_t *>(a.q) +
                           (row0 + min(query, S - 1)) * a.q_tok + head * a.q_head + 8 * lh;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) qf[s] = *reinterpret_cast<const bf16x8 *>(qp + 16 * s);
    }
    load_rows(vp, a.v_tok, 0, xv);
    f32x16 o[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    // What the exponents of this query's scores are taken from, its running maximum
    // times scale_log2 as rounded: the exponentials and the factors that rescale them
    // use the same value, which is finite before the first key (where a masked score
    // is -inf) at every scale.  Then this lane's sum.
    float base = -FLT_MAX, total = 0.0f;

    // operands from LDS: K's piece n of key lq of tile u; V^T's rows 32 t .. 32 t + 31
    // and 16 keys (s of the step), by two transposing reads of 4 keys each per lane
    const int koff = lq * KLD + 8 * lh;
    const int voff = (4 * lh + (l % 16) / 4) * VLD + 16 * ((l / 16) & 1) + 4 * (l % 4);
    auto key_piece = [&](const bf16_t *k, int u, int n) {
        return *reinterpret_cast<const bf16x8 *>(k + koff + u * kKeys * KLD + 16 * n);
    };
    auto value_piece = [&](const bf16_t *v, int s, int t) {
        s16x4 h[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const bf16_t *src = v + voff + (16 * s + 8 * e) * VLD + 32 * t;
            h[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4 *)src);
        }
        const s16x8 x = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(bf16x8, x);
    };
    // the weights of 16 keys: p[r] is key 8 (r / 4) + 4 lh + r % 4
    auto weights = [&](const float (&p)[8]) {
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = pack_bf16x2(p[2 * j], p[2 * j + 1]);
        return __builtin_bit_cast(bf16x8, w);
    };
    auto mfma = [](bf16x8 x, bf16x8 y, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    };
    // keeps the issue order of the steps below as written
    auto issue = [] { __builtin_amdgcn_sched_barrier(0); };
    // an output tile stays in accumulator registers: without this the rare rescaling
    // below has all of them moved out and back at every step (HD = 256)
    auto keep = [](f32x16 &x) {
        if constexpr (HD > 128) asm volatile("" : "+a"(x));
    };
    // this lane's mask entries of step t, loaded a step ahead
    int kept[SUBS];
    auto load_mask = [&](int t) {
#pragma unroll
        for (int u = 0; u < SUBS; ++u) {
            const int key = t * KEYS + u * kKeys + lq;
            kept[u] = key < S ? mp[key] : 0;
        }
    };
    // step t's mask, and the maximum the exponentials are taken from
    auto admit = [&](int t, f32x16 (&s)[SUBS]) {
        if (t + 1 == mine || mp) {
#pragma unroll
            for (int u = 0; u < SUBS; ++u) {
                const int tile = SUBS * t + u;
                // bit i: key 32 tile + i is kept
                const uint32_t on = mp ? (uint32_t)__ballot(kept[u] != 0) : ~0u;
                // keys <= the query
                const uint32_t seen = tile < qb ? ~0u : tile == qb ? (2u << lq) - 1u : 0u;
                const uint32_t see = (on & seen) >> (4 * lh);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[u][r] = (see >> (8 * (r / 4) + r % 4)) & 1u ? s[u][r] : -__builtin_inff();
            }
        }
        float top = s[0][0];
#pragma unroll
        for (int r = 1; r < 16 * SUBS; ++r) top = fmaxf(top, s[r / 16][r % 16]);
        // a new maximum rescales what is summed so far; one within 2^8 of the old
        // is left, its exponentials are at most 2^8 and lose nothing
        if (__ballot(__builtin_fmaf(top, a.scale_log2, -base) > 8.0f)) {
            const float next = fmaxf(base, swap_max32(top) * a.scale_log2);
            const float f = __builtin_amdgcn_exp2f(base - next);
            base = next;
            total *= f;
#pragma unroll
            for (int n = 0; n < TILES; ++n) {
                keep(o[n]);
                o[n] *= f;
                keep(o[n]);
                issue();
            }
        }
    };

    if (mp) load_mask(0);
    stage_rows(xk, sk[0], KLD);
    load_rows(kp, a.k_tok, 1, xk);
    stage_rows(xv, sv[0], VLD);
    __syncthreads();
    f32x16 s[SUBS] = {};
    if (mine > 0) {
#pragma unroll
        for (int u = 0; u < SUBS; ++u)
#pragma unroll
            for (int n = 0; n < STEPS; ++n) s[u] = mfma(key_piece(sk[0], u, n), qf[n], s[u]);
        admit(0, s);
    }
    stage_rows(xk, sk[1], KLD);
    __syncthreads();
    // One step of the loop: the exponentials of step t, its product with V, and the
    // scores of step t + 1, which need neither, so that the exponentials of one
    // step run beside the matrix products of the next in a single wavefront (the
    // accumulators leave room for one per SIMD); then the mask and maximum of t + 1.
    for (int t = 0; t < nsteps; ++t) {
        // in flight during this step (past the last step: loaded, not used)
        load_rows(kp, a.k_tok, t + 2, xk);
        load_rows(vp, a.v_tok, t + 1, xv);
        if (mp) load_mask(t + 1);
        if (t < mine) {
            constexpr int LEAD = 4;  // products between an LDS read and its use
            constexpr int ALL = SUBS * STEPS, PER = 16 / STEPS;
            const bf16_t *k = sk[(t + 1) & 1], *v = sv[t & 1];
            float p[8];
            bf16x8 kf[ALL], vf[ALL], pf[2 * SUBS];
            f32x16 next[SUBS] = {};  // past the last step: of old rows, not used
#pragma unroll
            for (int n = 0; n < LEAD; ++n) kf[n] = key_piece(k, n / STEPS, n % STEPS);
            issue();
#pragma unroll
            for (int n = 0; n < ALL; ++n) {
                const int m = n + LEAD;
                if (m < ALL) kf[m] = key_piece(k, m / STEPS, m % STEPS);
                else vf[m - ALL] = value_piece(v, (m - ALL) / TILES, (m - ALL) % TILES);
                next[n / STEPS] = mfma(kf[n], qf[n % STEPS], next[n / STEPS]);
#pragma unroll
                for (int r = PER * n; r < PER * (n + 1); ++r) {
                    p[r % 8] = __builtin_amdgcn_exp2f(
                        __builtin_fmaf(s[r / 16][r % 16], a.scale_log2, -base));
                    total += p[r % 8];
                    if (r % 8 == 7) pf[r / 8] = weights(p);
                }
                issue();
            }
#pragma unroll
            for (int n = 0; n < ALL; ++n) {
                const int m = n + LEAD;
                if (m < ALL) vf[m] = value_piece(v, m / TILES, m % TILES);
                o[n % TILES] = mfma(vf[n], pf[n / TILES], o[n % TILES]);
                issue();
            }
#pragma unroll
            for (int u = 0; u < SUBS; ++u) s[u] = next[u];
            if (t + 1 < mine) admit(t + 1, s);
        }
        stage_rows(xk, sk[t & 1], KLD);  // steps t and t - 1 are done with these buffers
        stage_rows(xv, sv[(t + 1) & 1], VLD);
        __syncthreads();
    }
    total = swap_sum32(total);
    // a query that saw no key weighs every key of the sequence alike
    if (mp) {
        const bool none = live && query < S && total == 0.0f;
        if (__syncthreads_or(none)) {
            for (int t = 0; t * KEYS < S; ++t) {
                load_rows(vp, a.v_tok, t, xv);
                stage_rows(xv, sv[0], VLD);
                __syncthreads();
#pragma unroll
                for (int h = 0; h < 2 * SUBS; ++h) {
                    float p[8];
#pragma unroll
                    for (int r = 0; r < 8; ++r)
                        p[r] = none && t * KEYS + 16 * h + 8 * (r / 4) + 4 * lh + r % 4 < S ? 1.0f
                                                                                            : 0.0f;
#pragma unroll
                    for (int n = 0; n < TILES; ++n)
                        o[n] = mfma(value_piece(sv[0], h, n), weights(p), o[n]);
                }
                __syncthreads();
            }
            if (none) total = (float)S;
        }
    }
    if (!live || query >= S) return;
    const float inv = 1.0f / total;
    // lane halves exchange groups of 4 rows, so that a lane holds 8 in a row: piece
    // i of tile t is columns 32 t + 16 i + 8 lh .. + 7
    const bf16_t *gp = reinterpret_cast<const bf16_t *>(a.gate) + (row0 + query) * a.gate_tok +
                       (int64_t)head * a.gate_head + 8 * lh;
    TO *op = reinterpret_cast<TO *>(a.out) + (row0 + query) * a.out_tok + (int64_t)head * HD +
             8 * lh;
    u32x4 gf[TILES][2];  // all in flight before the first is used
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) gf[t][i] = load_raw(gp + 32 * t + 16 * i);
    issue();
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float g[8], y[8];
            unpack(gf[t][i], g);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const auto r = __builtin_amdgcn_permlane32_swap(
                    __float_as_uint(o[t][8 * i + j]), __float_as_uint(o[t][8 * i + 4 + j]), false,
                    false);
                y[j] = __uint_as_float(r[0]) * inv * sigmoid(g[j]);
                y[4 + j] = __uint_as_float(r[1]) * inv * sigmoid(g[4 + j]);
            }
            store_frag<8>(op + 32 * t + 16 * i, y);
        }
}

// fp32 heads on the fp32 matrix cores (32x32x2).  The four wavefronts of a
// workgroup share one unit of 32 queries and deal its key tiles round-robin, so
// a short sequence still fills the chip, then add their sums through LDS.  A
// product runs 64 cycles, so K and V need no LDS: each lane's operands come from
// L2 a group of kGroup products ahead.  K's columns are dealt so that a lane reads
// 16 bytes: product (m, j) contracts columns 8m + j and 8m + 4 + j.
template <int HD, typename TO>
__global__ __launch_bounds__(kBlock, 1) void attention_fused_f32(Attention a) {
    constexpr int TILES = HD / 32, M = HD / 8, NW = kBlock / kWave;
    constexpr int KGROUP = 4;  // 16-byte pieces of K per group (16 products)
    constexpr int VGROUP = 2;  // keys (per half-wavefront) of V per group
    __shared__ float part[NW][4][16][kWave];  // partial outputs; first the maxima and sums
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), l = threadIdx.x % kWave;
    const int lq = l % 32, lh = l / 32;
    const int b = blockIdx.x / a.KV, kv = blockIdx.x - b * a.KV;
    const int S = a.S;
    const int unit = (int)(gridDim.y - 1 - blockIdx.y);  // the longest key ranges first
    const int head = kv * a.G + unit % a.G, qb = unit / a.G;
    const int query = qb * kQ + lq;
    const int all_tiles = (S + kKeys - 1) / kKeys;
    const int64_t row0 = (int64_t)b * S;
    const float *kp = reinterpret_cast<const float *>(a.k) + row0 * a.k_tok + kv * a.k_head +
                      4 * lh;
    const float *vp = reinterpret_cast<const float *>(a.v) + row0 * a.v_tok + kv * a.v_head + lq;
    const int32_t *mp = a.mask ? a.mask + row0 : nullptr;

    f32x4 qf[M];
    {
        const float *qp = reinterpret_cast<const float *>(a.q) +
                          (row0 + min(query, S - 1)) * a.q_tok + head * a.q_head + 4 * lh;
#pragma unroll
        for (int m = 0; m < M; ++m) qf[m] = *reinterpret_cast<const f32x4 *>(qp + 8 * m);
    }
    f32x16 o[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    float peak = -FLT_MAX, total = 0.0f;
    // an output tile stays in accumulator registers, as in the bf16 form
    auto keep = [](f32x16 &x) {
        if constexpr (HD > 128) asm volatile("" : "+a"(x));
    };

    // V of tile t: group g is the keys p[VGROUP g ..] weigh, every column; p[r] weighs
    // key 8 (r / 4) + 4 lh + r % 4
    constexpr int VG = 16 / VGROUP, KG = M / KGROUP;
    float vf[VG][VGROUP][TILES];
    auto fetch_v = [&](int t, int g) {
#pragma unroll
        for (int e = 0; e < VGROUP; ++e) {
            const int r = VGROUP * g + e;
            const int key = min(t * kKeys + 8 * (r / 4) + 4 * lh + r % 4, S - 1);
#pragma unroll
            for (int n = 0; n < TILES; ++n) vf[g][e][n] = vp[(int64_t)key * a.v_tok + 32 * n];
        }
    };
    auto issue = [] { __builtin_amdgcn_sched_barrier(0); };
    // O^T += V^T P^T of tile t, whose first two groups have been fetched
    auto product = [&](int t, const float (&p)[16]) {
#pragma unroll
        for (int g = 0; g < VG; ++g) {
            if (g + 2 < VG) fetch_v(t, g + 2);
            issue();
#pragma unroll
            for (int e = 0; e < VGROUP; ++e)
#pragma unroll
                for (int n = 0; n < TILES; ++n)
                    o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[g][e][n], p[VGROUP * g + e],
                                                                o[n], 0, 0, 0);
        }
    };
    auto mask_of = [&](int t) {  // this lane's mask entry, loaded a tile ahead
        const int key = t * kKeys + lq;
        return key < S ? mp[key] : 0;
    };

    int kept = mp ? mask_of(wv) : 0;
    for (int t = wv; t <= qb; t += NW) {
        // bit i: key 32 t + i is kept
        const uint32_t on = mp ? (uint32_t)__ballot(kept != 0) : ~0u;
        if (mp) kept = mask_of(t + NW);
        f32x16 s0, s1;
#pragma unroll
        for (int r = 0; r < 16; ++r) s0[r] = s1[r] = 0.0f;
        {
            const float *krow = kp + (int64_t)min(t * kKeys + lq, S - 1) * a.k_tok;
            f32x4 kf[M];
            auto fetch = [&](int g) {
#pragma unroll
                for (int e = 0; e < KGROUP; ++e)
                    kf[KGROUP * g + e] =
                        *reinterpret_cast<const f32x4 *>(krow + 8 * (KGROUP * g + e));
            };
            fetch(0);
            fetch(1);
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                if (g + 2 < KG) fetch(g + 2);
                else fetch_v(t, g + 2 - KG);  // lands during the last products and the softmax
                issue();
#pragma unroll
                for (int e = 0; e < KGROUP; ++e) {
                    const int m = KGROUP * g + e;
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[m][j], qf[m][j], s0, 0, 0, 0);
                        s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[m][j + 1], qf[m][j + 1], s1,
                                                                  0, 0, 0);
                    }
                }
            }
        }
        float p[16];
        const uint32_t seen = t == qb ? (2u << lq) - 1u : ~0u;  // keys <= the query
        const uint32_t see = (on & seen) >> (4 * lh);
#pragma unroll
        for (int r = 0; r < 16; ++r)
            p[r] = (see >> (8 * (r / 4) + r % 4)) & 1u ? s0[r] + s1[r] : -__builtin_inff();
        float top = p[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) top = fmaxf(top, p[r]);
        // a new maximum rescales what is summed so far; one within 2^8 of the old is
        // left, its exponentials are at most 2^8 and lose nothing
        if (__ballot((top - peak) * a.scale_log2 > 8.0f)) {
            const float next = fmaxf(peak, swap_max32(top));
            const float f = __builtin_amdgcn_exp2f((peak - next) * a.scale_log2);
            peak = next;
            total *= f;
#pragma unroll
            for (int n = 0; n < TILES; ++n) {
                keep(o[n]);
                o[n] *= f;
                keep(o[n]);
                issue();
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = __builtin_amdgcn_exp2f((p[r] - peak) * a.scale_log2);
            total += p[r];
        }
        product(t, p);
    }
    // the wavefronts' maxima and sums: every wavefront holds the same 32 queries
    total = swap_sum32(total);
    part[wv][0][0][l] = peak;
    part[wv][0][1][l] = total;
    __syncthreads();
    float top = part[0][0][0][l];
#pragma unroll
    for (int w = 1; w < NW; ++w) top = fmaxf(top, part[w][0][0][l]);
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
        sum += part[w][0][1][l] *
               __builtin_amdgcn_exp2f((part[w][0][0][l] - top) * a.scale_log2);
    __syncthreads();
    float f = __builtin_amdgcn_exp2f((peak - top) * a.scale_log2);
    // a query that saw no key weighs every key of the sequence alike
    const bool none = query < S && sum == 0.0f;
    if (mp && __ballot(none)) {  // the same in the four wavefronts
        for (int t = wv; t < all_tiles; t += NW) {
            float p[16];
#pragma unroll
            for (int r = 0; r < 16; ++r)
                p[r] = none && t * kKeys + 8 * (r / 4) + 4 * lh + r % 4 < S ? 1.0f : 0.0f;
            fetch_v(t, 0);
            fetch_v(t, 1);
            product(t, p);
        }
        if (none) {
            sum = (float)S;
            f = 1.0f;
        }
    }
    const float inv = f / sum;
    const bool store = query < S;
    const int64_t row = row0 + min(query, S - 1);
    const float *gp = reinterpret_cast<const float *>(a.gate) + row * a.gate_tok +
                      (int64_t)head * a.gate_head + 4 * lh;
    TO *op = reinterpret_cast<TO *>(a.out) + row * a.out_tok + (int64_t)head * HD + 4 * lh;
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += 4) {
#pragma unroll
        for (int n = 0; n < 4 && t0 + n < TILES; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[wv][n][r][l] = o[t0 + n][r] * inv;
        __syncthreads();
        if (t0 + wv < TILES && store) {  // wavefront wv adds and writes tile t0 + wv
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float g[4], y[4];
                unpack(load_frag<float, 4>(gp + 32 * (t0 + wv) + 8 * i), g);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float v = part[0][wv][4 * i + j][l];
#pragma unroll
                    for (int w = 1; w < NW; ++w) v += part[w][wv][4 * i + j][l];
                    y[j] = v * sigmoid(g[j]);
                }
                store_frag<4>(op + 32 * (t0 + wv) + 8 * i, y);
            }
        }
        __syncthreads();
    }
}

}  // namespace
}  // namespace qdc

using namespace qdc;

extern "C" int32_t qdc_attention_fused(void *out, int32_t out_dtype, const void *q, const void *k,
                                       const void *v, const void *gate, const int32_t *mask,
                                       int64_t batch, int64_t seq, int64_t heads, int64_t kv_heads,
                                       int64_t head_dim, int64_t q_tok, int64_t q_head,
                                       int64_t k_tok, int64_t k_head, int64_t v_tok,
                                       int64_t v_head, int64_t gate_tok, int64_t gate_head,
                                       int64_t out_tok, float scale, int32_t dtype,
                                       hipStream_t stream) {
    const bool split = out_dtype == QDC_BF16X2;
    if (!(valid_dtype(out_dtype) || split) || !valid_dtype(dtype)) return QDC_ERR_DTYPE;
    // a row's maximum is that of its unscaled scores
    const float scale_log2 = scale * 1.4426950408889634f;
    if (!(scale_log2 > 0.0f && scale_log2 < __builtin_inff())) return QDC_ERR_RANGE;
    if (batch < 0 || seq < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads)
        return QDC_ERR_SHAPE;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return QDC_ERR_SHAPE;
    if (batch == 0 || seq == 0) return QDC_OK;
    const int64_t tokens = batch * seq, lim = (int64_t)1 << 31;
    if (batch >= lim || seq >= lim / 64 || heads >= lim / 64 || batch * kv_heads >= lim / kBlock)
        return QDC_ERR_SHAPE;
    const int64_t units = heads / kv_heads * ceil_div(seq, (int64_t)kQ);
    const int64_t blocks = dtype == QDC_BF16 ? ceil_div(units, (int64_t)4) : units;
    if (blocks > 65535) return QDC_ERR_SHAPE;
    // 16-byte pieces of every input, groups of 4 of the output
    const int64_t strides16[] = {q_tok, q_head, k_tok, k_head, v_tok, v_head};
    const int64_t es = elem_size(dtype);
    for (int64_t s : strides16)
        if (s < head_dim || s * es % 16) return QDC_ERR_SHAPE;
    if (gate_tok < head_dim || gate_head < head_dim || gate_tok * es % 16 || gate_head * es % 16 ||
        out_tok < heads * head_dim || out_tok * elem_size(out_dtype) % 16)
        return QDC_ERR_SHAPE;
    if (!out || !q || !k || !v || !gate) return QDC_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(gate) || !aligned16(out) ||
        ((uintptr_t)mask & 3u))
        return QDC_ERR_SHAPE;
    const int64_t out_bytes = ((tokens - 1) * out_tok + heads * head_dim) * elem_size(out_dtype);
    auto span = [&](int64_t tok, int64_t head, int64_t n) {
        return ((tokens - 1) * tok + (n - 1) * head + head_dim) * es;
    };
    if (overlaps(out, out_bytes, q, span(q_tok, q_head, heads)) ||
        overlaps(out, out_bytes, k, span(k_tok, k_head, kv_heads)) ||
        overlaps(out, out_bytes, v, span(v_tok, v_head, kv_heads)) ||
        overlaps(out, out_bytes, gate, span(gate_tok, gate_head, heads)) ||
        (mask && overlaps(out, out_bytes, mask, tokens * 4)))
        return QDC_ERR_ALIAS;
    Attention a{};
    a.out = out;
    a.q = q;
    a.k = k;
    a.v = v;
    a.gate = gate;
    a.mask = mask;
    a.q_tok = q_tok;
    a.q_head = q_head;
    a.k_tok = k_tok;
    a.k_head = k_head;
    a.v_tok = v_tok;
    a.v_head = v_head;
    a.gate_tok = gate_tok;
    a.gate_head = gate_head;
    a.out_tok = out_tok;
    a.S = (int)seq;
    a.KV = (int)kv_heads;
    a.G = (int)(heads / kv_heads);
    a.units = (int)units;
    a.scale_log2 = scale_log2;
    const dim3 grid((uint32_t)(batch * kv_heads), (uint32_t)blocks);
#define QDC_ATTENTION(HD, TO)                                                                   \
    if (dtype == QDC_BF16)                                                                      \
        hipLaunchKernelGGL((attention_fused_bf16<HD, TO>), grid, dim3(kBlock), 0, stream, a);   \
    else                                                                                        \
        hipLaunchKernelGGL((attention_fused_f32<HD, TO>), grid, dim3(kBlock), 0, stream, a);    \
    return launch_status();
#define QDC_ATTENTION_HD(HD)                                                                    \
    if (head_dim == HD) {                                                                       \
        if (split) { QDC_ATTENTION(HD, split_t) }                                               \
        if (out_dtype == QDC_BF16) { QDC_ATTENTION(HD, bf16_t) }                                \
        QDC_ATTENTION(HD, float)                                                                \
    }
    QDC_ATTENTION_HD(64)
    QDC_ATTENTION_HD(128)
    QDC_ATTENTION_HD(256)
#undef QDC_ATTENTION_HD
#undef QDC_ATTENTION
    return QDC_ERR_SHAPE;
}
