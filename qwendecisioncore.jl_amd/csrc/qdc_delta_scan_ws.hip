// qdc_delta_scan_ws.hip -- the gated delta rule recurrence as two launches.
//
// For chunks of 16 tokens with state S0 (kept transposed, S^T [kd, vd]),
// log-decays d and their running sums g, the recurrence (cpu_delta_recurrent_step!,
// src/backbone_cpu.jl:681-705) is exactly
//     A[i][p] = beta_i exp(g_i - g_p) (k_i . k_p)   (p < i),  T = (I + A)^-1
//     U = T diag(beta) (V - diag(e^g) Z),   Z = K S0^T        (the deltas u_i)
//     O = diag(e^g) Q S0^T + P U,   P[i][p] = exp(g_i - g_p) (q_i . k_p)  (p <= i)
//     S^T <- e^(g_15) S^T + K^T diag(e^(g_15 - g)) U
// T diag(beta), P and the exponentials do not involve the state: the first launch
// (delta_chunk_prepare) computes them for every chunk of the sequence at once,
// one wavefront per chunk and value head, into a record per chunk; the second
// (delta_chunk_scan) is left with the products that do.
//
// Column n of S^T, U and O depends on no other column, so the scan's unit is a
// slice of 16 value columns: one wavefront runs a whole slice with the state in
// its accumulators, or KSPLIT wavefronts share a slice's key rows and add their
// partial Z and Q S0^T through LDS.  Either way a workgroup meets once a chunk: four
// whole slices for the k and q rows that they read from LDS together.
//
// The fp32 matrix products of the scan (104 of 32 cycles per chunk and slice: 177 us
// at 2.4 GHz for 128 chunks, a slice a SIMD) bound it when the slices fill the chip,
// the chain from one chunk's state to the next when they do not.  Kernel times in a
// trace that alternates the one-launch form of qdc_delta_scan.hip, which runs 64
// columns in eight wavefronts that meet twice a chunk, with these two, medians, kd =
// vd = 128, bf16 outputs, us, one launch / scan + prepare: 8 x 2048 tokens, 16 heads
// 494 / 307 + 57; the same with 32 heads 848 / 479 + 93; 2 x 1501, 32 heads 303 / 147 +
// 21; 1 x 777, 16 heads 159 / 47 + 6; 1 x 411, 4 heads 85 / 26 + 5.  (Inside a forward
// of 8 x 2048 tokens 297 + 67.)  Uniform bases and lane offsets for the running
// addresses of rows and outputs took 27 us off the first and 39 off the second; without
// the operands' refills (timing only) the scan of the first took 227 us, so what its
// loads cost beside the products is the next thing to gain.
#include "qdc_common.hpp"
#include "qdc_hip_workspace.h"

namespace qdc {
namespace {

constexpr int kC = 16;  // tokens per chunk: one MFMA tile edge
// One chunk's record (floats): T diag(beta) and P in operand order (lane l's four
// values, row l%16 and columns 4(l/16) .. +3, at 4l), then e^g and e^(g_15 - g).
constexpr int kRecTb = 0, kRecP = 256, kRecEg = 512, kRecEt = 528, kRecord = 544;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Inclusive prefix sum over each 16-lane row of a wavefront (DPP row shifts;
// lanes shifted in from outside the row contribute 0).
__device__ __forceinline__ float row_prefix_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));
    return v;
}

struct ChunkArgs {
    void *out;
    const float *q, *k, *v, *beta, *decay;
    float *ws;
    int64_t ld_qk, ld_v;  // elements between the token rows of q and k, and of v
    int S, H, vd, groups, chunks, slices;  // slices = vd / 16
    int64_t units;        // batch * heads * chunks (prepare)
    FastDiv by_chunks, by_heads, by_groups;  // by_groups: workgroups per head (scan)
};

__device__ __forceinline__ f32x4 load4(const float *p) {
    return *reinterpret_cast<const f32x4 *>(p);
}

// Records of all chunks: a wavefront per (sequence, head, chunk), chunks fastest.
// K K^T is symmetric and K Q^T is computed instead of Q K^T, so both land with
// lane l, register j holding row l%16, column 4(l/16) + j: the operand order of
// the record.  Bound by the reads of q and k when the batch is large.
template <int KB>
__global__ __launch_bounds__(kBlock) void delta_chunk_prepare(ChunkArgs a) {
    constexpr int RS = 20;  // LDS row stride: the four 16-lane groups on disjoint banks
    __shared__ __align__(16) float lds_a[kBlock / kWave][kC][RS], lds_t[kBlock / kWave][kC][RS];
    const int wv = threadIdx.x / kWave, l = threadIdx.x % kWave, lr = l % 16, lg = l / 16;
    const int64_t unit = (int64_t)blockIdx.x * (kBlock / kWave) + wv;
    if (unit >= a.units) return;  // uniform per wavefront; nothing below crosses wavefronts
    float(*sA)[RS] = lds_a[wv], (*sT)[RS] = lds_t[wv];
    const uint32_t bh = fastdiv((uint32_t)unit, a.by_chunks);
    const int c = (int)((uint32_t)unit - bh * a.by_chunks.d);
    const uint32_t b = fastdiv(bh, a.by_heads);
    const int h = (int)(bh - b * a.by_heads.d), g = h / a.groups;
    const int t0 = c * kC, tok = t0 + lr;
    const bool in = tok < a.S;
    // tokens past the end: any row in range (beta = 0 and d = 0 take it out)
    const int64_t row = (int64_t)b * a.S + min(tok, a.S - 1);
    const float *kp = a.k + row * a.ld_qk + (int64_t)g * (16 * KB) + 4 * lg;
    const float *qp = a.q + row * a.ld_qk + (int64_t)g * (16 * KB) + 4 * lg;
    f32x4 kf[KB], qf[KB];
#pragma unroll
    for (int i = 0; i < KB; ++i) kf[i] = load4(kp + 16 * i);
#pragma unroll
    for (int i = 0; i < KB; ++i) qf[i] = load4(qp + 16 * i);
    const float beta = in ? a.beta[row * a.H + h] : 0.0f;
    const float run = row_prefix_sum(in ? a.decay[row * a.H + h] : 0.0f);
    float g_col[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) g_col[j] = __shfl(run, 4 * lg + j, kWave);
    const float g_last = __shfl(run, kC - 1, kWave);

    f32x4 kk[4] = {}, kq[4] = {};
#pragma unroll
    for (int i = 0; i < KB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            kk[j] = mfma4(kf[i][j], kf[i][j], kk[j]);
            kq[j] = mfma4(kf[i][j], qf[i][j], kq[j]);
        }
    const f32x4 KK = (kk[0] + kk[1]) + (kk[2] + kk[3]);
    const f32x4 KQ = (kq[0] + kq[1]) + (kq[2] + kq[3]);
    f32x4 A, P;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int p = 4 * lg + j;
        const bool keep = p <= lr;
        const float e = expf(keep ? run - g_col[j] : 0.0f);
        A[j] = p < lr ? beta * e * KK[j] : 0.0f;
        P[j] = keep ? e * KQ[j] : 0.0f;
    }
    *reinterpret_cast<f32x4 *>(&sA[lr][4 * lg]) = A;
    // LDS operations of one wavefront complete in order; the fence keeps the
    // compiler from reordering them
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // T = (I + A)^-1, blocked: with A = [[A11, 0], [A21, A22]] in 8x8 blocks,
    // D = diag(T11, T22) by forward substitution on both blocks at once (lane
    // m < 16 owns column m), then T = D - D (N D) with N = [[0, 0], [A21, 0]]
    if (l < kC) {
        const int m = l, b0 = m & 8, mm = m & 7;
        float arow[8][8];
#pragma unroll
        for (int i = 1; i < 8; ++i)
#pragma unroll
            for (int p = 0; p < i; ++p) arow[i][p] = sA[b0 + i][b0 + p];
        float col[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) col[i] = i == mm ? 1.0f : 0.0f;
#pragma unroll
        for (int i = 1; i < 8; ++i) {
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
            for (int p = 0; p < i; p += 2) {
                s0 = __builtin_fmaf(arow[i][p], col[p], s0);
                if (p + 1 < i) s1 = __builtin_fmaf(arow[i][p + 1], col[p + 1], s1);
            }
            if (i > mm) col[i] = -(s0 + s1);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sT[b0 + i][m] = col[i];
            sT[(b0 ^ 8) + i][m] = 0.0f;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    float db[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) db[i] = sT[4 * lg + i][lr];       // D[k][lr]
    const f32x4 da = *reinterpret_cast<const f32x4 *>(&sT[lr][4 * lg]);  // D[lr][k]
    const bool lower = lr >= 8 && lg < 2;  // N[lr][k] nonzero only for lr >= 8, k < 8
    f32x4 X = {0.f, 0.f, 0.f, 0.f}, Y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) X = mfma4(lower ? A[i] : 0.0f, db[i], X);
#pragma unroll
    for (int i = 0; i < 4; ++i) Y = mfma4(da[i], X[i], Y);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
    for (int j = 0; j < 4; ++j) sT[4 * lg + j][lr] = (db[j] - Y[j]) * beta;  // column lr
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const f32x4 Tb = *reinterpret_cast<const f32x4 *>(&sT[lr][4 * lg]);
    float *rec = a.ws + unit * kRecord;
    *reinterpret_cast<f32x4 *>(rec + kRecTb + 4 * l) = Tb;
    *reinterpret_cast<f32x4 *>(rec + kRecP + 4 * l) = P;
    if (lg == 0) rec[kRecEg + lr] = expf(run);
    else if (lg == 1) rec[kRecEt + lr] = expf(g_last - run);
}

// The operands of one chunk held by one wavefront: its KBW 16-row blocks of the
// key dimension, in groups of V = min(2, KBW).  Key row of block t, row m:
//     base + 16 V (t / V) + V m + t % V
// so that both reads of k are vectors: as the A operand of Z (row = token l%16,
// k-slot l/16 of step j = row 4(l/16) + j of block t) 4V consecutive keys per
// lane, and as the A operand of the state update (row m = l%16, k-slot = token
// 4(l/16) + i) V consecutive keys.
template <int KBW, int PARTS> struct ChunkOperands {
    static constexpr int V = KBW < 2 ? KBW : 2, N = KBW / V;
    f32x4 k[N][V], q[N][V];        // 4V keys of token l%16 per group of V blocks
    float kt[N][4][V];             // V keys of tokens 4(l/16) + i
    f32x4 tb, eg, et;
    float v[4], p[PARTS];          // p: this key part's columns 4(l/16) + ...
};

// A uniform base and a lane's byte offset: one scalar-base load, no address math.
__device__ __forceinline__ const float *at(const float *base, uint32_t bytes) {
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + bytes);
}
template <int V> __device__ __forceinline__ void load_vec(const float *p, float (&o)[V]) {
    if constexpr (V == 4) {
        const f32x4 x = load4(p);
        o[0] = x[0]; o[1] = x[1]; o[2] = x[2]; o[3] = x[3];
    } else if constexpr (V == 2) {
        const f32x2 x = *reinterpret_cast<const f32x2 *>(p);
        o[0] = x[0]; o[1] = x[1];
    } else {
        o[0] = p[0];
    }
}

// One set of operands, each refilled for the next chunk as soon as this one has
// used it (two or three sets in turn measured no faster).  A wavefront has its SIMD
// all but to itself, so what is not a matrix product has to issue between them: a
// group of key blocks' products, then its refill.
//
// KSPLIT = 1: the workgroup's four slices are of one head.  Its wavefronts load a
// chunk's k and q rows once between them, two chunks ahead, into one of two LDS
// tiles, and refill their operands from the tile of the next chunk: the same loads
// from memory by every wavefront took a third of the kernel's time to issue.
template <int KB, int KSPLIT, typename TO>
__global__ __launch_bounds__(KSPLIT > 1 ? KSPLIT * kWave : kBlock, 2) void delta_chunk_scan(
    ChunkArgs a) {
    constexpr int KBW = KB / KSPLIT;
    constexpr int PARTS = 4 / KSPLIT;  // output rows and P's columns (of 4) per key part
    typedef ChunkOperands<KBW, PARTS> Ops;
    constexpr int V = Ops::V, N = Ops::N;
    constexpr bool SHARED = KSPLIT == 1;
    constexpr int LD = 16 * KB + 4;                       // LDS row stride: rows 4 banks apart
    constexpr int TILE16 = kC * 4 * KB;                   // 16-byte pieces of a tile
    constexpr int PIECES = (TILE16 + kBlock - 1) / kBlock;  // per thread
    __shared__ __align__(16) float tile[SHARED ? 2 : 1][2][SHARED ? kC * LD : 4];  // k, q
    // the key parts' shares of Z and of the output, two chunks' worth
    __shared__ f32x4 part_z[KSPLIT > 1 ? 2 : 1][KSPLIT][kWave];
    __shared__ float part_o[KSPLIT > 1 ? 2 : 1][KSPLIT][4][kWave];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int l = threadIdx.x % kWave, lr = l % 16, lg = l / 16;
    const int ks = KSPLIT > 1 ? wv : 0;
    // consecutive slices on one XCD (workgroups are dealt round-robin over the 8),
    // so the slices of a head share its L2's copy of k, q and the records
    const uint32_t nwg = gridDim.x, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const uint32_t per = nwg / 8, rem = nwg % 8;
    const uint32_t wg = xcd * per + min(xcd, rem) + slot;
    const uint32_t bh = fastdiv(wg, a.by_groups);  // groups of 4 slices, or slices
    const int slice = (int)(wg - bh * a.by_groups.d) * (SHARED ? 4 : 1) + (SHARED ? wv : 0);
    const bool live = slice < a.slices;
    const int col = 16 * min(slice, a.slices - 1) + lr;
    const uint32_t b = fastdiv(bh, a.by_heads);
    const int h = (int)(bh - b * a.by_heads.d), g = h / a.groups;
    const int S = a.S, chunks = a.chunks;
    const int64_t row0 = (int64_t)b * S, o_tok = (int64_t)a.H * a.vd;
    // where the output rows of the chunk to be stored start (uniform)
    TO *oc = reinterpret_cast<TO *>(a.out) + row0 * o_tok + (int64_t)h * a.vd;
    uint32_t off_o[PARTS];  // this lane's byte offsets from there
#pragma unroll
    for (int j = 0; j < PARTS; ++j)
        off_o[j] = (uint32_t)sizeof(TO) *
                   ((uint32_t)(4 * lg + ks * PARTS + j) * (uint32_t)o_tok + (uint32_t)col);

    // where the operands of the chunk being fetched start (uniform), and this
    // lane's byte offsets from there; in the last chunk, tokens past the end read
    // the last row (T diag(beta), P and the state update's U are zero there)
    const float *kc = a.k + row0 * a.ld_qk + (int64_t)g * (16 * KB) + ks * (16 * KBW);
    const float *qc = a.q + row0 * a.ld_qk + (int64_t)g * (16 * KB) + ks * (16 * KBW);
    const float *vc = a.v + row0 * a.ld_v + (int64_t)h * a.vd;
    const float *rc = a.ws + (int64_t)bh * chunks * kRecord;
    const int64_t kstep = kC * a.ld_qk, vstep = kC * a.ld_v;
    int fetched = 0;  // the chunk they point to
    uint32_t off, off_t[4], off_v[4];
    auto offsets = [&](int top) {  // top: last row in range
        off = 4u * ((uint32_t)min(lr, top) * (uint32_t)a.ld_qk + 4 * V * lg);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = min(4 * lg + i, top);
            off_t[i] = 4u * (r * (uint32_t)a.ld_qk + V * lr);
            off_v[i] = 4u * (r * (uint32_t)a.ld_v + col);
        }
    };
    auto advance = [&] {  // past the end: the last chunk again, loaded and never used
        if (fetched + 1 < chunks) {
            if (!SHARED) {
                kc += kstep;
                qc += kstep;
            }
            vc += vstep;
            rc += kRecord;
            if (++fetched + 1 == chunks) offsets(S - 1 - fetched * kC);
        }
    };
    // SHARED: chunk c's rows to registers, and from there to its tile
    f32x4 stage[2][PIECES];
    const float *kr = kc, *qr = qc;  // rows of the chunk to be loaded (uniform)
    uint32_t off_r[PIECES];          // this thread's byte offsets from there
    auto row_offsets = [&](int top) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int i = threadIdx.x + p * kBlock;
            off_r[p] = 4u * ((uint32_t)min(i / (4 * KB), top) * (uint32_t)a.ld_qk +
                             4u * (i % (4 * KB)));
        }
    };
    auto load_rows = [&](int c) {  // the chunks in order; past the end: not used
        if (c + 1 == chunks) row_offsets(S - 1 - c * kC);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            stage[0][p] = load4(at(kr, off_r[p]));
            stage[1][p] = load4(at(qr, off_r[p]));
        }
        if (c + 1 < chunks) {
            kr += kstep;
            qr += kstep;
        }
    };
    auto write_rows = [&](int c) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int i = threadIdx.x + p * kBlock, o = i / (4 * KB) * LD + 4 * (i % (4 * KB));
            if (TILE16 % kBlock == 0 || i < TILE16) {
                *reinterpret_cast<f32x4 *>(&tile[c & 1][0][o]) = stage[0][p];
                *reinterpret_cast<f32x4 *>(&tile[c & 1][1][o]) = stage[1][p];
            }
        }
    };
    const int lk = lr * LD + 4 * V * lg, lt = 4 * lg * LD + V * lr;
    auto fetch_k = [&](Ops &x, int n) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            x.k[n][e] = SHARED ? load4(&tile[fetched & 1][0][lk + 16 * V * n + 4 * e])
                               : load4(at(kc + 16 * V * n + 4 * e, off));
    };
    auto fetch_q = [&](Ops &x, int n) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            x.q[n][e] = SHARED ? load4(&tile[fetched & 1][1][lk + 16 * V * n + 4 * e])
                               : load4(at(qc + 16 * V * n + 4 * e, off));
    };
    auto fetch_kt = [&](Ops &x, int n) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            load_vec<V>(SHARED ? &tile[fetched & 1][0][lt + i * LD + 16 * V * n]
                               : at(kc + 16 * V * n, off_t[i]), x.kt[n][i]);
    };
    auto fetch_v = [&](Ops &x) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x.v[i] = *at(vc, off_v[i]);
    };
    auto fetch_tb = [&](Ops &x) { x.tb = load4(at(rc + kRecTb, 16u * l)); };
    auto fetch_p = [&](Ops &x) {
        load_vec<PARTS>(at(rc + kRecP + ks * PARTS, 16u * l), x.p);
    };
    auto fetch_e = [&](Ops &x) {
        x.eg = load4(at(rc + kRecEg, 16u * lg));
        x.et = load4(at(rc + kRecEt, 16u * lg));
    };
    // this key part's rows of the output of chunk c, the chunks in order
    auto store = [&](int c, const float (&o)[PARTS]) {
        char *dst = reinterpret_cast<char *>(oc);
        oc += kC * o_tok;
        if (!live) return;
        const int left = S - c * kC - 4 * lg - ks * PARTS;
        if ((c + 1) * kC <= S) {
#pragma unroll
            for (int j = 0; j < PARTS; ++j)
                *reinterpret_cast<TO *>(dst + off_o[j]) = from_f32<TO>(o[j]);
        } else {
#pragma unroll
            for (int j = 0; j < PARTS; ++j)
                if (j < left) *reinterpret_cast<TO *>(dst + off_o[j]) = from_f32<TO>(o[j]);
        }
    };

    f32x4 st[KBW];
#pragma unroll
    for (int i = 0; i < KBW; ++i) st[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read_output = [&](int c, float (&o)[PARTS]) {  // KSPLIT > 1
#pragma unroll
        for (int j = 0; j < PARTS; ++j) {
            o[j] = part_o[c & 1][0][ks * PARTS + j][l];
#pragma unroll
            for (int s = 1; s < KSPLIT; ++s) o[j] += part_o[c & 1][s][ks * PARTS + j][l];
        }
    };

    // between the last use of an operand and its refill, and after it: the loads
    // go into the registers just read (no second set, no copies) and leave at once
    auto refill = [] { __builtin_amdgcn_sched_barrier(0); };
    auto done = [](f32x4 &v) { asm volatile("" : "+v"(v)); };  // computed here, not later
    auto step = [&](int c, Ops &x) {
        advance();
        if constexpr (SHARED) load_rows(c + 2);
        f32x4 z[4] = {}, y[4] = {};
#pragma unroll
        for (int n = 0; n < N; ++n) {
#pragma unroll
            for (int m = 0; m < 4 * V; ++m) {
                const int t = V * n + m % V, j = m / V, e = V * j + m % V;
                z[m % 4] = mfma4(x.k[n][e / 4][e % 4], st[t][j], z[m % 4]);
            }
            refill();
            fetch_k(x, n);
            refill();
        }
        f32x4 Z = (z[0] + z[1]) + (z[2] + z[3]);
        float due[PARTS];
        if constexpr (KSPLIT > 1) {
            part_z[c & 1][ks][l] = Z;
            __syncthreads();
            Z = part_z[c & 1][0][l];
#pragma unroll
            for (int s = 1; s < KSPLIT; ++s) Z += part_z[c & 1][s][l];
            read_output(c - 1, due);  // of the first chunk: nothing yet, not stored
        }
        // e^(g_15), the chunk's whole decay: the last row's lanes hold it
        const float whole = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x.eg[3]), 48));
        f32x4 R, U = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) R[j] = x.v[j] - x.eg[j] * Z[j];
        // U's four dependent products between those of Q S0^T; a block of the state
        // is scaled once its products are done
#pragma unroll
        for (int n = 0; n < N; ++n) {
#pragma unroll
            for (int m = 0; m < 4 * V; ++m) {
                const int t = V * n + m % V, j = m / V, e = V * j + m % V;
                if (n == 0 && m < 4) U = mfma4(x.tb[m], R[m], U);
                y[m % 4] = mfma4(x.q[n][e / 4][e % 4], st[t][j], y[m % 4]);
            }
            refill();
            fetch_q(x, n);
            if (n == 0) {
                fetch_v(x);
                fetch_tb(x);
            }
            refill();
#pragma unroll
            for (int t = V * n; t < V * (n + 1); ++t) st[t] *= whole;
        }
        f32x4 Ue = U * x.et;
        f32x4 O = ((y[0] + y[1]) + (y[2] + y[3])) * x.eg;
        float u[PARTS];
#pragma unroll
        for (int j = 0; j < PARTS; ++j)
            u[j] = KSPLIT == 1 ? U[j]
                   : KSPLIT == 2 ? (ks ? U[(2 + j) % 4] : U[j])
                                 : (ks & 2 ? (ks & 1 ? U[3] : U[2]) : (ks & 1 ? U[1] : U[0]));
        done(O);
        done(Ue);
#pragma unroll
        for (int t = 0; t < KBW; ++t) done(st[t]);
        refill();
        fetch_e(x);
        refill();
#pragma unroll
        for (int n = 0; n < N; ++n) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int t = V * n; t < V * (n + 1); ++t)
                    st[t] = mfma4(x.kt[n][i][t % V], Ue[i], st[t]);
                if (n == 0 && i < PARTS) O = mfma4(x.p[i], u[i], O);
            }
            refill();
            fetch_kt(x, n);
            if (n == 0) fetch_p(x);
            refill();
        }
        if constexpr (KSPLIT > 1) {
#pragma unroll
            for (int j = 0; j < 4; ++j) part_o[c & 1][ks][j][l] = O[j];
            if (c > 0) store(c - 1, due);
        } else {
            // over chunk c's tile: every wavefront has read its operands from it before
            // the last barrier (at the end of step c - 1, or before step 0)
            if (c + 2 < chunks) write_rows(c + 2);
            const float o[4] = {O[0], O[1], O[2], O[3]};
            store(c, o);
            __syncthreads();
        }
        refill();
    };

    offsets(min(kC, S) - 1);
    if constexpr (SHARED) {
        row_offsets(kC - 1);
        load_rows(0);
        write_rows(0);
        load_rows(1);
        write_rows(1);
        __syncthreads();
    }
    Ops x;  // the first chunk's, in the order in which the steps refill them
    refill();
#pragma unroll
    for (int n = 0; n < N; ++n) fetch_k(x, n);
    refill();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        fetch_q(x, n);
        refill();
        if (n == 0) {
            fetch_v(x);
            fetch_tb(x);
        }
        refill();
    }
    fetch_e(x);
    refill();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        fetch_kt(x, n);
        if (n == 0) fetch_p(x);
        refill();
    }
    // step 0 writes chunk 2's rows over chunk 0's tile: not before every wavefront
    // has its operands out of it
    if constexpr (SHARED) __syncthreads();
    for (int c = 0; c < chunks; ++c) step(c, x);
    if constexpr (!SHARED) {
        __syncthreads();
        float due[PARTS];
        read_output(chunks - 1, due);
        store(chunks - 1, due);
    }
}

}  // namespace
}  // namespace qdc

using namespace qdc;

extern "C" int64_t qdc_delta_scan_workspace(int64_t batch, int64_t seq, int64_t heads,
                                            int64_t key_dim, int64_t value_dim) {
    if (batch <= 0 || seq <= 0 || heads <= 0 || value_dim <= 0 || value_dim % 16) return 0;
    if (key_dim != 32 && key_dim != 64 && key_dim != 128) return 0;
    const int64_t lim = (int64_t)1 << 31;
    if (batch > 65535 || heads > 65535 || seq >= lim || value_dim >= ((int64_t)1 << 24)) return 0;
    // wavefront counts of both launches stay below 2^25 (grids below 2^31 work-items)
    const int64_t chunks = ceil_div(seq, (int64_t)kC), lanes = (int64_t)1 << 25;
    if (batch * heads >= lanes || batch * heads * chunks >= lanes ||
        batch * heads * (value_dim / 16) >= lanes / 4)
        return 0;
    return batch * heads * chunks * kRecord * 4;
}

extern "C" int32_t qdc_delta_scan_ws(void *out, int32_t out_dtype, const float *q, const float *k,
                                     const float *v, const float *beta, const float *decay,
                                     int64_t batch, int64_t seq, int64_t heads, int64_t key_heads,
                                     int64_t key_dim, int64_t value_dim, int64_t ld_qk,
                                     int64_t ld_v, void *workspace, int64_t workspace_bytes,
                                     hipStream_t stream) {
    if (!valid_dtype(out_dtype)) return QDC_ERR_DTYPE;
    if (batch < 0 || seq < 0 || heads <= 0 || key_heads <= 0 || value_dim <= 0 ||
        heads % key_heads)
        return QDC_ERR_SHAPE;
    if (ld_qk < key_heads * key_dim || ld_v < heads * value_dim) return QDC_ERR_SHAPE;
    if (batch == 0 || seq == 0) return QDC_OK;
    const int64_t need = qdc_delta_scan_workspace(batch, seq, heads, key_dim, value_dim);
    if (need == 0 || workspace_bytes < need || ld_qk % 4 || ld_v % 4 ||
        ld_qk >= ((int64_t)1 << 25) || ld_v >= ((int64_t)1 << 25))  // 32-bit chunk offsets
        return QDC_ERR_SHAPE;
    if (!out || !q || !k || !v || !beta || !decay || !workspace) return QDC_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(workspace))
        return QDC_ERR_SHAPE;
    const int64_t tokens = batch * seq;
    const int64_t out_bytes = tokens * heads * value_dim * elem_size(out_dtype);
    const int64_t qk_bytes = ((tokens - 1) * ld_qk + key_heads * key_dim) * 4;
    const int64_t v_bytes = ((tokens - 1) * ld_v + heads * value_dim) * 4;
    if (overlaps(workspace, need, out, out_bytes) || overlaps(workspace, need, q, qk_bytes) ||
        overlaps(workspace, need, k, qk_bytes) || overlaps(workspace, need, v, v_bytes) ||
        overlaps(workspace, need, beta, tokens * heads * 4) ||
        overlaps(workspace, need, decay, tokens * heads * 4))
        return QDC_ERR_ALIAS;
    ChunkArgs a{};
    a.out = out;
    a.q = q;
    a.k = k;
    a.v = v;
    a.beta = beta;
    a.decay = decay;
    a.ws = reinterpret_cast<float *>(workspace);
    a.ld_qk = ld_qk;
    a.ld_v = ld_v;
    a.S = (int)seq;
    a.H = (int)heads;
    a.vd = (int)value_dim;
    a.groups = (int)(heads / key_heads);
    a.chunks = (int)ceil_div(seq, (int64_t)kC);
    a.slices = (int)(value_dim / 16);
    a.by_chunks = make_fastdiv((uint32_t)a.chunks);
    a.by_heads = make_fastdiv((uint32_t)heads);
    a.units = batch * heads * a.chunks;
    const dim3 pgrid((uint32_t)ceil_div(a.units, (int64_t)(kBlock / kWave)));
    const int64_t slices = batch * heads * a.slices;
    // Whole slices where they fill the chip's 1024 SIMDs more than half; below, the
    // time is that of the chain of chunks, and four wavefronts a slice shorten it.
    // Whole scan, kd = vd = 128, whole slices / four wavefronts, microseconds:
    // 32 slices, 411 tokens 60 / 32; 128 slices, 777 tokens 108 / 55; 512 slices,
    // 1501 tokens 214 / 167; 640 slices, 1501 tokens 222 / 242; 1024 slices, 2048
    // tokens 350 / 474.  (Two wavefronts a slice lost to one of these everywhere.)
    const bool whole = slices > 512;
#define QDC_CHUNK_SCAN(KB, KSPLIT)                                                              \
    {                                                                                           \
        const int64_t groups = KSPLIT > 1 ? a.slices : ceil_div(a.slices, (int64_t)4);          \
        a.by_groups = make_fastdiv((uint32_t)groups);                                           \
        const dim3 grid((uint32_t)(batch * heads * groups));                                    \
        const dim3 block(KSPLIT > 1 ? KSPLIT * kWave : kBlock);                                 \
        if (out_dtype == QDC_BF16)                                                              \
            hipLaunchKernelGGL((delta_chunk_scan<KB, KSPLIT, bf16_t>), grid, block, 0, stream,  \
                               a);                                                              \
        else                                                                                    \
            hipLaunchKernelGGL((delta_chunk_scan<KB, KSPLIT, float>), grid, block, 0, stream,   \
                               a);                                                              \
        return launch_status();                                                                 \
    }
#define QDC_CHUNKED(KB, PARTS)                                                                  \
    if (key_dim == 16 * KB) {                                                                   \
        hipLaunchKernelGGL((delta_chunk_prepare<KB>), pgrid, dim3(kBlock), 0, stream, a);       \
        const int32_t status = launch_status();                                                 \
        if (status != QDC_OK) return status;                                                    \
        if (whole) QDC_CHUNK_SCAN(KB, 1)                                                        \
        QDC_CHUNK_SCAN(KB, PARTS)                                                               \
    }
    QDC_CHUNKED(8, 4)
    QDC_CHUNKED(4, 4)
    QDC_CHUNKED(2, 2)
#undef QDC_CHUNKED
#undef QDC_CHUNK_SCAN
    return QDC_ERR_SHAPE;
}
