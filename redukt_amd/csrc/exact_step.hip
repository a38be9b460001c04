// exact_step.hip — the Mamba step in the reference CPU path's own arithmetic: the
// reference-order tier.
//
// Weight profile bit 6 selects it with numeric contract 1 (the reference's "Plain" kernel
// family: every product and every sum rounded on its own), bit 7 with numeric contract 2
// (fma-v1, src/domain/gemv_fma.rs:1-26: every acc + w * x of a GEMV one fused
// multiply-add).  Every projection output (row r, stream b) is the reference GEMV of that
// row, f32_rows / q8w_rows (src/domain/gemv.rs:181-194, 459-502) or their contract-2
// twins (gemv_fma.rs:98-134): eight accumulators by column residue from +0 over the
// 8-aligned body in column order, the horizontal sum ((l0+l4)+(l2+l6)) + ((l1+l5)+(l3+l7))
// (the tail is empty: every matrix here has whole 32-column blocks); Q8 rows fold
// dot_g * scale_g over the column groups from +0.  Eight lanes of a wave hold an output's
// eight accumulators, so nothing depends on the launch shape, the batch or the slot.  The norms are the reference's sequential sums (rms_norm_into,
// layer_norm_into: src/domain/tensor.rs:900-908, 1390-1398), the scan takes the portable exp, and the
// element-wise code (conv, SiLU, softplus, the d16 recurrence, the gate, softmax) is the
// other tiers', already the CPU path's bit for bit; so the logits are the CPU path's
// logits.  Per layer:
//   k_norm_e  : the layer's RMSNorm (LayerNorm with a bias) of the residual stream;
//   k_gemv_e  : in_proj, then conv1d + SiLU (conv_silu_block order) on the conv-branch rows;
//   k_gemv_e  : x_proj, each stream's complete outputs;
//   k_scan    : shared with the other tiers (dt_proj in the contract's order);
//   k_gemv_e  : out_proj and the residual add;
// and per step k_embed_e (row gather or Q8 dequantisation, device argument check), the
// final norm, the head, and optionally the shared softmax.  exact_gemv_launch hands the same
// F32 projection to the RWKV-7 step of this tier (rwkv_a8.hip).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfma_common.h"
#include "model.h"
#include "portable_math.h"
#include "rwkv_common.h"
#include "step.h"

#pragma clang fp contract(off)

namespace rdk {

namespace {

constexpr int kEBlock = 256;      // threads (outputs) per workgroup
constexpr int kNormMax = 1024;    // d_model limit of the loader

// ---------------------------------------------------------------- embedding

struct EmbedEArgs {
    RowMat emb;
    float* x;
    const uint32_t* tokens;
    const uint32_t* slots_in;
    uint32_t* slots;
    uint32_t n, cap;
    int check;
    uint32_t* err;
};

// x[b] = emb[token[b]]: the row as stored (F32) or q * scale of its group (MambaMatrix::
// row_into, model.rs:93-101; Q8wMatrix::dequant_row_into, gemv.rs:285-295).  Block b also
// checks its entry (check_entry).
__global__ __launch_bounds__(kEBlock) void k_embed_e(EmbedEArgs a) {
    const uint32_t b = blockIdx.x;
    const RowMat& e = a.emb;
    uint32_t tok = a.tokens[b];
    check_entry(a.slots_in, a.slots, a.n, b, tok < (uint32_t)e.rows, a.cap, a.check, a.err);
    if (tok >= (uint32_t)e.rows) tok = e.rows - 1;
    const int cols = e.cols;
    float* xo = a.x + (size_t)b * cols;
    if (e.group == 0) {
        for (int c = threadIdx.x; c < cols; c += kEBlock) xo[c] = ((const float*)e.w)[rowmat_at((int)tok, c, cols, false)];
    } else {
        const int ng = cols / e.group;
        for (int c = threadIdx.x; c < cols; c += kEBlock)
            xo[c] = (float)((const int8_t*)e.w)[rowmat_at((int)tok, c, cols, true)] *
                    e.scales[rowmat_scale_at((int)tok, c / e.group, ng)];
    }
}

// ---------------------------------------------------------------- norms

struct NormEArgs {
    const float* x;     // [n][d]
    const float* w;
    const float* bias;  // LayerNorm bias, or null for RMSNorm
    float* out;         // [n][d]
    int d;
};

// One stream per workgroup: the row through LDS, the sums by one thread in index order
// (the reference's sequential loops), the scale to every thread, then the element-wise
// output.  RMSNorm (tensor.rs:900-908): inv = 1 / sqrt(sum(x^2) / d + 1e-5),
// out = x * inv * w.  LayerNorm (tensor.rs:1390-1398, two passes): mean = sum(x) / d,
// var = sum((x - mean)^2) / d, out = (x - mean) * (1 / sqrt(var + 1e-5)) * w + b.
// The sequential sum of t[0 .. d) (d a multiple of 4) by one thread, in index order: the
// reads go ahead in float4s, only the adds form the chain.
__device__ __forceinline__ float seq_sum(const float* t, int d) {
    float s = 0.0f;
#pragma unroll 8
    for (int i = 0; i < d; i += 4) {
        const float4 v = *(const float4*)(t + i);
        s = s + v.x;
        s = s + v.y;
        s = s + v.z;
        s = s + v.w;
    }
    return s;
}

__global__ __launch_bounds__(kEBlock) void k_norm_e(NormEArgs a) {
    __shared__ __align__(16) float xs[kNormMax];
    __shared__ __align__(16) float tv[kNormMax];   // the terms of the sum in flight
    __shared__ float stat[2];
    const int d = a.d;
    const float* x = a.x + (size_t)blockIdx.x * d;
    for (int i = threadIdx.x; i < d; i += kEBlock) xs[i] = x[i];
    __syncthreads();
    if (a.bias == nullptr) {
        // each term x * x rounded on its own, as in ss += x * x
        for (int i = threadIdx.x; i < d; i += kEBlock) tv[i] = xs[i] * xs[i];
        __syncthreads();
        if (threadIdx.x == 0) {
            const float rms = sqrtf(seq_sum(tv, d) / (float)d + 1e-5f);
            stat[0] = 0.0f;
            stat[1] = 1.0f / rms;
        }
    } else {
        if (threadIdx.x == 0) stat[0] = seq_sum(xs, d) / (float)d;
        __syncthreads();
        const float mean = stat[0];
        for (int i = threadIdx.x; i < d; i += kEBlock) tv[i] = (xs[i] - mean) * (xs[i] - mean);
        __syncthreads();
        if (threadIdx.x == 0) stat[1] = 1.0f / sqrtf(seq_sum(tv, d) / (float)d + 1e-5f);
    }
    __syncthreads();
    float* o = a.out + (size_t)blockIdx.x * d;
    if (a.bias == nullptr) {
        const float inv = stat[1];
        for (int i = threadIdx.x; i < d; i += kEBlock) o[i] = xs[i] * inv * a.w[i];
    } else {
        const float mean = stat[0], inv = stat[1];
        for (int i = threadIdx.x; i < d; i += kEBlock) o[i] = (xs[i] - mean) * inv * a.w[i] + a.bias[i];
    }
}

// ---------------------------------------------------------------- projections

enum : int { kEpiPlain = EXACT_STORE, kEpiIn = 1, kEpiRes = EXACT_RESID, kEpiRelu2 = EXACT_RELU2, kEpiAct = 4 };

struct GemvEArgs {
    RowMat w;               // [rows][cols]
    const float* act;       // [n][cols] input rows
    uint32_t n;
    float* out;             // kEpiPlain, kEpiRelu2: out[b * ostride + r]; kEpiRes: the residual x [n][rows]
    uint32_t ostride;
    // kEpiIn: rows below di are the conv branch (conv1d + SiLU into u, the conv state
    // updated), the rest the gate branch (z).
    float* conv_st;         // this layer's conv state [slot][di][3]
    const float* conv_w;    // [di][4]
    const float* conv_b;
    const uint32_t* slots;
    uint32_t scap;
    float* u;
    float* z;
    int di;
    uint32_t chunks;        // chunks of 4 C streams
    int stride;             // LDS row stride of the staged activations
};

// One of the products of k_gemv_multi: out[b * ostride + r] = act of row r times stream b's
// input row at x + b * ldx; its workgroups from blk0 on.
struct GemvProduct {
    RowMat w;
    const float* x;
    float* out;
    uint32_t ldx, ostride, blk0;
    int act, stride;
};
struct GemvMultiArgs {
    GemvEArgs base;   // n and chunks
    int count;
    GemvProduct prod[kExactProducts];
};

// acc + w * x in the contract's arithmetic.
template <bool FMA>
__device__ __forceinline__ float madd(float w, float x, float acc) {
    return FMA ? __builtin_fmaf(w, x, acc) : acc + w * x;
}

// One 32-column block of one tile: for each of its four columns j of every residue, x[q][j]
// (of four streams) times w[h][j] (of the lane's row h) added to acc[h][q] in the contract's
// arithmetic.  v_mfma_f32_4x4x1_16b_f32 is sixteen blocks of a 4 x 1 times 1 x 4 product: each
// of its 256 outputs is one fused multiply-add, rounded once as fmaf rounds (subnormals,
// infinities and zeros too: tests/test_gpu_exact.py holds 31 million products of operands of
// every kind to the oracle's bits).  That is contract 2; contract 1 takes the rounded products from it (accumulator +0; an exact product
// of -0 comes out +0, which an accumulator that starts at +0 and so never holds -0 cannot
// tell apart) and adds them on the vector unit, eight products issued before the first add.
// S of the four streams are live.
template <bool FMA, int R, int C, int S>
__device__ __forceinline__ void rank1_block(const f32x4 (&x)[C], const float (&w)[R][4], f32x4 (&acc)[R][C]) {
    if (FMA) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int q = 0; q < C; q++)
#pragma unroll
                for (int h = 0; h < R; h++) acc[h][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[q][j], w[h][j], acc[h][q], 0, 0, 0);
        return;
    }
    constexpr int JB = R * C <= 2 ? 4 : 8 / (R * C);
#pragma unroll
    for (int j0 = 0; j0 < 4; j0 += JB) {
        f32x4 p[JB][R][C];
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
            for (int q = 0; q < C; q++)
#pragma unroll
                for (int h = 0; h < R; h++)
                    p[j][h][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[q][j0 + j], w[h][j0 + j],
                                                                    f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < JB; j++)
#pragma unroll
            for (int q = 0; q < C; q++)
#pragma unroll
                for (int h = 0; h < R; h++)
#pragma unroll
                    for (int i = 0; i < S; i++) acc[h][q][i] = acc[h][q][i] + p[j][h][q][i];
    }
}

// Lanes 0 .. 31: a of the lane plus a of lane + 32; lanes 32 .. 63: b of lane - 32 plus b of
// the lane.  pair16: the same within each half, 16 lanes apart; pair8: within each 16, 8 apart.
__device__ __forceinline__ float pair32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float pair16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
constexpr int kDppRowRor8 = 0x128;   // lane i of a row of 16 reads lane i ^ 8
__device__ __forceinline__ float pair8(float a, float b, bool upper) {
    const float keep = upper ? b : a, give = upper ? a : b;
    return keep + dpp_move<kDppRowRor8>(give);
}

// The weights of one 32-column block: the lane's four columns of its R rows (R = 2: the tile's
// two, R = 1: row h), and the scale that folds the column group the block ends (GB blocks a
// group; sc is the tile's scales at the lane's output row).
template <bool Q8, int R>
struct TileRaw {
    uint32_t q[R];
    float4 f[R];
    float sc;
};
template <bool Q8, int R, int GB>
__device__ __forceinline__ TileRaw<Q8, R> tile_load(const RowMat& m, size_t t0, int k, int h, int lane, const float* sc) {
    TileRaw<Q8, R> r;
    const size_t blk = t0 + k;
    if (Q8) {
        const uint32_t* q = (const uint32_t*)m.w + (blk * 64 + lane) * 2;
        if (R == 2) {
            const uint2 v = *(const uint2*)q;
            r.q[0] = v.x, r.q[R - 1] = v.y;
        } else {
            r.q[0] = q[h];
        }
        if (GB > 0) r.sc = sc[(size_t)(k / (GB > 0 ? GB : 1)) * kRowTile];
    } else {
#pragma unroll
        for (int i = 0; i < R; i++) r.f[i] = ((const float4*)m.w)[blk * 128 + 64 * (R == 2 ? i : h) + lane];
    }
    return r;
}
template <bool Q8, int R>
__device__ __forceinline__ void tile_decode(const TileRaw<Q8, R>& r, float (&w)[R][4]) {
#pragma unroll
    for (int h = 0; h < R; h++) {
        if (Q8) {
#pragma unroll
            for (int j = 0; j < 4; j++) w[h][j] = (float)(int8_t)(r.q[h] >> (8 * j));
        } else {
            w[h][0] = r.f[h].x, w[h][1] = r.f[h].y, w[h][2] = r.f[h].z, w[h][3] = r.f[h].w;
        }
    }
}

constexpr int kEWaves = kEBlock / kWave;
constexpr int kEAhead = 8;        // 32-column blocks of weights in flight per wave
constexpr int kEAheadShort = 4;   // the same where no row of a launch of several products is longer

// One wave computes 8 R rows x 4 C streams.  Lane 8 l + r holds the reference's accumulators
// l of row r of each octet, one register per stream: each step of a 32-column block adds one
// column of every residue (rank1), so an accumulator takes the columns c = l (mod 8) of a
// column group in order from +0.  The horizontal sum ((l0+l4)+(l2+l6)) + ((l1+l5)+(l3+l7)) is
// pair32, pair16, pair8 (each level also folds two registers into one, so lane 16 s + i ends
// with row i of stream s); Q8 rows then take sum = sum + dot * scale from +0, in the
// contract's arithmetic.  Workgroup: four waves of different rows, the 4 C streams' input
// rows staged in LDS, interleaved by residue (column 32 k + 8 j + l at 32 k + 4 l + j) so that
// a lane reads its four columns of a block at once.  GB: 32-column blocks per scale group (0:
// the whole row is one sum).
//
// Bound by vector instructions once the batch fills the chip (the head of 100 F32 streams,
// contract 1: they take 86 % of the cycles that its CUs are busy, SQ_ACTIVE_INST_VALU over
// SQ_BUSY_CU_CYCLES; 71 % of them are the adds themselves), by the chain of dependent products and the load latencies below that.  The version before this
// one (eight lanes an output on the vector unit, each product reading its activation from
// LDS) was bound by LDS.  us a launch, before and now: F32 contract 1 at 100 streams in_proj
// 28.5 -> 19.6, x_proj 16.6 -> 6.9, out_proj 19.6 -> 12.0, head 357 -> 187; int8 groups of 64
// contract 2 at 32 streams 14.5 -> 8.0, 14.3 -> 5.2, 17.2 -> 7.2, 87.8 -> 51.5.
//
// (Two workgroups a CU at least: at most 256 registers, so the products land in vector
// registers, not in accumulation registers that the adds would have to be copied from.)
template <bool Q8, bool FMA, int R, int C, int S, int EPI, int GB, int AHEAD>
__device__ __forceinline__ void gemv_e_body(const GemvEArgs& a, const RowMat& m, const float* act, uint32_t ldx, float* out,
                                            uint32_t ostride, int stride, int actv, uint32_t lin) {
    extern __shared__ __align__(16) float acts[];   // [4 C][stride]
    const int parts = m.tiles() * (2 / R);   // tiles (R = 2) or their halves of 8 rows
    const XcdTile job = xcd_tile(lin, a.chunks, (uint32_t)((parts + kEWaves - 1) / kEWaves));
    if (!job.live) return;
    const int lane = threadIdx.x % kWave, wave = wave_index();
    const int cols = m.cols, nb = cols / 32;
    const int p_raw = (int)job.unit * kEWaves + wave;
    const int part = min(p_raw, parts - 1), t = R == 2 ? part : part / 2, half = R == 2 ? 0 : part % 2;
    const uint32_t b0 = job.part * (4 * C);
    const size_t w0 = (size_t)t * nb;
    // the row of the lane's outputs; R = 1: lanes 8 .. 15 of each 16 hold copies
    const int r16 = R == 2 ? lane % 16 : 8 * half + lane % 8;
    const int r = t * kRowTile + r16;
    const bool row_live = p_raw < parts && r < m.rows && (R == 2 || (lane & 8) == 0);
    constexpr int kGB = GB > 0 ? GB : 1;   // (no division by zero in the other instantiation)
    const int ng = GB > 0 ? nb / kGB : 1;
    const float* scales = Q8 ? m.scales + (size_t)t * ng * kRowTile + r16 : nullptr;
    TileRaw<Q8, R> raw[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) raw[i] = tile_load<Q8, R, GB>(m, w0, min(i, nb - 1), half, lane, scales);
    const float sc_row = Q8 && GB == 0 ? scales[0] : 0.0f;
    // the epilogue's operands, requested with the products'
    float old[C], cs[C][3], cb = 0.0f;
    float4 cw = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    size_t cst[C];
    const bool conv = EPI == kEpiIn && row_live && r < a.di;
#pragma unroll
    for (int q = 0; q < C; q++) {
        const uint32_t b = b0 + 4 * q + (uint32_t)lane / 16;
        old[q] = EPI == kEpiRes && row_live && b < a.n ? out[(size_t)b * ostride + r] : 0.0f;
        cs[q][0] = cs[q][1] = cs[q][2] = 0.0f;
        cst[q] = 0;
        if (conv && b < a.n) {
            cst[q] = ((size_t)clamp_slot(a.slots[b], a.scap) * a.di + r) * 3;
#pragma unroll
            for (int k = 0; k < 3; k++) cs[q][k] = a.conv_st[cst[q] + k];
        }
    }
    if (conv) {
        cw = *(const float4*)(a.conv_w + (size_t)r * 4);
        cb = a.conv_b[r];
    }
#pragma unroll
    for (int s = 0; s < C; s++) {
        const int sr = wave + kEWaves * s;   // the wave's streams; S == 1: only the first is read
        const float* src = act + (size_t)min(b0 + (uint32_t)sr, a.n - 1) * ldx;
        if (S == 4 || sr < S) {
#pragma unroll 3
            for (int q = lane; q < cols / 4; q += kWave) {
                const float* p = src + 32 * (q / 8) + q % 8;
                const float4 v = make_float4(p[0], p[8], p[16], p[24]);
                *(float4*)(acts + sr * stride + 4 * q) = v;
            }
        }
    }
    __syncthreads();
    const float* xa = acts + (S == 1 ? 0 : lane % 4) * stride + 4 * (lane / 8);
    f32x4 acc[R][C];
    float res[C];
#pragma unroll
    for (int q = 0; q < C; q++) {
#pragma unroll
        for (int h = 0; h < R; h++) acc[h][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        res[q] = 0.0f;
    }
    auto finish = [&](float sc) {
#pragma unroll
        for (int q = 0; q < C; q++) {
            float h2[R];
#pragma unroll
            for (int h = 0; h < R; h++) {
                const f32x4 v = acc[h][q];
                h2[h] = S == 1 ? pair16(pair32(v[0], v[0]), pair32(v[0], v[0]))
                               : pair16(pair32(v[0], v[2]), pair32(v[1], v[3]));
                acc[h][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            const float v = pair8(h2[0], h2[R - 1], (lane & 8) != 0);
            res[q] = Q8 ? madd<FMA>(v, sc, res[q]) : v;
        }
    };
    f32x4 x[C];
#pragma unroll
    for (int q = 0; q < C; q++) x[q] = *(const f32x4*)(xa + (4 * q) * stride);
    // (the next block's activations are requested before this block's products)
    auto block = [&](const TileRaw<Q8, R>& rw, int k) {
        f32x4 xn[C];
#pragma unroll
        for (int q = 0; q < C; q++) xn[q] = *(const f32x4*)(xa + (4 * q) * stride + 32 * min(k + 1, nb - 1));
        __builtin_amdgcn_sched_barrier(0);
        float w[R][4];
        tile_decode<Q8, R>(rw, w);
        rank1_block<FMA, R, C, S>(x, w, acc);
        if (GB > 0 && (k + 1) % kGB == 0) finish(rw.sc);
#pragma unroll
        for (int q = 0; q < C; q++) x[q] = xn[q];
    };
    const int nbm = nb / AHEAD * AHEAD;
    for (int k0 = 0; k0 < nbm; k0 += AHEAD) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            block(raw[i], k0 + i);
            raw[i] = tile_load<Q8, R, GB>(m, w0, min(k0 + AHEAD + i, nb - 1), half, lane, scales);
        }
    }
    // the last nb % AHEAD blocks, already in raw[0 ..]
#pragma unroll
    for (int i = 0; i < AHEAD - 1; i++)
        if (nbm + i < nb) block(raw[i], nbm + i);
    if (GB == 0) finish(sc_row);
    if (!row_live) return;
#pragma unroll
    for (int q = 0; q < C; q++) {
        const uint32_t b = b0 + 4 * q + (uint32_t)lane / 16;
        if (b >= a.n) continue;
        const float y = res[q];
        if (EPI == kEpiAct) {
            out[(size_t)b * ostride + r] = activate(actv, y, r, m.rows);
        } else if (EPI == kEpiPlain) {
            out[(size_t)b * ostride + r] = y;
        } else if (EPI == kEpiRes) {
            // x += W_out * gated (model.rs:714-719): the residual add after the projection
            out[(size_t)b * ostride + r] = old[q] + y;
        } else if (EPI == kEpiRelu2) {
            // squared_relu_into (tensor.rs:1386-1388): max(y, 0)^2, a NaN to 0
            const float v = y > 0.0f ? y : 0.0f;
            out[(size_t)b * ostride + r] = v * v;
        } else if (r >= a.di) {
            a.z[(size_t)b * a.di + (r - a.di)] = y;
        } else {
            // conv_silu_block (model.rs:134-153) for channel r of stream b, then SiLU with the
            // lane sigmoid: d_inner comes in whole 64-channel blocks, so every channel is in
            // the 8-aligned body of its 256-channel block (tensor.rs:1197-1211).
            float* st = a.conv_st + cst[q];
            float val = 0.0f;
            val += cs[q][0] * cw.x;
            val += cs[q][1] * cw.y;
            val += cs[q][2] * cw.z;
            val += y * cw.w;
            val += cb;
            st[0] = cs[q][1];
            st[1] = cs[q][2];
            st[2] = y;
            a.u[(size_t)b * a.di + r] = val * lane_sigmoid_f(val);
        }
    }
}

template <bool Q8, bool FMA, int R, int C, int S, int EPI, int GB>
__global__ __launch_bounds__(kEBlock, 2) void k_gemv_e(GemvEArgs a) {
    gemv_e_body<Q8, FMA, R, C, S, EPI, GB, kEAhead>(a, a.w, a.act, (uint32_t)a.w.cols, a.out, a.ostride, a.stride, ACT_NONE,
                                           blockIdx.x);
}

// Several F32 contract-1 products that do not read each other's outputs in one launch: RWKV-7's
// receptance, key, value and first LoRA stages, then its second LoRA stages.  The LoRAs had a
// kernel of their own, a lane per accumulator and every operand from memory: at 64 streams
// 9.4 us a launch twice a layer beside 11.3 for the other three products; now 16.2 and 5.1.
template <int R, int C, int S, int AHEAD>
__global__ __launch_bounds__(kEBlock, 2) void k_gemv_multi(GemvMultiArgs a) {
    int i = 0;
    for (int k = 1; k < a.count; k++)
        if (blockIdx.x >= a.prod[k].blk0) i = k;
    const GemvProduct& p = a.prod[i];
    gemv_e_body<false, false, R, C, S, kEpiAct, 0, AHEAD>(a.base, p.w, p.x, p.ldx, p.out, p.ostride, p.stride, p.act,
                                                   blockIdx.x - p.blk0);
}

template <int R, int C, int S, int EPI>
const void* gemv_e_fn(const RowMat& w, bool fma) {
    if (w.group == 0) return fma ? (const void*)k_gemv_e<false, true, R, C, S, EPI, 0> : (const void*)k_gemv_e<false, false, R, C, S, EPI, 0>;
    if (w.group == w.cols) return fma ? (const void*)k_gemv_e<true, true, R, C, S, EPI, 0> : (const void*)k_gemv_e<true, false, R, C, S, EPI, 0>;
    constexpr int kGB = kRowMatGroup / 32;   // (make_rowmat takes no other group)
    return fma ? (const void*)k_gemv_e<true, true, R, C, S, EPI, kGB> : (const void*)k_gemv_e<true, false, R, C, S, EPI, kGB>;
}

// A wave's share of a product: 8 R rows and 4 C streams.
struct Share {
    int r, c;
};
typedef const void* (*GemvPick)(uint32_t n, Share s, const RowMat& w, bool fma);
template <int EPI>
const void* gemv_e_pick(uint32_t n, Share s, const RowMat& w, bool fma) {
    if (s.r == 1) return n == 1 ? gemv_e_fn<1, 1, 1, EPI>(w, fma) : gemv_e_fn<1, 1, 4, EPI>(w, fma);
    return s.c == 1 ? gemv_e_fn<2, 1, 4, EPI>(w, fma) : gemv_e_fn<2, 2, 4, EPI>(w, fma);
}

constexpr uint32_t kELdsMax = 64 * 1024;
// LDS row stride of the staged activations: 32 words more than the row, so that the four
// streams of a quad start in alternating halves of the banks; the row alone where that would
// not fit (4,096 columns).
int acts_stride(int cols, int quads) {
    return 16 * (uint32_t)quads * (uint32_t)(cols + 32) <= kELdsMax ? cols + 32 : cols;
}

// The smallest share (8 rows x 4 streams) up to ten waves a SIMD, since a lone wave issues at
// a third of the vector rate and its chain of products is the kernel's time; above that 16
// rows x 8 streams, which reads each operand half as often.  us a launch, shares of 8 x 4,
// 8 x 8, 16 x 4, 16 x 8, 16 x 16 (Mamba-130M; F32 contract 1 at 100 streams, then int8 groups
// of 64 contract 2 at 32): in_proj 19.6, 19.7, 19.6, 20.1, 25.3 and 8.0, 8.7, 8.1, 8.7, 13.2;
// x_proj 6.9, 10.9, 10.0, 16.4 and 5.2, 7.0, 6.8, 8.6; out_proj 12.0, 13.8, 14.4, 17.0 and 7.2,
// 9.4, 8.8, 12.0; the head 229, 191, 218, 187, 200 and 67.6, 55.4, 55.6, 51.5, 53.7.
Share exact_share(uint32_t tiles, int cols, uint32_t n) {
    const uint64_t waves = (uint64_t)tiles * 2 * ((n + 3) / 4);
    if (waves <= 10 * 1024) return Share{1, 1};
    return Share{2, 32u * (uint32_t)cols <= kELdsMax ? 2 : 1};
}

uint32_t gemv_e_grid(const RowMat& w, Share s, uint32_t chunks) {
    return xcd_grid(chunks, (uint32_t)((w.tiles() * (2 / s.r) + kEWaves - 1) / kEWaves));
}

Launch gemv_e_launch(GemvPick pick, bool fma, int cls, const RowMat& w, const float* act, uint32_t n, GemvEArgs a) {
    const Share s = exact_share((uint32_t)w.tiles(), w.cols, n);
    a.w = w;
    a.act = act;
    a.n = n;
    a.chunks = (n + 4 * s.c - 1) / (4 * s.c);
    a.stride = acts_stride(w.cols, s.c);
    const uint32_t lds = 16u * (uint32_t)s.c * (uint32_t)a.stride;
    return Launch::make(pick(n, s, w, fma), dim3(gemv_e_grid(w, s, a.chunks)), dim3(kEBlock), lds, (uint32_t)cls, a);
}

}  // namespace

Launch exact_gemv_launch(const RowMat& w, const float* act, uint32_t n, float* out, uint32_t ostride, int epi,
                         uint32_t cls) {
    GemvEArgs a{};
    a.out = out;
    a.ostride = ostride;
    const GemvPick pick = epi == EXACT_RESID   ? gemv_e_pick<kEpiRes>
                          : epi == EXACT_RELU2 ? gemv_e_pick<kEpiRelu2>
                                               : gemv_e_pick<kEpiPlain>;
    return gemv_e_launch(pick, false, (int)cls, w, act, n, a);
}

namespace {
template <int AHEAD>
const void* gemv_multi_fn(uint32_t n, Share s) {
    if (s.r == 1) return n == 1 ? (const void*)k_gemv_multi<1, 1, 1, AHEAD> : (const void*)k_gemv_multi<1, 1, 4, AHEAD>;
    static_assert(32 * kExactProductCols <= (int)kELdsMax, "a share of 16 rows takes 8 streams (exact_share)");
    return (const void*)k_gemv_multi<2, 2, 4, AHEAD>;
}
}  // namespace

Launch exact_gemv_multi_launch(const ExactProduct* prod, int count, uint32_t n, uint32_t cls) {
    uint32_t tiles = 0;
    int cols = 0;
    for (int k = 0; k < count; k++) {
        tiles += (uint32_t)prod[k].w->tiles();
        cols = std::max(cols, prod[k].w->cols);
    }
    const Share s = exact_share(tiles, cols, n);
    GemvMultiArgs a{};
    a.base.n = n;
    a.base.chunks = (n + 4 * s.c - 1) / (4 * s.c);
    a.count = count;
    uint32_t grid = 0, lds = 0;
    for (int k = 0; k < count; k++) {
        const ExactProduct& p = prod[k];
        const int stride = acts_stride(p.w->cols, s.c);
        a.prod[k] = GemvProduct{*p.w, p.x, p.out, p.ldx, p.ostride, grid, p.act, stride};
        grid += gemv_e_grid(*p.w, s, a.base.chunks);
        lds = std::max(lds, 16u * (uint32_t)s.c * (uint32_t)stride);
    }
    const void* fn = cols <= 32 * kEAheadShort ? gemv_multi_fn<kEAheadShort>(n, s) : gemv_multi_fn<kEAhead>(n, s);
    return Launch::make(fn, dim3(grid), dim3(kEBlock), lds, cls, a);
}

void ExactStep::build(Pool& p, const StepIO& io, std::vector<Launch>& out, int& io_i, int& head_i, int& sm_i) const {
    const Dims& D = *m.dims;
    const uint32_t n = io.n;
    const int d = (int)D.d, di = (int)D.di;
    const bool fma = m.fma;
    out.clear();
    io_i = (int)out.size();
    EmbedEArgs ea{*m.emb, p.x, io.tokens, io.slots, p.slots, n, p.cap, io.check ? 1 : 0, io.err};
    out.push_back(Launch::make((const void*)k_embed_e, dim3(n), dim3(kEBlock), 0, KC_EMBED, ea));
    const size_t conv_layer = (size_t)p.scap * di * (D.dc - 1);
    const size_t ssm_layer = (size_t)p.scap * di * 16;
    const uint32_t xr_pad = (uint32_t)(m.layers[0].x_proj.rt * kRowTile);
    for (uint32_t li = 0; li < D.nl; li++) {
        const DLayer& L = m.layers[li];
        out.push_back(Launch::make((const void*)k_norm_e, dim3(n), dim3(kEBlock), 0, KC_NORM,
                                   NormEArgs{p.x, L.norm_w, L.norm_b, p.normed, d}));
        GemvEArgs gi{};
        gi.conv_st = p.conv + li * conv_layer;
        gi.conv_w = L.conv_w;
        gi.conv_b = L.conv_b;
        gi.slots = p.slots;
        gi.scap = p.scap;
        gi.u = p.u;
        gi.z = p.z;
        gi.di = di;
        out.push_back(gemv_e_launch(gemv_e_pick<kEpiIn>, fma, KC_MIX_IN, L.e_in, p.normed, n, gi));
        GemvEArgs gx{};
        gx.out = p.xpart;
        gx.ostride = xr_pad;
        out.push_back(gemv_e_launch(gemv_e_pick<kEpiPlain>, fma, KC_XPROJ, L.e_xp, p.u, n, gx));
        out.push_back(scan_exact_launch(L, D, p, n, fma, p.g32, p.ssm + li * ssm_layer));
        GemvEArgs go{};
        go.out = p.x;
        go.ostride = (uint32_t)d;
        out.push_back(gemv_e_launch(gemv_e_pick<kEpiRes>, fma, KC_MIX_OUT, L.e_out, p.g32, n, go));
    }
    out.push_back(Launch::make((const void*)k_norm_e, dim3(n), dim3(kEBlock), 0, KC_NORM,
                               NormEArgs{p.x, m.norm_f_w, m.norm_f_b, p.normed, d}));
    head_i = (int)out.size();
    GemvEArgs gh{};
    gh.out = io.out;
    gh.ostride = D.vocab;
    out.push_back(gemv_e_launch(gemv_e_pick<kEpiPlain>, fma, KC_HEAD, *m.head, p.normed, n, gh));
    sm_i = -1;
    if (io.probs) {
        sm_i = (int)out.size();
        out.push_back(softmax_launch(io.out, (int)D.vocab, n));
    }
}

}  // namespace rdk
