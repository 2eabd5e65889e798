// fp32 NT GEMM on gfx950 MFMA: out[m][n] = epilogue(sum_t a[m][t] * b[n][t]).
//
// The contraction is GemmBackend::matmul_nt (crates/raya-kernels/src/gemm.rs:2-11):
// a is [m, k] row-major, b is a Linear weight [n, k] row-major, so both
// operands are contiguous along k.
//
// Arithmetic.  Every fp32 operand, times 2^23 (exact), is written as the sum of three bfloat16
// parts: x0 = x rounded to 8 bits, x1 = x - x0 rounded to 8 bits, x2 = x - x0 - x1.  Both
// differences are exact in fp32 and the second has at most 7 bits, so x = x0 + x1 + x2
// exactly, with |x1| <= 2^-8 |x| and |x2| <= 2^-17 |x|.  The scale lifts the last bit of the
// smallest fp32 subnormal (2^-149) to bfloat16's smallest normal number: unscaled, the lower
// parts of an operand below 2^-110 fell below bfloat16's smallest subnormal (the product was off
// by 2e-6 at 2^-116 and 6e-4 at 2^-124), and the matrix instruction aligns a subnormal part as
// if its leading bit were set, which costs the sum up to 7 bits.  The sums leave the scale by
// 2^-46 after the K loop.  The scaling takes 1% of a large product (QKV at 21,405 rows 380 ->
// 384 us) and gives the same bits wherever the unscaled parts were exact.  Of the nine part
// products the six
// a2 b0 + a0 b2 + a1 b1 + a1 b0 + a0 b1 + a0 b0 are summed, each exact in the fp32
// accumulator of v_mfma_f32_32x32x16_bf16; a1 b2 and a2 b1 (each at most 2^-25 of |a b|,
// typically 2^-28) and a2 b2 are left out.  The accumulator takes 6 roundings per 16 k where
// v_mfma_f32_32x32x2_f32 takes 16, so the result is nearer to the 64-bit product than the
// fp32 instruction's: relative 2-norm error 4.2e-7 against 5.0e-7 at k = 768, 8.7e-7
// against 1.1e-6 at k = 3072 (N(0, 1) rows, N(0, 0.02) weights).  The bfloat16
// instruction runs 16 times the fp32 one's rate (dense peaks 2.5 PFLOP/s and 157
// TFLOP/s), so six of them take 6 / 16 of the time.  What bounds the large tiles is the
// chip's power: the shader clock falls from 2.4 to about 1.75 GHz while they run, and a
// plain library bfloat16 product reaches 1,430 TFLOP/s (238 in these terms; its fp32 one
// 155).  At M = 21,405, [N, K] = 2304 x 768: 550-587 us by card (138-129 TFLOP/s) on the fp32
// instruction, 368-398 (206-190) here; on the slower card 768 x 768 189 -> 129 us, GeGLU
// 6144 x 768 1,479 -> 929, 768 x 3072 724 -> 448.
//
// Parts of Inf and NaN (and of |x| from 2^105 on, whose scaled value is above the largest
// bfloat16) are not sums of anything, so such an operand leaves every output of its row or column
// not finite, and so does a scaled sum past the largest float (2^82 unscaled); those outputs, and
// only those, are computed again with the fp32 instruction over the unsplit operands
// (exact_subtile).
//
// Register layouts (lane l, half h = l / 32):
//   v_mfma_f32_32x32x16_bf16: A[i][8h .. 8h + 7] in lane i + 32 h, B[.][j] in lane j + 32 h;
//   v_mfma_f32_32x32x2_f32:   A[i][h] in lane i + 32 h, B[h][j] in lane j + 32 h;
//   both: D[i][j] in lane j + 32 ((i / 4) % 2), register 4 (i / 8) + i % 4.
//
// Epilogues (ops.rs:91-109 bias add, encoder.rs:139-146 GeGLU, head.rs:392
// ReLU, encoder.rs:132-134 residual add): y = acc + bias; y = act(y);
// out = y + residual.  For GeGLU the weight has 2n rows; a workgroup loads the
// "input" rows j and the "gate" rows n + j side by side so that both halves of
// an output element land in the same lane and register.  The plain epilogue can
// also apply rotary embedding (ops.rs:118-141) to the q and k sections of a
// packed QKV projection, so encoder::attend's split_qkv + rope_in_place pass
// (encoder.rs:36-71) is not needed.
#pragma once

#include <algorithm>
#include <type_traits>

#include "internal.hpp"
#include "parts.hpp"
#include "row_norm.hpp"

namespace raya {
namespace gemm {

__device__ __forceinline__ floatx16 mfma_f32(float a, float b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float gelu_erf(float x) {
    return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}

// The plain activations, one branch for the wave.
__device__ __forceinline__ float activate(int act, float x) {
    if (act == RAYA_EPI_GELU) return gelu_erf(x);
    if (act == RAYA_EPI_RELU) return fmaxf(x, 0.0f);
    return x;
}

// The biases of this lane's columns of the wave's 64 (GeGLU: input column and gate).
template <bool GEGLU>
__device__ __forceinline__ void load_bias(const GemmLaunch &g, int c0, int li, float (&bias)[2]) {
    bias[0] = bias[1] = 0.f;
    if (!g.bias) return;
    if constexpr (GEGLU) {
        const int col = min(c0 + li, g.n - 1);
        bias[0] = g.bias[col];
        bias[1] = g.bias[g.n + col];
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) bias[j] = g.bias[min(c0 + 32 * j + li, g.n - 1)];
    }
}

constexpr int kXcds = 8;     // workgroup i runs on XCD i mod 8, each with its own L2

// Output tile of workgroup `bid`.  Each XCD takes a contiguous range of the
// tile sequence, and the sequence walks GROUP_M row blocks at a time, column
// by column, so a B column tile is reused GROUP_M times and the A row blocks of
// a group stay in that XCD's L2 while all of B streams past them.
template <int GROUP_M>
__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int total = tiles_m * tiles_n;
    const int per = total / kXcds, rem = total % kXcds;
    const int xcd = bid % kXcds, slot = bid / kXcds;
    const int t = xcd * per + min(xcd, rem) + slot;
    const int width = GROUP_M * tiles_n;
    const int group = t / width, first = group * GROUP_M;
    const int size = min(tiles_m - first, GROUP_M);
    const int r = t - group * width;
    tm = first + r % size;
    tn = r / size;
}

// Epilogue for out or residual rows that are not 16-byte aligned, on biased sums.
// Register r of acc[i][j] is row wm + 32 i + 8 (r / 4) + 4 h + r % 4 and column
// c0 + 32 j + li; a wave holds TM x 2 such 32 x 32 subtiles.
template <bool GEGLU, int TM>
__device__ __forceinline__ void epilogue(const GemmLaunch &g, const float (&acc)[TM][2][16], int m0, int wm, int c0,
                                         int li, int h) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row >= g.m) continue;
            float y[2] = {acc[i][0][r], acc[i][1][r]};
            if constexpr (GEGLU) {
                y[0] = gelu_erf(y[0]) * y[1];
            } else {
                y[0] = activate(g.act, y[0]);
                y[1] = activate(g.act, y[1]);
                // Columns c and c + 32 of one 64-wide head sit in the same lane and
                // register of acc[i][0] and acc[i][1].
                if (g.rope_cos && c0 < g.rope_cols) {
                    const int64_t t = (int64_t)g.positions[row] * (kRopeHeadDim / 2) + li;
                    const float c = g.rope_cos[t], sn = g.rope_sin[t];
                    const float x0 = y[0], x1 = y[1];
                    y[0] = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, sn));
                    y[1] = __fadd_rn(__fmul_rn(x1, c), __fmul_rn(x0, sn));
                }
            }
#pragma unroll
            for (int j = 0; j < (GEGLU ? 1 : 2); ++j) {
                const int col = c0 + 32 * j + li;
                if (col >= g.n) continue;
                float v = y[j];
                if (g.residual) v += g.residual[(int64_t)row * g.ldr + col];
                g.out[(int64_t)row * g.ldo + col] = v;
            }
        }
    }
}

// Sum over each 16-lane row of the wave with DPP moves (no LDS crossbar): lane
// pairs (quad_perm [1,0,3,2]), quads ([2,3,0,1]), then the row's halves of 8
// (row_half_mirror pairs quad 0 with 1 and 2 with 3) and the row (row_mirror
// pairs quad 0 with 3 and 1 with 2).  Every step adds the same two values in
// each lane of a pair, in the other order, and addition commutes, so all 16
// lanes hold the same bits.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_sum(float x) {
    x += dpp<0xB1>(x);   // quad_perm [1, 0, 3, 2]
    x += dpp<0x4E>(x);   // quad_perm [2, 3, 0, 1]
    x += dpp<0x141>(x);  // row_half_mirror
    x += dpp<0x140>(x);  // row_mirror
    return x;
}

// Epilogue through LDS, for out (and residual) with row strides a multiple of 4
// floats and 16-byte aligned bases: each wave writes its biased sums to its own
// LDS area and reads them back row-major, where the activation is applied (GeGLU: columns
// 0-31 are the inputs, 32-63 their gates) and RoPE reads its tables as float4,
// and the residual reads and the stores are float4 with 256-byte (GeGLU: 128-byte)
// row segments: a quarter of the store instructions of the accumulator layout.
// Staged row strides: lanes i and i + 32 of a write are 4 rows apart, and
// 4 * stride = 32 (mod 64) puts them on disjoint banks.
constexpr int kStageStride = 72;  // 64 columns per wave
constexpr int kStageFloats = 32 * kStageStride;  // per wave: 32 rows at a time

//
// With g.out_stats, each wave's 64 output columns are one chunk: the 16 lanes that
// hold a row reduce its sum to the chunk mean c (the same bits in every lane), then the
// deviations from c and their squares.
//
// RES false: the launch has no residual.  (With the rows' registers and the branch round them left in,
// QKV at 21,405 rows took 375 us instead of 368, the act head's 64 x 256 x 772 19.3 instead of 18.7.)
template <bool GEGLU, bool STATS, int TM, bool RES>
__device__ __forceinline__ void epilogue_staged(const GemmLaunch &g, const float (&acc)[TM][2][16], int m0, int wm,
                                                int c0, int li, int h, int lane, float *stg) {
    constexpr int COLS = GEGLU ? 32 : 64;  // output columns of this wave
    constexpr int S = kStageStride;
    constexpr int C4 = COLS / 4;           // float4 per output row
    constexpr int NT = 32 * C4 / 64;       // of them, per lane
    const bool ahead = RES && g.residual && g.n >= 4;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        // The 32 rows' residual is fetched together, before the staging: one latency instead of one
        // for each float4 (17,809 x 4,404: k = 112 275 -> 218 us, k = 768 677 -> 641; the 12-layer
        // forward of 512 tokens 1,825 -> 1,782).
        float4 add[NT] = {};
        if (ahead) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int idx = t * 64 + lane, col = c0 + 4 * (idx % C4), row = m0 + wm + 32 * i + idx / C4;
                const bool whole = row < g.m && col + 4 <= g.n;
                add[t] = *(const float4 *)(g.residual + (whole ? (int64_t)row * g.ldr + col : 0));
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int rr = 8 * (r >> 2) + 4 * h + (r & 3);
            stg[rr * S + li] = acc[i][0][r];
            stg[rr * S + 32 + li] = acc[i][1][r];
        }
        // LDS accesses of one wave complete in order: the reads below see the
        // writes above, and the next half's writes follow these reads.
        if (!GEGLU && !STATS && g.rope_cos) {
            // RoPE on row-major data: this wave's 64 columns are one head (c0 is a
            // multiple of 64), so a lane takes the 16-byte chunks c4 and c4 + 8 of a row,
            // columns c .. c + 3 and c + 32 .. c + 35 with c = 4 c4, and rotates each pair
            // at frequencies c .. c + 3: one float4 of each table per 8 outputs.  Bias and
            // activation came first, as in epilogue(); launch_gemm takes no residual with RoPE.
            const bool rot = c0 < g.rope_cols;  // the q and k sections: whole heads
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int idx = t * 64 + lane, rr = idx >> 3, c4 = idx & 7;
                const int row = m0 + wm + 32 * i + rr;
                if (row >= g.m) continue;
                float4 x0 = *(const float4 *)&stg[rr * S + 4 * c4];
                float4 x1 = *(const float4 *)&stg[rr * S + 32 + 4 * c4];
                if (rot) {
                    const int64_t tb = (int64_t)g.positions[row] * (kRopeHeadDim / 2) + 4 * c4;
                    const float4 cs4 = *(const float4 *)(g.rope_cos + tb), sn4 = *(const float4 *)(g.rope_sin + tb);
                    const auto turn = [](float &a, float &b, float c, float sn) {
                        const float a0 = a, b0 = b;
                        a = __fsub_rn(__fmul_rn(a0, c), __fmul_rn(b0, sn));
                        b = __fadd_rn(__fmul_rn(b0, c), __fmul_rn(a0, sn));
                    };
                    turn(x0.x, x1.x, cs4.x, sn4.x);
                    turn(x0.y, x1.y, cs4.y, sn4.y);
                    turn(x0.z, x1.z, cs4.z, sn4.z);
                    turn(x0.w, x1.w, cs4.w, sn4.w);
                }
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int col = c0 + 32 * half + 4 * c4;
                    if (col >= g.n) continue;
                    const float4 v = half ? x1 : x0;
                    float *o = g.out + (int64_t)row * g.ldo + col;
                    if (col + 4 <= g.n) {
                        *(float4 *)o = v;
                    } else {
                        const float e[4] = {v.x, v.y, v.z, v.w};
                        for (int q = 0; q < 4 && col + q < g.n; ++q) o[q] = e[q];
                    }
                }
            }
            continue;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int idx = t * 64 + lane, rr = idx / C4, c4 = idx % C4;
            const int row = m0 + wm + 32 * i + rr, col = c0 + 4 * c4;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < g.m && col < g.n) {
                v = *(const float4 *)&stg[rr * S + 4 * c4];
                if constexpr (GEGLU) {
                    const float4 gate = *(const float4 *)&stg[rr * S + 32 + 4 * c4];
                    v.x = gelu_erf(v.x) * gate.x;
                    v.y = gelu_erf(v.y) * gate.y;
                    v.z = gelu_erf(v.z) * gate.z;
                    v.w = gelu_erf(v.w) * gate.w;
                } else if (g.act != RAYA_EPI_NONE) {
                    v.x = activate(g.act, v.x);
                    v.y = activate(g.act, v.y);
                    v.z = activate(g.act, v.z);
                    v.w = activate(g.act, v.w);
                }
                float *o = g.out + (int64_t)row * g.ldo + col;
                const float *res = RES && g.residual ? g.residual + (int64_t)row * g.ldr + col : nullptr;
                if (col + 4 <= g.n) {
                    if (res) {
                        v.x += add[t].x;
                        v.y += add[t].y;
                        v.z += add[t].z;
                        v.w += add[t].w;
                    }
                    *(float4 *)o = v;
                } else {
                    const float e[4] = {v.x, v.y, v.z, v.w};
                    for (int q = 0; q < 4 && col + q < g.n; ++q) o[q] = res ? e[q] + res[q] : e[q];
                }
            }
            if constexpr (STATS && !GEGLU) {
                // n is a multiple of 64, so this wave's 64 columns are either all in range
                // (a chunk of the row) or all past n (a tile wider than the matrix: no chunk).
                if (c0 < g.n) {
                    const float c = row16_sum((v.x + v.y) + (v.z + v.w)) * (1.0f / 64.0f);
                    const float dx = v.x - c, dy = v.y - c, dz = v.z - c, dw = v.w - c;
                    const float r1 = row16_sum((dx + dy) + (dz + dw));
                    const float r2 = row16_sum((dx * dx + dy * dy) + (dz * dz + dw * dw));
                    if (c4 == 0 && row < g.m)
                        g.out_stats[(int64_t)row * (g.n / 64) + (c0 >> 6)] = make_float4(c, r1, r2, 0.0f);
                }
            }
        }
    }
}

// The folded LayerNorm's centre of an input row with statistics st = (mean_hi,
// mean_lo, rstd, 0): the row enters the product as x - centre.  A row
// within one standard deviation of zero (|mean| rstd <= 1) is not centred: the
// mean comes out afterwards as mean colsum, whose cancellation then costs at most
// about as much as the product's own rounding (mean_lo, below half a unit of
// mean_hi, is dropped there).  Rows further out are centred by mean_hi (exact for
// x within a factor 2 of it), so that only mean_lo colsum is subtracted
// afterwards.  A function of the row alone: a row's result does not depend on the
// rows it shares a workgroup with.
__device__ __forceinline__ float norm_centre(float4 st) { return fabsf(st.x) * st.z > 1.0f ? st.x : 0.0f; }

// A workgroup's tile: WM x WN waves of 32 TM x 64 outputs each, with WK such groups that
// share the tile's k between them (their sums meet in LDS, added in group order); slabs of
// BK k in a two-stage LDS ring, PF slabs ahead of it in registers; OCC waves per SIMD.
template <int WM_, int WN_, int WK_, int TM_, int BK_, int PF_, int OCC_>
struct Tile {
    static constexpr int WM = WM_, WN = WN_, WK = WK_, TM = TM_, BK = BK_, PF = PF_, OCC = OCC_;
    static constexpr int BM = WM * TM * 32, BN = WN * 64, ROWS = BM + BN;
    static constexpr int GROUP = WM * WN, THREADS = 64 * GROUP * WK;
    static constexpr bool PADS = TM < 4;          // takes depths that BK does not divide, and any rows
    static constexpr bool SPLIT = TM < 4;         // may share an output tile's k among workgroups
    static constexpr int KS = BK / 16;            // MFMA steps of a slab
    static constexpr int PLANE = ROWS * BK * 2;   // bytes of one part of a slab
    static constexpr int STAGE = 3 * PLANE;
    // After the K loop the ring holds the other groups' sums, then each wave's epilogue
    // staging.
    static constexpr int SUMS = (WK - 1) * GROUP * TM * 32 * 64 * 4;
    static constexpr int STAGING = SUMS + GROUP * kStageFloats * 4;
    static constexpr int NORMS = std::max(2 * STAGE, STAGING);  // the input rows' norms, past both
    static constexpr int LDS = NORMS + BM * 16;
    static_assert(KS % WK == 0, "every group takes whole MFMA steps of a slab");
};

// The chunk of 8 k values (2s + h) of row r of a slab sits in 16 bytes at row slot
// r ^ lds_swizzle of its [32 rows][8 k] block: the 16 lanes that write a row's (BK = 64), two
// rows' (32) or four rows' (16) chunks then cover 128 consecutive bytes, and an MFMA operand
// is one contiguous 1 KB read either way.
template <class T>
__device__ __forceinline__ int lds_swizzle(int chunk) { return T::KS <= 4 ? chunk * (4 / T::KS) : chunk & 7; }

// One 32 x 32 output subtile in fp32 from the unsplit operands, for outputs that the parts
// left not finite: the lane's A row (less its folded-norm centre) and B row, in the order of k
// (infinities of either sign in a row meet in the reference's order).  32 k are fetched ahead of the
// products (96: no faster, and spills).  Of rows of 16-byte chunks (VEC) a lane takes 4 consecutive k
// of each 8, half h from 4 h on, and the halves exchange elements to make operands of consecutive k.
// With single loads per k and two of them in flight, 21,405 x 2304 x 768 of NaN took 4,273 us, with Inf
// in every 64th row 2,351 and with one NaN in b 714; now 1,334, 870 and 595 (all finite 378).
template <bool VEC>
__device__ __forceinline__ floatx16 exact_subtile(const float *arow, const float *brow, int depth, uint32_t h, float cen) {
    constexpr uint32_t SPAN = 32;
    const uint32_t k = depth;
    const auto load = [&](const float *row, uint32_t t0, float (&x)[SPAN / 2]) {
        if constexpr (VEC) {  // k is a multiple of 4
#pragma unroll
            for (uint32_t s = 0; s < SPAN / 8; ++s) {
                const float4 u = *(const float4 *)(row + min(t0 + 8 * s + 4 * h, k - 4));
                x[4 * s] = u.x, x[4 * s + 1] = u.y, x[4 * s + 2] = u.z, x[4 * s + 3] = u.w;
            }
        } else {
#pragma unroll
            for (uint32_t p = 0; p < SPAN / 2; ++p) x[p] = row[min(t0 + 2 * p + h, k - 1)];
        }
    };
    // x[p]: the element of k = t0 + 2 p + h.
    const auto order = [&](float (&x)[SPAN / 2]) {
        if constexpr (VEC) {
            const auto swap = [](float &lo, float &hi) {
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
                lo = __uint_as_float(r[0]);
                hi = __uint_as_float(r[1]);
            };
#pragma unroll
            for (uint32_t s = 0; s < SPAN / 2; s += 4) {
                swap(x[s], x[s + 1]);
                swap(x[s + 2], x[s + 3]);
                const float t = x[s + 1];
                x[s + 1] = x[s + 2];
                x[s + 2] = t;
            }
        }
    };
    floatx16 y;
#pragma unroll
    for (int r = 0; r < 16; ++r) y[r] = 0.f;
    if (k == 0) return y;
    float a[SPAN / 2], b[SPAN / 2], an[SPAN / 2], bn[SPAN / 2];
    load(arow, 0, an);
    load(brow, 0, bn);
    for (uint32_t t0 = 0; t0 < k; t0 += SPAN) {
#pragma unroll
        for (uint32_t p = 0; p < SPAN / 2; ++p) a[p] = an[p], b[p] = bn[p];
        load(arow, t0 + SPAN, an);
        load(brow, t0 + SPAN, bn);
        order(a);
        order(b);
#pragma unroll
        for (uint32_t p = 0; p < SPAN / 2; ++p) {
            const bool in = t0 + 2 * p + h < k;
            y = mfma_f32(in ? a[p] - cen : 0.f, in ? b[p] : 0.f, y);
        }
    }
    return y;
}

// The operands' scale, and the sums'.
constexpr float kScale = 0x1p23f, kUnscale = 0x1p-46f;

// 16-byte loads of whole chunks of 4 k.
__host__ __device__ __forceinline__ bool aligned_rows(const GemmLaunch &g) {
    return ((g.lda | g.ldb | g.k) & 3) == 0 && (((uintptr_t)g.a | (uintptr_t)g.b) & 15) == 0;
}

// Row of b behind column `col` of the workgroup's tile.  GeGLU: tile rows
// [64t, 64t + 32) are input columns, [64t + 32, 64t + 64) their gates.
template <bool GEGLU>
__device__ __forceinline__ int b_row(const GemmLaunch &g, int n0, int row) {
    if constexpr (GEGLU) {
        const int within = row & 63, col = min(n0 + 32 * (row >> 6) + (within & 31), g.n - 1);
        return within < 32 ? col : col + g.n;
    } else {
        return min(n0 + row, g.n_rows_b - 1);
    }
}

// NORM: the input rows' LayerNorm is folded in (GemmLaunch::in_stats); STATS:
// the output rows' chunk statistics are written (GemmLaunch::out_stats); PAD: a depth
// that BK does not divide is padded with zeros (1: rows of 16-byte chunks, 2: any rows); RES: there
// may be a residual.
//
// Each slab's rows come from memory as fp32 (rows past m, or past b's, repeat the last one; the
// epilogue drops them), are split into their parts in registers and written to LDS as three
// planes.  Iteration kt multiplies slab kt out of one stage while slab kt + 1, fetched PF
// iterations ago, is split into the other between the MFMAs, so the splitting's VALU work
// (6.5 operations an element) runs beside the matrix cores; one barrier per slab.
template <class T, bool GEGLU, bool NORM, bool STATS, int PAD, bool RES>
__global__ void __launch_bounds__(T::THREADS, T::OCC) gemm_kernel(const GemmLaunch g) {
    __shared__ __attribute__((aligned(16))) char ring[T::LDS];
    constexpr int OUT_BN = GEGLU ? T::BN / 2 : T::BN;
    constexpr int TM = T::TM, BK = T::BK, KS = T::KS, PF = T::PF;
    const int tiles_n = (g.n + OUT_BN - 1) / OUT_BN;
    const int tiles_m = (g.m + T::BM - 1) / T::BM;
    // Split-K: workgroups tile * S .. tile * S + S - 1 share one output tile (the
    // reducing launch: one workgroup per tile).
    const int S = T::SPLIT && g.splits > 1 ? g.splits : 1;
    const int tile = T::SPLIT && g.reduce ? (int)blockIdx.x : (int)blockIdx.x / S;
    const int split = (int)blockIdx.x - tile * S;
    int tm, tn;
    // About 1,024 rows of A a group: 4 blocks of 256 (8: encoder B = 64 x 512 25.00 -> 25.14 ms).
    tile_of<T::BM == 256 ? 4 : 8>(tile, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * T::BM, n0 = tn * OUT_BN;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int group = wave / T::GROUP, wg = wave % T::GROUP;
    const int wm = wg / T::WN * 32 * TM, wn = wg % T::WN * 64;
    const int li = lane & 31, h = lane >> 5;

    // The input rows' (mean_hi, mean_lo, rstd), one row per thread.
    float4 *norms = (float4 *)(ring + T::NORMS);
    if constexpr (NORM) {
        static_assert(T::BM <= T::THREADS, "a thread per row");
        if (tid < T::BM) {
            const int row = min(m0 + tid, g.m - 1), chunks = g.k / 64;
            norms[tid] = g.in_stats ? g.in_stats[row] : row_norm(g.in_chunks + (int64_t)row * chunks, chunks, g.in_eps);
        }
        __syncthreads();
    }

    floatx16 acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    constexpr int kPartial4 = T::BM * T::BN / 4, kWave4 = TM * 32 * 64 / 4;  // float4 of a partial tile
    if (T::SPLIT && g.reduce) {
        // The partials of this tile, summed in split order, a whole partial's loads in
        // flight at a time.
        const float4 *all = (const float4 *)g.partials + (int64_t)tile * S * kPartial4 + wg * kWave4;
        if (group == 0)
            for (int s = 0; s < S; ++s) {
                float4 u[TM * 8];
#pragma unroll
                for (int q = 0; q < TM * 8; ++q) u[q] = all[(int64_t)s * kPartial4 + q * 64 + lane];
#pragma unroll
                for (int q = 0; q < TM * 8; ++q) {
                    floatx16 &x = acc[q >> 3][(q >> 2) & 1];
                    const int r = 4 * (q & 3);
                    x[r] = s ? x[r] + u[q].x : u[q].x;
                    x[r + 1] = s ? x[r + 1] + u[q].y : u[q].y;
                    x[r + 2] = s ? x[r + 2] + u[q].z : u[q].z;
                    x[r + 3] = s ? x[r + 3] + u[q].w : u[q].w;
                }
            }
    } else {
        // Staging: LPR lanes take the 16-byte chunks of one row, RPP rows a pass.
        constexpr int LPR = BK / 4, RPP = T::THREADS / LPR, PASS = T::ROWS / RPP, APASS = T::BM / RPP;
        static_assert(T::ROWS % RPP == 0 && T::BM % RPP == 0, "whole passes of A and of B");
        const int c = tid % LPR, r0 = tid / LPR, chunk = c >> 1;
        const float *src[PASS];
        float cen[APASS];
#pragma unroll
        for (int p = 0; p < PASS; ++p) {
            if (p < APASS) {
                const int row = min(m0 + r0 + p * RPP, g.m - 1);
                src[p] = g.a + (int64_t)row * g.lda + 4 * c;
                cen[p] = 0.f;
                if constexpr (NORM) cen[p] = norm_centre(norms[r0 + p * RPP]) * kScale;
            } else {
                src[p] = g.b + (int64_t)b_row<GEGLU>(g, n0, r0 + p * RPP - T::BM) * g.ldb + 4 * c;
            }
        }
        const int slabs = g.k / BK + (g.k % BK != 0);
        const int slab0 = (int)((int64_t)slabs * split / S), nk = (int)((int64_t)slabs * (split + 1) / S) - slab0;
        float4 st[PF][PASS];
        const auto load = [&](int kt, float4 (&x)[PASS]) {
            const int k0 = (slab0 + kt) * BK;
            if constexpr (PAD == 0) {
#pragma unroll
                for (int p = 0; p < PASS; ++p) x[p] = *(const float4 *)(src[p] + k0);
            } else if constexpr (PAD == 1) {  // a chunk past k reads the last one instead (put() zeroes it)
                const int at = min(k0, g.k - 4 - 4 * c);
#pragma unroll
                for (int p = 0; p < PASS; ++p) x[p] = *(const float4 *)(src[p] + at);
            } else {
                const int left = g.k - 1 - k0 - 4 * c;  // of this chunk's elements, the last below k
#pragma unroll
                for (int p = 0; p < PASS; ++p) {
                    const float *s = src[p] + k0;
                    x[p] = make_float4(s[min(0, left)], s[min(1, left)], s[min(2, left)], s[min(3, left)]);
                }
            }
        };
        const auto put = [&](int kt, int p, float4 x) {
            if constexpr (PAD != 0) {
                const int left = (int)((uint32_t)g.k - (uint32_t)(slab0 + kt) * BK) - 4 * c;
                x = make_float4(left > 0 ? x.x : 0.f, left > 1 ? x.y : 0.f, left > 2 ? x.z : 0.f, left > 3 ? x.w : 0.f);
            }
            const float o = NORM && p < APASS ? cen[p < APASS ? p : 0] : 0.f;
            const auto scaled = [&](float v) {
                return NORM && p < APASS ? __builtin_fmaf(v, kScale, -o) : v * kScale;
            };
            uint32_t lo[3], hi[3];
            split3(scaled(x.x), scaled(x.y), lo);
            split3(scaled(x.z), scaled(x.w), hi);
            const int r = r0 + p * RPP;
            char *d = ring + (kt & 1) * T::STAGE + ((r >> 5) * KS + (chunk >> 1)) * 1024 + (chunk & 1) * 512 +
                      ((r & 31) ^ lds_swizzle<T>(chunk)) * 16 + (c & 1) * 8;
#pragma unroll
            for (int q = 0; q < 3; ++q) *(uint32x2 *)(d + q * T::PLANE) = uint32x2{lo[q], hi[q]};
        };
        const auto part = [&](const char *base, int q, int row, int s) {
            return *(const bf16x8 *)(base + q * T::PLANE + ((row >> 5) * KS + s) * 1024 + h * 512 +
                                     ((li ^ lds_swizzle<T>(2 * s + h)) * 16));
        };
        const auto multiply = [&](const char *base, int s) {
            bf16x8 a[TM][3], b[2][3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
#pragma unroll
                for (int i = 0; i < TM; ++i) a[i][q] = part(base, q, wm + 32 * i, s);
#pragma unroll
                for (int j = 0; j < 2; ++j) b[j][q] = part(base, q, T::BM + wn + 32 * j, s);
            }
            // The smallest products first.
            constexpr int qa[6] = {2, 0, 1, 1, 0, 0}, qb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = mfma_bf16(a[i][qa[q]], b[j][qb[q]], acc[i][j]);
        };
        constexpr int STEPS = KS / T::WK;  // this group's MFMA steps of a slab
        // One slab's turn.  Loads past the last slab repeat it and its last turn splits one that
        // nobody reads: a branch around either would make the registers in flight wait.
        const auto turn = [&](int kt, float4 (&next)[PASS]) {
            const char *base = ring + (kt & 1) * T::STAGE;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                multiply(base, group * STEPS + s);
#pragma unroll
                for (int p = s * PASS / STEPS; p < (s + 1) * PASS / STEPS; ++p) put(kt + 1, p, next[p]);
            }
            load(min(kt + 1 + PF, nk - 1), next);
            __syncthreads();
        };
        if (nk > 0) {
#pragma unroll
            for (int u = 0; u < PF; ++u) load(min(u, nk - 1), st[u]);
#pragma unroll
            for (int p = 0; p < PASS; ++p) put(0, p, st[0][p]);
            load(min(PF, nk - 1), st[0]);
            __syncthreads();
            int kt = 0;
            for (; kt + PF <= nk; kt += PF)
#pragma unroll
                for (int u = 0; u < PF; ++u) turn(kt + u, st[(u + 1) % PF]);
#pragma unroll
            for (int u = 0; u < PF - 1; ++u)
                if (kt + u < nk) turn(kt + u, st[(u + 1) % PF]);
        }
        if constexpr (T::WK > 1) {
            // Every wave is past its last read of the ring.
            float *sums = (float *)ring + wg * TM * 32 * 64 + lane;
            constexpr int kGroupFloats = T::GROUP * TM * 32 * 64;
            if (group > 0) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            sums[(group - 1) * kGroupFloats + ((i * 2 + j) * 16 + r) * 64] = acc[i][j][r];
            }
            __syncthreads();
            if (group == 0) {
#pragma unroll
                for (int o = 0; o < T::WK - 1; ++o)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                acc[i][j][r] += sums[o * kGroupFloats + ((i * 2 + j) * 16 + r) * 64];
            }
        }
        if (T::SPLIT && S > 1) {
            // The partial tile goes out in the accumulator layout (each wave's outputs as
            // lane-contiguous float4 rows); the reducing launch reads it back.
            if (group > 0) return;
            float4 *mine = (float4 *)g.partials + ((int64_t)tile * S + split) * kPartial4 + wg * kWave4;
#pragma unroll
            for (int q = 0; q < TM * 8; ++q) {
                const floatx16 &x = acc[q >> 3][(q >> 2) & 1];
                const int r = 4 * (q & 3);
                mine[q * 64 + lane] = make_float4(x[r], x[r + 1], x[r + 2], x[r + 3]);
            }
            return;
        }
    }
    if (group > 0) return;

    // One product has one rounding on the fp32 instruction, and the parts that the six products
    // leave out show (largest error 1.5 units of 2^-24 |ab| instead of 1; from k = 2 on it is below the
    // fp32 instruction's): depth 1 takes every output from there.
    const bool exact = g.k == 1;
    // From here on single floats: a 16-register vector changed in a branch would be held twice.
    float y[TM][2][16];
    uint32_t redo = 0;  // subtiles 2 i + j with outputs to compute again
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float z = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                y[i][j][r] = acc[i][j][r] * kUnscale;
                z = __builtin_fmaf(y[i][j][r], 0.f, z);  // NaN where one of them is not finite
            }
            if (exact || __any(z != 0.f)) redo |= 1u << (2 * i + j);
        }
    // One copy of the code for all of them: a copy each made every launch 1-2% slower.
    while (redo) {
        const int at = __builtin_ctz(redo), i = at >> 1, j = at & 1;
        redo &= redo - 1;
        const int row = min(m0 + wm + 32 * i + li, g.m - 1);
        float cen = 0.f;
        if constexpr (NORM) cen = norm_centre(norms[wm + 32 * i + li]);
        const floatx16 e = exact_subtile<PAD != 2>(
            g.a + (int64_t)row * g.lda, g.b + (int64_t)b_row<GEGLU>(g, n0, wn + 32 * j + li) * g.ldb, g.k, h, cen);
#pragma unroll
        for (int q = 0; q < 2 * TM; ++q)
            if (q == at)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float &x = y[q >> 1][q & 1][r];
                    x = exact || !(fabsf(x) <= 3.40282347e38f) ? e[r] : x;
                }
    }

    const bool vec_out = (g.ldo & 3) == 0 && ((uintptr_t)g.out & 15) == 0 &&
                         (!g.residual || ((g.ldr & 3) == 0 && ((uintptr_t)g.residual & 15) == 0));
    const int c0 = n0 + (GEGLU ? wn >> 1 : wn);  // first output column of this wave
    float bias[2], cs[2] = {0.f, 0.f};
    load_bias<GEGLU>(g, c0, li, bias);
    if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            cs[j] = GEGLU ? g.colsum[min(c0 + li, g.n - 1) + j * g.n] : g.colsum[min(c0 + 32 * j + li, g.n - 1)];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (NORM) {
                // rstd (y - rest colsum), rest = (mean_hi - centre) + mean_lo the part of the
                // mean that the centring left (norm_centre).
                const float4 st = norms[wm + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3)];
                const float rest = (st.x - norm_centre(st)) + st.y;
#pragma unroll
                for (int j = 0; j < 2; ++j) y[i][j][r] = st.z * (y[i][j][r] - rest * cs[j]);
            }
            // Without a bias the sum is used as it is (x + 0 would turn -0 into +0).
#pragma unroll
            for (int j = 0; j < 2; ++j) y[i][j][r] = g.bias ? y[i][j][r] + bias[j] : y[i][j][r];
            // A few rows at a time: the temporaries of all of them would not fit beside the sums.
            if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    if (vec_out)
        epilogue_staged<GEGLU, STATS, TM, RES>(g, y, m0, wm, c0, li, h, lane, (float *)(ring + T::SUMS) + wg * kStageFloats);
    else
        epilogue<GEGLU, TM>(g, y, m0, wm, c0, li, h);
}

// The tiles, from the one with the fewest operand bytes per product to the ones that give small
// outputs enough workgroups (more groups, so that a workgroup's 8 waves still hide each other's
// splitting and LDS latency).  plan_of (gemm.hip) chooses among them.
using Tile256 = Tile<2, 4, 1, 4, 16, 1, 2>;     // 256 x 256: 8 waves of 128 x 64
using Tile256x128 = Tile<4, 2, 1, 2, 16, 2, 2>; // 256 x 128: 8 waves of 64 x 64
using Tile128 = Tile<2, 2, 2, 2, 32, 1, 2>;     // 128 x 128: 4 waves of 64 x 64, two groups
using Tile64x128 = Tile<2, 2, 2, 1, 32, 1, 2>;  // 64 x 128: 4 waves of 32 x 64, two groups
using Tile64 = Tile<2, 1, 4, 1, 64, 1, 2>;      // 64 x 64: 2 waves of 32 x 64, four groups
using Tile32 = Tile<1, 1, 8, 1, 128, 1, 2>;     // 32 x 64: one wave's outputs, eight groups

// Defined per tile in gemm_large.hip and gemm_small.hip.
template <class T, bool GEGLU>
hipError_t launch_tile(const GemmLaunch &g, unsigned grid, hipStream_t stream);

#ifdef RAYA_GEMM_INSTANTIATE
template <class T, bool GEGLU>
hipError_t launch_tile(const GemmLaunch &g, unsigned grid, hipStream_t stream) {
    const dim3 blocks(grid), threads(T::THREADS);
    const bool vec = aligned_rows(g), pad = !vec || g.k % T::BK != 0;
    const auto go = [&](auto norm, auto stats, auto padding, auto res) {
        hipLaunchKernelGGL((gemm_kernel<T, GEGLU, norm(), stats(), padding(), res()>), blocks, threads, 0, stream, g);
    };
    const auto residual = [&](auto norm, auto padding) {
        if (g.residual)
            go(norm, std::false_type{}, padding, std::true_type{});
        else
            go(norm, std::false_type{}, padding, std::false_type{});
    };
    using Whole = std::integral_constant<int, 0>;
    if (g.in_stats || g.in_chunks) {  // folded LayerNorm: QKV (with or without RoPE) and GeGLU
        if (pad) return hipErrorInvalidValue;
        residual(std::true_type{}, Whole{});
    } else if (g.out_stats) {  // the residual GEMMs
        if constexpr (GEGLU) return hipErrorInvalidValue;
        if (pad) return hipErrorInvalidValue;
        go(std::false_type{}, std::bool_constant<!GEGLU>{}, Whole{}, std::true_type{});
    } else if (!pad) {
        residual(std::false_type{}, Whole{});
    } else if constexpr (!T::PADS) {
        return hipErrorInvalidValue;
    } else if (vec) {
        residual(std::false_type{}, std::integral_constant<int, 1>{});
    } else {
        residual(std::false_type{}, std::integral_constant<int, 2>{});
    }
    return hipGetLastError();
}
#endif

}  // namespace gemm
}  // namespace raya
