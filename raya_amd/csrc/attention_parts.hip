// Attention at head_dim 64 and 128 on three-part bfloat16 products: 128 query rows per workgroup.
//
// The fp32 matrix instruction bounds the multi-tile masks (Block3 at 16 x 8192 rows ran at
// 113 of its 155 TFLOP/s).  Here every operand of both products is the exact sum of three
// bfloat16 parts and a product the six part products that carry it, as in gemm_kernel.hpp:
// 6 / 16 of the fp32 instruction's time, fewer roundings, and the probabilities keep all their
// 24 bits (down to 2^-110 of a row's largest; below, see the checks).  Splitting costs 5.5 VALU
// operations an element, so a workgroup takes 128 rows: each K and V element is split once for all of
// them, and each wave's 32 rows fill the 32 x 32 x 16 instruction.  At head_dim 64 a wave's tile of
// 64 keys is 96 matrix instructions (3,072 clocks) and about 500 VALU operations (2,400 at the 4.7
// clocks they sustain); two waves a SIMD overlap them to about 3,900 clocks a tile.
//
// Measured (us, the 64-row fp32 kernel -> this one, on one card): Block3 16 x 8192 119 -> 80 (159 TFLOP/s),
// Block3 32 x 12 x 2048 610 -> 450, Full 4 x 12 x 2048 (1024 to 2048 valid) 329 -> 194, Full
// 1 x 12 x 4096 439 -> 303 (170 TFLOP/s); head_dim 128: Block3 8 x 8 x 2048 229 -> 163, Full
// 2 x 8 x 2048 289 -> 185 (186 TFLOP/s); relative 2-norm error against float64 4.6e-7 -> 3.9e-7
// (Block3), 7.7e-7 -> 7.0e-7 (Full).
//
//   S^T = K Q^T (32 keys x 32 queries per subtile), online softmax as in attention_body.hpp,
//   O^T += V^T P^T, P^T taken straight from the S^T registers.
//
// Layouts of v_mfma_f32_32x32x16_bf16 (lane l, li = l % 32, h = l / 32): A[li][8h + e],
// B[8h + e][li] for e = 0 .. 7, D[8 (r / 4) + 4h + r % 4][li] in register r.  The score of key
// 8 (r / 4) + 4h + r % 4 of a subtile is register r, so registers 8s .. 8s + 7 are the
// B operand of PV step s when its contraction index (h, e) is key 16s + 8 (e / 4) + 4h + e % 4;
// V is written to LDS transposed in that order.
//
// LDS holds one tile of 64 keys: K's parts while the scores are formed, V's while they are
// used.  Phase A forms the scores of tile j while V of tile j is split into place, phase B takes
// the softmax and PV while K of tile j + 1 is: the VALU work of the splitting runs beside the
// matrix cores, with one barrier after each phase.  Rows are fetched into registers two phases
// ahead.
//
// What the parts lose, a half of 64 rows leaves to the fp32 body, in the same workgroup and before
// anything of it is stored (q may be out):
// - an output that is not finite: an operand that is not finite, or above the largest bfloat16, has no
//   parts;
// - operands so small that their lower parts fall below bfloat16's smallest subnormal, where a part is
//   off by up to 2^-134 whatever its size.  In K that moves a score by up to 2^-134 |q| a dim, so
//   |q scale| has to be below kHugeQ; in Q by 2^-134 |k|, so a Q element has to be zero or at least kTinyQ; in
//   V and the weights it moves an output by up to 2^-134 (1 + |v|) a key, so V has to be below kHugeV
//   and an output at least kTinyOut (2^-94 a key against 2^-40) or zero in a row that is not all zeros.
// The checks take 2-3% (Block3 16 x 8192 70.8 -> 73.0 us, head_dim 128 2 x 8 x 3000 74.2 -> 76.1), half of it
// V's largest element.  Scaling K, V and the weights as the GEMM does, which loses nothing, takes an
// operation an element: 75.0 -> 80.2 us without the weights.
#include "attention_body.hpp"
#include "parts.hpp"

namespace raya {
namespace attn {
namespace {

// Orders the values that are not zero by size, zero above all of them.
__device__ __forceinline__ uint32_t small_key(float x) { return 2 * __float_as_uint(x) - 1; }

constexpr float kTinyQ = 0x1p-100f, kHugeQ = 0x1p90f, kHugeV = 0x1p40f, kTinyOut = 0x1p-40f;

// acc[i] += a[i] b over the parts, the smallest products first; the sums alternate, so that
// no instruction waits for the one before it.
template <int N>
__device__ __forceinline__ void products(const bf16x8 (&a)[N][3], const bf16x8 (&b)[3], floatx16 (&acc)[N]) {
    constexpr int qa[6] = {2, 0, 1, 1, 0, 0}, qb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] = mfma_bf16(a[i][qa[q]], b[qb[q]], acc[i]);
}
__device__ __forceinline__ void product(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx16 &acc) {
    constexpr int qa[6] = {2, 0, 1, 1, 0, 0}, qb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q) acc = mfma_bf16(a[qa[q]], b[qb[q]], acc);
}

// Bytes of one part of a K or V tile, and of a tile.
template <int D>
constexpr int kPlane = kKeys * D * 2;
template <int D>
constexpr int kPartTile = 3 * kPlane<D>;

// K part blocks: [32-key subtile][step][h][32 keys][8 dims]; key row r of the block at slot
// r ^ ((2 step + h) mod 8), so that the 16 lanes that write one row's chunks cover 128 bytes.
template <int D>
__device__ __forceinline__ int k_slot(int key, int step, int h) {
    return ((key >> 5) * (D / 16) + step) * 1024 + h * 512 + ((key & 31) ^ ((2 * step + h) & 7)) * 16;
}
// V part blocks: [32-dim tile][16-key step][h][32 dims][8 keys]; dim row d at slot
// d ^ ((d / 4) & 7), so that 8 lanes writing dims 4 apart hit 8 different slots mod 8.
__device__ __forceinline__ int v_slot(int dim, int step, int h) {
    const int d = dim & 31;
    return ((dim >> 5) * (kKeys / 16) + step) * 1024 + h * 512 + (d ^ ((d >> 2) & 7)) * 16;
}

// Item `item` with the sequences taken longest first (ties in order).  Under Full an item's work
// is its sequence's length, and a long one that starts last is waited for alone: 4 sequences of
// 1024 to 2048 rows x 12 heads in the caller's order 224 us, longest first 208; 8 of 100 to 300
// rows 27.0 -> 22.4.  Batches past kMaxSorted keep their order: their tails are too short to pay
// for the ranking (64 of 128 to 512 rows: 194 -> 198 us).
constexpr int kMaxSorted = 16;
__device__ __forceinline__ Item decode_longest_first(const AttnLaunch &a, const Plan &p, int item) {
    const int bh = fdiv(item, p.by_qt), slot = fdiv(bh, p.by_heads), lane = threadIdx.x & 63;
    const int mine = lane < a.batch ? min(max(a.valid_len[min(lane, a.batch - 1)], 0), a.seq) : -1;
    int rank = 0;
    for (int b = 0; b < a.batch; ++b) {
        const int other = __builtin_amdgcn_readlane(mine, b);
        rank += other > mine || (other == mine && b < lane);
    }
    const int seq = __builtin_ctzll(__ballot(lane < a.batch && rank == slot));
    return decode<kPartRows, RAYA_MASK_FULL>(a, p, item + (seq - slot) * a.heads * p.n_qt);
}

// Whole (sequence, head) pairs per XCD (item_of): the tiles of a pair start one further on than those
// of the XCD's pair before.  An XCD deals its workgroups to four shader engines in turn, so that
// with a multiple of four tiles a pair (two, by halves) the same engines would get every pair's padding:
// 64 x 12 x 512 with 128 to 256 valid rows took 114 us under Full instead of 76, with 128 to 512 under
// Block3 163 instead of 129, at head_dim 128 304 instead of 190 and 401 instead of 320.
__device__ __forceinline__ int rotate_tiles(const Plan &p, int item) {
    if (p.pairs_per_xcd == 0 || p.rot_units > 0) return item;
    const int bh = fdiv(item, p.by_qt), t = item - bh * p.n_qt + bh / kXcds;
    return bh * p.n_qt + t - fdiv(t, p.by_qt) * p.n_qt;
}

template <int D, int MK, bool TIMED>
__device__ __forceinline__ void parts_body(const AttnLaunch &a, const Plan &p, char *lds, StageClock *clk) {
    constexpr int DS = D / 16, DT = D / 32, CH = D / 4;  // MFMA steps, 32-wide tiles and 16-byte chunks of a row
    constexpr int PLANE = kPlane<D>;
    // Windows leave each wave whole subtiles outside its rows' keys; the block masks' items see
    // every key of their range.
    constexpr bool WINDOW = MK == RAYA_MASK_SLIDING;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int li = lane & 31, h = lane >> 5;
    const int item = rotate_tiles(p, item_of(blockIdx.x, p));
    const bool sorted = MK == RAYA_MASK_FULL && a.valid_len && a.batch > 1 && a.batch <= kMaxSorted;
    const Item it = sorted ? decode_longest_first(a, p, item) : decode<kPartRows, MK>(a, p, item);
    const bool packed = a.seq_start != nullptr;
    const int64_t row0 = packed ? (int64_t)a.seq_start[it.b] : 0;
    const auto base = [&](int64_t bs, int64_t hs, int64_t rs) {
        return (packed ? row0 * rs : (int64_t)it.b * bs) + (int64_t)it.h * hs;
    };
    float *ob = a.out + base(a.o_bs, a.o_hs, a.o_rs);
    if (it.k_lo >= it.k_hi) {  // every row is padding: write zeros
        if (packed) return;
        for (int c = tid; c < kPartRows * CH; c += kThreads) {
            const int r = it.q0 + c / CH;
            if (r < a.seq) store_stream(ob + (int64_t)r * a.o_rs + 4 * (c % CH), make_float4(0.f, 0.f, 0.f, 0.f));
        }
        return;
    }
    const float c_exp = fmaxf(fabsf(a.scale) * kLog2e, 1.17549435e-38f);
    const float q_sign = a.scale < 0.f ? -1.f : 1.f;
    const int valid = it.valid, arg = a.mask_arg;
    const int qw = it.q0 + 32 * wave, qi = qw + li;
    const Range rr = qi < valid ? key_range(MK, arg, p.by_arg, qi, valid) : Range{0, 0};
    const bool wave_live = qw < valid, wave_full = qw + 31 < valid;
    const Range w_first = key_range(MK, arg, p.by_arg, min(qw, valid - 1), valid);
    const Range w_last = key_range(MK, arg, p.by_arg, min(qw + 31, valid - 1), valid);
    const float *kb = a.k + base(a.k_bs, a.k_hs, a.k_rs), *vb = a.v + base(a.v_bs, a.v_hs, a.v_rs);

    // The item's tiles, walked from the one whose index is a multiple of their count
    // (attention_body.hpp: neighbours' first touches spread over the steps).
    const int n_tiles = (it.k_hi - it.k_lo + kKeys - 1) / kKeys;
    int rot = (it.k_lo / kKeys) % n_tiles;
    rot = rot == 0 ? 0 : n_tiles - rot;
    const auto tile_at = [&](int j) {
        j += rot;
        return it.k_lo + (j >= n_tiles ? j - n_tiles : j) * kKeys;
    };

    // Staging.  K: CH lanes take a row's 16-byte chunks.  V: each thread takes 4 keys x 4 dims
    // (key quad 4 s + 2 half + vh of PV step s), for every 64 dims, so that it can write 4 keys
    // of a dim together.
    constexpr int KR = kThreads / CH, PUTS = kKeys / KR;  // rows a pass and passes; V: PUTS dims a thread
    const int kc = tid % CH, kr = tid / CH;
    const int vs = wave, half = (lane >> 3) & 1, vh = (lane >> 4) & 1, dq = (lane & 7) + 8 * (lane >> 5);
    const int vkey = 16 * vs + 8 * half + 4 * vh;
    float4 kreg[PUTS], vreg[PUTS];
    // Keys past the item's last one are fetched as copies of it (they weigh 0), tiles past the
    // last one as copies of that (a branch would make the registers in flight wait).
    const auto load_k = [&](int j) {
        const int kt = tile_at(min(j, n_tiles - 1)), last = it.k_hi - 1 - kt;
        const float *src = kb + (int64_t)kt * a.k_rs;
#pragma unroll
        for (int i = 0; i < PUTS; ++i)
            kreg[i] = *(const float4 *)(src + (uint32_t)(min(kr + KR * i, last) * (int)a.k_rs) + 4 * kc);
    };
    const auto load_v = [&](int j) {
        const int kt = tile_at(min(j, n_tiles - 1)), last = it.k_hi - 1 - kt;
        const float *src = vb + (int64_t)kt * a.v_rs;
#pragma unroll
        for (int i = 0; i < PUTS; ++i)
            vreg[i] = *(const float4 *)(src + (uint32_t)(min(vkey + i % 4, last) * (int)a.v_rs) + 64 * (i / 4) + 4 * dq);
    };
    char *kl = lds, *vl = lds + kPartTile<D>;
    const auto put_k = [&](int i) {
        uint32_t lo[3], hi[3];
        split3(kreg[i].x, kreg[i].y, lo);
        split3(kreg[i].z, kreg[i].w, hi);
        char *d = kl + k_slot<D>(kr + KR * i, kc >> 2, (kc >> 1) & 1) + (kc & 1) * 8;
#pragma unroll
        for (int q = 0; q < 3; ++q) *(uint32x2 *)(d + q * PLANE) = uint32x2{lo[q], hi[q]};
    };
    // Dim 64 (i / 4) + 4 dq + i % 4 of this thread's four keys.
    float vmax = 0.f;
    const auto put_v = [&](int i) {
        const auto at = [&](int k) {
            const float4 &x = vreg[i / 4 * 4 + k];
            return i % 4 == 0 ? x.x : i % 4 == 1 ? x.y : i % 4 == 2 ? x.z : x.w;
        };
        uint32_t lo[3], hi[3];
        split3(at(0), at(1), lo);
        split3(at(2), at(3), hi);
        // (fmaxf(fmaxf()) of these took head_dim 128 to 81 us.)
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(vmax) : "v"(at(0)), "v"(at(1)));
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(vmax) : "v"(at(2)), "v"(at(3)));
        char *d = vl + v_slot(64 * (i / 4) + 4 * dq + i % 4, vs, vh) + half * 8;
#pragma unroll
        for (int q = 0; q < 3; ++q) *(uint32x2 *)(d + q * PLANE) = uint32x2{lo[q], hi[q]};
    };

    load_k(0);
    load_v(0);
    // Q's parts: dims 16 s + 8 h .. + 7 of this lane's row (rows at or beyond valid take the last
    // one's, and all their keys are masked), negated for a negative scale.
    bf16x8 qf[DS][3];
    uint32_t q_lo = ~0u;
    float q_hi = 0.f;
    {
        const float *qp = a.q + base(a.q_bs, a.q_hs, a.q_rs) + (int64_t)min(qi, valid - 1) * a.q_rs + 8 * h;
#pragma unroll
        for (int s = 0; s < DS; ++s) {
            const float4 x = *(const float4 *)(qp + 16 * s), y = *(const float4 *)(qp + 16 * s + 4);
            const float e[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int c = 0; c < 8; c += 2) {
                q_lo = min(q_lo, min(small_key(e[c]), small_key(e[c + 1])));
                q_hi = fmaxf(q_hi, fmaxf(fabsf(e[c]), fabsf(e[c + 1])));
            }
            uint32x4 w[3];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                uint32_t part[3];
                split3(e[2 * c] * q_sign, e[2 * c + 1] * q_sign, part);
#pragma unroll
                for (int q = 0; q < 3; ++q) w[q][c] = part[q];
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) qf[s][q] = __builtin_bit_cast(bf16x8, w[q]);
        }
    }
#pragma unroll
    for (int i = 0; i < PUTS; ++i) put_k(i);
    load_k(1);
    __syncthreads();

    floatx16 oacc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;
    float m = -INFINITY;  // running max of the scores times c_exp, rounded: the weights' reference
    float l = 0.f;        // this lane's partial sum of weights
    if constexpr (TIMED) clk->last = clock_now();

#pragma unroll 1
    for (int j = 0; j < n_tiles; ++j) {
        const int kt = tile_at(j);
        int live = wave_live ? 3 : 0;  // subtiles with a key of some row of the wave
        if constexpr (WINDOW) {
            live = 0;
#pragma unroll
            for (int t = 0; t < 2; ++t)
                if (wave_live && kt + 32 * t < w_last.hi && kt + 32 * t + 32 > w_first.lo) live |= 1 << t;
        }
        // Phase A: scores.
        floatx16 s[2];
        if constexpr (TIMED) clk->tiles += live ? (wave_full || qw + 16 < valid ? 2 : 1) : 0;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
        if constexpr (WINDOW) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (live >> t & 1) {
#pragma unroll
                    for (int d = 0; d < DS; ++d) {
                        bf16x8 kf[3];
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            kf[q] = *(const bf16x8 *)(kl + q * PLANE + k_slot<D>(32 * t + li, d, h));
                        product(kf, qf[d], s[t]);
                    }
                }
#pragma unroll
                for (int i = t * PUTS / 2; i < (t + 1) * PUTS / 2; ++i) put_v(i);
            }
        } else {
#pragma unroll
            for (int d = 0; d < DS; ++d) {
                bf16x8 kf[2][3];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        kf[t][q] = *(const bf16x8 *)(kl + q * PLANE + k_slot<D>(32 * t + li, d, h));
                products(kf, qf[d], s);
                put_v(d);  // PUTS = DS
            }
        }
        load_v(j + 1);
        if constexpr (TIMED) {
            settle(s[0][15]);
            settle(s[1][15]);
            lap(clk, clk->qk);
        }
        __syncthreads();
        if constexpr (TIMED) lap(clk, clk->load_wait);

        // Phase B: the softmax update, then PV.
        if (!WINDOW || live) {
            if (WINDOW || !(wave_full && kt >= w_last.lo && kt + kKeys <= w_first.hi)) {
                const int lo = rr.lo - kt - 4 * h, hi = rr.hi - kt - 4 * h;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = 32 * t + 8 * (r >> 2) + (r & 3);
                        if (key < lo || key >= hi || (WINDOW && !(live >> t & 1))) s[t][r] = -INFINITY;
                    }
            }
            float tmax = s[0][0];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[t][r]);
            tmax = max_xor32(tmax);
            const float m_new = fmaxf(m, tmax * c_exp);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;
            if (__any(m_new > m)) {  // otherwise every factor is 1
                const float alpha = fast_exp2(m - m_use);
                l *= alpha;
#pragma unroll
                for (int t = 0; t < DT; ++t) oacc[t] *= alpha;
            }
            m = m_new;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                if (WINDOW && !(live >> t & 1)) continue;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[t][r] = fast_exp2(__builtin_fmaf(s[t][r], c_exp, -m_use));
                    l += s[t][r];
                }
            }
            if constexpr (TIMED) {
                settle(l);
                settle(oacc[0][15]);
                lap(clk, clk->softmax);
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (!WINDOW || (live >> t & 1)) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    uint32x4 w[3];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        uint32_t part[3];
                        split3(s[t][8 * u + 2 * c], s[t][8 * u + 2 * c + 1], part);
#pragma unroll
                        for (int q = 0; q < 3; ++q) w[q][c] = part[q];
                    }
                    bf16x8 pf[3], vf[DT][3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) pf[q] = __builtin_bit_cast(bf16x8, w[q]);
#pragma unroll
                    for (int d = 0; d < DT; ++d)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            vf[d][q] = *(const bf16x8 *)(vl + q * PLANE + v_slot(32 * d + li, 2 * t + u, h));
                    products(vf, pf, oacc);
                }
            }
#pragma unroll
            for (int i = t * PUTS / 2; i < (t + 1) * PUTS / 2; ++i) put_k(i);
        }
        load_k(j + 2);
        if constexpr (TIMED) {
            settle(oacc[0][15]);
            settle(oacc[DT - 1][15]);
            lap(clk, clk->pv);
        }
        __syncthreads();
        if constexpr (TIMED) lap(clk, clk->load_wait);
    }

    // Dims 32 t + 8 r + 4 h .. + 3 of row qi are registers 4 r .. 4 r + 3 of oacc[t].  Each
    // wave's 32 x 64 outputs go through LDS and leave as whole rows (attention_body.hpp).
    l = sum_xor32(l);
    float *st = (float *)lds + wave * 32 * D;
    const bool zero_row = qi >= valid || l == 0.f;
    const float inv = zero_row ? 0.f : 1.f / l;
    const bool bad_v = vmax >= kHugeV;
    bool bad = q_lo < small_key(kTinyQ) || !(q_hi * fmaxf(1.f, fabsf(a.scale)) < kHugeQ);
    uint32_t out_lo = ~0u;
    float out_nan = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!zero_row)
                y = make_float4(oacc[t][4 * r] * inv, oacc[t][4 * r + 1] * inv, oacc[t][4 * r + 2] * inv,
                                oacc[t][4 * r + 3] * inv);
            out_lo = min(min(out_lo, min(small_key(y.x), small_key(y.y))), min(small_key(y.z), small_key(y.w)));
            out_nan = __builtin_fmaf(y.x, 0.f, __builtin_fmaf(y.y, 0.f, out_nan));
            out_nan = __builtin_fmaf(y.z, 0.f, __builtin_fmaf(y.w, 0.f, out_nan));
            *(float4 *)(st + li * D + 4 * ((8 * t + 2 * r + h) ^ (li & 15))) = y;
        }
    // The row's smallest output that is not zero: its dims are in lanes li and li + 32.
    const auto halves = __builtin_amdgcn_permlane32_swap(out_lo, out_lo, false, false);
    out_lo = min(halves[0], halves[1]);
    if (!zero_row) bad |= out_lo < small_key(kTinyOut) || out_lo == ~0u || out_nan != 0.f;
    int redo = 0;  // halves
    if (__syncthreads_or(bad || bad_v)) {
        redo = (__syncthreads_or(bad && wave < 2) ? 1 : 0) | (__syncthreads_or(bad && wave >= 2) ? 2 : 0);
        if (__syncthreads_or(bad_v)) redo = 3;
        if (it.q0 + kQRows >= valid) redo &= 1;  // the second half has padding only, stored as zeros
    }
    const int rows = packed ? valid : a.seq;
    if (!(redo >> (wave >> 1) & 1)) {
#pragma unroll
        for (int i = 0; i < CH / 2; ++i) {
            const int at = i * 64 + lane, r = at / CH, c = at % CH;
            const float4 y = *(const float4 *)(st + r * D + 4 * (c ^ (r & 15)));
            if (qw + r < rows) store_stream(ob + (int64_t)(qw + r) * a.o_rs + 4 * c, y);
        }
    }
#pragma unroll 1
    for (; redo; redo &= redo - 1) {
        Item half_item = it;
        half_item.q0 = it.q0 + (redo & 1 ? 0 : kQRows);
        half_item.k_lo = key_range(MK, arg, p.by_arg, half_item.q0, valid).lo;
        half_item.k_hi = key_range(MK, arg, p.by_arg, min(half_item.q0 + kQRows, valid) - 1, valid).hi;
        __syncthreads();
        attend_body<D, D == 64, false, WINDOW && D == 64, false, MK, false, 0, WINDOW>(
            a, p, half_item, (float *)lds, (float *)lds + kKeys * D, nullptr);
    }
}

// Waves per SIMD: at head_dim 128 Q's parts and the output take 160 registers by themselves.
template <int D>
constexpr int kPartWaves = D == 64 ? 2 : 1;

template <int D, int MK>
__global__ void __launch_bounds__(kThreads, kPartWaves<D>) attend_parts_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kPartTile<D>];
    parts_body<D, MK, false>(a, p, lds, nullptr);
}

// The same with the stage clock (attention.hip's attend_timed_kernel).
template <int D, int MK>
__global__ void __launch_bounds__(kThreads, kPartWaves<D>) attend_parts_timed_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kPartTile<D>];
    __shared__ uint64_t part[kWaves][5];
    StageClock c{};
    parts_body<D, MK, true>(a, p, lds, &c);
    add_stage_totals(a, c, part);
}

template <int D, int MK>
hipError_t launch_mask(const AttnLaunch &a, const Plan &p, hipStream_t stream) {
    const dim3 grid((unsigned)p.total), block(kThreads);
    if (a.stage_cycles)
        hipLaunchKernelGGL((attend_parts_timed_kernel<D, MK>), grid, block, 0, stream, a, p);
    else
        hipLaunchKernelGGL((attend_parts_kernel<D, MK>), grid, block, 0, stream, a, p);
    return hipGetLastError();
}

template <int D>
hipError_t launch_dim(const AttnLaunch &a, const Plan &p, hipStream_t stream) {
    switch (a.mask_kind) {
    case RAYA_MASK_BLOCK3: return launch_mask<D, RAYA_MASK_BLOCK3>(a, p, stream);
    case RAYA_MASK_FULL: return launch_mask<D, RAYA_MASK_FULL>(a, p, stream);
    case RAYA_MASK_SLIDING: return launch_mask<D, RAYA_MASK_SLIDING>(a, p, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_parts(const AttnLaunch &a, const Plan &p, hipStream_t stream) {
    if (a.head_dim == 64) return launch_dim<64>(a, p, stream);
    if (a.head_dim == 128) return launch_dim<128>(a, p, stream);
    return hipErrorInvalidValue;
}

}  // namespace attn
}  // namespace raya
