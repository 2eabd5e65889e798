// The attention kernels of the fp32 matrix instruction (attention_body.hpp) and the choice of
// kernel, item height and item order for a launch.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "attention_body.hpp"

namespace raya {
namespace {

using namespace attn;

template <int DP, bool FUSED, bool EXACTV>
__global__ void __launch_bounds__(kThreads, kMinWaves<DP>) attend_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * DP];
    const Item it = decode<kQRows>(a, p, item_of(blockIdx.x, p));
    attend_body<DP, FUSED, false, false, false, -1, false, 0, EXACTV>(a, p, it, ks, vs, nullptr);
}

// Head_dim 64 under Window64 and Sliding(w): the fused kernel with subtile
// skipping (+7% on Window64 at L = 8192; no use for the block masks, whose
// items' key ranges cover whole subtiles).
// BlockDiag(b) with b dividing 64 at head_dim 64: every item is one 64-key tile,
// and the mask is known, so the item decode and key ranges compile to a few
// scalar instructions (the general kernel's first K/V load sits behind the
// decode of every mask kind and the tile walk's set-up): 64 VGPRs instead of
// 126, and the first load about 420 instructions earlier.  Blocks narrower than 64
// (SKIP) leave each wave's rows whole 16-key subtiles of other blocks' keys, which it
// skips: a quarter (b <= 16) or half (b = 32) of the matrix work, and no other block's
// V enters its rows even at weight 0 (0 * Inf would be NaN) when b is 16 or 32.
template <int DP, bool SKIP>
__global__ void __launch_bounds__(kThreads, kMinWaves<DP>) attend_blockdiag_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * DP];
    const Item it = decode<kQRows, RAYA_MASK_BLOCKDIAG>(a, p, item_of(blockIdx.x, p));
    // BlockDiag(64) rows of a wave share one range; narrower blocks may not.
    attend_body<DP, true, false, SKIP, false, RAYA_MASK_BLOCKDIAG, true, 0, SKIP>(a, p, it, ks, vs, nullptr);
}

template <int DP, int MK>
__global__ void __launch_bounds__(kThreads, kMinWaves<DP>) attend_sliding_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * DP];
    const Item it = decode<kQRows, MK>(a, p, item_of(blockIdx.x, p));
    attend_body<DP, true, false, true, false, MK>(a, p, it, ks, vs, nullptr);
}

// 16-row items with the key tiles split over the four waves, for grids that
// leave most compute units idle with 64-row items.
template <int DP, bool FUSED, int MK = -1, bool SINGLE = false, bool EXACTV = true>
__global__ void __launch_bounds__(kThreads, (kMinWavesOf<DP, true, FUSED>)) attend_split_kernel(const AttnLaunch a,
                                                                                               const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * DP];
    const Item it = decode<kSplitRows, MK>(a, p, item_of(blockIdx.x, p));
    attend_body<DP, FUSED, false, false, true, MK, SINGLE, 0, EXACTV>(a, p, it, ks, vs, nullptr);
}

// The split kernel at head_dim 64 for items of at most MAXT tiles, every tile's K/V
// loads issued before the first tile is computed.  2 waves per SIMD hold the MAXT
// register sets (239 VGPRs at MAXT = 6); the small grids this kernel serves place at
// most two workgroups per compute unit.
template <int MAXT, bool EXACTV>
__global__ void __launch_bounds__(kThreads, 2) attend_split_all_kernel(const AttnLaunch a, const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * 64];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * 64];
    const Item it = decode<kSplitRows>(a, p, item_of(blockIdx.x, p));
    attend_body<64, true, false, false, true, -1, false, MAXT, EXACTV>(a, p, it, ks, vs, nullptr);
}

// The same kernel with the stage clock.  Per-wave totals are summed in LDS,
// then one thread per stage adds the workgroup's sum to the caller's totals.
// An item whose rows are all padding returns from the body in every wave with
// zero totals.
template <int DP, bool FUSED, bool SKIP, bool SPLIT = false>
__global__ void __launch_bounds__(kThreads, (kMinWavesOf<DP, SPLIT, FUSED>)) attend_timed_kernel(const AttnLaunch a,
                                                                                                const Plan p) {
    __shared__ __attribute__((aligned(16))) float ks[kKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kKeys * DP];
    __shared__ uint64_t part[kWaves][5];
    StageClock c{};
    const Item it = decode<(SPLIT ? kSplitRows : kQRows)>(a, p, item_of(blockIdx.x, p));
    attend_body<DP, FUSED, true, SKIP, SPLIT>(a, p, it, ks, vs, &c);
    add_stage_totals(a, c, part);
}

// Half the bit width of the scatter domain: the smallest h with 4^h >= total.
int scatter_half_bits(int64_t total) {
    int h = 1;
    while ((int64_t(1) << (2 * h)) < total) ++h;
    return h;
}

// Grids of fewer 64-row items than this take the split kernel (16-row items,
// each tile's keys split over the waves).  At 192 items the two kernels take
// the same time; below, the split kernel is faster, above, the 64-row one (the
// split kernel runs 3 workgroups per compute unit).
constexpr int64_t kSplitBelow = 192;

// Whether a launch at head_dim 64 or 128 takes the 128-row kernel on three-part products
// (attention_parts.hip), by the masks and grids where it is the faster one.  Its items are twice
// as long as the 64-row kernel's, so what it loses is a last round that few of them fill: the
// grid is measured in rounds of one item a compute unit.  us, 128-row / 64-row / 16-row items:
// - Full and Block3 at head_dim 64, from 144 items: 16 x 8192 Block3 80 / 122, 4 x 12 x 2048 Full
//   193 / 326; just past a round (2 x 13 x 1161 Block3, 260 items) 35.4 / 36.5, before it
//   (2 x 14 x 1109, 252) 26.0 / 37.2.  Fewer items are worth it on one long sequence only, from 80 (12 x 896,
//   84 items: Full 42.1 / 49.2 / 43.2, Block3 22.2 / 22.6 / 22.9; 8 x 1152, 72 items: Block3 21.6 / 22.2 / 20.3, Full
//   51.5 / 57.4 / 52.3; 4 x 2304, 72 items: Full 97.0 / 117 / 95.3; 12 x 640 Full 32.2 / 34.8 / 26.0); in padded
//   batches the 16-row items have less to do (3 x 8 x 388 Full 27.4 / 27.3 / 24.6).
// - head_dim 128 (one wave a SIMD: Q's parts and the output alone fill 160 registers): Block3
//   2 x 8 x 3000 79 / 92, Full 2 x 8 x 2048 183 / 290, from 144 items (Block3 8 x 1536, 96 items,
//   39.0 / 37.1).  Past one round only where the rounds are 70% full: Full 23 x 3 x 442 (276 items)
//   92 / 73, Block3 12 x 15 x 227 (360) 63 / 67.
// - Sliding(w) from w = 128: part of an item's keys lie outside each wave's windows.  8 x 12 x 2048
//   at w = 64 77 / 76, 128 106 / 136, 256 172 / 239; 13 x 8 x 652 at 107 54 / 56.  Past one
//   round at 75% (8 x 5 x 1217 at 205, 400 items, 53 / 62).  At head_dim 128 from w = 256, past one round
//   at 90% (18 x 4 x 541 at 237, 360 items, 126 / 113): 4 x 8 x 2048 at 256 150 / 169 and 16 x 8 x 1024 of 256
//   to 1024 valid rows 213 / 228, but at 128 100 / 102 and 153 / 142, and 32 x 12 x 1024 at 128 402 / 383.
// - not BlockDiag: one or two tiles an item leave nothing to gain from cheaper products (64 is
//   bound by memory).
// Items that hold few rows waste them: 64 x 130 rows Block3 39 / 36, 64 x 100 25 / 34.  The lengths of a
// device batch are not known here: with valid rows from a quarter to half of seq the 128-row kernel is
// the faster one too (64 x 12 x 512 of 128 to 256 rows: Full 74 / 108, Block3 76 / 108, Sliding(128)
// 78 / 100), and so with fewer (of 16 to 32: Full 28 / 37, Sliding(128) 25 / 28; 16 x 8 x 1024 of
// 32 to 64, Full 17.8 / 16.9).
constexpr int64_t kPartsFrom = 144, kPartsFromAlone = 80, kAloneSeq = 768;
constexpr int64_t kPartsWindow = 128, kPartsWindowWide = 256, kRound = 256;

bool takes_parts(const AttnLaunch &a) {
    const bool block = a.mask_kind == RAYA_MASK_FULL || a.mask_kind == RAYA_MASK_BLOCK3;
    const bool wide = a.head_dim > 64;
    if (!block && !(a.mask_kind == RAYA_MASK_SLIDING && a.mask_arg >= (wide ? kPartsWindowWide : kPartsWindow)))
        return false;
    const int64_t tiles = (a.seq + kPartRows - 1) / kPartRows;
    if (5 * (int64_t)a.seq < 3 * kPartRows * tiles) return false;  // under 60% of the items' rows
    const int64_t items = tiles * a.heads * a.batch;
    if (items < (block && !wide && a.batch == 1 && a.seq >= kAloneSeq ? kPartsFromAlone : kPartsFrom)) return false;
    const int64_t percent = wide ? (block ? 70 : 90) : (block ? 0 : 75);
    const int64_t rounds = (items + kRound - 1) / kRound;
    return rounds == 1 || 100 * items >= percent * rounds * kRound;
}

// Query rows of an item.  RAYA_ATTN_ITEMS=16, 64 or 128 forces the height where the kernel
// exists (as the reference's RAYA_BACKEND forces a micro-kernel backend); anything else selects
// by grid.
int64_t item_rows(const AttnLaunch &a, bool parts_dim) {
    const bool parts_ok = parts_dim && a.mask_kind != RAYA_MASK_BLOCKDIAG && a.mask_kind != RAYA_MASK_WINDOW64;
    if (const char *e = std::getenv("RAYA_ATTN_ITEMS")) {
        if (!std::strcmp(e, "16")) return kSplitRows;
        if (!std::strcmp(e, "64")) return kQRows;
        if (!std::strcmp(e, "128") && parts_ok) return kPartRows;
    }
    if (parts_ok && takes_parts(a)) return kPartRows;
    return (a.seq + kQRows - 1) / kQRows * a.heads * a.batch < kSplitBelow ? kSplitRows : kQRows;
}

// The most 64-key tiles one 16-row item's key interval spans (every row valid; a
// shorter valid length only clips intervals).
int64_t max_item_tiles(const AttnLaunch &a) {
    const int64_t b = a.mask_arg;
    int64_t span;
    switch (a.mask_kind) {
    case RAYA_MASK_BLOCK3: span = 3 * RAYA_BLOCK; break;  // the rows share one 128-block
    case RAYA_MASK_WINDOW64: span = kSplitRows + 2 * RAYA_WINDOW; break;
    case RAYA_MASK_FULL: span = a.seq; break;
    case RAYA_MASK_SLIDING: span = kSplitRows + 2 * b; break;
    default:  // BlockDiag(b): one block when 16 divides b, else the blocks 16 rows touch
        span = b % kSplitRows == 0 ? b : b * ((kSplitRows - 1) / b + 2);
        break;
    }
    span = std::min<int64_t>(span, a.seq);
    return (span + kKeys - 1) / kKeys;
}

// RAYA_ATTN_PREFETCH=0 keeps the one-tile-ahead loads of the split kernel on items of
// up to six tiles.
bool prefetch_all() {
    const char *e = std::getenv("RAYA_ATTN_PREFETCH");
    return !(e && !std::strcmp(e, "0"));
}

// Item order of the 64-row kernels.  XCD x taking whole (sequence, head) pairs
// gives each XCD the padding of the sequences whose heads it holds: with 12
// heads on 8 XCDs, even sequences put two heads on XCDs 0-3 and odd ones on
// XCDs 4-7, so the XCDs' shares of the work differ by the two halves' valid
// lengths (7% on a batch of 32 sequences of U[512, 2048] valid rows).  Dealing
// each pair's units of 4 consecutive tiles round the XCDs, rotated by the
// pair's index, gives every XCD an equal share of every pair while a unit's
// items still share their key tiles in one L2: the MFMA-bound multi-tile lines
// gain about 1% (Block3 and BlockDiag(128) at 4 x 12 x 16384, Block3 at 32 x
// 12 x 2048).  A batch of one sequence gives every pair the same valid length
// and keeps whole pairs (16 heads x 2048 rows under Block3 ran 1% slower in
// units).  Single-tile BlockDiag(b <= 64) keeps whole pairs: HBM-bound, it runs
// the same either way (the XCD that finishes early leaves its bandwidth to the
// others), and units of 1 or 2 tiles, which scatter neighbouring rows over the
// XCDs, run it 16-20% slower.  Window64 and Sliding keep whole pairs too (units
// of 4 tiles: 0.4-1.5% slower on 16 heads x 4096 and 8192 rows).
// RAYA_ATTN_ORDER=pairs keeps whole pairs, rot1/rot2/rot4/rot8 deal units of
// that many tiles for any mask; the units must divide a pair's tiles 8 times
// over, else whole pairs.  Returns the shift, or -1 for whole pairs.
int rotate_shift(const AttnLaunch &a) {
    if (const char *e = std::getenv("RAYA_ATTN_ORDER")) {
        if (!std::strcmp(e, "pairs")) return -1;
        if (!std::strcmp(e, "rot1")) return 0;
        if (!std::strcmp(e, "rot2")) return 1;
        if (!std::strcmp(e, "rot4")) return 2;
        if (!std::strcmp(e, "rot8")) return 3;
    }
    const bool wide_block = a.mask_kind == RAYA_MASK_BLOCKDIAG && kKeys % a.mask_arg != 0;
    // One sequence gives every pair the same valid length: whole pairs are balanced.
    return (a.mask_kind == RAYA_MASK_BLOCK3 || wide_block) && a.batch > 1 ? 2 : -1;
}

template <bool EXACTV>
void launch_split_all(int64_t t, dim3 grid, dim3 block, hipStream_t stream, const AttnLaunch &a, const Plan &p) {
    if (t <= 2)
        hipLaunchKernelGGL((attend_split_all_kernel<2, EXACTV>), grid, block, 0, stream, a, p);
    else if (t <= 3)
        hipLaunchKernelGGL((attend_split_all_kernel<3, EXACTV>), grid, block, 0, stream, a, p);
    else if (t <= 4)
        hipLaunchKernelGGL((attend_split_all_kernel<4, EXACTV>), grid, block, 0, stream, a, p);
    else
        hipLaunchKernelGGL((attend_split_all_kernel<6, EXACTV>), grid, block, 0, stream, a, p);
}

template <int DP, bool FUSED = false>
hipError_t launch_dp(const AttnLaunch &a, hipStream_t stream) {
    // (The same row strides as the fused issue's: the parts' rows are addressed within a tile too.)
    constexpr bool PARTS = FUSED || DP == 128;
    const int64_t rows = item_rows(a, PARTS && a.head_dim == DP && a.k_rs < kMaxFusedRowStride && a.v_rs < kMaxFusedRowStride);
    const bool split = rows == kSplitRows;
    const int64_t n_qt = (a.seq + rows - 1) / rows;
    const int64_t total = n_qt * a.heads * a.batch;
    if (total > 0x7fffffff) return hipErrorInvalidValue;
    Plan p;
    p.total = (int)total;
    p.half_bits = scatter_half_bits(total);
    p.n_qt = (int)n_qt;
    p.by_qt = make_fastdiv((uint32_t)n_qt);
    p.by_heads = make_fastdiv((uint32_t)a.heads);
    p.by_arg = make_fastdiv(a.mask_kind == RAYA_MASK_BLOCKDIAG ? (uint32_t)a.mask_arg : 1u);
    const int64_t pairs = (int64_t)a.heads * a.batch;
    p.pairs_per_xcd = pairs % kXcds == 0 ? (int)(pairs / kXcds) : 0;
    p.quads = split && p.pairs_per_xcd == 0 && total % (4 * kXcds) == 0;
    if (p.quads) {
        const char *e = std::getenv("RAYA_ATTN_QUADS");
        if (!(e && !std::strcmp(e, "plain"))) p.quads = 2;
    }
    p.rot_units = p.rot_shift = 0;
    p.by_rot = make_fastdiv(1u);
    const int shift = split ? -1 : rotate_shift(a);
    if (shift >= 0 && n_qt % (kXcds << shift) == 0) {
        p.rot_shift = shift;
        p.rot_units = (int)(n_qt / (kXcds << shift));
        p.by_rot = make_fastdiv((uint32_t)(p.rot_units << shift));
    }
    if constexpr (PARTS) {
        if (rows == kPartRows) return launch_parts(a, p, stream);
    }
    const dim3 grid((unsigned)total), block(kThreads);
    const bool sliding = a.mask_kind == RAYA_MASK_SLIDING || a.mask_kind == RAYA_MASK_WINDOW64;
    // Masks whose key ranges differ between the 16 rows of a wave take the kernels
    // that recompute non-finite output chunks (exact_chunk).
    const bool ragged = sliding || (a.mask_kind == RAYA_MASK_BLOCKDIAG && a.mask_arg % 16 != 0);
    if (split) {
        if (a.stage_cycles)
            hipLaunchKernelGGL((attend_timed_kernel<DP, FUSED, false, true>), grid, block, 0, stream, a, p);
        else if (FUSED && a.mask_kind == RAYA_MASK_BLOCKDIAG && kKeys % a.mask_arg == 0)
            if (a.mask_arg < 16)
                hipLaunchKernelGGL((attend_split_kernel<DP, FUSED, RAYA_MASK_BLOCKDIAG, true, true>), grid, block, 0, stream, a, p);
            else
                hipLaunchKernelGGL((attend_split_kernel<DP, FUSED, RAYA_MASK_BLOCKDIAG, true, false>), grid, block, 0, stream, a, p);
        else if (FUSED && prefetch_all() && max_item_tiles(a) >= 2 && max_item_tiles(a) <= 6) {
            // (Single-tile items have no later load to overlap.)
            const int64_t t = max_item_tiles(a);
            if (ragged)
                launch_split_all<true>(t, grid, block, stream, a, p);
            else
                launch_split_all<false>(t, grid, block, stream, a, p);
        }
        else if (ragged)
            hipLaunchKernelGGL((attend_split_kernel<DP, FUSED, -1, false, true>), grid, block, 0, stream, a, p);
        else
            hipLaunchKernelGGL((attend_split_kernel<DP, FUSED, -1, false, false>), grid, block, 0, stream, a, p);
        return hipGetLastError();
    }
    if constexpr (FUSED) {
        if (a.stage_cycles && sliding)
            hipLaunchKernelGGL((attend_timed_kernel<DP, true, true>), grid, block, 0, stream, a, p);
        else if (a.stage_cycles)
            hipLaunchKernelGGL((attend_timed_kernel<DP, true, false>), grid, block, 0, stream, a, p);
        else if (a.mask_kind == RAYA_MASK_WINDOW64)
            hipLaunchKernelGGL((attend_sliding_kernel<DP, RAYA_MASK_WINDOW64>), grid, block, 0, stream, a, p);
        else if (sliding)
            hipLaunchKernelGGL((attend_sliding_kernel<DP, RAYA_MASK_SLIDING>), grid, block, 0, stream, a, p);
        else if (a.mask_kind == RAYA_MASK_BLOCKDIAG && a.mask_arg == kKeys)
            hipLaunchKernelGGL((attend_blockdiag_kernel<DP, false>), grid, block, 0, stream, a, p);
        else if (a.mask_kind == RAYA_MASK_BLOCKDIAG && kKeys % a.mask_arg == 0)
            hipLaunchKernelGGL((attend_blockdiag_kernel<DP, true>), grid, block, 0, stream, a, p);
        else if (ragged)
            hipLaunchKernelGGL((attend_kernel<DP, true, true>), grid, block, 0, stream, a, p);
        else
            hipLaunchKernelGGL((attend_kernel<DP, true, false>), grid, block, 0, stream, a, p);
    } else {
        if (a.stage_cycles)
            hipLaunchKernelGGL((attend_timed_kernel<DP, false, false>), grid, block, 0, stream, a, p);
        else if (ragged)
            hipLaunchKernelGGL((attend_kernel<DP, false, true>), grid, block, 0, stream, a, p);
        else
            hipLaunchKernelGGL((attend_kernel<DP, false, false>), grid, block, 0, stream, a, p);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_attention(const AttnLaunch &a, hipStream_t stream) {
    const int dp = (a.head_dim + 15) / 16 * 16;
    switch (dp) {
    case 16: return launch_dp<16>(a, stream);
    case 32: return launch_dp<32>(a, stream);
    case 48: return launch_dp<48>(a, stream);
    case 64:
        // The fused issue forms K/V offsets within a tile in 32 bits: 63 rows of the
        // row stride plus the last chunk must stay below 2^31 bytes.
        return a.head_dim == 64 && a.k_rs < kMaxFusedRowStride && a.v_rs < kMaxFusedRowStride
                   ? launch_dp<64, true>(a, stream)
                   : launch_dp<64>(a, stream);
    case 80: return launch_dp<80>(a, stream);
    case 96: return launch_dp<96>(a, stream);
    case 112: return launch_dp<112>(a, stream);
    case 128: return launch_dp<128>(a, stream);
    // Above 128 the contraction is padded to the next of four widths (at most 1/8 of it
    // zeros from 144 up): K/V tiles of 64 keys take 2 x 64 x DP floats of LDS (128 KB at
    // 256, one workgroup per compute unit).
    case 144:
    case 160: return launch_dp<160>(a, stream);
    case 176:
    case 192: return launch_dp<192>(a, stream);
    case 208:
    case 224: return launch_dp<224>(a, stream);
    case 240:
    case 256: return launch_dp<256>(a, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace raya

// The query rows of an item that a launch of these sizes takes (16, 64, or 128 on three-part products),
// for the tests and the bench's choice of matrix peak; -1 for a head_dim without a kernel.  Row strides
// short enough for every kernel.
extern "C" int raya_attention_item_rows(int batch, int heads, int seq, int head_dim, int mask_kind, int mask_arg) {
    using namespace raya;
    if (head_dim <= 0 || head_dim > kMaxHeadDim) return -1;
    AttnLaunch a{};
    a.batch = batch, a.heads = heads, a.seq = seq, a.head_dim = head_dim;
    a.mask_kind = mask_kind, a.mask_arg = mask_arg;
    return (int)item_rows(a, head_dim == 64 || head_dim == 128);
}
