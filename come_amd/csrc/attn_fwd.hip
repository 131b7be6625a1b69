// Forward attention over packed variable-length sequences with an additive per-key
// bias, head_dim 64, for gfx950 (wave64, v_mfma_f32_32x32x16 bf16/f16; 16x16x32 where a launch fills the
// chip, attn_block16).
//
// Work decomposition
//   A wavefront owns 64 consecutive queries (two tiles of 32) of one (segment, head) and walks
//   keys in tiles of 64.  A workgroup is NW wavefronts: NW / KS query tiles times KS key groups,
//   group g taking every KS-th key tile.  The wavefronts of a group share its K and V tiles in LDS
//   (a ring of half-tiles, one barrier per tile); Q stays in registers; the partial results of the
//   groups meet in LDS at the end.  Long segments run as 8 x 1 (512 queries), short ones as 4 x 1
//   (256 queries, two workgroups per CU) with the last, mostly empty block of a segment as 2 x 2,
//   launches that would leave the chip idle as 2 x 2 or 2 x 4 (128 queries).  In launches of many short segments a
//   workgroup computes several blocks one after another and asks for the first K, V and Q of the next one before it
//   writes out the present one.
//
// Orientation
//   Scores are produced transposed, S^T = K (c Q)^T, so that in the MFMA accumulator
//   layout a lane holds ONE query (lane % 32) and 16 keys per 32x32 tile: the row max
//   and row sum of the online softmax are in-lane reductions plus one exchange between
//   lane l and lane l ^ 32.  The same registers, rounded to 16 bit, are the B operand
//   of O^T += V^T P^T without any data movement; V^T fragments come out of the
//   row-major V tile with the transposing LDS read ds_read_b64_tr_b16.
//
// Bias, reference point and tail masking
//   The accumulator of a score tile does not start from zero but from the bias of its keys (read from LDS, -inf beyond
//   the end of the segment: such keys get probabilities of exactly 0).  Default arithmetic (EXACT): the accumulator
//   starts from bias / scale and collects the raw scores; one fused multiply-add per score, c s - m, gives the exponent
//   of exp2, with c = softmax_scale log2(e) in fp32 and m the reference point of the query's row: a lane holds one query
//   column, so a reference point per row costs nothing.  (The reference adds bias / scale to the raw scores,
//   flash_fwd_kernel.h:30-55, and subtracts the scaled running maximum inside exp2, softmax.h:76-88.)  m starts from the
//   row's maximum over the first 32 keys (fp16: the whole number above it).  COME_ATTN_FOLD_SCALE (bf16): Q is multiplied by c once and rounded back, the
//   accumulator starts from bias log2(e) minus a constant and is the exponent itself; all reference points start from that
//   constant, which the bound on the logits that the flag promises allows.  fp16 has neither the range nor the need for that form and always runs the
//   default one.
//   The reference point of a row moves lazily, by powers of two (only when its row sum - bf16: the running one, fp16:
//   that of a half-tile - leaves the range the 16-bit probabilities keep their precision in).  A workgroup in which a
//   stored probability left the 16-bit range altogether raises a flag in LDS and then computes its query block again,
//   tile by tile, with a running maximum per row: any finite scores are exact.
#include "attn_common.h"
#include "attn_deal.h"
#include "qk_math.h"

#include <algorithm>
#include <cmath>
#include <mutex>

// Work buffer of come_attn_varlen_fwd_static: pieces of the key-split tail (unnormalised outputs, reference
// points and row sums).  Every GPU the library runs on holds its own copy of the array at its own address.
constexpr int64_t kStaticWorkBytes = 64ll << 20;
static __device__ __align__(256) unsigned char scratch[kStaticWorkBytes];

namespace come {
namespace {

constexpr int kHeadDim = 64;
constexpr int kPieceExtra = 2;       // per query row of a piece: 64 unnormalised outputs, reference point, row sum

// What the scores of the folded arithmetic are relative to before any row's reference point (log2 units; 0 in the default
// arithmetic).  A little below zero the accumulators of a score tile keep their sign from key to key and step to step; the
// matrix pipe draws less power for it, and long launches are limited by power: segments of 25 536 and 21 848 tokens, 16 heads,
// 3.70 ms with 0, 3.60 with 4, 3.59 with 20.  No further, because a score is rounded at the size it has with the constant.
// Emulated against 64 bits (q, k of unit variance or out of a LayerNorm, gains of 1, bias log 9 on a tenth of the keys), rms in
// log2 units: 7e-8 with 0, 2.0e-7 with 4, 1.1e-6 with 20; relative to the largest score of a query block's first keys, as
// with COME_ATTN_BLOCK_REFERENCE, 4.2e-7.
constexpr float kFoldedBase = 4.f;
constexpr int kHalf = kBlockN / 2;   // keys of a half-tile, the unit of the ring and of the software pipeline

// Range of the probabilities relative to the reference point of their row.  They are stored in the 16-bit type of
// the inputs: bf16 has the exponent range of fp32, fp16 reaches only 65504 and loses precision below 2^-14.
//   kSumLimit  a row sum above this (bf16: the running sum, fp16: the sum over a half-tile) moves the reference point
//              of the row up
template <int DT> struct Range;
//   kLowLimit  a row sum below this at the end has lost its largest terms (possible where the reference point was not taken
//              from scores of the row: the constant of the folded arithmetic, a row or key group whose first 32 keys are
//              all masked): computed again as well
//   kHardLimit a row sum above this may come from probabilities that left the 16-bit type's range
//              (infinite, or saturated): the workgroup then computes its block again with a running maximum
template <> struct Range<COME_BF16> {
    static constexpr float kSumLimit = 1099511627776.f;   // 2^40
    static constexpr float kLowLimit = 7.8886091e-31f;     // 2^-100
    // bf16 has the exponent range of fp32, but the fp32 outputs collect p * v over the 32 keys of a step: 2^100
    // leaves 2^27 of headroom for |v| and the accumulation, and is still far above kSumLimit
    static constexpr float kHardLimit = 1.2676506e30f;     // 2^100
};
template <> struct Range<COME_F16> {
    // with reference points that leave the first keys' maximum in [1/2, 1): a row moves its reference when a half-tile's sum
    // (32 at most to begin with) has grown to 2^9; a probability may grow by 2^7 more before fp16 saturates.  Lower limits make
    // more rows of ordinary logits move: 2^5, 40 segments of 1374 tokens, 16 heads, 446 us instead of 363; 2^8, one of 1596
    // merged tokens 24.6 us instead of 24.1.  Reference points further up ([1/8, 1/4)) save moves where logits follow the
    // positions (2 x 798 keys as one 28.6 us instead of 31.0) and lose the last bits of all that is small beside the first keys: with
    // five keys at the head of a segment 11 nats above N(0, 1), relative error of the outputs against 64 bits 1.11e-3 instead of
    // 3.6e-4 (12 768 keys), 2.12e-3 instead of 5.7e-4 (25 536).
    static constexpr float kSumLimit = 512.f;
    static constexpr float kHardLimit = 32768.f;           // one probability near 65504 (where the conversion saturates)
    // A reference point that was taken from scores of the row leaves a sum of at least 1/2 (the largest of the first 32
    // probabilities), a move of it one of 2.  One that was not (see kLowLimit) has to leave probabilities of 2^-13 on
    // average: they keep their eleven bits down to 2^-14 and lose them one by one below.  (1100 keys of which the first 40 are
    // masked, N(0, 1) logits shifted by -14 nats: relative error of the outputs below 2e-3, without the limit 0.56.)
    static constexpr float kLowLimit = 0.25f, kLowMean = 1.220703125e-4f;
};
// The reference point of a row that no score gave.  fp16 tells it from every other one, all whole numbers; no probability notices.
template <int DT> constexpr float kNoScore = DT == COME_F16 ? 9.094947e-13f : 0.f;          // 2^-40

// -------------------------------------------------------------------------------------
// Software pipeline of a wavefront, in slots of 32 keys (half-tiles).  While the vector ALU turns the scores of one
// half-tile (both query tiles) into probabilities, the matrix pipe adds the P V products of the half-tile before it
// and builds the scores of the one behind it:
//
//   slot h:   VALU P(h) = exp2(c S(h) - m)      MFMA O += V(h-1)^T P(h-1) ; S(h+1) = K(h+1) Q^T
//
// A key tile is two slots and one barrier.  In the two slots of tile j the half-tiles 2j+1, 2j+2 of K and 2j-1, 2j of V
// are read (and, ahead of the next tile, 2j+1 of V); rings of half-tiles hold them and what is on its way.  Set s is
// half-tiles 2s+1, 2s+2 of K and 2s, 2s+1 of V: what tile s needs beyond the sets before it.  Tile j stages set
// j + kDeep: two tiles ahead where a key group has 64 KiB of LDS, one where it has to do with 36.
// Row sums are taken on the matrix pipe too (the rounded probabilities times a matrix of ones, v_mfma_f32_16x16x32), so
// the steady state spends one exp2, half a pack and (EXACT) one multiply-add per score on the vector ALU.
// One wavefront alone can issue such a slot in 600 cycles (668 with the multiply-adds) against 576 cycles of the matrix
// pipe (measured on a stream without memory), so nothing may stand between the slots: V fragments are requested across
// the slot border, staging loads and bias conversion go out between the chunks of a slot, the range check looks at sums
// that are complete.
// -------------------------------------------------------------------------------------
template <int NW, int KS, bool DEEP = KS == 1> struct Shape {
    static constexpr int kQTiles = NW / KS;                          // 64-query tiles of a workgroup
    static constexpr int kBlockM = 64 * kQTiles;
    static constexpr int kDeep = DEEP ? 2 : 1;
    // half-tiles per key group.  In tile j half-tiles up to 2j+2+2 kDeep of K are on their way while 2j+1 is read, of V up
    // to 2j+1+2 kDeep while 2j-1 is
    static constexpr int kRingK = DEEP ? 8 : 4, kRingV = DEEP ? 8 : 5;
    static constexpr int kDma = 8 / kQTiles;                         // direct loads per wavefront for a pair of half-tiles
    static constexpr int kKvElems = KS * (kRingK + kRingV) * kHalf * kHeadDim;
};

// One query block: `rows` of the packed tensors it belongs to, the key tiles to walk, where a key share goes to.
struct Item {
    int seq_start, L, head, q0;
    int tile_base, n_tiles;      // key tiles of this workgroup (all of the segment's unless it computes a key share)
    float *piece;                // unnormalised result of a key share (nullptr: the output itself)
};

// For a kernel with a loop over blocks (AGAIN): the same value, but computed again where it is used, and the kernel's
// arguments, read again from where the launch left them (cached scalar loads).  Keeps what only the two ends of a block need
// out of the registers of the key loop between them; kept there, it cost more than the chaining of blocks gains.
template <bool AGAIN, class T> __device__ __forceinline__ T afresh(T x) {
    if constexpr (AGAIN) asm volatile("" : "+v"(x));
    return x;
}
template <bool AGAIN, class T> __device__ __forceinline__ T afresh_s(T x) {
    if constexpr (AGAIN) asm volatile("" : "+s"(x));
    return x;
}
typedef const AttnArgs __attribute__((address_space(4))) *ArgsAfresh;
template <bool AGAIN> __device__ __forceinline__ ArgsAfresh args_afresh() {
    return afresh_s<AGAIN>(reinterpret_cast<ArgsAfresh>(reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr())));
}

__device__ inline int blocks_of(int len, int block_m) { return (len + block_m - 1) / block_m; }

// Which query block a workgroup computes.  Workgroup i is dispatched to XCD i % 8, each XCD with its own L2: the query
// blocks of one (segment, head) unit run back to back on one XCD and share that unit's K / V there.
//
// compact: the grid holds no empty blocks (but for a few at its very end).  Every wavefront counts the blocks of all
// segments itself, one segment per lane, and takes item (xcd, local) of two head-major lists of blocks that are dealt to
// the XCDs in equal contiguous ranges: first the full ones, then the last blocks of segments that run in half the steps
// (at most short_block queries), so that a launch ends on its short workgroups (32 segments around 800 keys: 1 % faster
// than in natural order).  With the segment lengths' upper bound in the grid instead, a third of the workgroups of a
// merged model's frame attention is empty and, an XCD dealing its workgroups to its shader engines in turn, real ones
// wait behind them: 8 segments of 800 tokens ran as two rounds although their 512 blocks fit one.
//   before -> now, us, 16 heads, bf16 default arithmetic: 2 x 800 18.9 -> 14.5, 8 x 800 45.0 -> 34.3,
//   32 x 800 123.6 -> 117.2, 32 x 1374 285.7 -> 278.4, 128 x 390 157.2 -> 153.8, 1 x 1600 33 -> 20
//
// Blocks of long segments are dealt the same way; the second list then holds the shares of the key-split tail (the last nb_tail blocks of
// every unit in `splits` pieces).  Whole units to the XCDs in turn leave up to half of the chip idle where the heads are no multiple of eight: us,
// 6 heads, 2 x 10 000 keys 512 -> 282, 2 x 12 000 617 -> 416, 2 x 14 000 766 -> 551; 12 heads, 4 x 12 000 944 -> 814.  With heads that are
// one, more than eight segments, default arithmetic: 8 heads, 12 x 4096 keys 410 -> 381, 10 of 9000 - 1000 621 -> 592; 16 heads, 10 of 4500 - 3000
// 586 -> 556, 16 of 5083 - 2541 957 -> 925, 40 of 5000 - 1500 1888 -> 1836; equal segments of 16 and 24 heads are alike.
//
// few (at most kFewSegments of them): every segment's blocks are dealt to the XCDs on their own, in contiguous ranges of the
// head-major list (attn_deal.h), and an XCD starts with the longest segment.  One list of all blocks gives the XCDs the same number of
// blocks, which is not the same work where segments differ (12 heads: every other XCD has the first half of a head, every other the second).
//   us, default arithmetic / folded: 6 heads, 7000 and 5000 keys 170 -> 142, 149 -> 124; 12 heads, 4500 - 3000 keys 181 -> 169, 165 -> 153;
//   20 000, 15 000 and 30 000 keys 4280 -> 3970, 3910 -> 3530
// With the same XCDs first in every segment's list the blocks left over added up there: 12 heads, 3 x 801 keys (one round of workgroups as one
// list) 25.8 and 24.7 us, with the lists going on where the one before ended 15.9 and 15.3; 6 heads, 3 x 7200 396 and 354, 244 and 222.
//
// Otherwise (more than 64 kCompactChunks segments): units are dealt to the XCDs round-robin and every unit has n_mblocks blocks.
// The workgroups of an XCD are dealt to its four shader engines in turn (position mod 4, measured: a fixed assignment,
// also while the engines are full).  Short segments leave the same query blocks of every unit empty, so with an even
// number of blocks per unit the empty ones would keep landing on the same engines; with `rotate`, set for even block
// counts, unit u starts its blocks at position u.  A split workgroup (behind the n_full_wg ordinary ones) gets the index
// of its query block among the unit's tail blocks and its key share; the pieces of one query block are neighbours.
constexpr int kCompactChunks = 4;        // 64 segments each
constexpr int kTable = 64 * kCompactChunks;
// Against one list of all blocks.  Up to 8 segments, over 504 launches of 1 - 8 segments of 300 - 3344 keys and 6, 12 and 16 heads, 1.6 % faster by geometric
// mean: segments of different lengths up to 1.28 (16 heads, 1374 and 700 keys 25.8 -> 20.1 us; 12 heads, 6 of 1374 - 700 35.6 -> 31.1),
// 5 - 8 short ones of one length up to 5 % slower, since the heads of every segment are spread over all XCDs and each K / V is read by more of them (12
// heads, 6 x 631 16.4 -> 17.4, 7 x 798 23.9 -> 24.4; 6 heads, 8 of 1374 - 700 28.1 -> 29.4): the host knows no lengths to tell these apart.  Beyond 8
// segments short ones lose more than that (16 heads, 64 of 862 - 686, fp16 212 -> 245; 6 heads, 9 x 801 18.9 -> 20.9) and long ones gain (12
// heads, 16 of 3000 - 1500 263 -> 247; 12 of 6000 - 2000 622 -> 589; 6 heads, 12 of 30 000 - 9000 7780 -> 7000; equal ones nothing).
constexpr int kFewSegments = 8;
constexpr int kListed = 64;              // blocks of a workgroup at most
typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int NW, int KS>
__device__ inline bool locate_block(const AttnArgs &a, Item &it, int *table, bool &listed) {
    constexpr bool kLoop = NW == 4 && KS == 1, kSplit = NW == 8 && KS == 1;
    const int block_m = a.block_m;
    it.piece = nullptr;
    it.tile_base = 0;
    if (a.few) {
        const int lane = static_cast<int>(threadIdx.x & 63), n_seq = a.n_seq, n_heads = a.n_heads;
        int start, len;
        segment_of(a, min(lane, n_seq - 1), start, len);
        if (lane >= n_seq) len = 0;
        const int blocks = blocks_of(len, block_m), left = len % block_m;
        const int apart = kSplit && a.splits > 1 ? min(blocks, a.nb_tail) : left > 0 && left <= a.short_block ? 1 : 0;
        const int per_head[2] = {blocks - apart, kSplit && a.splits > 1 ? apart * a.splits : apart};           // of either list
        const int xcd = static_cast<int>(blockIdx.x & 7u);
        const int items[2] = {per_head[0] * n_heads, per_head[1] * n_heads}, over = (items[0] & 7) | ((items[1] & 7) << 16);
        int in_front[2] = {0, 0}, over_front = 0, of_all[2] = {0, 0}, over_all = 0;      // items of longer segments, and of all; left over among them
        for (int t = 0; t < n_seq; ++t) {
            const int n0 = __builtin_amdgcn_readlane(items[0], t), n1 = __builtin_amdgcn_readlane(items[1], t), o = __builtin_amdgcn_readlane(over, t);
            if (__builtin_amdgcn_readlane(len, t) > len - (t < lane ? 1 : 0)) in_front[0] += n0, in_front[1] += n1, over_front += o;
            of_all[0] += n0, of_all[1] += n1, over_all += o;
        }
        const int over_full = over_all & 0xffff, front0 = over_front & 0xffff, front1 = over_full + (over_front >> 16), over_both = over_full + (over_all >> 16);
        const XcdShare mine[2] = {share_of(items[0], front0, xcd), share_of(items[1], front1, xcd)};         // of the segment's items
        const int full = items_to(of_all[0], 0, over_full, xcd), all = full + items_to(of_all[1], over_full, over_both, xcd);
        const int local = static_cast<int>(blockIdx.x >> 3);
        if (local >= all) return false;
        const bool is_rest = local >= full;
        const int before = is_rest ? full + items_to(in_front[1], over_full, front1, xcd) : items_to(in_front[0], 0, front0, xcd);
        const int at = local - before, per = is_rest ? per_head[1] : per_head[0];
        const int l = __builtin_ctzll(__ballot(lane < n_seq && at >= 0 && at < (is_rest ? mine[1].count : mine[0].count)));
        const int item = __builtin_amdgcn_readlane(at + (is_rest ? mine[1].first : mine[0].first), l);
        const int per_l = __builtin_amdgcn_readlane(per, l);
        it.seq_start = __builtin_amdgcn_readlane(start, l);
        it.L = __builtin_amdgcn_readlane(len, l);
        it.head = item / per_l;
        const int b = item - it.head * per_l, all_tiles = (it.L + kBlockN - 1) / kBlockN;
        it.q0 = is_rest ? it.L / block_m * block_m : b * block_m;
        it.n_tiles = all_tiles;
        if (kSplit && is_rest) {                                      // one of the unit's last query blocks, and which keys
            const int apart_l = __builtin_amdgcn_readlane(apart, l), t = b / a.splits, keys = b - t * a.splits;
            it.q0 = (blocks_of(it.L, block_m) - apart_l + t) * block_m;
            it.tile_base = static_cast<int>(static_cast<int64_t>(keys) * all_tiles / a.splits);
            it.n_tiles = static_cast<int>(static_cast<int64_t>(keys + 1) * all_tiles / a.splits) - it.tile_base;
            const int64_t piece = (static_cast<int64_t>(l * n_heads + it.head) * a.nb_tail + t + a.nb_tail - apart_l) * a.splits + keys;
            it.piece = a.work + piece * (Shape<NW, KS>::kBlockM * (kHeadDim + kPieceExtra));
        }
        listed = false;
        return true;
    }
    if (a.compact) {
        const int lane = afresh<kLoop>(static_cast<int>(threadIdx.x & 63));
        const int n_seq = afresh_s<kLoop>(a.n_seq), block_m = afresh_s<kLoop>(a.block_m), short_block = afresh_s<kLoop>(a.short_block), n_heads = afresh_s<kLoop>(a.n_heads);
        int start[kCompactChunks], len[kCompactChunks], full[kCompactChunks], rest[kCompactChunks];
#pragma unroll
        for (int c = 0; c < kCompactChunks; ++c) {                   // (all loads in flight before the first is looked at)
            start[c] = len[c] = 0;
            if (64 * c < n_seq) segment_of(a, min(64 * c + lane, n_seq - 1), start[c], len[c]);
            if (64 * c + lane >= n_seq) len[c] = 0;
        }
        int total_full = 0, total_rest = 0;                          // blocks per head
#pragma unroll
        for (int c = 0; c < kCompactChunks; ++c) {
            full[c] = rest[c] = 0;
            if (64 * c >= n_seq) continue;
            const int left = len[c] % block_m;                       // queries of the last, partial block
            const bool is_short = left > 0 && left <= short_block;
            if (kSplit && a.splits > 1) {
                const int blocks = blocks_of(len[c], block_m), apart = min(blocks, a.nb_tail);
                full[c] = static_cast<int>(wave_scan_add(static_cast<uint32_t>(blocks - apart)));
                rest[c] = static_cast<int>(wave_scan_add(static_cast<uint32_t>(apart * a.splits)));
            } else {
                full[c] = static_cast<int>(wave_scan_add(static_cast<uint32_t>(blocks_of(len[c], block_m) - (is_short ? 1 : 0))));
                rest[c] = static_cast<int>(wave_scan_add(is_short ? 1u : 0u));
            }
            total_full += __builtin_amdgcn_readlane(full[c], 63);
            total_rest += __builtin_amdgcn_readlane(rest[c], 63);
        }
        const int xcd = static_cast<int>(blockIdx.x & 7u);
        int local = static_cast<int>(blockIdx.x >> 3);
        const int full_items = total_full * n_heads, rest_items = total_rest * n_heads;
        const int full_per_xcd = (full_items + 7) / 8, rest_per_xcd = (rest_items + 7) / 8;
        const int in_front = a.chained > 0 ? min(a.chained, full_per_xcd) : full_per_xcd;       // workgroups of the full blocks
        const bool is_rest = local >= in_front;
        if (is_rest) local -= in_front;
        listed = !is_rest && a.chained > 0 && full_per_xcd > a.chained;
        if (listed) {
            // What next_block looks up: the blocks of this workgroup, lane t finds number t (every wavefront writes the same
            // values).  In front of them, for the search: blocks up to and with each segment, where it starts, its length.
            int *const starts = table + kTable, *const lens = table + 2 * kTable;
            int before = 0;
#pragma unroll
            for (int c = 0; c < kCompactChunks; ++c) {
                if (64 * c >= n_seq) continue;
                table[64 * c + lane] = before + full[c];
                starts[64 * c + lane] = start[c];
                lens[64 * c + lane] = len[c];
                before += __builtin_amdgcn_readlane(full[c], 63);
            }
            const int mine = local + lane * a.chained, at = xcd * full_per_xcd + mine;
            const bool valid = mine < full_per_xcd && at < full_items;
            const int in_head = valid ? at % total_full : 0;
            int seg = 0;                                              // segments whose blocks all lie in front of it: < n_seq
#pragma unroll
            for (int step = kTable / 2; step > 0; step >>= 1)
                if (seg + step < n_seq && table[seg + step - 1] <= in_head) seg += step;
            *reinterpret_cast<i32x4 *>(table + 3 * kTable + 4 * lane) =
                i32x4{valid ? at / total_full : -1, starts[seg], lens[seg], (in_head - (seg > 0 ? table[seg - 1] : 0)) * block_m};
        }
        const int per_xcd = is_rest ? rest_per_xcd : full_per_xcd;
        const int idx = xcd * per_xcd + local;
        if (local >= per_xcd || idx >= (is_rest ? rest_items : full_items)) return false;
        const int total = is_rest ? total_rest : total_full;
        it.head = idx / total;
        int b = idx - it.head * total;                                // block b of the list, of this head
        bool found = false;
        int share = -1;                                               // key share of a split block
        int64_t piece = 0;
#pragma unroll
        for (int c = 0; c < kCompactChunks; ++c) {
            if (64 * c >= n_seq || found) continue;
            const int incl = is_rest ? rest[c] : full[c];
            const int in_chunk = __builtin_amdgcn_readlane(incl, 63);
            if (b >= in_chunk) {
                b -= in_chunk;
                continue;
            }
            found = true;
            const int l = __builtin_ctzll(__ballot(incl > b));         // the first such lane's segment holds it
            it.seq_start = __builtin_amdgcn_readlane(start[c], l);
            it.L = __builtin_amdgcn_readlane(len[c], l);
            const int before = l > 0 ? __builtin_amdgcn_readlane(incl, l - 1) : 0;
            it.q0 = is_rest ? it.L / block_m * block_m : (b - before) * block_m;
            if (kSplit && is_rest && a.splits > 1) {                  // one of the unit's last query blocks, and which keys
                const int blocks = blocks_of(it.L, block_m), apart = min(blocks, a.nb_tail);
                const int t = (b - before) / a.splits;
                share = (b - before) - t * a.splits;
                it.q0 = (blocks - apart + t) * block_m;
                piece = (static_cast<int64_t>((64 * c + l) * n_heads + it.head) * a.nb_tail + t + a.nb_tail - apart) * a.splits + share;
            }
        }
        const int all_tiles = (it.L + kBlockN - 1) / kBlockN;
        it.n_tiles = all_tiles;
        if (kSplit && share >= 0) {
            it.tile_base = static_cast<int>(static_cast<int64_t>(share) * all_tiles / a.splits);
            it.n_tiles = static_cast<int>(static_cast<int64_t>(share + 1) * all_tiles / a.splits) - it.tile_base;
            it.piece = a.work + piece * (Shape<NW, KS>::kBlockM * (kHeadDim + kPieceExtra));
        }
        return true;
    }
    // one straight-line computation for both kinds of workgroup (branches that assign different outputs made the
    // compiler keep the outputs in scratch memory)
    const bool split = static_cast<int64_t>(blockIdx.x) >= a.n_full_wg;
    const int e = split ? static_cast<int>(blockIdx.x - a.n_full_wg) : static_cast<int>(blockIdx.x);
    const int xcd = e & 7;
    const int local = e >> 3;
    const int per_unit = split ? a.nb_tail * a.splits : a.n_mblocks;
    const int unit_on_xcd = local / per_unit;
    const int unit = xcd + 8 * unit_on_xcd;
    const int within = local % per_unit;
    int mblk = split ? 0 : (a.rotate ? (within + unit_on_xcd) % per_unit : within);
    const int tail = split ? within / a.splits : -1;
    const int ks = split ? within % a.splits : 0;
    it.head = unit % a.n_heads;
    const int seq = unit / a.n_heads;
    if (unit >= a.n_units) return false;
    segment_of(a, seq, it.seq_start, it.L);
    const int n_qblocks = blocks_of(it.L, block_m);
    if (tail >= 0) {
        mblk = n_qblocks - a.nb_tail + tail;          // split workgroup: one of the unit's last query blocks
        if (mblk < 0) return false;
    } else if (a.splits > 1 && mblk >= n_qblocks - a.nb_tail) {
        return false;                                 // left to the split workgroups (or beyond the segment)
    }
    it.q0 = mblk * block_m;
    if (it.q0 >= it.L) return false;
    // keys of this workgroup: all tiles, or share ks of them
    const int all_tiles = (it.L + kBlockN - 1) / kBlockN;
    it.tile_base = tail >= 0 ? static_cast<int>(static_cast<int64_t>(ks) * all_tiles / a.splits) : 0;
    it.n_tiles = (tail >= 0 ? static_cast<int>(static_cast<int64_t>(ks + 1) * all_tiles / a.splits) : all_tiles) - it.tile_base;
    if (tail >= 0) {
        const int64_t index = (static_cast<int64_t>(seq * a.n_heads + it.head) * a.nb_tail + tail) * a.splits + ks;
        it.piece = a.work + index * (Shape<NW, KS>::kBlockM * (kHeadDim + kPieceExtra));
    }
    return true;
}

// Block number `turn` of this workgroup.
__device__ inline bool next_block(Item &it, const int *table, int turn) {
    if (turn >= kListed) return false;
    const i32x4 e = *reinterpret_cast<const i32x4 *>(table + 3 * kTable + 4 * turn);
    it.head = __builtin_amdgcn_readfirstlane(e[0]);
    it.seq_start = __builtin_amdgcn_readfirstlane(e[1]);
    it.L = __builtin_amdgcn_readfirstlane(e[2]);
    it.q0 = __builtin_amdgcn_readfirstlane(e[3]);
    it.n_tiles = (it.L + kBlockN - 1) / kBlockN;
    return it.head >= 0;
}

// Computes `it` and, one after another, the blocks that `next` names (it returns false at the last one).  A block's first
// K, V, Q and bias loads are issued between the key loop and the epilogue of the block before it.  By timestamps, a block of
// its own workgroup spends 7.2 - 8 us around its key loop (finding its block 1.6 - 2, issuing and waiting for the first loads
// 3, first scores 0.4, sums and barrier 0.8, writing out 1.8) next to 17 us (800 keys) or 9 us (390 keys) in it; a chained one
// 5.2 - 6 us.  us before -> now, 16 heads, folded: 128 x 390 147 -> 139, 32 x 800 104 -> 100, 200 x 100 - 1400 662 -> 632,
// 20 x 800 (default arithmetic) 67.3 -> 65.4.
template <int DT, int NW, int KS, bool EXACT, bool DEEP, class Next>
__device__ __forceinline__ void attn_block(const AttnArgs &a, Item it, uint16_t *lds_kv, float *lds_seed, uint32_t *lds_raw,
                                           uint32_t *lds_words, Next next) {
    using E = Elem<DT>;
    using S = Shape<NW, KS, DEEP>;
    static_assert(EXACT || DT == COME_BF16, "fp16 runs the default arithmetic");
    constexpr float kSumLimit = Range<DT>::kSumLimit;
    constexpr int RK = S::kRingK, RV = S::kRingV, kDma = S::kDma, kBlockM = S::kBlockM, kThreads = 64 * NW;
    constexpr int kHalfElems = kHalf * kHeadDim;
    constexpr float kLog2e = 1.4426950408889634f;
    constexpr bool kChained = KS == 1 && NW == 4 && DT == COME_BF16;          // several blocks (the others' `next` has none)
    float *const piece = it.piece;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = KS == 1 ? wave : wave % S::kQTiles, group = KS == 1 ? 0 : wave / S::kQTiles;     // query tile and key group of this wavefront
    const int h = lane >> 5;
    const int r = lane & 31;
    // K and V half-tiles: 32 rows of 128 bytes, unpadded, filled by direct global->LDS loads (a wavefront's load lands as
    // 1 KiB, eight rows, in lane order); bank conflicts are avoided by permuting the 16-byte chunks inside a row: K chunk
    // c of row r sits at slot c ^ ((r >> 1) & 7), V chunk c at c ^ (((r >> 1) & 1) << 2).
    uint16_t *const lds_k = lds_kv + group * (RK * kHalfElems);
    uint16_t *const lds_v = lds_kv + (KS * RK + group * RV) * kHalfElems;
    if (it.n_tiles <= 0) {                         // a key share without tiles (segment shorter than the split count)
        for (int i = tid; i < kBlockM; i += kThreads) {
            piece[kBlockM * kHeadDim + i] = -1e30f;               // reference point
            piece[kBlockM * (kHeadDim + 1) + i] = 0.f;            // row sum
        }
        return;
    }

    // ---- global -> LDS staging.  Pair of half-tiles: loads 0 .. 3 bring the first one, 4 .. 7 the second, so that all of
    // a wavefront's loads of a pair lie in one of them (my_half).  A key index beyond the segment is redirected to its last
    // key (finite data); such keys start from -inf, so their probabilities are exactly 0 and neither their K nor
    // their V row can reach the output.
    const char *k_seg, *v_seg;
    const uint32_t k_rs_b = static_cast<uint32_t>(a.k_rs) * 2u, v_rs_b = static_cast<uint32_t>(a.v_rs) * 2u;
    const int my_half = (qi * kDma) >> 2, my_rows = ((qi * kDma) & 3) * 8;       // (uniform)
    const int st_row = my_rows + (lane >> 3);
    const uint32_t k_chunk = static_cast<uint32_t>((lane & 7) ^ ((st_row >> 1) & 7)) * 16u;      // load i: ^ 64 for odd i
    const uint32_t v_chunk = static_cast<uint32_t>((lane & 7) ^ (((st_row >> 1) & 1) << 2)) * 16u;
    // Byte offsets from the segment's first row fit 32 bits (the host has checked).  The first keys of a wavefront's
    // half-tiles of K and V advance by one step per set, up to the half-tile that holds the segment's last key; rows are
    // clamped to that key, additions saturate.
    uint32_t k_end, v_end;
    const uint32_t k_step = static_cast<uint32_t>(KS * kBlockN) * k_rs_b, v_step = static_cast<uint32_t>(KS * kBlockN) * v_rs_b;
    auto first_row = [&](int hf, uint32_t rs_b) __attribute__((always_inline)) {      // half-tile hf of this group
        return static_cast<uint32_t>(min((it.tile_base + KS * (hf >> 1) + group) * kBlockN + (hf & 1) * kHalf, it.L - 1)) * rs_b;
    };
    // per parity of the load: offset of this lane's chunk in the first of its rows, and in the segment's last row
    const uint32_t k_at[2] = {static_cast<uint32_t>(st_row) * k_rs_b + k_chunk, static_cast<uint32_t>(st_row) * k_rs_b + (k_chunk ^ 64u)};
    const uint32_t v_at_row = static_cast<uint32_t>(st_row) * v_rs_b + v_chunk;
    uint32_t k_last[2], v_last;
    auto load_k = [&](uint32_t first, uint32_t lds, int i) __attribute__((always_inline)) {
        const uint32_t at = __builtin_elementwise_add_sat(k_at[i & 1] + 8u * i * k_rs_b, first);
        dma_b128(k_seg, min(at, k_last[i & 1]), lds + 1024u * i);
    };
    auto load_v = [&](uint32_t first, uint32_t lds, int i) __attribute__((always_inline)) {
        const uint32_t at = __builtin_elementwise_add_sat(v_at_row + 8u * i * v_rs_b, first);
        dma_b128(v_seg, min(at, v_last), lds + 1024u * i);
    };
    // LDS address of this wavefront's part of ring stage `stage`
    const uint32_t k_part = lds_address(lds_k) + static_cast<uint32_t>(my_rows) * 128u, v_part = lds_address(lds_v) + static_cast<uint32_t>(my_rows) * 128u;
    constexpr uint32_t kStageBytes = kHalfElems * 2u;
    // Initial values of the scores ("seeds"), one float per key: bias in the unit of the accumulators, -inf beyond the
    // end of the segment.  NW tiles at a time, one per wavefront: wavefront w brings the aligned 32-bit words that hold
    // the 16-bit biases of tile NW m + w, and converts them a group of tiles later.
    const float c_scale = a.scale_log2;
    const float unit = EXACT ? kLog2e / a.scale_log2 : kLog2e;                    // EXACT: accumulators hold raw scores
    const char *b_seg;
    uint32_t b_mis;
    auto seed_key = [&](int m) __attribute__((always_inline)) { return (it.tile_base + NW * m + wave) * kBlockN + lane; };
    auto request_bias = [&](int m) __attribute__((always_inline)) {
        if (a.bias == nullptr) return;
        const uint32_t key = static_cast<uint32_t>(min(seed_key(m), it.L - 1));
        dma_b32(b_seg, ((b_mis + 2u * key) & ~3u), lds_address(lds_raw + wave * 64));
    };
    auto seed_of = [&](int key, uint32_t word) __attribute__((always_inline)) {
        const uint32_t at = b_mis + 2u * static_cast<uint32_t>(min(key, it.L - 1));
        const float bias = a.bias ? E::to_f32(static_cast<uint16_t>((at & 2u) ? (word >> 16) : (word & 0xffffu))) : 0.f;
        return key < it.L ? bias * unit : -INFINITY;
    };
    // The point (log2 units) all scores of the block are relative to: a constant, or with COME_ATTN_BLOCK_REFERENCE the
    // largest score of the block's rows over the first 32 keys.
    constexpr bool kBlockRef = !EXACT && KS == 1;
    constexpr float kBase = EXACT ? 0.f : kFoldedBase;
    float base = kBase;
    auto write_seeds = [&](int m, uint32_t word) __attribute__((always_inline)) {
        lds_seed[((m & 1) * NW + wave) * kBlockN + lane] = seed_of(seed_key(m), word) - (EXACT ? 0.f : base);
    };

    // ---- everything the first tile of block `it` needs is requested before anything is waited for
    uint32_t bias_word[2];                  // of the first two groups of tiles
    uint32_t k_first, v_first;              // of the next set to stage
    u32x4 qf[2][4];                         // Q fragments (B operand: n = query r, k = head-dim 16 ks + 8 h ..)
    auto stage_set = [&](uint32_t k_lds, uint32_t v_lds) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kDma; ++i) load_k(k_first, k_lds, i);
#pragma unroll
        for (int i = 0; i < kDma; ++i) load_v(v_first, v_lds, i);
    };
    auto next_set = [&]() __attribute__((always_inline)) {
        k_first += min(k_step, k_end - k_first);
        v_first += min(v_step, v_end - v_first);
    };
    auto begin = [&]() __attribute__((always_inline)) {
        const ArgsAfresh ka = args_afresh<kChained>();
        k_seg = reinterpret_cast<const char *>(ka->k + static_cast<int64_t>(it.seq_start) * ka->k_rs + it.head * ka->k_hs);
        v_seg = reinterpret_cast<const char *>(ka->v + static_cast<int64_t>(it.seq_start) * ka->v_rs + it.head * ka->v_hs);
        k_end = static_cast<uint32_t>(it.L - 1) * k_rs_b;
        v_end = static_cast<uint32_t>(it.L - 1) * v_rs_b;
        k_last[0] = k_end + k_chunk;
        k_last[1] = k_end + (k_chunk ^ 64u);
        v_last = v_end + v_chunk;
        const uintptr_t b_addr = reinterpret_cast<uintptr_t>(ka->bias) + 2u * static_cast<uintptr_t>(it.seq_start);
        b_seg = reinterpret_cast<const char *>(b_addr & ~static_cast<uintptr_t>(3));
        b_mis = static_cast<uint32_t>(b_addr & 3);
        bias_word[0] = bias_word[1] = 0u;
        if (ka->bias)
#pragma unroll
            for (int m = 0; m < 2; ++m)
                bias_word[m] = *reinterpret_cast<const uint32_t *>(b_seg + ((b_mis + 2u * static_cast<uint32_t>(min(seed_key(m), it.L - 1))) & ~3u));
        k_first = first_row(1 + my_half, k_rs_b);
        v_first = first_row(my_half, v_rs_b);
        if (my_half == 0) {
            const uint32_t k0 = first_row(0, k_rs_b);
#pragma unroll
            for (int i = 0; i < kDma; ++i) load_k(k0, k_part, i);
        }
        stage_set(k_part + (1 + my_half) * kStageBytes, v_part + my_half * kStageBytes);
        next_set();
        const int r = afresh<kChained>(lane) & 31, h = afresh<kChained>(lane) >> 5;
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            const uint16_t *qp = ka->q + static_cast<int64_t>(it.seq_start + min(it.q0 + 64 * qi + 32 * qt + r, it.L - 1)) * ka->q_rs + it.head * ka->q_hs + 8 * h;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) qf[qt][ks] = *reinterpret_cast<const u32x4 *>(qp + 16 * ks);
        }
    };
    __builtin_amdgcn_s_setprio(2);          // (until the loop: a starting workgroup beside a running one gets through faster)
    begin();
    for (int turn = 0;; ++turn) {           // one block; the body, which is the rest of the function, keeps its indentation
    const int seq_start = it.seq_start, L = it.L, head = it.head, q0 = it.q0;
    const int qw0 = q0 + 64 * qi;                                    // first query of this wavefront
    const int n_it = (it.n_tiles + KS - 1) / KS;                     // iterations: group g walks tiles tile_base + KS j + g
    // "some row has to be computed again": a word of its own for every other block, so that it can be cleared while slower
    // wavefronts still look at the one of the block before
    uint32_t *const lds_redo = lds_words + (turn & 1);
    {   // V half-tile "-1": zeros (its probabilities are zero as well)
        u32x4 *z = reinterpret_cast<u32x4 *>(lds_v + (RV - 1) * kHalfElems);
        for (int i = qi * 64 + lane; i < kHalfElems / 8; i += 64 * S::kQTiles) z[i] = zero4();
    }
    if (tid == 0) *lds_redo = 0;
    base = kBase;
    write_seeds(0, bias_word[0]);
    write_seeds(1, bias_word[1]);
    // The prologue of the attention (q LayerNorm + 2-D rotary embedding, qkv.py:31-39 of the reference's common
    // package) on the fragments just loaded, with the arithmetic and the summation order of the stand-alone pass, so
    // that the fragments hold the bits that pass would have written to memory.  A lane holds chunks 2 ks + h of its
    // query's head (ks = 0 .. 3): the rotation partner of a chunk (c ^ 2) is in the same lane, the neighbour in the
    // sums (c ^ 1) in lane l ^ 32.
    if (const ArgsAfresh ka = args_afresh<kChained>(); ka->qp_on) {
        using C = QkChunk<DT>;
        using V = Vec16<DT>;
        const int r = afresh<kChained>(lane) & 31, h = afresh<kChained>(lane) >> 5;
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            uint4 word[4];
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) word[ks] = __builtin_bit_cast(uint4, qf[qt][ks]);
            if (ka->qp_norm) {
                float part[4];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) part[ks] = sum_across_halves(C::sum(word[ks]));
                const float mean = C::mean_of((part[0] + part[1]) + (part[2] + part[3]));
                float f[4][8];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    V::unpack(word[ks], f[ks]);
                    part[ks] = sum_across_halves(C::center(f[ks], mean));
                }
                const float rstd = C::inv_std((part[0] + part[1]) + (part[2] + part[3]), ka->qp_eps);
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    float g[8], b[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) g[i] = 1.f, b[i] = 0.f;
                    if (ka->qp_gamma != nullptr) V::unpack(static_cast<const uint4 *>(ka->qp_gamma)[2 * ks + h], g);
                    if (ka->qp_beta != nullptr) V::unpack(static_cast<const uint4 *>(ka->qp_beta)[2 * ks + h], b);
                    word[ks] = C::scale(f[ks], rstd, g, b);
                }
            }
            if (ka->qp_pos != nullptr) {
                const int64_t token = seq_start + min(qw0 + 32 * qt + r, L - 1);
#pragma unroll
                for (int half = 0; half < 2; ++half) {                 // y: chunks 0 - 3 (ks 0, 1), x: chunks 4 - 7 (ks 2, 3)
                    const int entry = (C::table_row(ka->qp_pos[token * 2 + half], ka->qp_n_pos) * 16 + h * 8) * V::ELEM_BYTES;
                    float c[8], sn[8], lo[8], hi[8];
                    V::unpack(*reinterpret_cast<const uint4 *>(static_cast<const char *>(ka->qp_cos) + entry), c);
                    V::unpack(*reinterpret_cast<const uint4 *>(static_cast<const char *>(ka->qp_sin) + entry), sn);
                    V::unpack(word[2 * half], lo);
                    V::unpack(word[2 * half + 1], hi);
                    word[2 * half] = C::rotate(lo, hi, c, sn, C::one_and_sign(false));
                    word[2 * half + 1] = C::rotate(hi, lo, c, sn, C::one_and_sign(true));
                }
            }
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) qf[qt][ks] = __builtin_bit_cast(u32x4, word[ks]);
        }
    }
    if constexpr (!EXACT) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t raw = qf[qt][ks][w];
                    qf[qt][ks][w] = E::pack2(E::to_f32(static_cast<uint16_t>(raw & 0xffffu)) * a.scale_log2,
                                             E::to_f32(static_cast<uint16_t>(raw >> 16)) * a.scale_log2);
                }
    }
    // (the compiler's wait for Q, which counts only the loads it knows, belongs in front of the loads that may stay in flight)
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(qf[qt][ks]));
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    request_bias(2);
#pragma unroll
    for (int s = 1; s < S::kDeep; ++s) {
        stage_set(k_part + (2 * s + 1 + my_half) * kStageBytes, v_part + (2 * s + my_half) * kStageBytes);
        next_set();
    }
    asm volatile("s_barrier" ::: "memory");            // set 0 and the first seeds have landed

    // LDS read offsets (in elements) of this lane
    int k_rd[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) k_rd[ks] = r * kHeadDim + (((2 * ks + h) ^ ((r >> 1) & 7)) << 3);
    const int b_rd = 4 * h;                // keys 8 g + 4 h .. + 3 of a half-tile are accumulator elements 4 g .. 4 g + 3
    const int i16 = lane & 15;
    int v_rd[2];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
        v_rd[dt] = (4 * h + (i16 >> 2)) * kHeadDim +
                   (((4 * dt + 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1)) ^ (((i16 >> 3) & 1) << 2)) << 3) + 4 * (i16 & 1);
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // s_acc[b][qt]: scores of query tile qt for one half-tile; buffer b alternates between "being turned into
    // probabilities" and "being built by the matrix pipe".  p_frag[b][qt][u]: the probabilities of that half-tile as B
    // operands (u = 16-key step).
    f32x16 s_acc[2][2];
    f32x16 o_acc[2][2];          // [query tile][head-dim half]
    u32x4 p_frag[2][2][2];
    float delta[2] = {0.f, 0.f};  // reference point of the row, log2 units
    float l_run[2] = {0.f, 0.f};  // row sum, both half-waves together (outside the key loop)
    // Row sums in the key loop come from the matrix pipe: with the probabilities of a 16-key step as the A operand of
    // v_mfma_f32_16x16x32 (row m = lane % 16, eight keys per lane: lane group g = lane / 16 holds query m + 16 (g & 1),
    // keys 8 (g >> 1) ..) and a B operand whose lane group g is all ones in column g & 1 and zero elsewhere, the result
    // column n = 0 / 1 holds the sums of queries m / m + 16 over the step's 16 keys, whatever order the unit gives the
    // keys inside a lane.  In the 16 x 16 result a lane holds column lane % 16, rows 4 (lane / 16) .. + 3: the sums of
    // queries 0 .. 15 sit in lanes 0, 16, 32, 48, those of queries 16 .. 31 in lanes 1, 17, 33, 49, four per lane, and
    // every other lane holds zeros.  Four such MFMAs per slot (64 cycles of the matrix pipe) replace 16 v_dot2c_f32,
    // which hold the matrix pipe for as long as eight of them and the vector ALU on top.
    // bf16 (kChain): the MFMAs accumulate straight onto the running sums and the range check looks at those - a running
    // sum beyond 2^40 moves the reference point just as well as a half-tile sum beyond it.  fp16: its limit (2^9) is
    // about the size of the current probabilities, which a running sum says nothing about, so the sums of a slot are
    // formed on their own and added afterwards (those of the second query tile one slot later: they are not waited for).
    constexpr bool kChain = DT == COME_BF16;
    f32x4 l_acc[2];               // running row sums in that layout
    f32x4 s_late = {0.f, 0.f, 0.f, 0.f};      // fp16: the second query tile's sums of the slot before
    const u32x4 ones_sel = ((lane & 15) == ((lane >> 4) & 1))
                               ? u32x4{E::kOne | (E::kOne << 16), E::kOne | (E::kOne << 16), E::kOne | (E::kOne << 16), E::kOne | (E::kOne << 16)}
                               : zero4();
    const int sum_lane = (r >> 4) + 16 * ((r & 15) >> 2);         // where this lane's query keeps its row sum (element r & 3)
    // row sum of this lane's query out of that layout (a few LDS permutes: rare path and loop exit only)
    auto row_value = [&](const f32x4 &v) __attribute__((always_inline)) -> float {
        float out = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float t = __shfl(v[j], sum_lane);
            out = (r & 3) == j ? t : out;
        }
        return out;
    };
    auto seed_at = [&](const float *seeds, int half, int g) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4 *>(seeds + kHalf * half + 8 * g + b_rd);
    };
    // scores of both query tiles against the K half-tile in ring stage `stage`, into buffer b
    auto score_mfma = [&](int b, int stage, const float *seeds, int half) __attribute__((always_inline)) {
        f32x16 seed;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 bq = seed_at(seeds, half, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) seed[4 * g + e] = bq[e];
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const u32x4 kf = *reinterpret_cast<const u32x4 *>(lds_k + stage * kHalfElems + k_rd[ks]);
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
                s_acc[b][qt] = E::mfma(kf, qf[qt][ks], ks == 0 ? seed : s_acc[b][qt]);
        }
    };
    // V^T fragment f = 2 u + dt of the half-tile in ring stage `stage` (u: 16-key step, dt: head-dim half)
    auto read_v = [&](int stage, int f) __attribute__((always_inline)) {
        const uint16_t *vp = lds_v + stage * kHalfElems + v_rd[f & 1] + 16 * (f >> 1) * kHeadDim;
        const u32x2 lo2 = __builtin_bit_cast(u32x2, lds_read_tr(vp));
        const u32x2 hi2 = __builtin_bit_cast(u32x2, lds_read_tr(vp + 8 * kHeadDim));
        return u32x4{lo2[0], lo2[1], hi2[0], hi2[1]};
    };
    // O^T += V^T P^T of both query tiles for the V half-tile in ring stage `stage`, probabilities of buffer b
    auto pv_mfma = [&](int b, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const u32x4 vf = read_v(stage, f);
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) o_acc[qt][f & 1] = E::mfma(vf, p_frag[b][qt][f >> 1], o_acc[qt][f & 1]);
        }
    };

    // One slot in explicit issue order.  The vector ALU turns the scores in buffer X (one half-tile, both query tiles)
    // into probabilities.  Meanwhile the matrix pipe adds the previous half-tile's P V (8 MFMAs on 4 V fragments,
    // probabilities of buffer Y from the previous slot) and builds the scores of the next half-tile in buffer Y (8 MFMAs
    // on 4 K fragments, each fragment shared by both query tiles).  Every MFMA is followed by a chunk of vector work and
    // fragments are requested kAhead fragments (two chunks each) ahead - a dependent LDS read takes 165 cycles, a
    // transposing one 215 - so an in-order wavefront always has independent work behind each MFMA.  The first V fragments
    // of a slot come from the slot before (v_ahead): nothing at the top of a slot waits for LDS.  `between(c)` is issued in
    // chunk c.  sched_barrier keeps the compiler from regrouping the chunks.
    // fp16: returns through ssum[qt] the row sums of the half-tile (layout of l_acc); bf16 adds them to l_acc.
    constexpr int kAhead = 3;
    u32x4 v_ahead[kAhead];
    auto slot = [&](int X, int Y, int k_stage, const float *seeds, int half, int v_stage, int next_v_stage, f32x4 (&ssum)[2],
                    auto between) __attribute__((always_inline)) {
        // fragments 0..3: V (u, dt) of the P V MFMAs 0..7; fragments 4..7: K k-steps of the score MFMAs 8..15.
        // P V goes first: the probabilities of buffer Y die while those of buffer X are born, and the score
        // registers of buffer Y are not needed before half of buffer X has been consumed.
        u32x4 frag[8];
        f32x16 seed;                  // initial values of this lane's 16 keys of the half-tile being scored
        auto request = [&](int f) __attribute__((always_inline)) {
            if (f < 4) frag[f] = read_v(v_stage, f);
            else if (f < 8) frag[f] = *reinterpret_cast<const u32x4 *>(lds_k + k_stage * kHalfElems + k_rd[f - 4]);
            else v_ahead[f - 8] = read_v(next_v_stage, f - 8);
        };
        auto issue = [&](int m) __attribute__((always_inline)) {
            const int f = m >> 1, qt = m & 1;
            // empty asm statements are ordering pins: MFMAs and exponentials are pure operations which the
            // compiler would otherwise float out of their chunk (sched_barrier only fences what is already there)
            if (qt == 0) asm volatile("" : "+v"(frag[f]));
            if (f < 4) {
                const int u = f >> 1, dt = f & 1;
                o_acc[qt][dt] = E::mfma(frag[f], p_frag[Y][qt][u], o_acc[qt][dt]);
            } else {
                s_acc[Y][qt] = E::mfma(frag[f], qf[qt][f - 4], f == 4 ? seed : s_acc[Y][qt]);
            }
        };
#pragma unroll
        for (int f = 0; f < kAhead; ++f) frag[f] = v_ahead[f];
        const f32x4 zero4f = {0.f, 0.f, 0.f, 0.f};
        f32x4 &dst0 = kChain ? l_acc[0] : ssum[0];
        f32x4 &dst1 = kChain ? l_acc[1] : ssum[1];
        float p0 = 0.f, p1 = 0.f;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            // one MFMA per chunk: P V MFMAs 0..7, score MFMAs 8..15
            issue(c);
            if ((c & 1) == 0) request((c >> 1) + kAhead);            // the last chunks: the next slot's first fragments
            between(c);
            if (c >= 1 && c <= 4) {                                  // initial values of the scores, needed by chunk 8
                const f32x4 bq = seed_at(seeds, half, c - 1);
#pragma unroll
                for (int e = 0; e < 4; ++e) seed[4 * (c - 1) + e] = bq[e];
            }
            if (c > 0) {                    // pack and add the pair whose exponentials were issued one chunk ago
                const int pc = c - 1, qt = pc >> 3, w = pc & 7;
                const uint32_t pw = E::pack2_prob(p0, p1);
                p_frag[X][qt][w >> 2][w & 3] = pw;
                // a 16-key step of a query tile is complete: its row sums
                if (pc == 3) dst0 = E::mfma16(p_frag[X][0][0], ones_sel, kChain ? l_acc[0] : zero4f);
                if (pc == 7) dst0 = E::mfma16(p_frag[X][0][1], ones_sel, dst0);
                if (pc == 11) {
                    dst1 = E::mfma16(p_frag[X][1][0], ones_sel, kChain ? l_acc[1] : zero4f);
                }
            }
            float s0 = s_acc[X][c >> 3][2 * (c & 7)], s1 = s_acc[X][c >> 3][2 * (c & 7) + 1];
            if (EXACT) {
                s0 = fmaf(s0, c_scale, -delta[c >> 3]);
                s1 = fmaf(s1, c_scale, -delta[c >> 3]);
            }
            p0 = __builtin_amdgcn_exp2f(s0);
            p1 = __builtin_amdgcn_exp2f(s1);
            asm volatile("" : "+v"(p0), "+v"(p1));
            __builtin_amdgcn_sched_barrier(0);
        }
        {
            const uint32_t pw = E::pack2_prob(p0, p1);
            p_frag[X][1][1][3] = pw;
            dst1 = E::mfma16(p_frag[X][1][1], ones_sel, dst1);
        }
        // the decision that follows the slot is tied to its end, so that the branch cannot be moved
        // above the probability chunks
        asm volatile("" : "+v"(dst1) : "v"(p_frag[X][1][1][3]));
    };

    // O[qt] *= f, in place.  Written as asm so that the accumulator tuples keep their registers across a
    // rarely taken branch (plain arithmetic makes the register allocator copy the 16-register tuples).
    auto scale_o = [&](int qt, float f) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                float t = o_acc[qt][dt][e];
                asm volatile("v_mul_f32 %0, %1, %0" : "+v"(t) : "v"(f));
                o_acc[qt][dt][e] = t;
            }
    };

    // End of a slot.  Steady state: the range check (fp16: and adding the slot's row sums).
    // When a row sum leaves the safe range the reference point of the row moves up by a power of two, 2^shift:
    //  - the row sum is rescaled now;
    //  - O is rescaled one slot later (o_pending), after the P V MFMAs of the probabilities just made,
    //    which are relative to the old reference, have been accumulated.
    // EXACT: the next exponentials subtract the new reference.  Folded: the scores of buffer Y, just built relative to `base`,
    // are corrected here, from then on in every slot (ordinary logits of that mode never get there).
    float o_pending[2] = {1.f, 1.f};
    bool any_pending = false;                  // wave-uniform
    bool busy = false;                         // wave-uniform: every slot has to take the branch below
    // Whether a row sum is out of range.  Sums are not negative: if the rows of a lane together stay within the limit, each of
    // them does (written so that a NaN counts as beyond it: an infinite probability times a zero of the ones matrix is one).
    // kChain: the running sums only grow between two moves of the reference point, so they are looked at once per key tile,
    // in the middle of its second slot, where neither is being added to (the second query tile's as of the first slot).  A
    // comparison at the end of either slot, with the branch right behind it, was 11 % of the loop of a wavefront alone.  Folded,
    // us: one segment of 25 536 keys, 16 heads 2057 -> 2038, 1 % on average over launches of 6 heads and 100 - 8000 rows;
    // default arithmetic: no change.
    bool beyond = false;                       // wave-uniform
    auto check_sums = [&]() __attribute__((always_inline)) {
        float t = ((l_acc[0][0] + l_acc[0][1]) + (l_acc[0][2] + l_acc[0][3])) + ((l_acc[1][0] + l_acc[1][1]) + (l_acc[1][2] + l_acc[1][3]));
        asm volatile("" : "+v"(t));
        beyond = __any(!(t <= kSumLimit)) || busy;
    };
    auto finish_slot = [&](int Y, const f32x4 (&ssum)[2]) __attribute__((always_inline)) {
        if constexpr (kChain) {
            if (Y == 1) beyond = busy;
        } else {
            const float t = ((ssum[0][0] + ssum[0][1]) + (ssum[0][2] + ssum[0][3])) + ((s_late[0] + s_late[1]) + (s_late[2] + s_late[3]));
            beyond = __any(!(t <= kSumLimit)) || busy;
        }
        if (beyond) {
            // the asm arithmetic below reads MFMA results; the compiler cannot see that, so the wait states an
            // MFMA result needs before a vector instruction may read it are spent here explicitly
            asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
            bool moved = false;
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                if (any_pending) scale_o(qt, o_pending[qt]);
                // of this lane's query: over the half-tile, or (kChain) over all keys so far
                f32x4 sums = kChain ? l_acc[qt] : ssum[qt];
                const f32x4 s_prev = s_late;
                if (!kChain && qt == 1) {
                    l_acc[1] += s_late;                   // (not yet added)
                    s_late = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                if (!kChain && qt == 1) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) sums[j] += s_prev[j];          // (a maximum would lose a NaN)
                }
                float row_sum = row_value(sums);
                asm volatile("" : "+v"(row_sum));       // keeps the arithmetic of this rare path inside the branch
                if (__any(!(row_sum <= Range<DT>::kHardLimit))) {
                    *lds_redo = 1;                      // read behind the barrier that follows the loop
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                const int shift = row_sum <= kSumLimit ? 0 : max(__builtin_amdgcn_frexp_expf(row_sum) - 2, 1);
                const float down = __builtin_amdgcn_exp2f(static_cast<float>(-shift));
                delta[qt] += static_cast<float>(shift);
                if constexpr (!EXACT) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        float v = s_acc[Y][qt][e];
                        asm volatile("v_sub_f32 %0, %0, %1" : "+v"(v) : "v"(delta[qt]));
                        s_acc[Y][qt][e] = v;
                    }
                }
                // the running sums, where they live: element j of a lane belongs to query 16 (lane % 16) + 4 (lane / 16) + j
                // (lanes whose column is neither 0 nor 1 hold zeros and stay zero)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float dj = __shfl(down, (16 * (lane & 15) + 4 * (lane >> 4) + j) & 31);
                    l_acc[qt][j] = (kChain ? l_acc[qt][j] : l_acc[qt][j] + ssum[qt][j]) * dj;
                }
                o_pending[qt] = down;
                moved = moved || __any(shift != 0);
            }
            any_pending = moved;
            const bool keep = moved || (!EXACT && __any(delta[0] != 0.f || delta[1] != 0.f));
            busy = keep;
        } else if (!kChain) {
            l_acc[0] += ssum[0];
            l_acc[1] += s_late;
            s_late = ssum[1];
        }
    };

#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
        o_acc[qt][0] = zero16;
        o_acc[qt][1] = zero16;
        l_acc[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            p_frag[b][qt][0] = zero4();
            p_frag[b][qt][1] = zero4();
        }
    }
    int seed_at_tile = group * kBlockN;          // where the seeds of the current tile lie
    // A wavefront whose 64 queries all lie beyond the end of the segment (last workgroup of a segment) only
    // helps with the staging: it has nothing to compute and nothing to write.
    const bool idle = qw0 >= L;
    if constexpr (kBlockRef) {
        if (a.block_ref) {
            base = 0.f;
            write_seeds(0, bias_word[0]);
            write_seeds(1, bias_word[1]);
            __syncthreads();
            // the largest score of the block's rows over the first 32 keys (rows beyond the segment repeat its last one)
            float *const refs = reinterpret_cast<float *>(lds_words + 2);
            score_mfma(0, 0, lds_seed, 0);
            float wave_max = -INFINITY;
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                float mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s_acc[0][qt][e]);
                mx = max_across_halves(mx);
                wave_max = fmaxf(wave_max, (mx == -INFINITY || mx != mx) ? 0.f : mx);
            }
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1) wave_max = fmaxf(wave_max, __shfl_xor(wave_max, d));
            if (lane == 0) refs[wave] = wave_max;
            __syncthreads();
            float m = refs[0];
#pragma unroll
            for (int w = 1; w < NW; ++w) m = fmaxf(m, refs[w]);
            base = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, m)));
            write_seeds(0, bias_word[0]);
            write_seeds(1, bias_word[1]);
            __syncthreads();
        }
    }
    constexpr int kUnroll = RK / 2;              // iterations after which the K ring's stages (DEEP: both rings') repeat
    constexpr int kRefill = NW / KS;             // iterations a group of NW tiles lasts
    static_assert(kRefill >= 2 && kRefill % 2 == 0, "a tile's bias has one iteration to arrive");
    // V ring: stage of half-tile 2 j + d in iteration j.  DEEP: a constant of J = j % kUnroll.  Otherwise (a ring of
    // five) counted from v_at, the stage of half-tile 2 j - 1.
    int v_at = RV - 1;
    auto v_stage_of = [&](int J, int d) __attribute__((always_inline)) {
        if (DEEP) return (2 * J + d) & (RV - 1);
        const int x = v_at + 1 + d;
        return x >= RV ? x - RV : x;
    };
    auto end_iteration = [&]() __attribute__((always_inline)) {
        // what iteration j + 1 reads has landed: everything but (kDeep == 2) the 2 kDma loads of this iteration
        if (S::kDeep == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kDma) : "memory");
        asm volatile("s_barrier" ::: "memory");
        if (!DEEP) v_at = v_at + 2 >= RV ? v_at + 2 - RV : v_at + 2;
    };
    if (idle) {
        __builtin_amdgcn_s_setprio(0);
        if (!DEEP) asm volatile("s_barrier" ::: "memory");
        for (int j = 0; j < n_it; ++j) {
            if (j % kRefill == 0 && j > 0) {
                const int m = j / kRefill;
                const uint32_t word = a.bias ? lds_raw[wave * 64 + lane] : 0u;
                write_seeds(m + 1, word);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                request_bias(m + 2);
            }
            stage_set(k_part + ((2 * (j + S::kDeep) + 1 + my_half) & (RK - 1)) * kStageBytes,
                      v_part + v_stage_of(j % kUnroll, 2 * S::kDeep + my_half) * kStageBytes);
            next_set();
            end_iteration();
        }
    } else {
        if (kBlockRef && a.block_ref) {
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                for (int e = 0; e < 16; ++e) s_acc[0][qt][e] -= base;
        } else {
            score_mfma(0, 0, lds_seed + seed_at_tile, 0);
        }
        if constexpr (EXACT) {          // reference point of a row: its maximum over the first 32 keys of the group
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                float mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s_acc[0][qt][e]);
                mx = max_across_halves(mx) * c_scale;                  // c > 0: the maximum commutes with the scale
                // (none of them finite: kNoScore, see kLowLimit.)  fp16 probabilities are truncated, and what they lose on average
                // cancels against the row sum, unless the largest is a power of two and loses nothing: a whole number, then,
                // that leaves it anywhere in its binary order.  Relative error of the outputs against 64 bits, segments of 700,
                // 333 and 90 tokens: 2.99e-4 with the maximum itself, 2.85e-4 with the whole number; one of 16 000: 3.02e-4, 3.01e-4.
                delta[qt] = (mx == -INFINITY || mx != mx) ? kNoScore<DT> : kChain ? mx : floorf(mx) + 1.f;
            }
        }
#pragma unroll
        for (int f = 0; f < kAhead; ++f) v_ahead[f] = read_v(RV - 1, f);
        __builtin_amdgcn_s_setprio(0);
        // ring of four: every wavefront has read half-tile 0 of K, whose stage the first iteration fills again
        if (!DEEP) asm volatile("s_barrier" ::: "memory");
        // one key tile; J: j modulo kUnroll, a constant, so that the fragment reads address LDS through their offset fields
        auto iteration = [&](int j, int J) __attribute__((always_inline)) {
            f32x4 sum[2];
            uint32_t word = 0;
            const bool refill = (kRefill <= kUnroll ? J % kRefill : j % kRefill) == 0 && j > 0;
            const int m = j / kRefill;
            // (sets beyond the end: the segment's last rows again; no branch in the slots)
            const uint32_t k_lds = k_part + ((2 * (J + S::kDeep) + 1 + my_half) & (RK - 1)) * kStageBytes;
            const uint32_t v_lds = v_part + v_stage_of(J, 2 * S::kDeep + my_half) * kStageBytes;
            const float *const seeds_a = lds_seed + seed_at_tile;
            seed_at_tile = (seed_at_tile + KS * kBlockN) & (2 * NW * kBlockN - 1);
            const float *const seeds_b = lds_seed + seed_at_tile;
            // (what a set overwrites was last read in the iteration before)
            slot(0, 1, (2 * J + 1) & (RK - 1), seeds_a, 1, v_stage_of(J, -1), v_stage_of(J, 0), sum,
                 [&](int c) __attribute__((always_inline)) {
                     if (c == 1 && refill && a.bias) word = lds_raw[wave * 64 + lane];
                     if (c >= 5 && c < 5 + kDma) load_k(k_first, k_lds, c - 5);
                     if (c >= 10 && c < 10 + kDma) load_v(v_first, v_lds, c - 10);
                     if (c == 14) next_set();
                 });
            finish_slot(1, sum);
            slot(1, 0, (2 * J + 2) & (RK - 1), seeds_b, 0, v_stage_of(J, 0), v_stage_of(J, 1), sum,
                 [&](int c) __attribute__((always_inline)) {
                     if (kChain && c == 12) check_sums();
                     if (c == 2 && refill) {
                         write_seeds(m + 1, word);        // visible behind the barrier, needed kRefill - 1 iterations from now
                         request_bias(m + 2);             // (the word it overwrites has been read)
                     }
                 });
            finish_slot(0, sum);
            // The bare barrier leaves the V fragments just requested in flight; what this wavefront has written to LDS in
            // the iteration is older than fragments it has already waited for.
            end_iteration();
        };
        int j = 0;
        for (; j + kUnroll <= n_it; j += kUnroll) {
            iteration(j, 0);
            iteration(j + 1, 1);
            if constexpr (kUnroll == 4) {
                iteration(j + 2, 2);
                iteration(j + 3, 3);
            }
        }
        if (j < n_it) {          // (leaving the loop in its middle instead costs 1 % on long segments)
            iteration(j, 0);
            if constexpr (kUnroll == 4) {
                if (j + 1 < n_it) {
                    iteration(j + 1, 1);
                    if (j + 2 < n_it) iteration(j + 2, 2);
                }
            }
        }
    }
    __builtin_amdgcn_s_setprio(2);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // nothing is on its way into LDS any more (behind the next barrier)

    // ---- Probabilities are stored in the 16-bit type relative to a reference point that follows the scores lazily.
    // A key that beats everything its row has seen by more than that type can hold (2^127 for bf16, about 2^15 for
    // fp16) within one 32-key step leaves an infinite or saturated probability behind.  The wavefront that saw such a
    // row sum has said so, and the workgroup then computes its block once more with the textbook running maximum
    // (one tile at a time, no pipelining: slow, exact for any scores, and never taken by ordinary attention logits).
    if (!idle) {
        if (!kChain) l_acc[1] += s_late;
        bool redo = false;
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            if (!EXACT) delta[qt] += base;
            l_run[qt] = row_value(l_acc[qt]);
            // what the last slots added has not been looked at (fp16: limit on a half-tile's sum, checked as it was made,
            // but for the very last one of the second query tile, whose probabilities saturate rather than overflow)
            if (kChain) redo = redo || !(l_run[qt] <= Range<DT>::kHardLimit);
            else if (qt == 1) redo = redo || !(row_value(s_late) <= Range<DT>::kHardLimit);
            // a sum that vanished, or probabilities too small for their type (groups without keys of their own have none)
            float low = Range<DT>::kLowLimit;
            if constexpr (DT == COME_F16) low = delta[qt] == kNoScore<DT> ? fmaxf(low, Range<DT>::kLowMean * static_cast<float>(n_it * kBlockN)) : low;
            redo = redo || (group < it.n_tiles && !(l_run[qt] >= low));
        }
        if (__any(redo)) *lds_redo = 1;
        pv_mfma(1, DEEP ? (2 * n_it - 1) & (RV - 1) : v_at);      // the last half-tile
        if (any_pending) {
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o_acc[qt][dt][e] *= o_pending[qt];
        }
    }
    __syncthreads();
    const bool again = __builtin_amdgcn_readfirstlane(static_cast<int>(*lds_redo)) != 0;
    if (again) {
        float m_row[2] = {-INFINITY, -INFINITY};
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            o_acc[qt][0] = zero16;
            o_acc[qt][1] = zero16;
            l_run[qt] = 0.f;
        }
        for (int j = 0; j < n_it; ++j) {
            __syncthreads();                                    // stages 0 and 1 are free again
#pragma unroll
            for (int i = 0; i < kDma; ++i) {
                load_k(first_row(2 * j + my_half, k_rs_b), k_part + my_half * kStageBytes, i);
                load_v(first_row(2 * j + my_half, v_rs_b), v_part + my_half * kStageBytes, i);
            }
            if (qi == 0) {
                const int key = (it.tile_base + KS * j + group) * kBlockN + lane;
                uint32_t word = 0;
                if (a.bias) word = *reinterpret_cast<const uint32_t *>(b_seg + ((b_mis + 2u * static_cast<uint32_t>(min(key, L - 1))) & ~3u));
                lds_seed[group * kBlockN + lane] = seed_of(key, word);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (idle) continue;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                score_mfma(0, half, lds_seed + group * kBlockN, half);
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) {
                    float ex[16];
                    float mx = -INFINITY;
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        ex[e] = EXACT ? s_acc[0][qt][e] * c_scale : s_acc[0][qt][e];
                        mx = fmaxf(mx, ex[e]);
                    }
                    mx = fmaxf(max_across_halves(mx), m_row[qt]);
                    const float ref = mx == -INFINITY ? 0.f : mx;          // a row that has seen masked keys only
                    const float down = __builtin_amdgcn_exp2f(m_row[qt] - ref);
                    m_row[qt] = mx;
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                        for (int e = 0; e < 16; ++e) o_acc[qt][dt][e] *= down;
                    float part = 0.f;
#pragma unroll
                    for (int w = 0; w < 8; ++w) {
                        const uint32_t pw = E::pack2_prob(__builtin_amdgcn_exp2f(ex[2 * w] - ref),
                                                          __builtin_amdgcn_exp2f(ex[2 * w + 1] - ref));
                        p_frag[0][qt][w >> 2][w & 3] = pw;
                        part = E::dot2_ones(pw, part);
                    }
                    l_run[qt] = l_run[qt] * down + sum_across_halves(part);
                }
                pv_mfma(0, half);
            }
        }
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) delta[qt] = m_row[qt] == -INFINITY ? 0.f : m_row[qt];
        __syncthreads();                                        // the epilogue reuses the stages
    }
    const bool more = kChained && next(it);
    if (more) {
        begin();                 // (nobody reads K stages 0 - 4, V stages 0 - 3 any more, and the epilogue does not write them)
    }

    // ---- the key groups meet in LDS (the ring: nothing is in flight any more).  Every wavefront leaves its part there and
    // takes 4 / KS of the four 8-column strips (g) of its query tile's output halves from all groups: with m* the largest
    // reference point, O = sum of 2^(m_i - m*) O_i over sum of 2^(m_i - m*) l_i.  A lane then holds 8-byte pieces of
    // output rows, 8 / KS per query tile: few enough to store as they are.
    if constexpr (KS > 1) {
        float *const parts = reinterpret_cast<float *>(lds_kv);
        constexpr int kPart = 64 * (64 + 4);                    // floats of one wavefront: 64 of O, 2 reference points, 2 sums a lane
        static_assert(NW * kPart * 4 <= S::kKvElems * 2, "the parts fit the ring");
        if (!idle) {
            float *p = parts + wave * kPart + 4 * lane;
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<f32x4 *>(p + ((2 * qt + dt) * 4 + g) * 256) =
                            f32x4{o_acc[qt][dt][4 * g], o_acc[qt][dt][4 * g + 1], o_acc[qt][dt][4 * g + 2], o_acc[qt][dt][4 * g + 3]};
            *reinterpret_cast<f32x4 *>(p + 16 * 256) = f32x4{delta[0], delta[1], l_run[0], l_run[1]};
        }
        __syncthreads();
        if (idle) return;
        f32x4 ml[KS];
#pragma unroll
        for (int g2 = 0; g2 < KS; ++g2)
            ml[g2] = *reinterpret_cast<const f32x4 *>(parts + (g2 * S::kQTiles + qi) * kPart + 4 * lane + 16 * 256);
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            float m_star = -INFINITY, l_tot = 0.f, w[KS];
#pragma unroll
            for (int g2 = 0; g2 < KS; ++g2) m_star = ml[g2][2 + qt] > 0.f ? fmaxf(m_star, ml[g2][qt]) : m_star;     // (a group without keys has no say)
#pragma unroll
            for (int g2 = 0; g2 < KS; ++g2) {
                w[g2] = ml[g2][2 + qt] > 0.f ? __builtin_amdgcn_exp2f(ml[g2][qt] - m_star) : 0.f;
                l_tot += ml[g2][2 + qt] * w[g2];
            }
            const float inv = 1.0f / l_tot;
            const int row = qw0 + qt * 32 + r;
            if (row < L && group == 0 && h == 0 && a.lse)
                a.lse[static_cast<int64_t>(head) * a.total + seq_start + row] = (m_star + __log2f(l_tot)) * 0.6931471805599453f;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int i = 0; i < 4 / KS; ++i) {
                    const int g = group * (4 / KS) + i;
                    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int g2 = 0; g2 < KS; ++g2)
                        o += *reinterpret_cast<const f32x4 *>(parts + (g2 * S::kQTiles + qi) * kPart + ((2 * qt + dt) * 4 + g) * 256 + 4 * lane) * w[g2];
                    if (row < L)
                        *reinterpret_cast<u32x2 *>(a.out + static_cast<int64_t>(seq_start + row) * a.o_rs + head * a.o_hs + 32 * dt + 8 * g + 4 * h) =
                            u32x2{E::pack2(o[0] * inv, o[1] * inv), E::pack2(o[2] * inv, o[3] * inv)};
                }
        }
        return;
    }
    if (!kChained && idle) return;

    // ---- epilogue of a split workgroup: unnormalised outputs, reference point and row sum of its key share
    if (piece != nullptr) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            const int local_row = (2 * qi + qt) * 32 + r;
            if (q0 + local_row < L) {
                float *op = piece + local_row * kHeadDim + 4 * h;
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<f32x4 *>(op + 32 * dt + 8 * g) =
                            f32x4{o_acc[qt][dt][4 * g], o_acc[qt][dt][4 * g + 1], o_acc[qt][dt][4 * g + 2],
                                  o_acc[qt][dt][4 * g + 3]};
                if (h == 0) {
                    piece[kBlockM * kHeadDim + local_row] = delta[qt];
                    piece[kBlockM * (kHeadDim + 1) + local_row] = l_run[qt];
                }
            }
        }
        return;
    }

    // ---- epilogue: normalise, write O (and LSE).  In the accumulators a lane holds 8-byte pieces of one output row,
    // 32 rows per store instruction; written like that, a wavefront's 32 stores touch 32 rows each and queue up in the
    // memory pipeline for microseconds.  Each wavefront therefore passes its two 32 x 64 tiles through 4 KiB of LDS
    // (16-byte chunk c of row r at chunk c ^ (r & 7)) and stores whole 128-byte rows, eight rows per instruction.  Chained:
    // stages that the next block's first loads leave alone (K 5 - 7 and V 4).
    uint16_t *const slot_base = lds_kv + (kChained ? (wave < 3 ? 5 + wave : RK + 4) : wave) * kHalfElems;
    const ArgsAfresh ka = args_afresh<kChained>();
    if (!idle) {
        const int el = afresh<kChained>(lane), er = el & 31, eh = el >> 5;
        u32x4 rows[2][4];                                            // rows 8 i + el / 8 of the query tiles, one chunk each
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            const float l_tot = l_run[qt];
            const float inv = 1.0f / l_tot;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    u32x2 w;
                    w[0] = E::pack2(o_acc[qt][dt][4 * g] * inv, o_acc[qt][dt][4 * g + 1] * inv);
                    w[1] = E::pack2(o_acc[qt][dt][4 * g + 2] * inv, o_acc[qt][dt][4 * g + 3] * inv);
                    *reinterpret_cast<u32x2 *>(slot_base + er * 64 + (((4 * dt + g) ^ (er & 7)) << 3) + 4 * eh) = w;
                }
            const int row = qw0 + qt * 32 + er;
            if (row < L && eh == 0 && ka->lse)
                ka->lse[static_cast<int64_t>(head) * ka->total + seq_start + row] = (delta[qt] + __log2f(l_tot)) * 0.6931471805599453f;
#pragma unroll
            for (int i = 0; i < 4; ++i) rows[qt][i] = *reinterpret_cast<const u32x4 *>(slot_base + 64 * (8 * i) + 8 * el);
        }
        // the chunk this lane finds at position el % 8 of rows el / 8 + 8 i
        const int c = (el & 7) ^ ((el >> 3) & 7);
        const int64_t o_rs = ka->o_rs;
        uint16_t *op = ka->out + (seq_start + qw0 + (el >> 3)) * o_rs + head * ka->o_hs + 8 * c;
        const bool out_wide = ka->out_wide != 0;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const u32x4 v = rows[n >> 2][n & 3];
            if (qw0 + 8 * n + (el >> 3) < L) {
                if (out_wide) {
                    *reinterpret_cast<u32x4 *>(op) = v;
                } else {
                    *reinterpret_cast<u32x2 *>(op) = u32x2{v[0], v[1]};
                    *reinterpret_cast<u32x2 *>(op + 4) = u32x2{v[2], v[3]};
                }
            }
            op += 8 * o_rs;
        }
    }
    if (!more) return;
    }
}

// -------------------------------------------------------------------------------------
// The same for one key group, 8 x 1 or 4 x 1, in tiles of 16 x 16: v_mfma 16x16x32 in place of 32x32x16.
//
// A launch that fills the chip runs at the clock its power allows, not at the rate of its instructions (25 536 and 21 848 keys, 16
// heads: 4.13 ms of N(0, 1) values, 3.18 of zeros), and 16x16x32 draws less: it moves 8 registers of sums in and out for
// 16 cycles of the matrix pipe, 32x32x16 moves 32 for 32.  A slot of this pipeline without loads and barriers, two wavefronts a
// SIMD on the whole chip, TFLOP/s: default arithmetic 1255 with 32x32x16 and 1317, folded 1396 and 1480.  It takes twice the
// matrix instructions, which a wavefront alone on its SIMD has no room for (13 us of slots 0.469 -> 0.486 us each, folded 0.421 ->
// 0.425), so the shapes of several key groups keep 32x32x16; so do chained blocks, which have no registers for it (14 - 21
// spilled; us, folded, 32 x 798 keys 98.6 -> 104.9, 128 x 390 142.5 -> 152.6), and launches with COME_ATTN_BLOCK_REFERENCE, whose callers
// ask for the same bits from one launch to the next.  What the clock gives differs from card to card: 25 536 and 21 848 keys, 16 heads, on
// three of them 4.14 -> 3.96 ms, 4.03 -> 3.86 and 4.07 -> 3.93, folded 3.72 -> 3.56 and 3.61 -> 3.47, on a fourth 4.04 -> 4.03; one segment of
// 25 536 2.33 -> 2.23 and 2.09 -> 2.01; 7713 keys 222 -> 214 us and 200 -> 193.
//
// What differs from attn_block.  Lane l = 16 g + r holds query r of four tiles (n) and, of a half-tile, keys 16 (g / 2) + 8 kt + 4 (g % 2) + e
// in two score tiles (kt).  The eight keys a lane gives to a P V instruction are all of those, so the instruction's sum takes the keys in
// the order in which two of attn_block's take them, and a row has the same bits from either: an output does not depend on which pipeline
// the size of a launch asks for.  (Keys 4 g + e of two tiles of consecutive rows, as fast, gave other last bits, 3e-3 behind 48 blocks.  In fp16 a
// reference point may move a slot earlier or later, since the sums that one lane looks at together are those of other rows: 5 rows in 10 000 of
// logits three times as large as a LayerNorm's.)
// V^T fragments come from two transposing reads 8 rows apart, one per kt.  Row sums are the products of a matrix of ones with the probabilities:
// every lane receives the sum of its own query.  K chunk c of row x sits at c ^ (x / 2 % 4) ^ 4 (x / 16), V chunk c at c ^ 4 (x / 2 % 2)
// ^ 2 (x / 4 % 2): the rows that one phase of a fragment's reads takes lie in different banks.
// -------------------------------------------------------------------------------------
template <int DT, int NW, bool EXACT>
__device__ __forceinline__ void attn_block16(const AttnArgs &a, Item it, uint16_t *lds_kv, float *lds_seed, uint32_t *lds_raw,
                                             uint32_t *lds_redo) {
    using E = Elem<DT>;
    using S = Shape<NW, 1>;
    static_assert(EXACT || DT == COME_BF16, "fp16 runs the default arithmetic");
    constexpr float kSumLimit = Range<DT>::kSumLimit;
    constexpr int RK = S::kRingK, RV = S::kRingV, kDma = S::kDma, kBlockM = S::kBlockM, kThreads = 64 * NW;
    constexpr int kHalfElems = kHalf * kHeadDim;
    constexpr float kLog2e = 1.4426950408889634f;
    float *const piece = it.piece;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);       // query tile of 64
    const int g = lane >> 4;
    const int r = lane & 15;
    uint16_t *const lds_k = lds_kv;
    uint16_t *const lds_v = lds_kv + RK * kHalfElems;
    if (it.n_tiles <= 0) {                         // a key share without tiles (segment shorter than the split count)
        for (int i = tid; i < kBlockM; i += kThreads) {
            piece[kBlockM * kHeadDim + i] = -1e30f;               // reference point
            piece[kBlockM * (kHeadDim + 1) + i] = 0.f;            // row sum
        }
        return;
    }

    // ---- global -> LDS staging, as in attn_block
    const char *k_seg, *v_seg;
    const uint32_t k_rs_b = static_cast<uint32_t>(a.k_rs) * 2u, v_rs_b = static_cast<uint32_t>(a.v_rs) * 2u;
    const int my_half = (wave * kDma) >> 2, my_rows = ((wave * kDma) & 3) * 8;       // (uniform)
    const int st_row = my_rows + (lane >> 3);
    static_assert(kDma <= 2, "the 8 i rows that load i is further on do not reach the next 16");
    const uint32_t k_chunk = static_cast<uint32_t>((lane & 7) ^ ((st_row >> 1) & 3) ^ (st_row >> 4 << 2)) * 16u;
    const uint32_t v_chunk = static_cast<uint32_t>((lane & 7) ^ (((st_row >> 1) & 1) << 2) ^ (((st_row >> 2) & 1) << 1)) * 16u;
    uint32_t k_end, v_end;
    const uint32_t k_step = static_cast<uint32_t>(kBlockN) * k_rs_b, v_step = static_cast<uint32_t>(kBlockN) * v_rs_b;
    auto first_row = [&](int hf, uint32_t rs_b) __attribute__((always_inline)) {      // half-tile hf
        return static_cast<uint32_t>(min((it.tile_base + (hf >> 1)) * kBlockN + (hf & 1) * kHalf, it.L - 1)) * rs_b;
    };
    const uint32_t k_at_row = static_cast<uint32_t>(st_row) * k_rs_b + k_chunk, v_at_row = static_cast<uint32_t>(st_row) * v_rs_b + v_chunk;
    uint32_t k_last, v_last;
    auto load_k = [&](uint32_t first, uint32_t lds, int i) __attribute__((always_inline)) {
        const uint32_t at = __builtin_elementwise_add_sat(k_at_row + 8u * i * k_rs_b, first);
        dma_b128(k_seg, min(at, k_last), lds + 1024u * i);
    };
    auto load_v = [&](uint32_t first, uint32_t lds, int i) __attribute__((always_inline)) {
        const uint32_t at = __builtin_elementwise_add_sat(v_at_row + 8u * i * v_rs_b, first);
        dma_b128(v_seg, min(at, v_last), lds + 1024u * i);
    };
    const uint32_t k_part = lds_address(lds_k) + static_cast<uint32_t>(my_rows) * 128u, v_part = lds_address(lds_v) + static_cast<uint32_t>(my_rows) * 128u;
    constexpr uint32_t kStageBytes = kHalfElems * 2u;
    const float c_scale = a.scale_log2;
    const float unit = EXACT ? kLog2e / a.scale_log2 : kLog2e;                    // EXACT: accumulators hold raw scores
    const char *b_seg;
    uint32_t b_mis;
    auto seed_key = [&](int m) __attribute__((always_inline)) { return (it.tile_base + NW * m + wave) * kBlockN + lane; };
    auto request_bias = [&](int m) __attribute__((always_inline)) {
        if (a.bias == nullptr) return;
        const uint32_t key = static_cast<uint32_t>(min(seed_key(m), it.L - 1));
        dma_b32(b_seg, ((b_mis + 2u * key) & ~3u), lds_address(lds_raw + wave * 64));
    };
    auto seed_of = [&](int key, uint32_t word) __attribute__((always_inline)) {
        const uint32_t at = b_mis + 2u * static_cast<uint32_t>(min(key, it.L - 1));
        const float bias = a.bias ? E::to_f32(static_cast<uint16_t>((at & 2u) ? (word >> 16) : (word & 0xffffu))) : 0.f;
        return key < it.L ? bias * unit : -INFINITY;
    };
    constexpr float kBase = EXACT ? 0.f : kFoldedBase;             // what all scores are relative to (log2 units)
    auto write_seeds = [&](int m, uint32_t word) __attribute__((always_inline)) {
        lds_seed[((m & 1) * NW + wave) * kBlockN + lane] = seed_of(seed_key(m), word) - kBase;
    };

    // ---- everything the first tile of block `it` needs is requested before anything is waited for
    uint32_t bias_word[2];                  // of the first two groups of tiles
    uint32_t k_first, v_first;              // of the next set to stage
    u32x4 qf[4][2];                         // Q fragments (B operand: query 16 n + r, head-dim 32 d + 8 g ..)
    auto stage_set = [&](uint32_t k_lds, uint32_t v_lds) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kDma; ++i) load_k(k_first, k_lds, i);
#pragma unroll
        for (int i = 0; i < kDma; ++i) load_v(v_first, v_lds, i);
    };
    auto next_set = [&]() __attribute__((always_inline)) {
        k_first += min(k_step, k_end - k_first);
        v_first += min(v_step, v_end - v_first);
    };
    __builtin_amdgcn_s_setprio(2);          // (until the loop: a starting workgroup beside a running one gets through faster)
    k_seg = reinterpret_cast<const char *>(a.k + static_cast<int64_t>(it.seq_start) * a.k_rs + it.head * a.k_hs);
    v_seg = reinterpret_cast<const char *>(a.v + static_cast<int64_t>(it.seq_start) * a.v_rs + it.head * a.v_hs);
    k_end = static_cast<uint32_t>(it.L - 1) * k_rs_b;
    v_end = static_cast<uint32_t>(it.L - 1) * v_rs_b;
    k_last = k_end + k_chunk;
    v_last = v_end + v_chunk;
    const uintptr_t b_addr = reinterpret_cast<uintptr_t>(a.bias) + 2u * static_cast<uintptr_t>(it.seq_start);
    b_seg = reinterpret_cast<const char *>(b_addr & ~static_cast<uintptr_t>(3));
    b_mis = static_cast<uint32_t>(b_addr & 3);
    bias_word[0] = bias_word[1] = 0u;
    if (a.bias)
#pragma unroll
        for (int m = 0; m < 2; ++m)
            bias_word[m] = *reinterpret_cast<const uint32_t *>(b_seg + ((b_mis + 2u * static_cast<uint32_t>(min(seed_key(m), it.L - 1))) & ~3u));
    k_first = first_row(1 + my_half, k_rs_b);
    v_first = first_row(my_half, v_rs_b);
    if (my_half == 0) {
        const uint32_t k0 = first_row(0, k_rs_b);
#pragma unroll
        for (int i = 0; i < kDma; ++i) load_k(k0, k_part, i);
    }
    stage_set(k_part + (1 + my_half) * kStageBytes, v_part + my_half * kStageBytes);
    next_set();
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const uint16_t *qp = a.q + static_cast<int64_t>(it.seq_start + min(it.q0 + 64 * wave + 16 * n + r, it.L - 1)) * a.q_rs + it.head * a.q_hs + 8 * g;
#pragma unroll
        for (int d = 0; d < 2; ++d) qf[n][d] = *reinterpret_cast<const u32x4 *>(qp + 32 * d);
    }
    const int seq_start = it.seq_start, L = it.L, head = it.head, q0 = it.q0;
    const int qw0 = q0 + 64 * wave;                                  // first query of this wavefront
    const int n_it = it.n_tiles;
    {   // V half-tile "-1": zeros (its probabilities are zero as well)
        u32x4 *z = reinterpret_cast<u32x4 *>(lds_v + (RV - 1) * kHalfElems);
        for (int i = tid; i < kHalfElems / 8; i += kThreads) z[i] = zero4();
    }
    if (tid == 0) *lds_redo = 0;
    write_seeds(0, bias_word[0]);
    write_seeds(1, bias_word[1]);
    // The prologue of the attention on the fragments just loaded (attn_block).  A lane holds chunks 4 d + g of its query's head: the
    // neighbour in the sums (c ^ 1) is in lane l ^ 16, the rotation partner (c ^ 2) in lane l ^ 32.
    if (a.qp_on) {
        using C = QkChunk<DT>;
        using V = Vec16<DT>;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            uint4 word[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) word[d] = __builtin_bit_cast(uint4, qf[n][d]);
            if (a.qp_norm) {
                float part[2];
#pragma unroll
                for (int d = 0; d < 2; ++d) part[d] = sum_across_quarters(C::sum(word[d]));
                const float mean = C::mean_of(part[0] + part[1]);
                float f[2][8];
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    V::unpack(word[d], f[d]);
                    part[d] = sum_across_quarters(C::center(f[d], mean));
                }
                const float rstd = C::inv_std(part[0] + part[1], a.qp_eps);
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    float gain[8], b[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) gain[i] = 1.f, b[i] = 0.f;
                    if (a.qp_gamma != nullptr) V::unpack(static_cast<const uint4 *>(a.qp_gamma)[4 * d + g], gain);
                    if (a.qp_beta != nullptr) V::unpack(static_cast<const uint4 *>(a.qp_beta)[4 * d + g], b);
                    word[d] = C::scale(f[d], rstd, gain, b);
                }
            }
            if (a.qp_pos != nullptr) {
                const int64_t token = seq_start + min(qw0 + 16 * n + r, L - 1);
                const bool second = (g & 2) != 0;                      // chunks 2, 3 of a half
                const uint32_t sign = second ? C::one_and_sign(true) : C::one_and_sign(false);
#pragma unroll
                for (int d = 0; d < 2; ++d) {                          // y: chunks 0 - 3, x: chunks 4 - 7
                    const int entry = (C::table_row(a.qp_pos[token * 2 + d], a.qp_n_pos) * 16 + (g & 1) * 8) * V::ELEM_BYTES;
                    float c[8], sn[8], own[8], partner[8];
                    V::unpack(*reinterpret_cast<const uint4 *>(static_cast<const char *>(a.qp_cos) + entry), c);
                    V::unpack(*reinterpret_cast<const uint4 *>(static_cast<const char *>(a.qp_sin) + entry), sn);
                    V::unpack(word[d], own);
                    V::unpack(uint4{other_half(word[d].x), other_half(word[d].y), other_half(word[d].z), other_half(word[d].w)}, partner);
                    word[d] = C::rotate(own, partner, c, sn, sign);
                }
            }
#pragma unroll
            for (int d = 0; d < 2; ++d) qf[n][d] = __builtin_bit_cast(u32x4, word[d]);
        }
    }
    if constexpr (!EXACT) {
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t raw = qf[n][d][w];
                    qf[n][d][w] = E::pack2(E::to_f32(static_cast<uint16_t>(raw & 0xffffu)) * a.scale_log2,
                                           E::to_f32(static_cast<uint16_t>(raw >> 16)) * a.scale_log2);
                }
    }
    // (the compiler's wait for Q, which counts only the loads it knows, belongs in front of the loads that may stay in flight)
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int d = 0; d < 2; ++d) asm volatile("" : "+v"(qf[n][d]));
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    request_bias(2);
#pragma unroll
    for (int s = 1; s < S::kDeep; ++s) {
        stage_set(k_part + (2 * s + 1 + my_half) * kStageBytes, v_part + (2 * s + my_half) * kStageBytes);
        next_set();
    }
    asm volatile("s_barrier" ::: "memory");            // set 0 and the first seeds have landed

    // LDS read offsets (in elements) of this lane
    const int key0 = 16 * (g >> 1) + 4 * (g & 1);                    // the lane's first key of score tile 0
    int k_rd[2];                            // key of score row r of tile 0, head-dim 32 d + 8 g .. + 7
#pragma unroll
    for (int d = 0; d < 2; ++d) k_rd[d] = (16 * (r >> 3) + (r & 7)) * kHeadDim + (((4 * d + g) ^ (r >> 1)) << 3);
    int v_rd[4];                            // head-dim 16 dt + r, keys key0 .. + 3
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
        v_rd[dt] = (key0 + (r >> 2)) * kHeadDim + (((2 * dt + ((r & 3) >> 1)) ^ (((r >> 3) & 1) << 2) ^ ((g & 1) << 1)) << 3) + 4 * (r & 1);
    const f32x4 zero4f = {0.f, 0.f, 0.f, 0.f};

    // s_acc[b][kt][n]: scores of query tile n for the 16 keys of score tile kt; p_frag[b][n]: the probabilities of the half-tile
    f32x4 s_acc[2][2][4];
    f32x4 o_acc[4][4];           // [query tile][16 of the head-dim]
    u32x4 p_frag[2][4];
    float delta[4] = {0.f, 0.f, 0.f, 0.f};  // reference point of the row, log2 units
    float l_run[4] = {0.f, 0.f, 0.f, 0.f};  // row sum (outside the key loop; fp16: everywhere)
    // bf16 (kChain): the row sums' instructions accumulate straight onto the running sums, whose four registers are alike.
    // fp16, whose limit is about the size of the current probabilities: the sums of a slot are formed on their own and added
    // afterwards (those of the last query tile one slot later: they are not waited for).
    constexpr bool kChain = DT == COME_BF16;
    f32x4 l_acc[4];
    float s_late = 0.f;          // fp16: the last query tile's sums of the slot before
    constexpr uint32_t kOnes = E::kOne | (E::kOne << 16);
    const u32x4 ones = {kOnes, kOnes, kOnes, kOnes};
    auto seed_at = [&](const float *seeds, int half, int kt) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4 *>(seeds + kHalf * half + 8 * kt + key0);
    };
    auto read_k = [&](int stage, int f) __attribute__((always_inline)) {              // fragment f = 2 d + kt
        return *reinterpret_cast<const u32x4 *>(lds_k + stage * kHalfElems + k_rd[f >> 1] + 8 * kHeadDim * (f & 1));
    };
    auto read_v = [&](int stage, int dt) __attribute__((always_inline)) {
        const uint16_t *vp = lds_v + stage * kHalfElems + v_rd[dt];
        const u32x2 lo2 = __builtin_bit_cast(u32x2, lds_read_tr(vp));
        const u32x2 hi2 = __builtin_bit_cast(u32x2, lds_read_tr(vp + 8 * kHeadDim));
        return u32x4{lo2[0], lo2[1], hi2[0], hi2[1]};
    };
    // scores of all query tiles against the K half-tile in ring stage `stage`, into buffer b
    auto score_mfma = [&](int b, int stage, const float *seeds, int half) __attribute__((always_inline)) {
        const f32x4 seed[2] = {seed_at(seeds, half, 0), seed_at(seeds, half, 1)};
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const u32x4 kf = read_k(stage, f);
#pragma unroll
            for (int n = 0; n < 4; ++n) s_acc[b][f & 1][n] = E::mfma16(kf, qf[n][f >> 1], f < 2 ? seed[f & 1] : s_acc[b][f & 1][n]);
        }
    };
    // O^T += V^T P^T for the V half-tile in ring stage `stage`, probabilities of buffer b
    auto pv_mfma = [&](int b, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            const u32x4 vf = read_v(stage, dt);
#pragma unroll
            for (int n = 0; n < 4; ++n) o_acc[n][dt] = E::mfma16(vf, p_frag[b][n], o_acc[n][dt]);
        }
    };

    // One slot in explicit issue order (attn_block): two MFMAs and the exponentials of two scores a chunk.
    constexpr int kAhead = NW == 8 ? 3 : 2;            // (3: 2 - 4 registers spilled with 4 wavefronts)
    u32x4 v_ahead[kAhead];
    auto slot = [&](int X, int Y, int k_stage, const float *seeds, int half, int v_stage, int next_v_stage, f32x4 (&ssum)[4],
                    auto between) __attribute__((always_inline)) {
        u32x4 frag[8];                // 0..3: V^T of 16 head-dims; 4..7: K (d, kt)
        f32x4 seed[2];
        auto request = [&](int f) __attribute__((always_inline)) {
            if (f < 4) frag[f] = read_v(v_stage, f);
            else if (f < 8) frag[f] = read_k(k_stage, f - 4);
            else v_ahead[f - 8] = read_v(next_v_stage, f - 8);
        };
        auto issue = [&](int m) __attribute__((always_inline)) {
            const int f = m >> 2, n = m & 3;
            if (n == 0) asm volatile("" : "+v"(frag[f]));            // (ordering pins, as below)
            if (f < 4) o_acc[n][f] = E::mfma16(frag[f], p_frag[Y][n], o_acc[n][f]);
            else s_acc[Y][f & 1][n] = E::mfma16(frag[f], qf[n][(f - 4) >> 1], f < 6 ? seed[f & 1] : s_acc[Y][f & 1][n]);
        };
        auto add_sums = [&](int n) __attribute__((always_inline)) {
            f32x4 &dst = kChain ? l_acc[n] : ssum[n];
            dst = E::mfma16(ones, p_frag[X][n], kChain ? l_acc[n] : zero4f);
        };
#pragma unroll
        for (int f = 0; f < kAhead; ++f) frag[f] = v_ahead[f];
        float p0 = 0.f, p1 = 0.f;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            issue(2 * c);
            issue(2 * c + 1);
            if ((c & 1) == 0) request((c >> 1) + kAhead);            // the last chunks: the next slot's first fragments
            between(c);
            if (c == 1 || c == 3) seed[c >> 1] = seed_at(seeds, half, c >> 1);        // needed by chunks 8 and 10
            if (c > 0) {                    // pack the pair whose exponentials were issued one chunk ago
                const int n = (c - 1) >> 2, w = (c - 1) & 3;
                p_frag[X][n][w] = E::pack2_prob(p0, p1);
                if (w == 3) add_sums(n);
            }
            float s0 = s_acc[X][(c >> 1) & 1][c >> 2][2 * (c & 1)], s1 = s_acc[X][(c >> 1) & 1][c >> 2][2 * (c & 1) + 1];
            if (EXACT) {
                s0 = fmaf(s0, c_scale, -delta[c >> 2]);
                s1 = fmaf(s1, c_scale, -delta[c >> 2]);
            }
            p0 = __builtin_amdgcn_exp2f(s0);
            p1 = __builtin_amdgcn_exp2f(s1);
            asm volatile("" : "+v"(p0), "+v"(p1));
            __builtin_amdgcn_sched_barrier(0);
        }
        p_frag[X][3][3] = E::pack2_prob(p0, p1);
        add_sums(3);
        // the decision that follows the slot is tied to its end, so that the branch cannot be moved above the chunks
        if (kChain) asm volatile("" : "+v"(l_acc[3]) : "v"(p_frag[X][3][3]));
        else asm volatile("" : "+v"(ssum[3]) : "v"(p_frag[X][3][3]));
    };

    // O[n] *= f, in place (as asm: see attn_block)
    auto scale_o = [&](int n, float f) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float t = o_acc[n][dt][e];
                asm volatile("v_mul_f32 %0, %1, %0" : "+v"(t) : "v"(f));
                o_acc[n][dt][e] = t;
            }
    };

    // End of a slot: the range check, and where a row sum leaves the range the reference point of the row moves (attn_block).
    // All of it is in the lane that holds the query.
    float o_pending[4] = {1.f, 1.f, 1.f, 1.f};
    bool any_pending = false;                  // wave-uniform
    bool busy = false;                         // wave-uniform: every slot has to take the branch below
    bool beyond = false;                       // wave-uniform
    auto check_sums = [&]() __attribute__((always_inline)) {
        float t = (l_acc[0][0] + l_acc[1][0]) + (l_acc[2][0] + l_acc[3][0]);
        asm volatile("" : "+v"(t));
        beyond = __any(!(t <= kSumLimit)) || busy;
    };
    auto finish_slot = [&](int Y, const f32x4 (&ssum)[4]) __attribute__((always_inline)) {
        if constexpr (kChain) {
            if (Y == 1) beyond = busy;
        } else {
            const float t = (ssum[0][0] + ssum[1][0]) + (ssum[2][0] + s_late);
            beyond = __any(!(t <= kSumLimit)) || busy;
        }
        if (beyond) {
            // (wait states of MFMA results read by the asm arithmetic below)
            asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
            bool moved = false;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                if (any_pending) scale_o(n, o_pending[n]);
                float row_sum = kChain ? l_acc[n][0] : ssum[n][0];
                if (!kChain && n == 3) {
                    l_run[3] += s_late;                   // (not yet added)
                    row_sum += s_late;                    // (a maximum would lose a NaN)
                    s_late = 0.f;
                }
                asm volatile("" : "+v"(row_sum));       // keeps the arithmetic of this rare path inside the branch
                if (__any(!(row_sum <= Range<DT>::kHardLimit))) {
                    *lds_redo = 1;                      // read behind the barrier that follows the loop
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
                const int shift = row_sum <= kSumLimit ? 0 : max(__builtin_amdgcn_frexp_expf(row_sum) - 2, 1);
                const float down = __builtin_amdgcn_exp2f(static_cast<float>(-shift));
                delta[n] += static_cast<float>(shift);
                if constexpr (!EXACT) {
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float v = s_acc[Y][kt][n][e];
                            asm volatile("v_sub_f32 %0, %0, %1" : "+v"(v) : "v"(delta[n]));
                            s_acc[Y][kt][n][e] = v;
                        }
                }
                if (kChain) l_acc[n] *= down;
                else l_run[n] = (l_run[n] + ssum[n][0]) * down;
                o_pending[n] = down;
                moved = moved || __any(shift != 0);
            }
            any_pending = moved;
            busy = moved || (!EXACT && __any(delta[0] != 0.f || delta[1] != 0.f || delta[2] != 0.f || delta[3] != 0.f));
        } else if (!kChain) {
#pragma unroll
            for (int n = 0; n < 3; ++n) l_run[n] += ssum[n][0];
            l_run[3] += s_late;
            s_late = ssum[3][0];
        }
    };

#pragma unroll
    for (int n = 0; n < 4; ++n) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o_acc[n][dt] = zero4f;
        l_acc[n] = zero4f;
        p_frag[0][n] = p_frag[1][n] = zero4();
    }
    int seed_at_tile = 0;                        // where the seeds of the current tile lie
    const bool idle = qw0 >= L;                  // all queries beyond the end of the segment: only helps with the staging
    constexpr int kUnroll = RK / 2;              // iterations after which the rings' stages repeat
    constexpr int kRefill = NW;                  // iterations a group of NW tiles lasts
    auto v_stage_of = [&](int J, int d) __attribute__((always_inline)) { return (2 * J + d) & (RV - 1); };      // of half-tile 2 j + d
    auto end_iteration = [&]() __attribute__((always_inline)) {
        // what iteration j + 1 reads has landed: everything but the 2 kDma loads of this iteration
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kDma) : "memory");
        asm volatile("s_barrier" ::: "memory");
    };
    if (idle) {
        __builtin_amdgcn_s_setprio(0);
        for (int j = 0; j < n_it; ++j) {
            if (j % kRefill == 0 && j > 0) {
                const int m = j / kRefill;
                const uint32_t word = a.bias ? lds_raw[wave * 64 + lane] : 0u;
                write_seeds(m + 1, word);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                request_bias(m + 2);
            }
            stage_set(k_part + ((2 * (j + S::kDeep) + 1 + my_half) & (RK - 1)) * kStageBytes,
                      v_part + v_stage_of(j % kUnroll, 2 * S::kDeep + my_half) * kStageBytes);
            next_set();
            end_iteration();
        }
    } else {
        score_mfma(0, 0, lds_seed + seed_at_tile, 0);
        if constexpr (EXACT) {          // reference point of a row: its maximum over the first 32 keys
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                float mx = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s_acc[0][kt][n][e]);
                mx = max_across_quarters(mx) * c_scale;                // c > 0: the maximum commutes with the scale
                // (none of them finite: kNoScore, see kLowLimit; fp16: a whole number, see attn_block)
                delta[n] = (mx == -INFINITY || mx != mx) ? kNoScore<DT> : kChain ? mx : floorf(mx) + 1.f;
            }
        }
#pragma unroll
        for (int f = 0; f < kAhead; ++f) v_ahead[f] = read_v(RV - 1, f);
        __builtin_amdgcn_s_setprio(0);
        // one key tile; J: j modulo kUnroll, a constant, so that the fragment reads address LDS through their offset fields
        auto iteration = [&](int j, int J) __attribute__((always_inline)) {
            f32x4 sum[4];
            uint32_t word = 0;
            const bool refill = (kRefill <= kUnroll ? J % kRefill : j % kRefill) == 0 && j > 0;
            const int m = j / kRefill;
            const uint32_t k_lds = k_part + ((2 * (J + S::kDeep) + 1 + my_half) & (RK - 1)) * kStageBytes;
            const uint32_t v_lds = v_part + v_stage_of(J, 2 * S::kDeep + my_half) * kStageBytes;
            const float *const seeds_a = lds_seed + seed_at_tile;
            seed_at_tile = (seed_at_tile + kBlockN) & (2 * NW * kBlockN - 1);
            const float *const seeds_b = lds_seed + seed_at_tile;
            // (what a set overwrites was last read in the iteration before)
            slot(0, 1, (2 * J + 1) & (RK - 1), seeds_a, 1, v_stage_of(J, -1), v_stage_of(J, 0), sum,
                 [&](int c) __attribute__((always_inline)) {
                     if (c == 1 && refill && a.bias) word = lds_raw[wave * 64 + lane];
                     if (c >= 5 && c < 5 + kDma) load_k(k_first, k_lds, c - 5);
                     if (c >= 10 && c < 10 + kDma) load_v(v_first, v_lds, c - 10);
                     if (c == 14) next_set();
                 });
            finish_slot(1, sum);
            slot(1, 0, (2 * J + 2) & (RK - 1), seeds_b, 0, v_stage_of(J, 0), v_stage_of(J, 1), sum,
                 [&](int c) __attribute__((always_inline)) {
                     if (kChain && c == 12) check_sums();
                     if (c == 2 && refill) {
                         write_seeds(m + 1, word);        // visible behind the barrier, needed kRefill - 1 iterations from now
                         request_bias(m + 2);             // (the word it overwrites has been read)
                     }
                 });
            finish_slot(0, sum);
            end_iteration();
        };
        int j = 0;
        for (; j + kUnroll <= n_it; j += kUnroll) {
            iteration(j, 0);
            iteration(j + 1, 1);
            iteration(j + 2, 2);
            iteration(j + 3, 3);
        }
        if (j < n_it) {          // (leaving the loop in its middle instead costs 1 % on long segments)
            iteration(j, 0);
            if (j + 1 < n_it) {
                iteration(j + 1, 1);
                if (j + 2 < n_it) iteration(j + 2, 2);
            }
        }
    }
    __builtin_amdgcn_s_setprio(2);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // nothing is on its way into LDS any more (behind the next barrier)

    // ---- rows whose probabilities left the 16-bit type's range, or were too small for it: see attn_block
    if (!idle) {
        bool redo = false;
        if (!kChain) {
            l_run[3] += s_late;
            redo = !(s_late <= Range<DT>::kHardLimit);       // (the very last sums have not been looked at)
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            if (!EXACT) delta[n] += kBase;
            if (kChain) {
                l_run[n] = l_acc[n][0];
                redo = redo || !(l_run[n] <= Range<DT>::kHardLimit);
            }
            float low = Range<DT>::kLowLimit;
            if constexpr (DT == COME_F16) low = delta[n] == kNoScore<DT> ? fmaxf(low, Range<DT>::kLowMean * static_cast<float>(n_it * kBlockN)) : low;
            redo = redo || !(l_run[n] >= low);
        }
        if (__any(redo)) *lds_redo = 1;
        pv_mfma(1, (2 * n_it - 1) & (RV - 1));               // the last half-tile
        if (any_pending) {
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o_acc[n][dt] *= o_pending[n];
        }
    }
    __syncthreads();
    const bool again = __builtin_amdgcn_readfirstlane(static_cast<int>(*lds_redo)) != 0;
    if (again) {
        float m_row[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int n = 0; n < 4; ++n) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) o_acc[n][dt] = zero4f;
            l_run[n] = 0.f;
        }
        for (int j = 0; j < n_it; ++j) {
            __syncthreads();                                    // stages 0 and 1 are free again
#pragma unroll
            for (int i = 0; i < kDma; ++i) {
                load_k(first_row(2 * j + my_half, k_rs_b), k_part + my_half * kStageBytes, i);
                load_v(first_row(2 * j + my_half, v_rs_b), v_part + my_half * kStageBytes, i);
            }
            if (wave == 0) {
                const int key = (it.tile_base + j) * kBlockN + lane;
                uint32_t word = 0;
                if (a.bias) word = *reinterpret_cast<const uint32_t *>(b_seg + ((b_mis + 2u * static_cast<uint32_t>(min(key, L - 1))) & ~3u));
                lds_seed[lane] = seed_of(key, word);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (idle) continue;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                score_mfma(0, half, lds_seed, half);
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    float ex[8];
                    float mx = -INFINITY;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float s = s_acc[0][e >> 2][n][e & 3];
                        ex[e] = EXACT ? s * c_scale : s;
                        mx = fmaxf(mx, ex[e]);
                    }
                    mx = fmaxf(max_across_quarters(mx), m_row[n]);
                    const float ref = mx == -INFINITY ? 0.f : mx;          // a row that has seen masked keys only
                    const float down = __builtin_amdgcn_exp2f(m_row[n] - ref);
                    m_row[n] = mx;
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) o_acc[n][dt] *= down;
                    float part = 0.f;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const uint32_t pw = E::pack2_prob(__builtin_amdgcn_exp2f(ex[2 * w] - ref), __builtin_amdgcn_exp2f(ex[2 * w + 1] - ref));
                        p_frag[0][n][w] = pw;
                        part = E::dot2_ones(pw, part);
                    }
                    l_run[n] = l_run[n] * down + sum_across_quarters(part);
                }
                pv_mfma(0, half);
            }
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) delta[n] = m_row[n] == -INFINITY ? 0.f : m_row[n];
        __syncthreads();                                        // the epilogue reuses the stages
    }
    if (idle) return;
    // (counted again: kept through the key loop they are three registers too many)
    const int out_lane = afresh<true>(static_cast<int>(threadIdx.x)) & 63, out_g = out_lane >> 4, out_r = out_lane & 15;

    // ---- epilogue of a split workgroup: unnormalised outputs, reference point and row sum of its key share
    if (piece != nullptr) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int local_row = 64 * wave + 16 * n + out_r;
            if (q0 + local_row < L) {
                float *op = piece + local_row * kHeadDim + 4 * out_g;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) *reinterpret_cast<f32x4 *>(op + 16 * dt) = o_acc[n][dt];
                if (out_g == 0) {
                    piece[kBlockM * kHeadDim + local_row] = delta[n];
                    piece[kBlockM * (kHeadDim + 1) + local_row] = l_run[n];
                }
            }
        }
        return;
    }

    // ---- epilogue: normalise, write O (and LSE) through 4 KiB of LDS a wavefront, as in attn_block
    uint16_t *const slot_base = lds_kv + wave * kHalfElems;
    u32x4 rows[2][4];                                            // rows 8 i + lane / 8 of 32 queries, one chunk each
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int n = 2 * half + x;
            const float l_tot = l_run[n];
            const float inv = 1.0f / l_tot;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const u32x2 w = {E::pack2(o_acc[n][dt][0] * inv, o_acc[n][dt][1] * inv), E::pack2(o_acc[n][dt][2] * inv, o_acc[n][dt][3] * inv)};
                *reinterpret_cast<u32x2 *>(slot_base + (16 * x + out_r) * 64 + (((2 * dt + (out_g >> 1)) ^ (out_r & 7)) << 3) + 4 * (out_g & 1)) = w;
            }
            const int row = qw0 + 16 * n + out_r;
            if (row < L && out_g == 0 && a.lse)
                a.lse[static_cast<int64_t>(head) * a.total + seq_start + row] = (delta[n] + __log2f(l_tot)) * 0.6931471805599453f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) rows[half][i] = *reinterpret_cast<const u32x4 *>(slot_base + 64 * (8 * i) + 8 * out_lane);
    }
    // the chunk this lane finds at position lane % 8 of rows lane / 8 + 8 i
    const int c = (out_lane & 7) ^ ((out_lane >> 3) & 7);
    const int64_t o_rs = a.o_rs;
    uint16_t *op = a.out + (seq_start + qw0 + (out_lane >> 3)) * o_rs + head * a.o_hs + 8 * c;
    const bool out_wide = a.out_wide != 0;
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        const u32x4 v = rows[n >> 2][n & 3];
        if (qw0 + 8 * n + (out_lane >> 3) < L) {
            if (out_wide) {
                *reinterpret_cast<u32x4 *>(op) = v;
            } else {
                *reinterpret_cast<u32x2 *>(op) = u32x2{v[0], v[1]};
                *reinterpret_cast<u32x2 *>(op + 4) = u32x2{v[2], v[3]};
            }
        }
        op += 8 * o_rs;
    }
}

template <int NW, int KS, bool MIXED> struct KernelLds {
    static constexpr int kOwn = Shape<NW, KS, (KS < 4)>::kKvElems, kShort = Shape<NW, 2>::kKvElems;
    static constexpr int kElems = MIXED && kShort > kOwn ? kShort : kOwn;
};

// MIXED (4 wavefronts): a block of at most 128 queries - the last one of a segment, or any where the launch's blocks are
// that small - runs as 2 query tiles x 2 key groups, in half the steps, instead of leaving half of its wavefronts idle.
// T16: blocks of one key group in 16 x 16 tiles.
template <int DT, int NW, int KS, bool EXACT, bool MIXED, bool T16>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_fwd_pipe_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(1024))) uint16_t lds_kv[KernelLds<NW, KS, MIXED>::kElems];
    __shared__ __attribute__((aligned(16))) float lds_seed[2 * NW * kBlockN];
    __shared__ __attribute__((aligned(256))) uint32_t lds_raw[NW * 64];
    __shared__ uint32_t lds_words[2 + NW];                           // two redo words; one per wavefront for the prologue
    __shared__ __attribute__((aligned(16))) int lds_table[MIXED ? 3 * kTable + 4 * kListed : 4];
    Item it;
    bool listed = false;
    if (!locate_block<NW, KS>(a, it, lds_table, listed)) return;
    if constexpr (MIXED) {
        if (min(it.L - it.q0, a.block_m) <= a.short_block) {
            attn_block<DT, NW, 2, EXACT, false>(a, it, lds_kv, lds_seed, lds_raw, lds_words, [](Item &) { return false; });
            return;
        }
    }
    int turn = 0;
    auto next = [&](Item &i) __attribute__((always_inline)) { return MIXED && listed && next_block(i, lds_table, ++turn); };
    if constexpr (T16) attn_block16<DT, NW, EXACT>(a, it, lds_kv, lds_seed, lds_raw, lds_words);
    else attn_block<DT, NW, KS, EXACT, (KS < 4)>(a, it, lds_kv, lds_seed, lds_raw, lds_words, next);
}

// Combines the key shares of the split query blocks: with m* the largest reference point of a row,
// O = sum_i 2^(m_i - m*) O_i / sum_i 2^(m_i - m*) l_i.  One thread per (row, four output elements); a workgroup
// covers 16 rows of a split query block, so the grid is (split query blocks) x block_m / 16 workgroups.
template <int DT>
__global__ __launch_bounds__(256) void attn_combine_kernel(const AttnArgs a, int block_m) {
    using E = Elem<DT>;
    const int groups = block_m / 16;
    const int group = blockIdx.x % groups;
    const int block = blockIdx.x / groups;
    const int tail = block % a.nb_tail;
    const int unit = block / a.nb_tail;
    const int head = unit % a.n_heads;
    const int seq = unit / a.n_heads;
    int seq_start, L;
    segment_of(a, seq, seq_start, L);
    const int mblk = (L + block_m - 1) / block_m - a.nb_tail + tail;
    if (mblk < 0) return;
    const int q0 = mblk * block_m;
    const int64_t piece_floats = static_cast<int64_t>(block_m) * (kHeadDim + kPieceExtra);
    const float *first = a.work + (static_cast<int64_t>(unit) * a.nb_tail + tail) * a.splits * piece_floats;
    {
        const int idx = group * 256 + threadIdx.x;
        const int local_row = idx / (kHeadDim / 4);
        const int c4 = idx % (kHeadDim / 4);
        if (q0 + local_row >= L) return;
        float m_star = -INFINITY;
        for (int i = 0; i < a.splits; ++i) {
            const float *pc = first + i * piece_floats;
            if (pc[block_m * (kHeadDim + 1) + local_row] > 0.f) m_star = fmaxf(m_star, pc[block_m * kHeadDim + local_row]);
        }
        float l_sum = 0.f;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < a.splits; ++i) {
            const float *pc = first + i * piece_floats;
            const float l_i = pc[block_m * (kHeadDim + 1) + local_row];
            if (!(l_i > 0.f)) continue;
            const float w = __builtin_amdgcn_exp2f(pc[block_m * kHeadDim + local_row] - m_star);
            l_sum += w * l_i;
            const f32x4 v = *reinterpret_cast<const f32x4 *>(pc + local_row * kHeadDim + 4 * c4);
            o += v * w;
        }
        const float inv = 1.0f / l_sum;
        u32x2 packed;
        packed[0] = E::pack2(o[0] * inv, o[1] * inv);
        packed[1] = E::pack2(o[2] * inv, o[3] * inv);
        *reinterpret_cast<u32x2 *>(a.out + static_cast<int64_t>(seq_start + q0 + local_row) * a.o_rs + head * a.o_hs + 4 * c4) = packed;
        if (c4 == 0 && a.lse)
            a.lse[static_cast<int64_t>(head) * a.total + seq_start + q0 + local_row] =
                (m_star + __log2f(l_sum)) * 0.6931471805599453f;
    }
}

// How a launch is shaped.
//  - Long segments: 8 wavefronts per workgroup share every staged K / V tile among 512 queries (half the L2 -> LDS
//    traffic), but such a workgroup fills a whole CU, so a partly filled last round of workgroups costs a full round.
//    Without a work buffer it is used for long segments only when the expected number of workgroups nearly
//    fills its last round.  With a work buffer the query blocks of that last round are cut along the keys into `splits`
//    workgroups each, which fill the chip with short pieces instead; a small kernel combines the pieces.
//  - Everything else: one of the three small shapes (small_shape below).
enum SmallShape { kBlocks256 = 0, kBlocks128, kBlocks128Alone, kBlocks128x4 };
struct Plan {
    bool wide = false;
    int nb_tail = 0, splits = 1;
    SmallShape small = kBlocks256;
    int64_t work_bytes = 0;
};

enum class Arithmetic { kHalf, kExact, kFolded };        // fp16; bf16 with the scale in fp32; bf16, folded

// The shape of a launch of short or few segments, from what the host knows of it exactly (rows, segments, heads: the
// choice does not depend on how loose `max_seqlen` is).
//   256 queries, 4 x 1 wavefronts, two workgroups per CU: the least work per query
//   128 queries, 2 x 2 wavefronts, two per CU: half the steps per workgroup, twice the workgroups
//   128 queries, 2 x 2 wavefronts, one per CU, which has the LDS to stage two tiles ahead (bf16)
//   128 queries, 2 x 4 wavefronts, one per CU: a quarter of the steps, 2 us more in front and behind
// Where every 128-query workgroup gets a CU (counted with a block more per segment than the rows fill, the most there can
// be: one too many would be a second round), the last two (fp16: the second and the last).  us, 16 heads, folded, second / third /
// fourth: 480 keys 10.8, 10.6, 11.7; 766 12.9, 12.7, 13.4; 1400 18.1, 17.3, 18.2; 1596 20.4, 19.8, 20.1; 6 heads, third / fourth: 1596
// 18.3, 18.6; 2000 20.7, 20.0; 3200 28.7, 27.3.
// Otherwise by estimated time in us: rounds of workgroups (half a block and a little more per segment than the rows fill) times
// the time of one, from what it takes around the key loop and per step while a CU holds one workgroup and while it holds two.
// Fitted to 518 launches of 1 - 24 segments, equal and ragged, 100 - 4000 rows each, 6 - 16 heads, every shape timed.  Over 113 others
// of 1 - 24 segments of 150 - 4000 rows what is picked takes more than the best of all by 0.6 % (default arithmetic), 0.7 (folded) and 0.5 (fp16); by
// more than 2 % in ten, ten and nine of them.  The worst: 12 heads, 6 x 426 keys 14.6 us instead of 12.9, folded 14.2 and 12.3, fp16 14.9 and
// 13.2; 5 x 515 7 - 8 %; 16 heads, 8 x 237 7 %, 3 and 6; 6 heads, 4 x 3407 6 %, 0 and 8.
// fp16 had an estimate of its own, of whole rounds: 12 heads, 5 segments of 560 - 350 keys 21.5 -> 14.3 us, 3 of 2010 - 1430 50.0 -> 39.1, 8 of
// 1500 93.5 -> 76.9; against it 6 heads, 4 of 2363 - 1181 lose 4 % (40.6 -> 42.2), 7 of 773 - 386 3 %.
// The reference points of fp16 move often where the first keys of a group are the wrong ones for a row (logits of +-8 nats that
// follow the positions): there the third shape, with twice the steps a row of the fourth, lost what it gains otherwise (2 x 798 keys,
// us: ordinary logits 29.2 and 28.4, those 31.0 and 33.1), so it is not used, and the second one for fewer keys than in bf16.  us, second and fourth, 16 heads,
// ordinary logits / those that follow the positions: 766 keys 13.0 and 13.5 / 15.4 and 15.1, 1270 17.7 and 17.3 / 20.5 and 18.8,
// 1300 18.7 and 19.6 / 21.2 and 20.5, 1400 18.7 and 19.3 / 21.3 and 20.9, 1596 20.9 and 21.4 / 23.3 and 22.6, 1790 22.9 and 22.6 / 25.1 and 23.2.
SmallShape small_shape(Arithmetic how, int64_t n_seq, int64_t total, int64_t n_heads) {
    const double n_cu = cu_count(), len = static_cast<double>(total) / static_cast<double>(n_seq), tiles = std::ceil(len / 64.0);
    const double most128 = static_cast<double>(n_heads * (n_seq == 1 ? ceil_div(total, 128) : total / 128 + n_seq));
    if (most128 <= n_cu) {
        if (how == Arithmetic::kHalf) return tiles > 20 ? kBlocks128x4 : kBlocks128;
        return tiles > 28 ? kBlocks128x4 : kBlocks128Alone;
    }
    auto cost = [&](int64_t block, double around, double steps, double alone, double full) {
        const double blocks = n_seq == 1 ? static_cast<double>(ceil_div(total, block))
                                         : static_cast<double>(total) / static_cast<double>(block) + 0.65 * static_cast<double>(n_seq);
        const double wgs = static_cast<double>(n_heads) * blocks, rounds = wgs / (2 * n_cu);
        const double crowded = std::min(1.0, std::max(0.0, (wgs / n_cu - 1.1) / 0.5));
        return (rounds <= 1 ? 1.0 : rounds + (rounds < 4 ? 0.4 : 0.5)) * (around + steps * (alone + (full - alone) * crowded));
    };
    const double c256 = cost(256, 5.5, tiles, how == Arithmetic::kFolded ? 0.80 : how == Arithmetic::kExact ? 0.88 : 0.90, 1.43);
    const double c128 = cost(128, 6.3, tiles / 2 + 0.3, 1.08, 2.35);
    const double c128x4 = std::ceil(most128 / n_cu) * (7.0 + std::ceil(tiles / 4) * 1.7);
    if (c256 <= c128 && c256 <= c128x4) return kBlocks256;
    return c128 <= c128x4 ? kBlocks128 : kBlocks128x4;
}

Plan make_plan(Arithmetic how, int64_t n_seq, int64_t total, int64_t n_heads, int64_t max_seqlen, bool may_split) {
    Plan p;
    const int64_t units = n_seq * n_heads;
    p.small = small_shape(how, n_seq, total, n_heads);
    if (max_seqlen < 4096) return p;
    const int n_cu = cu_count();
    // one segment: exact; several: half a block of padding per segment on average
    const int64_t expected = n_seq == 1 ? n_heads * ceil_div(total, 512) : n_heads * ceil_div(total + n_seq * 256, 512);
    const int64_t rounds = ceil_div(expected, n_cu);
    if (expected * 100 >= rounds * n_cu * 95) {
        p.wide = true;
        return p;
    }
    if (!may_split) return p;
    const int64_t full = expected / n_cu;
    const int64_t tail = expected - full * n_cu;
    if (full == 0 || tail == 0) return p;
    const int64_t nb_tail = ceil_div(tail, units);
    const int64_t tiles = ceil_div(max_seqlen, kBlockN);
    int best = 0;
    double best_cost = 0.6;                          // what the partly filled last round of 256-query workgroups costs
    for (int sp = 2; sp <= 8; ++sp) {
        if (tiles / sp < 16) break;                  // pieces of at least 16 key tiles
        const double cost = static_cast<double>(ceil_div(nb_tail * units * sp, n_cu)) / sp + 0.02 * sp;
        if (cost < best_cost) {
            best_cost = cost;
            best = sp;
        }
    }
    if (best == 0 || nb_tail > ceil_div(max_seqlen, 512)) return p;
    p.wide = true;
    p.nb_tail = static_cast<int>(nb_tail);
    p.splits = best;
    p.work_bytes = units * nb_tail * best * 512 * (kHeadDim + kPieceExtra) * static_cast<int64_t>(sizeof(float));
    return p;
}

}  // namespace
}  // namespace come

using namespace come;

extern "C" int64_t come_attn_queue_bytes(int64_t, int64_t, int64_t) { return 0; }

extern "C" int64_t come_attn_work_bytes(int64_t n_seq, int64_t total, int64_t n_heads, int64_t max_seqlen) {
    if (n_seq <= 0 || total <= 0 || n_heads <= 0 || max_seqlen <= 0) return 0;
    return make_plan(Arithmetic::kFolded, n_seq, total, n_heads, max_seqlen, true).work_bytes;        // (the same for all)
}

// Address of this device's copy of `scratch` (nullptr + error message on failure).  The array's name is only a
// host-side handle: the device address is asked for once per device, with that device current, and kept.
static void *static_work_pointer() {
    constexpr int kMaxDevices = 64;
    static std::mutex lock;
    static void *known[kMaxDevices] = {};
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("come_attn_varlen_fwd_static: no usable current device (%s)", hipGetErrorString(e));
        return nullptr;
    }
    std::lock_guard<std::mutex> guard(lock);
    if (known[dev] == nullptr) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_error("come_attn_varlen_fwd_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            return nullptr;
        }
        known[dev] = p;
    }
    return known[dev];
}

// Shared body of the attention entry points.  static_work: the buffer is the library's own fixed-size array; a launch
// that needs more is an error instead of a launch without the key split.
static int attn_varlen_fwd_impl(const void *q, const void *k, const void *v, int dtype, int64_t q_row_stride,
                                int64_t q_head_stride, int64_t k_row_stride, int64_t k_head_stride,
                                int64_t v_row_stride, int64_t v_head_stride, const int32_t *cu_seqlens,
                                int64_t n_seq, int64_t total, int64_t n_heads, int64_t head_dim,
                                const void *perkey_bias, int64_t max_seqlen, float softmax_scale, void *out,
                                int64_t o_row_stride, int64_t o_head_stride, float *lse, void *work,
                                int64_t work_bytes, bool static_work, int flags, void *stream,
                                const come_q_prologue *qp = nullptr) {
    clear_error();
    COME_REQUIRE((flags & ~(COME_ATTN_FOLD_SCALE | COME_ATTN_WORK_QUEUE | COME_ATTN_BLOCK_REFERENCE)) == 0, COME_ERR_INVALID,
                 "come_attn_varlen_fwd: unknown bits in flags (%d)", flags);
    COME_REQUIRE(dtype == COME_BF16 || dtype == COME_F16, COME_ERR_UNSUPPORTED,
                 "come_attn_varlen_fwd: only fp16 and bf16 are supported");
    COME_REQUIRE(head_dim == 32 || head_dim == kHeadDim || head_dim == 128, COME_ERR_UNSUPPORTED,
                 "come_attn_varlen_fwd: head_dim must be 32, 64 or 128 (got %lld)", (long long)head_dim);
    COME_REQUIRE(n_seq > 0, COME_ERR_INVALID, "come_attn_varlen_fwd: batch size must be positive");
    COME_REQUIRE(total >= 0 && n_heads > 0 && max_seqlen >= 0, COME_ERR_INVALID,
                 "come_attn_varlen_fwd: negative size");
    COME_REQUIRE(total < (1ll << 31) && n_heads < 65536 && n_seq < (1ll << 24), COME_ERR_UNSUPPORTED,
                 "come_attn_varlen_fwd: problem too large");
    COME_REQUIRE(softmax_scale > 0.f && softmax_scale < INFINITY, COME_ERR_INVALID,
                 "come_attn_varlen_fwd: softmax_scale must be positive and finite");
    if (total == 0 || max_seqlen == 0) return COME_OK;
    // offsets inside a segment are 32-bit byte offsets from the segment's first row
    COME_REQUIRE(max_seqlen * (k_row_stride > v_row_stride ? k_row_stride : v_row_stride) * 2 < (1ll << 32),
                 COME_ERR_UNSUPPORTED, "come_attn_varlen_fwd: a segment may span at most 4 GiB of K or V rows");
    COME_REQUIRE(q && k && v && out && cu_seqlens, COME_ERR_INVALID, "come_attn_varlen_fwd: NULL tensor");
    const int64_t strides[8] = {q_row_stride, q_head_stride, k_row_stride, k_head_stride,
                                v_row_stride, v_head_stride, o_row_stride, o_head_stride};
    for (int i = 0; i < 8; ++i)
        COME_REQUIRE(strides[i] >= head_dim || (i % 2 == 1 && n_heads == 1), COME_ERR_INVALID,
                     "come_attn_varlen_fwd: stride %d is smaller than head_dim", i);
    for (int i = 0; i < 6; ++i)
        COME_REQUIRE(strides[i] % 8 == 0, COME_ERR_UNSUPPORTED,
                     "come_attn_varlen_fwd: q/k/v strides must be multiples of 8 elements (16-byte loads)");
    COME_REQUIRE(o_row_stride % 4 == 0 && o_head_stride % 4 == 0, COME_ERR_UNSUPPORTED,
                 "come_attn_varlen_fwd: out strides must be multiples of 4 elements");
    COME_REQUIRE((reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(k) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(v) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
                 COME_ERR_UNSUPPORTED, "come_attn_varlen_fwd: q/k/v must be 16-byte aligned, out 8-byte aligned");

    if (qp != nullptr) {
        COME_REQUIRE(head_dim == kHeadDim, COME_ERR_UNSUPPORTED, "come_attn_varlen_fwd_qp: head_dim must be 64");
        COME_REQUIRE((flags & COME_ATTN_WORK_QUEUE) == 0, COME_ERR_UNSUPPORTED,
                     "come_attn_varlen_fwd_qp: not available together with COME_ATTN_WORK_QUEUE");
        COME_REQUIRE(qp->eps >= 0.f, COME_ERR_INVALID, "come_attn_varlen_fwd_qp: eps must be >= 0");
        const void *aligned[] = {qp->weight, qp->bias, qp->cos_table, qp->sin_table};
        for (const void *p : aligned)
            COME_REQUIRE((reinterpret_cast<uintptr_t>(p) & 15) == 0, COME_ERR_INVALID,
                         "come_attn_varlen_fwd_qp: prologue pointers must be 16-byte aligned");
        if (qp->positions != nullptr)
            COME_REQUIRE(qp->cos_table != nullptr && qp->sin_table != nullptr && qp->n_pos > 0 && qp->n_pos < (1 << 24),
                         COME_ERR_INVALID, "come_attn_varlen_fwd_qp: positions need cos / sin tables with 0 < n_pos < 2^24");
    }
    if (head_dim != kHeadDim) {               // the other widths: one kernel, no work buffer
        AttnArgs a{};
        a.q = static_cast<const uint16_t *>(q);
        a.k = static_cast<const uint16_t *>(k);
        a.v = static_cast<const uint16_t *>(v);
        a.bias = static_cast<const uint16_t *>(perkey_bias);
        a.out = static_cast<uint16_t *>(out);
        a.lse = lse;
        a.cu = cu_seqlens;
        a.q_rs = q_row_stride; a.q_hs = q_head_stride;
        a.k_rs = k_row_stride; a.k_hs = k_head_stride;
        a.v_rs = v_row_stride; a.v_hs = v_head_stride;
        a.o_rs = o_row_stride; a.o_hs = o_head_stride;
        a.total = total;
        a.n_heads = static_cast<int>(n_heads);
        a.n_units = static_cast<int>(n_seq * n_heads);
        a.scale_log2 = softmax_scale * 1.4426950408889634f;
        a.splits = 1;
        return launch_attn_hd(a, dtype, static_cast<int>(head_dim), max_seqlen, static_cast<hipStream_t>(stream));
    }
    // fp16 has one arithmetic: the default one (its range asks for reference points per row, which cost nothing there)
    const bool exact = (flags & COME_ATTN_FOLD_SCALE) == 0 || dtype == COME_F16;
    const Arithmetic how = dtype == COME_F16 ? Arithmetic::kHalf : exact ? Arithmetic::kExact : Arithmetic::kFolded;
    Plan plan = make_plan(how, n_seq, total, n_heads, max_seqlen, work != nullptr || static_work);
    if (static_work && plan.splits > 1) {
        COME_REQUIRE(plan.work_bytes <= kStaticWorkBytes, COME_ERR_UNSUPPORTED,
                     "come_attn_varlen_fwd_static: this launch needs a work buffer of %lld bytes, the built-in one "
                     "holds %lld; use come_attn_varlen_fwd_ws with a buffer of come_attn_work_bytes() bytes",
                     (long long)plan.work_bytes, (long long)kStaticWorkBytes);
        work = static_work_pointer();
        if (work == nullptr) return COME_ERR_HIP;
        work_bytes = kStaticWorkBytes;
    }
    if (plan.splits > 1 && (work_bytes < plan.work_bytes || (reinterpret_cast<uintptr_t>(work) & 15) != 0))
        plan = make_plan(how, n_seq, total, n_heads, max_seqlen, false);             // buffer too small or misaligned: no split
    // one reference point per query block of one key group: the shapes with several groups are out
    const bool block_ref = (flags & COME_ATTN_BLOCK_REFERENCE) != 0 && (flags & COME_ATTN_FOLD_SCALE) != 0 && dtype == COME_BF16;
    if (block_ref) plan.small = kBlocks256;
    const bool wide = plan.wide;
    const int kBlockM = wide ? 512 : plan.small == kBlocks256 ? 256 : 128;
    AttnArgs a{};
    a.q = static_cast<const uint16_t *>(q);
    a.k = static_cast<const uint16_t *>(k);
    a.v = static_cast<const uint16_t *>(v);
    a.bias = static_cast<const uint16_t *>(perkey_bias);
    a.out = static_cast<uint16_t *>(out);
    a.lse = lse;
    a.cu = cu_seqlens;
    a.q_rs = q_row_stride; a.q_hs = q_head_stride;
    a.k_rs = k_row_stride; a.k_hs = k_head_stride;
    a.v_rs = v_row_stride; a.v_hs = v_head_stride;
    a.o_rs = o_row_stride; a.o_hs = o_head_stride;
    a.total = total;
    a.n_heads = static_cast<int>(n_heads);
    a.n_mblocks = static_cast<int>(ceil_div(max_seqlen, kBlockM));
    a.scale_log2 = softmax_scale * 1.4426950408889634f;
    a.n_units = static_cast<int>(n_seq * n_heads);
    a.n_seq = static_cast<int>(n_seq);
    a.rotate = (!wide && a.n_mblocks % 2 == 0) ? 1 : 0;
    a.out_wide = (o_row_stride % 8 == 0 && o_head_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) ? 1 : 0;
    a.nb_tail = plan.nb_tail;
    a.splits = plan.splits;
    a.work = static_cast<float *>(work);
    a.block_m = kBlockM;
    // the compact grid: every wavefront counts all segments, so not too many of them
    a.compact = n_seq <= 64 * kCompactChunks ? 1 : 0;
    a.short_block = block_ref || wide ? 0 : 128;
    a.block_ref = block_ref ? 1 : 0;
    if (qp != nullptr && (qp->apply_norm || qp->positions != nullptr)) {
        a.qp_on = 1;
        a.qp_norm = qp->apply_norm ? 1 : 0;
        a.qp_gamma = qp->weight;
        a.qp_beta = qp->bias;
        a.qp_eps = qp->eps;
        a.qp_pos = qp->positions;
        a.qp_cos = qp->cos_table;
        a.qp_sin = qp->sin_table;
        a.qp_n_pos = qp->n_pos;
    }
    // Chained blocks: what a block spends in front of and behind its key loop (7 - 8 us, two thirds of it waiting) is hidden
    // for all but the first of a workgroup.  Of short segments, where that is a fifth to a half of a block's time; with long
    // ones of different lengths a fixed share of the blocks costs more than it hides (four segments of 6000 - 3000 tokens,
    // 12 heads: 283 -> 299 us).  Not for fp16, whose key loop has no registers to spare (40 segments: 157 -> 159 us).
    a.chained = a.compact && !wide && plan.small == kBlocks256 && dtype == COME_BF16 && total <= 2048 * n_seq ? std::max(1, 2 * cu_count() / 8) : 0;
    if (n_heads * (total / kBlockM + n_seq) > kListed * 8 * static_cast<int64_t>(a.chained)) a.chained = 0;
    // compact: two lists, each dealt to eight XCDs in equal shares
    a.n_full_wg = a.compact ? 8 * (ceil_div(n_heads * (total / kBlockM + n_seq), 8) + 1) : ceil_div(n_seq * n_heads, 8) * 8 * a.n_mblocks;
    if (a.chained > 0) a.n_full_wg = std::min(a.n_full_wg, 8 * (a.chained + ceil_div(n_heads * n_seq, 8)));          // (at most one short block a segment)
    // Few segments: each dealt to the XCDs in equal shares.  (A list that is longer than the workgroups that chain its blocks is left to
    // those.)
    a.few = n_seq <= kFewSegments && (a.chained == 0 || n_heads * (total / kBlockM + n_seq) <= 8 * static_cast<int64_t>(a.chained)) ? 1 : 0;
    if (a.few) a.compact = 1, a.chained = 0;
    const int64_t n_split = n_seq * n_heads * (plan.splits > 1 ? plan.nb_tail * plan.splits : 0);
    int64_t n_wg = a.n_full_wg + (a.compact ? ceil_div(n_split, 8) * 8 : ceil_div(n_seq * n_heads, 8) * 8 * (n_split / (n_seq * n_heads)));
    if (a.few) n_wg = 8 * ceil_div(n_heads * (total / kBlockM + n_seq) + n_split, 8);         // (shares differ by one)
    const int64_t n_cwg = n_seq * n_heads * plan.nb_tail * (kBlockM / 16);       // combine kernel: 16 rows each
    COME_REQUIRE(n_wg < (1ll << 31) && n_cwg < (1ll << 31), COME_ERR_UNSUPPORTED,
                 "come_attn_varlen_fwd: grid too large");
    const dim3 grid(static_cast<unsigned>(n_wg));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 block(wide || plan.small == kBlocks128x4 ? 512 : 256);
    // 4 x 1 in 16 x 16 tiles: where every CU has two workgroups at a time, whose wavefronts hide each other's matrix instructions, and
    // none chains blocks.  us, 16 heads, folded / default / fp16: 6 x 2500 keys 139.4 -> 136.1, 154.7 -> 149.8, 164.4 -> 157.9; 32 x 798, fp16
    // 111.6 -> 108.7; 12 heads, 4500 - 3000 keys 172.9 -> 164.6, 184.3 -> 181.4.  With fewer: one of 3000 keys 44.0 -> 46.3, 49.8 -> 51.0;
    // 6 heads, 7000 and 5000 keys 150.2 -> 157.9, 171.0 -> 178.0.
    const bool tiles16 = plan.small == kBlocks256 && !block_ref && a.chained == 0 && n_heads * (total / 256 + n_seq / 2) >= 2 * cu_count();
#define COME_ATTN_LAUNCH(NW_, KS_, MIXED_, T16_)                                                                       \
    do {                                                                                                               \
        if (dtype == COME_F16) hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_F16, NW_, KS_, true, MIXED_, T16_>), grid, block, 0, s, a); \
        else if (exact) hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_BF16, NW_, KS_, true, MIXED_, T16_>), grid, block, 0, s, a);       \
        else hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_BF16, NW_, KS_, false, MIXED_, T16_>), grid, block, 0, s, a);     \
    } while (0)
    if (block_ref && wide) hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_BF16, 8, 1, false, false, false>), grid, block, 0, s, a);
    else if (wide) COME_ATTN_LAUNCH(8, 1, false, true);
    else if (plan.small == kBlocks128x4) COME_ATTN_LAUNCH(8, 4, false, false);
    else if (plan.small == kBlocks128Alone && exact) hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_BF16, 4, 2, true, false, false>), grid, block, 0, s, a);
    else if (plan.small == kBlocks128Alone) hipLaunchKernelGGL((attn_fwd_pipe_kernel<COME_BF16, 4, 2, false, false, false>), grid, block, 0, s, a);
    else if (tiles16) COME_ATTN_LAUNCH(4, 1, true, true);
    else COME_ATTN_LAUNCH(4, 1, true, false);
#undef COME_ATTN_LAUNCH
    COME_CHECK_LAUNCH("come_attn_varlen_fwd");
    if (plan.splits > 1) {
        static_assert(kHeadDim / 4 == 16, "a workgroup of the combine kernel covers 16 rows of 16 four-element chunks");
        const dim3 cgrid(static_cast<unsigned>(n_cwg));
        if (dtype == COME_BF16) hipLaunchKernelGGL(attn_combine_kernel<COME_BF16>, cgrid, dim3(256), 0, s, a, kBlockM);
        else hipLaunchKernelGGL(attn_combine_kernel<COME_F16>, cgrid, dim3(256), 0, s, a, kBlockM);
        COME_CHECK_LAUNCH("come_attn_varlen_fwd (combine)");
    }
    return COME_OK;
}

extern "C" int come_attn_varlen_fwd_ws(const void *q, const void *k, const void *v, int dtype, int64_t q_row_stride,
                                       int64_t q_head_stride, int64_t k_row_stride, int64_t k_head_stride,
                                       int64_t v_row_stride, int64_t v_head_stride, const int32_t *cu_seqlens,
                                       int64_t n_seq, int64_t total, int64_t n_heads, int64_t head_dim,
                                       const void *perkey_bias, int64_t max_seqlen, float softmax_scale, void *out,
                                       int64_t o_row_stride, int64_t o_head_stride, float *lse, void *work,
                                       int64_t work_bytes, int flags, void *stream) {
    return attn_varlen_fwd_impl(q, k, v, dtype, q_row_stride, q_head_stride, k_row_stride, k_head_stride,
                                v_row_stride, v_head_stride, cu_seqlens, n_seq, total, n_heads, head_dim,
                                perkey_bias, max_seqlen, softmax_scale, out, o_row_stride, o_head_stride, lse,
                                work, work_bytes, false, flags, stream);
}

extern "C" int come_attn_varlen_fwd_qp(const void *q, const void *k, const void *v, int dtype, int64_t q_row_stride,
                                       int64_t q_head_stride, int64_t k_row_stride, int64_t k_head_stride,
                                       int64_t v_row_stride, int64_t v_head_stride, const int32_t *cu_seqlens,
                                       int64_t n_seq, int64_t total, int64_t n_heads, int64_t head_dim,
                                       const void *perkey_bias, int64_t max_seqlen, float softmax_scale, void *out,
                                       int64_t o_row_stride, int64_t o_head_stride, float *lse, void *work,
                                       int64_t work_bytes, const come_q_prologue *prologue, int flags, void *stream) {
    return attn_varlen_fwd_impl(q, k, v, dtype, q_row_stride, q_head_stride, k_row_stride, k_head_stride,
                                v_row_stride, v_head_stride, cu_seqlens, n_seq, total, n_heads, head_dim,
                                perkey_bias, max_seqlen, softmax_scale, out, o_row_stride, o_head_stride, lse,
                                work, work_bytes, false, flags, stream, prologue);
}

extern "C" int come_attn_varlen_fwd(const void *q, const void *k, const void *v, int dtype, int64_t q_row_stride,
                                    int64_t q_head_stride, int64_t k_row_stride, int64_t k_head_stride,
                                    int64_t v_row_stride, int64_t v_head_stride, const int32_t *cu_seqlens,
                                    int64_t n_seq, int64_t total, int64_t n_heads, int64_t head_dim,
                                    const void *perkey_bias, int64_t max_seqlen, float softmax_scale, void *out,
                                    int64_t o_row_stride, int64_t o_head_stride, float *lse, int flags,
                                    void *stream) {
    return attn_varlen_fwd_impl(q, k, v, dtype, q_row_stride, q_head_stride, k_row_stride, k_head_stride,
                                v_row_stride, v_head_stride, cu_seqlens, n_seq, total, n_heads, head_dim,
                                perkey_bias, max_seqlen, softmax_scale, out, o_row_stride, o_head_stride, lse,
                                nullptr, 0, false, flags, stream);
}

// Also takes the address of the current device's copy of the array, so that a caller who asks for the size before
// its first launch (as a capturing caller has to, outside the capture) leaves nothing but kernel launches to the
// entry point itself.  Returns -1 when that fails (come_last_error() says why).
extern "C" int64_t come_attn_static_work_bytes(void) {
    clear_error();
    return static_work_pointer() != nullptr ? kStaticWorkBytes : -1;
}

extern "C" int come_attn_varlen_fwd_static(const void *q, const void *k, const void *v, int dtype,
                                           int64_t q_row_stride, int64_t q_head_stride, int64_t k_row_stride,
                                           int64_t k_head_stride, int64_t v_row_stride, int64_t v_head_stride,
                                           const int32_t *cu_seqlens, int64_t n_seq, int64_t total, int64_t n_heads,
                                           int64_t head_dim, const void *perkey_bias, int64_t max_seqlen,
                                           float softmax_scale, void *out, int64_t o_row_stride,
                                           int64_t o_head_stride, float *lse, int flags, void *stream) {
    return attn_varlen_fwd_impl(q, k, v, dtype, q_row_stride, q_head_stride, k_row_stride, k_head_stride,
                                v_row_stride, v_head_stride, cu_seqlens, n_seq, total, n_heads, head_dim,
                                perkey_bias, max_seqlen, softmax_scale, out, o_row_stride, o_head_stride, lse,
                                nullptr, 0, true, flags, stream);
}
