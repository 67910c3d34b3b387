// fa_api.hip - the extern "C" entry points declared in include/fa.h.
//
// Argument checking mirrors the reference's host wrappers
// (attention/fused/fused.py:69-71, attention/gqa/fused_gqa.py:71-77,
// attention/backward/fused_backward.py:151-158); the Python layer raises the
// reference's exception types before it ever reaches this ABI, so these
// checks are the last line of defence for C callers.
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <iterator>
#include <mutex>

#include "fa_launch.h"

namespace {

constexpr int kMaxGroupHeadsPerWg = 4;

bool tile_ok(int t) { return t == 64 || t == 128; }

fa::FwdFn fwd_table(int dtype, int D, int bm, int bn, int gh, int lse) {
  if (dtype == FA_F16) {
    if (D == 32) return fa_fwd_table_f16_32(bm, bn, gh, lse);
    if (D == 64) return fa_fwd_table_f16_64(bm, bn, gh, lse);
    if (D == 128) return fa_fwd_table_f16_128(bm, bn, gh, lse);
  } else if (dtype == FA_BF16) {
    if (D == 32) return fa_fwd_table_bf16_32(bm, bn, gh, lse);
    if (D == 64) return fa_fwd_table_bf16_64(bm, bn, gh, lse);
    if (D == 128) return fa_fwd_table_bf16_128(bm, bn, gh, lse);
  }
  return nullptr;
}

fa::BwdFn bwd_table(int dtype, int D, int bm, int bn) {
  if (dtype == FA_F16) {
    if (D == 32) return fa_bwd_table_f16_32(bm, bn);
    if (D == 64) return fa_bwd_table_f16_64(bm, bn);
    if (D == 128) return fa_bwd_table_f16_128(bm, bn);
  } else if (dtype == FA_BF16) {
    if (D == 32) return fa_bwd_table_bf16_32(bm, bn);
    if (D == 64) return fa_bwd_table_bf16_64(bm, bn);
    if (D == 128) return fa_bwd_table_bf16_128(bm, bn);
  }
  return nullptr;
}

// Query heads per workgroup for a GQA group: as many heads of one K/V group
// as fit in 8 waves (512 threads), each head taking block_m/32 waves.  With
// 128-key tiles a wave holds two 128-key score tiles in flight and needs more
// than the 256 VGPRs of two waves per SIMD, so the workgroup stays at 4 waves
// (no rule takes them any more: fa_fwd; the exact entries and fa_supported do).
// Counters (profiles/tile_study_mha_gqa_bwd.md, GQA B=2 H=32 H_kv=8 S=8192 D=128):
// one head of 64 rows 898 TFLOP/s, MFMA busy 48.2 %; two heads 1185 / 71.4 %; four
// heads 1236 / 68.4 %.
int heads_per_wg(int group, int block_m, int block_n) {
  int cap = (block_n == 128 ? 128 : 256) / block_m;  // waves / (block_m / 32)
  if (cap > kMaxGroupHeadsPerWg) cap = kMaxGroupHeadsPerWg;
  int gh = 1;
  while (gh * 2 <= cap && group % (gh * 2) == 0) gh *= 2;
  return gh;
}

int check_common(int B, int H, int S, int D, int dtype, int block_m, int block_n) {
  if (B <= 0 || H <= 0 || S <= 0) return FA_ERR_DIMS;
  if (dtype != FA_F16 && dtype != FA_BF16) return FA_ERR_DTYPE;
  if (D != 32 && D != 64 && D != 128) return FA_ERR_HEADDIM;
  if (!tile_ok(block_m) || !tile_ok(block_n)) return FA_ERR_TILE;  // any S >= 1: partial edge tiles
  // element offsets inside one tensor are formed in 32-bit for the per-row
  // parts and 64-bit for the (batch, head) base; keep the whole tensor
  // addressable with 32-bit row indices
  if ((long long)B * H * S > 0x7fffffffLL) return FA_ERR_DIMS;
  // the kernels form byte offsets inside one (batch, head) slice, and the byte
  // size of a slice's remaining rows, in 32-bit int: keep S * D * 2 below 2^31
  if ((long long)S * D * 2 > 0x7fffffffLL) return FA_ERR_DIMS;
  return FA_OK;
}

using fa::cu_count;
using fa::kMaxDevices;

// The rows per head that the heads are chosen for: up to three 64-row workgroups per CU a
// 128-row tile counts as 64, or a group's two heads of 128 rows would make half as many workgroups
// of twice the chain (bitwise equal; us of 128 / 64 rows, two heads each, groups of 4: D = 128 128 heads S=100 8.7 /
// 6.5, 128 heads S=256 12.9 / 9.8, 96 heads S=512 18.8 / 19.1; D = 64 256 heads S=64 4.9 / 4.6, 128 heads S=256 9.3 /
// 6.7, 76 heads S=640 14.9 / 11.0; D = 32 48 heads S=1024 15.8 / 14.2).
int fwd_tile_m(int B, int H, int S, int block_m) {
  return (long long)B * H * ((S + 63) / 64) <= 3LL * cu_count() ? 64 : block_m;
}

// Forward query heads per workgroup for this launch: heads_per_wg's choice, but four
// heads (64-row tiles) drop to two where the grid would leave the co-resident pair of
// workgroups per CU short: below two workgroups per CU, and at D = 32 below four, where
// the heavy-first order cannot balance the causal triangle with the fewer, longer
// workgroups.  Two heads of 64 rows still hold two waves per SIMD.  Measured
// (profiles/tile_study_mha_gqa_bwd.md, TFLOP/s of two / four heads): B=1 H=16 H_kv=4
// S=4096 D=128 (one workgroup per CU at four heads) 864 / 754; B=2 H=8 H_kv=1 S=8192 fp16
// (two per CU) D=128 1045 / 1134, D=64 899 / 915, D=32 650 / 602; the study's run before
// it read the same order (D=128 990 / 1053, D=64 868 / 897, D=32 662 / 629).
// A 128-row tile with 64 keys runs as 64-row workgroups of four heads wherever the
// 64-row tile would take four: each K/V tile is then staged for four heads instead of
// two, and every 32-row wave computes the same either way (results bitwise equal).
// Interleaved timings, two heads of 128 rows against four of 64: GQA B=2 H=32 H_kv=8
// S=8192 D=128 +0.8 %, B=1 H=32 H_kv=4 S=8192 +0.9 %, B=2 H=32 H_kv=8 S=4096 +1.5 %,
// MQA B=1 H=32 S=16384 D=64 fp16 +0.3 %, B=2 H=32 H_kv=8 S=8192 D=64 fp16 +0.7 %.
int fwd_heads_per_wg(int B, int H, int group, int S, int D, int block_m, int block_n) {
  auto four_fit = [&](int bm) {
    return (long long)B * (H / 4) * ((S + bm - 1) / bm) >= (D <= 32 ? 4LL : 2LL) * cu_count();
  };
  if (block_m == 128 && block_n == 64 && heads_per_wg(group, 64, 64) == 4 && four_fit(64)) return 4;
  int gh = heads_per_wg(group, block_m, block_n);
  if (gh == 4 && !four_fit(block_m)) gh = 2;
  return gh;
}

// tile_m only sets how many 32-row waves share a workgroup: each 32-row group runs
// the same arithmetic over the same key tiles either way, so results do not depend
// on it (bitwise).  A single-head workgroup of 64 rows holds two waves, and with
// its K and V tiles double-buffered in LDS it gets one wave per SIMD or less;
// where that is measured slower, tile_m = 64 runs as 128-row workgroups.
// Forward, MHA B=4 H=32 S=4096 bf16, TFLOP/s of tile 64 -> 128 rows
// (profiles/tile_study_mha_gqa_bwd.md): tile_n = 64: D=128 845 -> 1106 (MFMA busy
// 43.9 -> 66.8 %: a 64-row workgroup holds one wave per SIMD), D=64 649 -> 922, D=32
// 441 -> 675; tile_n = 128: D=128 464 -> 775, D=64 631 -> 654, D=32 447 -> 461 (the
// D <= 64 forward at 128 keys +1.7-3.6 % at six shapes of A/B runs, -0.3 % at
// B=4 H=32 D=32 bf16; four runs of the study read 128 rows 2-5 % faster).  dQ, every
// head dim: 64 -> 128 rows at D=128 870 -> 1144 (MFMA busy 42.4 -> 62.2 %), at D=64
// 973 -> 1003 with 64-key tiles and 681 -> 1019 with 128-key tiles, at D=32 739 -> 794
// (the D = 32 backward +0.9-2.3 % at four shapes in A/B runs, -0.3 % at B=2 H=16 S=4096).
int fwd_block_m(int block_m, int /*block_n*/, int /*D*/, int gh) {
  if (gh == 4) return 64;  // four heads run 64-row tiles (fwd_heads_per_wg)
  return (block_m == 64 && gh == 1) ? 128 : block_m;
}
// Short sequences at D <= 64: one-head forward workgroups and dQ workgroups of 64 rows (two waves)
// in place of 128.  With so few key tiles a workgroup is mostly start, diagonal and tail: smaller ones
// overlap them better, and half as many rows past S and masked tiles are computed (most where
// ceil(S / 64) is odd).  They stage K and V twice as often, though.  Past three tiles that pays only
// where the heads are a multiple of 8, so that each XCD finds its own heads' keys in its L2 and
// no other's; past seven (D = 32: eight) also only where the 128-row workgroups are more
// than two and a half per CU, below which they start all at once or nearly (four and a half at D = 64
// with an even number of tiles, whose last 128-row workgroups are full).
// Measured, us of 128 / 64 rows (bitwise equal):
//   forward D = 32: B=16 H=32 S=200 12.7 / 11.4, S=512 28.4 / 25.8, S=576 36.1 / 30.2, S=700 46.4 / 39.5;
//   B=8 H=16 S=1024 20.9 / 22.2; B=3 H=16 S=1500 17.0 / 19.4
//   forward D = 64: B=16 H=32 S=384 26.3 / 25.1, S=576 48.3 / 42.8, S=700 65.0 / 58.4; B=8 H=16 S=1024 28.3 /
//   30.9; B=3 H=16 S=1500 23.8 / 27.2; up to two 64-row workgroups per CU 128 rows stay (B=8 H=16
//   S=256 7.2 / 7.6, D = 32 5.9 / 6.1); 258 heads S=192 11.7 / 11.1, but past it, no multiple of 8: 133
//   heads S=384 10.3 / 12.8, 341 heads S=768 48.7 / 71.4, 585 heads S=896 97.3 / 157.5; and few 128-row
//   workgroups: 72 heads S=768 14.0 / 15.5, 96 heads S=705 14.5 / 16.3, 256 heads S=512 21.1 / 21.9
//   backward (dQ at 64 rows) D = 32 / 64: B=16 H=32 S=256 33.1 / 32.1, 52.7 / 51.5; B=16 H=32 S=576 87.2 / 82.3,
//   139 / 132; B=8 H=16 S=700 42.6 / 39.5, 64.9 / 60.0; 341 heads S=768 91.5 / 97.1, 141 / 163; 72 heads S=768
//   D = 32 26.5 / 28.3; B=8 H=16 S=1100 71.8 / 73.4, 106 / 107
bool short_rows(int B, int H, int S, int D) {
  if (D > 64 || S <= 192) return D <= 64;
  const long long heads = (long long)B * H;
  if (heads % 8 != 0 || S > 960) return false;
  const bool full = D == 64 && (S + 63) / 64 % 2 == 0;
  return S <= (D == 32 ? 512 : 448) || 2 * heads * ((S + 127) / 128) > (full ? 9LL : 5LL) * cu_count();
}
// Forward instance of a call.  Below a grid that fills the GPU the keys of a tile are split
// over groups of waves (fwd_kernel's KS): the call then waits for the serial chain of the
// last rows, and every other CU, or SIMD of a CU, idles.  By the number W of 64-row
// workgroups, which depends on neither tile_m nor H_kv (results still depend on neither):
//   W <= one per CU:  D <= 64: 32 rows x 4 groups over 128-key tiles; D = 128, whose 128-key
//     tiles allow one workgroup per CU: 64 rows x 4 groups
//   W <= three per CU: 64 rows x 2 groups over 64-key tiles (D = 128 at S >= 4096 and W <= two per
//     CU: 64 x 4 again)
// A chain must be long enough to pay for the merge and for workgroups of half the rows, which
// stage K and V twice as often; the more workgroups, the longer.  Where the heads are no multiple
// of 8 the XCDs share them, each staging every shared head's keys through its own L2, which the
// extra staging pays for again: at an odd number of heads each of the 8 streams all.
// Measured, us of unsplit / 64 x 2 / 64 x 4 / 32 x 4:
//   D = 64:  B=2 H=8 S=512 (W = 128) 8.6 / 6.6 / 6.9 / 5.8; B=8 H=1 S=1755 (224) 18.7 / 13.4 / 11.8 /
//   10.8; B=1 H=2 S=8192 (256) 68.8 / 48.3 / 36.9 / 34.5; B=2 H=8 S=2048 (512) 21.5 / 16.2 / 17.8 / 19.0;
//   B=2 H=16 S=1024 (512) 13.2 / 9.9 / 13.4 / 13.3
//   D = 128: B=3 H=5 S=1000 (240) 17.6 / 15.0 / 15.1 / 17.8; B=1 H=1 S=16384 (256) 201 / 153 / 120 / 119;
//   B=2 H=8 S=2048 (512) 31.2 / 28.1 / 28.0 / 43.7; B=1 H=8 S=4096 (512) 56.2 / 49.7 / 44.3 / 68.0;
//   GQA B=1 H=32 H_kv=8 S=1531 (768) 30.1 / 27.9 / 36.0 / 55.6; B=2 H=16 S=2048 (1024) 41.9 / 44.1 / 54 / 88
// and the lengths from which the split pays, us of unsplit / split (heads of all batches, W; graph
// replays, without the launches; at about 4000 sizes, groups of 1 to 32, the split calls lie between
// 0.29 and 1.03 of the unsplit ones, mean 0.81):
//   W <= half the CUs: D = 64 S=64, 128 heads 4.20 / 4.41, S=100, 64 heads 5.21 / 4.46
//   W <= one per CU: D = 64 S=64, 256 heads 4.39 / 5.33, GQA S=100, 128 heads 4.96 / 5.33, S=256, 64 heads 0.82 of it;
//   D = 128: S=64, 128 heads 5.27 / 7.07, S=128, 128 heads 6.89 / 7.59, S=320 1.07, S=384, 42 heads 10.47 / 10.29
//   W <= two: D = 64 S=512, 64 heads 9.66 / 7.56; D = 128 S=640, 48 heads 14.7 / 12.8, 51 heads 15.9 / 16.6,
//   S=1024, 31 heads 20.3 / 20.9, S=1100, 25 heads 0.88
//   W <= two and a quarter: D = 64 S=577, 56 heads 0.82 of it, GQA S=513, 62 heads 1.03; D = 128 S=640, 56
//   heads 0.87, S=576, 60 heads 0.95, S=833, 41 heads 1.13
//   W <= two and a half: D = 64 S=640, GQA, 64 heads 10.1 / 10.9, S=896, 45 heads 15.0 / 13.7; D = 128 S=833, 45
//   heads 20.9 / 24.2, S=1280, 32 heads 26.6 / 22.9, 31 heads 26.2 / 28.1
//   W <= three: GQA D = 64 S=640, 76 heads 10.6 / 12.5, S=1024, 48 heads 18.6 / 14.7, 44 heads 14.7 / 15.1, S=1531, 31
//   heads 21.2 / 19.0; D = 128 S=1024, 48 heads 27.3 / 22.8, 46 heads 24.8 / 26.3, S=1531, 31 heads 32.2 / 36.4
struct FwdShape {
  int block_m, block_n, gh;   // gh = -KS: key groups
};
constexpr int kNever = 0x7fffffff;
struct KeySplitBand {
  int quarters;             // up to this many quarters of a 64-row workgroup per CU
  int narrow[2], wide[4];   // the longest S not split: D <= 64, heads any / a multiple of 8;
                            // D = 128, heads odd / even / a multiple of 4 / of 8
};
constexpr KeySplitBand kKeySplit[] = {
    {2, {64, 64}, {320, 320, 320, 320}},      {4, {128, 128}, {320, 320, 320, 320}},
    {6, {511, 511}, {704, 511, 511, 511}},    {8, {511, 511}, {1024, 768, 511, 511}},
    {9, {576, 576}, {1400, 768, 640, 640}},   {10, {832, 768}, {1400, 832, 832, 768}},
    {12, {1280, 832}, {kNever, 1280, 1280, 832}},
};
bool fwd_key_split(int B, int H, int S, int D, FwdShape* out) {
  const long long heads = (long long)B * H, w = heads * ((S + 63) / 64), cus = cu_count();
  const int pow2 = heads % 8 == 0 ? 3 : heads % 4 == 0 ? 2 : heads % 2 == 0 ? 1 : 0;
  const KeySplitBand* band = kKeySplit;
  while (4 * w > band->quarters * cus)
    if (++band == std::end(kKeySplit)) return false;
  if (S <= (D == 128 ? band->wide[pow2] : band->narrow[pow2 == 3])) return false;
  const bool four = w <= cus || (D == 128 && S >= 4096 && w <= 2 * cus);
  if (out) *out = !four ? FwdShape{64, 64, -2} : D == 128 ? FwdShape{64, 128, -4} : FwdShape{32, 128, -4};
  return true;
}

int dq_block_m(int block_m, int /*D*/) { return block_m == 64 ? 128 : block_m; }
// Keys per dQ tile (bitwise the same either way): at D = 128 a 128-key tile leaves one wave per
// SIMD (backward, us of 128 / 64 keys: B=4 H=32 S=2048 579 / 520, B=2 H=16 H_kv=4 S=4096 499 / 470);
// at D <= 64 both hold two, and 128 keys are 0-2 % faster.
int dq_block_n(int block_n, int D) { return D == 128 ? 64 : block_n; }
fa::BwdFn bwd_fn(int dtype, int D, int B, int H, int S, int block_m, int block_n) {
  if (short_rows(B, H, S, D)) return bwd_table(dtype, D, 64, 64);
  return bwd_table(dtype, D, dq_block_m(block_m, D), dq_block_n(block_n, D));
}

// Work items (key-tile chunks) the dK/dV kernel should have for its heavy-first order
// to balance: two per workgroup slot the GPU holds at once, and one round more per
// 8192 keys beyond, since the heaviest key tile's pairs grow with S while the average
// does not keep up (a split costs an fp32 partial write, read and reduction, so it is
// kept to what load balance needs).  Slots: the paired D = 128 kernel runs one
// persistent workgroup per CU that walks its items; the one-wave kernel (D <= 64) two
// workgroups per CU, one per item.  Measured (profiles/dkdv_split_study.md, dK/dV +
// reduction, us, the rule's choice first):
//   paired: MQA B=1 H=32 S=4096 D=128, 16 / 8 / 32: 253 / 377 / 280; MHA B=1 H=4 S=8192,
//   2 / 1 / 4: 140 / 197 / 160; MHA B=1 H=8 S=4096, 2 / 1 / 4: 84 / 95 / 105; GQA B=1 H=32
//   H_kv=4 S=8192, 2 / 1 / 4: 913 / 1427 / 937; B=1 H=8 H_kv=1 S=16384, 8 / 4 / 16: 920 /
//   1170 / 965;
//   one-wave: MQA B=1 H=32 S=4096 D=64, 32 / 16 / 64: 179 / 212 / 188; MHA B=1 H=16 S=4096
//   D=64, 2 / 1 / 4: 98 / 108 / 113; B=2 H=16 S=4096 D=64, 1 / 2: 155 / 186; MQA B=1 H=32
//   S=16384 D=64, 16 / 8 / 32: 2039 / 2160 / 2074.
// (The previous rule, 2 x CU items per 4096 keys for both kernels, chose 4 for MHA
// B=1 H=4 S=8192 and for the GQA shape, 16 for B=1 H=8 H_kv=1 and for MQA S=4096 D=64, and
// 1 for MHA B=1 H=16 D=64: 14, 3, 5, 18 and 10 % slower.)  D = 32 runs the one-wave kernel
// and takes its rule unmeasured.
int dkdv_target_workgroups(int S, int D) {
  const int slots = cu_count() * (D == 128 ? 1 : 2);
  return 2 * slots * std::max(1, (S + 8191) / 8192);
}

size_t gqa_workspace_bytes(int B, int H_kv, int S, int D, int nsplit) {
  return nsplit > 1 ? 2 * (size_t)B * H_kv * nsplit * S * D * sizeof(float) : 0;
}

// -LSE/c and -Delta per query row ([2, B*H, S] fp32), rounded up to 256 bytes so
// the partial sums after them stay aligned
size_t rowb_bytes(int B, int H, int S) {
  return (2 * (size_t)B * H * S * sizeof(float) + 255) / 256 * 256;
}

// Chunks per key tile for dK/dV: enough that B * H_kv * (key tiles) * nsplit
// reaches the target number of work items, at most the pairs of the heaviest key
// tile (G query heads x all 64-row query tiles) and kMaxDkdvSplit; 1 when the key
// tiles alone already reach it, or when the heaviest tile has fewer than
// kMinSplitPairs pairs: then the partial-sum traffic and the extra pass cost more
// than the imbalance (profiles/tile_study_mha_gqa_bwd.md, dK/dV + reduction: B=2 H=8
// S=2048 D=128, 32 pairs, 57 us whole against 282 at split 16; B=1 H=8 S=4096, 64
// pairs, 98 -> 86 us at split 2; MQA B=1 H=32 S=4096 D=64 1748 -> 196 us at split 64).
constexpr int kMaxDkdvSplit = 64;
constexpr int kMinSplitPairs = 64;
int dkdv_nsplit(int B, int H, int H_kv, int S, int D) {
  const long long items = (long long)B * H_kv * ((S + fa::kDkdvKeys - 1) / fa::kDkdvKeys);
  const long long want = dkdv_target_workgroups(S, D);
  const long long pairs = (long long)(H / H_kv) * ((S + 63) / 64);
  if (items >= want || pairs < kMinSplitPairs) return 1;
  long long s = (want + items - 1) / items;
  if (s > pairs) s = pairs;
  if (s > kMaxDkdvSplit) s = kMaxDkdvSplit;
  return s < 1 ? 1 : (int)s;
}

// Whether the backward runs as bwd_small_kernel: dQ and dK/dV in one launch of 64-row and 64-key
// workgroups (a split dK/dV keeps its kernel behind that launch's dQ).  By the number W of dQ's 64-row
// workgroups: at D = 128, whose workgroup has a CU to itself, up to one per CU; at D <= 64 up to three.
// Within that the launch's dK/dV workgroups, W / group, bound it: the 128-key kernel has
// half as many, so the fewer there are, the longer the one launch is ahead.  For MHA the bound is the
// `quarters` of a workgroup per CU below: less for short sequences, where with one or two tiles to a
// chain there is little to halve and the two launches are already short; a dK/dV workgroup weighs
// five times a dQ one (fitted on groups of 1 to 8).  A split counts as MHA: there the launch is dQ alone.
// The workspace does not decide, so dQ is the same with and without one.
// Measured, us of the two kernels / the one launch (W):
//   D = 32:  B=2 H=8 S=1024 (256) 27.6 / 15.5, B=1 H=16 S=2240 (560) 52.6 / 42.0, B=3 H=8 S=2048 (768) 68.0 /
//   51.1, B=8 H=16 S=512 (1024) 24.3 / 25.5; 381 heads S=128 (762) 12.9 / 13.9; groups of 2 to 8, W up to 768: 0.49 to
//   0.99, mean 0.69; MQA 128 heads S=384 (768) 46.0 / 47.6
//   D = 64:  B=2 H=8 S=512 (128) 23.4 / 12.2, B=2 H=16 S=1024 (512) 37.8 / 32.6, B=3 H=16 S=832 (624) 40.4 /
//   34.7, B=4 H=16 S=1024 (1024) 54.9 / 58.3; 512 heads S=64 (512) 13.0 / 14.8, 251 heads S=128 (502) 15.4 /
//   17.1, 384 heads S=128 (768) 20.5 / 23.5, 125 heads S=320 (625) 24.1 / 25.3, 75 heads S=600 (750) 35.3 / 38.0,
//   24 heads S=2048 (768) 0.84, 16 heads S=3000 (752) 103 / 109; groups of 2 to 8: 0.49 to 1.02 (but of 2, 768 heads S=64
//   17.8 / 19.0), mean 0.75; MQA 160 heads S=256 (640) 53.2 / 56.8
//   D = 128: B=2 H=8 S=512 (128) 36.3 / 22.7, B=3 H=5 S=1000 (240) 56.5 / 46.3, B=2 H=8 S=1024 (256) 56.4 /
//   45.2, B=3 H=8 S=768 (288) 47.2 / 47.8, B=4 H=16 S=512 (512) 39.9 / 59.0; 256 heads S=64 (256) 15.3 / 20.1, 128
//   heads S=64 (128) 0.67; of groups 256 heads S=64: of 2 16.8 / 17.6, of 4 0.82
//   dQ alone of a split: B=1 H=4 S=4096 D=128 137 / 124, D=64 94 / 87; B=2 H=8 H_kv=2 S=2048 D=64 73 / 70
// At about 3700 sizes, groups of 1 to 32, the calls that take it lie between 0.44 and 1.04 of the
// two kernels' time, mean 0.73.
bool bwd_small(int B, int H, int H_kv, int S, int D) {
  const long long tiles = (S + 63) / 64, dq = (long long)B * H * tiles, cus = cu_count();
  if (dq > (D == 128 ? 1 : 3) * cus) return false;
  const long long dkdv = dkdv_nsplit(B, H, H_kv, S, D) > 1 ? dq : (long long)B * H_kv * tiles;
  int quarters;
  if (D == 128) quarters = S <= 64 ? 2 : 4;
  else if (D == 32) quarters = S > 64 && S <= 384 ? 10 : 12;
  else if (S <= 128) quarters = S <= 48 ? 12 : S <= 64 ? 6 : S <= 100 ? 10 : 7;
  else if (S <= 640) quarters = S <= 384 ? 9 : 10;
  else quarters = S <= 2048 && (long long)B * H % 8 == 0 ? 12 : 11;
  return 2 * (dq + 5 * dkdv) <= 3 * quarters * cus;
}

// ---------------------------------------------------------------------------
// Device scratch of the allocation-free backward (fa_bwd_gqa_noalloc): stands in
// for fa_bwd_gqa's caller workspace.  Each device that loads the library holds its
// own copy until the process ends.  On the host the array's name is only a
// stand-in for the symbol, never a device address: host code uses the address
// that hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
std::atomic<void*> g_scratch[kMaxDevices];
std::mutex g_scratch_mu;

}  // namespace

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

// This device's copy of `scratch`, looked up on the first call on the device (with
// it current) and kept; FA_ERR_LAUNCH if the runtime cannot name it.
int scratch_address(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FA_ERR_LAUNCH;
  void* p = g_scratch[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch[dev].load(std::memory_order_relaxed);
    if (!p) {
      if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FA_ERR_LAUNCH;
      g_scratch[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return FA_OK;
}

}  // namespace

extern "C" {

int fa_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
           int B, int H, int H_kv, int S, int D, int dtype, float scale_log2,
           int block_m, int block_n, void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, block_m, block_n);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H_kv > H || H % H_kv != 0) return FA_ERR_DIMS;
  if (!q || !k || !v || !o) return FA_ERR_NULL;
  FwdShape w;
  if (!fwd_key_split(B, H, S, D, &w)) {
    // 64-key tiles whatever block_n: a 128-key tile needs more registers than two waves per
    // SIMD have, and is slower everywhere (us of 128 x 128 / 128 x 64, D = 32, 64, 128: MHA B=4
    // H=32 S=2048 89 / 62, 112 / 87, 189 / 139; GQA B=2 H=16 H_kv=4 S=4096 73 / 56, 97 / 77, 167 / 129;
    // B=16 H=32 S=512 D=32 47 / 29)
    const int tile_m = fwd_tile_m(B, H, S, block_m);
    const int gh = fwd_heads_per_wg(B, H, H / H_kv, S, D, tile_m, 64);
    const bool few = gh == 1 && short_rows(B, H, S, D) && (long long)B * H * ((S + 63) / 64) > 2LL * cu_count();
    w = FwdShape{few ? 64 : fwd_block_m(tile_m, 64, D, gh), 64, gh};
  }
  fa::FwdFn fn = fwd_table(dtype, D, w.block_m, w.block_n, w.gh, lse != nullptr);
  if (!fn) return FA_ERR_UNSUPPORTED;
  fa::FwdArgs a{q, k, v, o, lse, B, H, H_kv, S, D, scale_log2, hip_stream};
  return fn(a);
}

int fa_bwd(const void* q, const void* k, const void* v, const void* o,
           const void* d_o, const float* lse, void* dq, void* dk, void* dv,
           int B, int H, int S, int D, int dtype, float scale_log2, float sm_scale,
           int block_m, int block_n, void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, block_m, block_n);
  if (st != FA_OK) return st;
  if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return FA_ERR_NULL;
  fa::BwdFn fn = bwd_fn(dtype, D, B, H, S, block_m, block_n);
  if (!fn) return FA_ERR_UNSUPPORTED;
  fa::BwdArgs a{q, k, v, o, d_o, lse, dq, dk, dv, B, H, H, S, D, scale_log2, sm_scale, hip_stream,
                nullptr, nullptr, 1, nullptr, false, bwd_small(B, H, H, S, D)};
  return fn(a);
}

size_t fa_bwd_gqa_workspace_size(int B, int H, int H_kv, int S, int D) {
  if (B <= 0 || H <= 0 || S <= 0 || H_kv <= 0 || H_kv > H || H % H_kv != 0) return 0;
  if (D != 32 && D != 64 && D != 128) return 0;
  return rowb_bytes(B, H, S) + gqa_workspace_bytes(B, H_kv, S, D, dkdv_nsplit(B, H, H_kv, S, D));
}

int fa_bwd_gqa(const void* q, const void* k, const void* v, const void* o,
               const void* d_o, const float* lse, void* dq, void* dk, void* dv,
               int B, int H, int H_kv, int S, int D, int dtype, float scale_log2, float sm_scale,
               int block_m, int block_n, void* workspace, size_t workspace_bytes, void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, block_m, block_n);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H_kv > H || H % H_kv != 0) return FA_ERR_DIMS;
  if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return FA_ERR_NULL;
  if (workspace && (reinterpret_cast<uintptr_t>(workspace) & 15)) return FA_ERR_WORKSPACE;
  fa::BwdFn fn = bwd_fn(dtype, D, B, H, S, block_m, block_n);
  if (!fn) return FA_ERR_UNSUPPORTED;
  // the workspace holds, in this order and as far as it reaches: the per-row terms
  // (dQ then runs first and dK/dV reads Delta instead of forming it), then the
  // partial sums of the split the shape asks for, or of the largest one that fits
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  size_t left = workspace ? workspace_bytes : 0;
  float* rowb = nullptr;
  if (left >= rowb_bytes(B, H, S)) {
    rowb = reinterpret_cast<float*>(ws);
    ws += rowb_bytes(B, H, S);
    left -= rowb_bytes(B, H, S);
  }
  int nsplit = workspace ? dkdv_nsplit(B, H, H_kv, S, D) : 1;
  while (nsplit > 1 && gqa_workspace_bytes(B, H_kv, S, D, nsplit) > left) --nsplit;
  float* wsk = nsplit > 1 ? reinterpret_cast<float*>(ws) : nullptr;
  float* wsv = nsplit > 1 ? wsk + (size_t)B * H_kv * nsplit * S * D : nullptr;
  fa::BwdArgs a{q, k, v, o, d_o, lse, dq, dk, dv, B, H, H_kv, S, D, scale_log2, sm_scale, hip_stream,
                wsk, wsv, nsplit, rowb, false, bwd_small(B, H, H_kv, S, D)};
  return fn(a);
}

int fa_bwd_gqa_noalloc(const void* q, const void* k, const void* v, const void* o,
                       const void* d_o, const float* lse, void* dq, void* dk, void* dv,
                       int B, int H, int H_kv, int S, int D, int dtype, float scale_log2, float sm_scale,
                       int block_m, int block_n, void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, block_m, block_n);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H_kv > H || H % H_kv != 0) return FA_ERR_DIMS;
  if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return FA_ERR_NULL;
  // the scratch is fa_bwd_gqa's workspace of kNoAllocScratchBytes: the per-row terms must
  // fit, and fa_bwd_gqa then takes the largest dK/dV split whose partial sums fit behind
  // them (the whole split the shape asks for when it fits), so the results are those of
  // fa_bwd_gqa given a workspace of that size.  Nothing in it needs clearing: dQ writes
  // every row's terms before dK/dV reads them, and every split chunk stores its whole
  // partial sum before the reduction reads it.
  if (rowb_bytes(B, H, S) > kNoAllocScratchBytes) return FA_ERR_SCRATCH;
  void* ws = nullptr;
  st = scratch_address(&ws);
  if (st != FA_OK) return st;
  return fa_bwd_gqa(q, k, v, o, d_o, lse, dq, dk, dv, B, H, H_kv, S, D, dtype, scale_log2, sm_scale,
                    block_m, block_n, ws, kNoAllocScratchBytes, hip_stream);
}

size_t fa_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes; }

int fa_fwd_exact(const void* q, const void* k, const void* v, void* o, float* lse,
                 int B, int H, int H_kv, int S, int D, int dtype, float scale_log2,
                 int block_m, int block_n, int heads_per_wg, void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, block_m, block_n);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H_kv > H || H % H_kv != 0) return FA_ERR_DIMS;
  // the heads of one workgroup share one K/V head
  if (heads_per_wg <= 0 || (H / H_kv) % heads_per_wg != 0) return FA_ERR_DIMS;
  if (!q || !k || !v || !o) return FA_ERR_NULL;
  fa::FwdFn fn = fwd_table(dtype, D, block_m, block_n, heads_per_wg, lse != nullptr);
  if (!fn) return FA_ERR_UNSUPPORTED;
  fa::FwdArgs a{q, k, v, o, lse, B, H, H_kv, S, D, scale_log2, hip_stream};
  return fn(a);
}

int fa_bwd_gqa_exact(const void* q, const void* k, const void* v, const void* o,
                     const void* d_o, const float* lse, void* dq, void* dk, void* dv,
                     int B, int H, int H_kv, int S, int D, int dtype, float scale_log2, float sm_scale,
                     int dq_block_m, int dq_block_n, int nsplit, void* workspace, size_t workspace_bytes,
                     void* hip_stream) {
  int st = check_common(B, H, S, D, dtype, dq_block_m, dq_block_n);
  if (st != FA_OK) return st;
  if (H_kv <= 0 || H_kv > H || H % H_kv != 0) return FA_ERR_DIMS;
  if (nsplit < 1 || nsplit > kMaxDkdvSplit) return FA_ERR_DIMS;
  if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return FA_ERR_NULL;
  if (workspace && (reinterpret_cast<uintptr_t>(workspace) & 15)) return FA_ERR_WORKSPACE;
  // the split's partial sums must fit behind the per-row terms; without a workspace
  // the reference's order runs (dK/dV forming Delta, then dQ)
  const size_t need = rowb_bytes(B, H, S) + gqa_workspace_bytes(B, H_kv, S, D, nsplit);
  if (nsplit > 1 && (!workspace || workspace_bytes < need)) return FA_ERR_WORKSPACE;
  fa::BwdFn fn = bwd_table(dtype, D, dq_block_m, dq_block_n);
  if (!fn) return FA_ERR_UNSUPPORTED;
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  const bool rows = workspace && workspace_bytes >= rowb_bytes(B, H, S);
  float* rowb = rows ? reinterpret_cast<float*>(ws) : nullptr;
  float* wsk = nsplit > 1 ? reinterpret_cast<float*>(ws + rowb_bytes(B, H, S)) : nullptr;
  float* wsv = nsplit > 1 ? wsk + (size_t)B * H_kv * nsplit * S * D : nullptr;
  fa::BwdArgs a{q, k, v, o, d_o, lse, dq, dk, dv, B, H, H_kv, S, D, scale_log2, sm_scale, hip_stream,
                wsk, wsv, nsplit, rowb, rowb == nullptr, false};
  return fn(a);
}

int fa_fwd_heads_per_wg(int B, int H, int H_kv, int S, int D, int block_m, int block_n) {
  if (B <= 0 || H <= 0 || S <= 0 || H_kv <= 0 || H_kv > H || H % H_kv != 0) return 0;
  if (D != 32 && D != 64 && D != 128) return 0;
  if (!tile_ok(block_m) || !tile_ok(block_n)) return 0;
  if (fwd_key_split(B, H, S, D, nullptr)) return 1;
  // (fa_fwd's tiles are 64 keys whatever block_n)
  return fwd_heads_per_wg(B, H, H / H_kv, S, D, fwd_tile_m(B, H, S, block_m), 64);
}

int fa_fwd_rows_per_wg(int block_m, int block_n, int D, int heads_per_wg) {
  if (!tile_ok(block_m) || !tile_ok(block_n)) return 0;
  return fwd_block_m(block_m, block_n, D, heads_per_wg);
}

int fa_bwd_dq_rows_per_wg(int block_m, int D) { return tile_ok(block_m) ? dq_block_m(block_m, D) : 0; }

int fa_bwd_dkdv_split(int B, int H, int H_kv, int S, int D) {
  if (B <= 0 || H <= 0 || S <= 0 || H_kv <= 0 || H_kv > H || H % H_kv != 0) return 0;
  if (D != 32 && D != 64 && D != 128) return 0;
  return dkdv_nsplit(B, H, H_kv, S, D);
}

int fa_supported(int dtype, int D, int block_m, int block_n, int group, int with_lse, int is_bwd) {
  if (check_common(1, 1, 256, D, dtype, block_m, block_n) != FA_OK) return 0;
  if (group <= 0) return 0;
  if (is_bwd) return bwd_table(dtype, D, block_m, block_n) ? 1 : 0;
  return fwd_table(dtype, D, block_m, block_n, heads_per_wg(group, block_m, block_n), with_lse) ? 1 : 0;
}

const char* fa_strerror(int status) {
  switch (status) {
    case FA_OK: return "ok";
    case FA_ERR_DIMS:
      return "invalid dimensions (B, H, H_kv, S must be positive, H_kv must divide H, B*H*S and "
             "S*D*2 must stay below 2^31)";
    case FA_ERR_DTYPE: return "unsupported dtype (expected float16 or bfloat16)";
    case FA_ERR_HEADDIM: return "unsupported head dim (expected 32, 64 or 128)";
    case FA_ERR_TILE: return "unsupported tile (block_m and block_n must be 64 or 128)";
    case FA_ERR_NULL: return "a required pointer is NULL";
    case FA_ERR_LAUNCH: return "HIP kernel launch failed";
    case FA_ERR_UNSUPPORTED: return "no kernel for this combination";
    case FA_ERR_WORKSPACE:
      return "workspace not 16-byte aligned (or, for fa_bwd_gqa_exact, too small for the requested split)";
    case FA_ERR_SCRATCH:
      return "this shape's per-row terms (8 * B * H * S bytes) exceed the library's device scratch "
             "(fa_bwd_gqa_noalloc); use fa_bwd_gqa with a caller workspace";
    default: return "unknown status";
  }
}

int fa_version(void) { return 140; }

}  // extern "C"
