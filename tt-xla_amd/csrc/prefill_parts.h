// Prefill passes of few query rows over many cached keys, split over the keys: several workgroups per row block, each
// with a share of the keys, hand float accumulators to prefill_merge_kernel.  Shared by the two loops
// (prefill_stream.hip, prefill.hip), whose lanes hold the accumulators alike.
#pragma once

#include "prefill_common.h"

#include <algorithm>

namespace ttpa {
namespace {

// ---- splitting over the keys --------------------------------------------------------------------
// Splitting costs a second launch (1.4 us, also where the kernel then does not split), the start of more
// workgroups, and 64 KiB of float accumulators written and read per part and workgroup; it saves about 0.48 us per
// 32-key block that a workgroup need not walk.  How many blocks there are is in device memory (the host sees the
// page table's width), so the host launches the most parts that may be wanted and the kernel decides, as does the
// merge kernel with the same function.  Attention of a pass in us, unsplit / split, by workgroups of the unsplit launch:
//    8 (32 rows, 32 / 8 heads):   10 blocks 12.8 / 13.6, 16 blocks 15.9 / 13.7, 64 blocks 38.9 / 16.1
//   32 (128 rows, 32 / 8 heads):  10 blocks 12.9 / 14.7, 16 blocks 16.0 / 15.2, 64 blocks 39.4 / 23.8
//   64 (4 x 64 rows, 32 / 8):     16 blocks 16.1 / 17.7, 32 blocks 24.0 / 21.9, 64 blocks 39.4 / 23.7
//  128 (512 rows, 32 / 8 heads):  32 blocks 23.6 / 27.1, 64 blocks 38.5 / 35.0, 128 blocks 68.8 / 46.9
//  192 (3 x 256 rows, 32 / 8):    64 blocks 40.0 / 41.8, 96 blocks 55.1 / 53.8, 256 blocks 131 / 115
//  256 (512 rows, 64 / 8 heads):  64 blocks 41.2 / 47.3, 128 blocks 76.9 / 77.8, 256 blocks 145 / 138
// so (the streaming loop) from 16 blocks on, or 7 / 16 of the number of workgroups, or half of it where a split leaves no CU to itself.  The last
// row block decides for all: where some are split and others are not, the launch is as long as without a split and the merge comes
// on top (4 x 64 rows of 32 / 8 heads, 23 and 24 blocks, the pass 27 us, 22 without a split).
// The plain loop's passes (prefill.hip) are longer per block: 0.49 us at head size 64, 1.2 at 256, 0.72 and 1.15 where it expands
// block-float-8 blocks of 64 and 128 on their way into LDS.  So its parts may be shorter and a launch is split from fewer blocks:
// whole passes (fill and attention), before there was a split / with it:
//   head size 64, 8 / 8 heads:   1 x 224 rows behind 320 tokens 17.1 / 13.5, 1216 30.5 / 15.1, 8192 136 / 18.9; 4 x 64 behind 640 20.5 / 14.5
//   head size 64, 64 / 8 heads:  1 x 128 rows behind 640 tokens 21.9 / 18.5, 2368 47.1 / 24.4
//   head size 256, 16 / 8 heads: 5 x 192 rows behind 832 tokens 67 / 49; 1 x 32 behind 256 23.8 / 20.7, 2368 97.9 / 32.9
//   block-float-8, 8 / 8 of 64:  1 x 128 rows behind 640 tokens 26.9 / 17.3, 2368 65 / 18.8
// The host knows how many blocks there may be from the page table, or closer from a caller who knows where the chunk lies
// (a.keys_bound): by a table of 8192 tokens alone a pass that reads few of them prepares a split that it does not make, which costs
// 1.5 us (whole passes, bounded / not: 32 rows of 8/8 heads of 64 behind 64 tokens 9.2 / 10.9, 512 rows of 64/8 behind 512 24.5 /
// 26.2, block-float-8, 128 rows of 16/16 of 128 behind 64 16.2 / 19.3).  Where
// a table holds little more than the blocks to split from, the parts would be few and the merge launch be there for nothing
// where the pass reads less: 1 x 32 rows behind 128 tokens 10.4 us, 12.4 with.
struct SplitRule {
  int wgs_per_cu;               // workgroup slots of a CU
  int min_part, min_split;      // 32-key blocks per part at least; blocks from which on a launch is split
  int table_percent;            // a page table holds at least this many hundredths of the blocks to split from
  int known_percent;            // ... or that the caller knows of: copies are better than the shortest split of block-float-8 blocks
  int block_cost;               // of a 32-key block, in hundredths of the streaming loop's
};
// At 64 and 256 the streaming loop keeps the parts of the plain one: with 128's rule (two thirds as many parts) 4 x 64 rows of 8 / 8 heads
// of 64 behind 1024 tokens took 16.0 us instead of 14.9, and the error against 64 bits was 1 ... 5 % larger, since a part starts from a
// maximum of its own.
constexpr SplitRule stream_split(int d) {
  return d == 128 ? SplitRule{2, 8, 16, 100, 100, 100} : SplitRule{d == 64 ? 2 : 1, 4, 8, 150, 100, d == 64 ? 150 : 300};
}
constexpr SplitRule plain_split(int d, bool bfp8) { return {d <= 128 ? 2 : 1, 4, 8, bfp8 ? 125 : 150, bfp8 && d == 128 ? 113 : 100, d == 256 ? 300 : bfp8 ? 225 : 150}; }
// Parts up to one workgroup per CU; twice as many, which then share a CU's matrix pipes, from this many blocks per part
// on (128 workgroups, 2 / 4 parts: 64 blocks 35.0 / 35.6 us, 80 blocks 43.5 / 41.5, 96 blocks 43.6 / 40.8, 256 blocks
// 82.5 / 77.3).
constexpr int kSharedPartBlocks = 20;
constexpr int kMaxParts = 16;
constexpr int kBlockKeys = 32;
constexpr int part_acc_floats(int d) { return kRowsPerWave * d; }  // accumulators of one (part, head, row block)

// Blocks of a part (whole 64-key tiles) in a launch whose first query row is at `offset`; a row block of no more is not split.
__host__ __device__ __forceinline__ int part_of_blocks(const PrefillArgs &a, int most) {
  if (most < a.split_from) return most;
  const int shared = quotient(a.by_parts, most + a.parts - 1);
  const int share = shared >= kSharedPartBlocks ? shared : max(quotient(a.by_parts_one, most + a.parts_one - 1), a.part_min);
  return (share + 1) & ~1;
}
__device__ __forceinline__ int blocks_per_part(const PrefillArgs &a, int offset) {
  return part_of_blocks(a, max(((a.causal ? min(a.skv, offset + a.sq) : a.skv) + kBlockKeys - 1) / kBlockKeys, 1));  // (of the last row block)
}

// Accumulators and (reference, sum) rows of the parts: [part][batch][head][row block], the statistics
// behind all accumulators.
struct PartLayout {
  int64_t slots;  // (part, batch entry, head, row block) combinations
  int row_blocks;
};
__host__ __device__ inline PartLayout part_layout(const PrefillArgs &a) {
  const int rb = (a.sq + kRowsPerWave - 1) / kRowsPerWave;
  return {(int64_t)a.parts * a.batch * a.hq * rb, rb};
}

// Merges the parts of a row block: out = sum_p 2^(m_p - M) acc_p / sum_p 2^(m_p - M) l_p.  One workgroup per
// (row block, head, batch entry); thread (n, g) takes row n and head-dim elements 16 g .. 16 g + 15, which lie in
// register groups 2 g and 2 g + 1 of lanes n and n + 32 (prefill_stream_kernel's lane holds elements
// 8 group + 4 (lane / 32) .. + 3): 512 consecutive bytes per read of 32 lanes, whole 32-byte pieces of a row per
// write.  Memory bound: 34 MB of accumulators (512 rows, 32 heads, 4 parts) in 7.9 us.  Parts past the last are zeros: repeated
// with weight 0 they needed as long at head sizes 64 and 128 and 5 us more at 256 (128 rows of 16/8 heads behind 2048 tokens 36.7 / 31.7).
template <int D>
__global__ __launch_bounds__(2 * D) void prefill_merge_kernel(PrefillArgs a) {
  const int rb = blockIdx.x, hq = blockIdx.y, b = blockIdx.z;
  const int pair = rb * a.head_group + hq - quotient(a.by_head_group, hq) * a.head_group;
  const int n = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int offset = a.causal ? chunk_offset(a.chunk_start, a.sq, a.skv) : 0;
  const int wg_last_row = min(a.sq, (last_row_block(a, pair >> 2) + 1) * kRowsPerWave) - 1;
  const int kv_end = a.causal ? min(a.skv, offset + wg_last_row + 1) : a.skv;
  const int nblk = (kv_end + kBlockKeys - 1) / kBlockKeys;
  const int share = blocks_per_part(a, offset);
  if (share >= nblk) return;  // one workgroup saw all keys and wrote the output
  const int active = (nblk + share - 1) / share;
  const PartLayout lay = part_layout(a);
  const int64_t step = (int64_t)a.batch * a.hq * lay.row_blocks;
  const int64_t at = ((int64_t)b * a.hq + hq) * lay.row_blocks + rb;
  const float *acc = a.part_acc + at * part_acc_floats(D) + (8 * g) * 64 + 4 * n;
  const float *stats = a.part_acc + lay.slots * part_acc_floats(D) + at * (2 * kRowsPerWave) + 2 * n;
  float m[kMaxParts], l[kMaxParts];
  float top = -INFINITY;
#pragma unroll
  for (int p = 0; p < kMaxParts; ++p) {
    const int q = min(p, active - 1);
    const float2 s = *reinterpret_cast<const float2 *>(stats + q * step * (2 * kRowsPerWave));
    m[p] = s.x, l[p] = p < active ? s.y : 0.f;
    top = fmaxf(top, m[p]);
  }
  float sum = 0.f;
  float o[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = 0.f;
  // four parts' accumulators in flight at a time; parts past the last are zeros with weight 0 (with the last one's values an
  // infinite one would become NaN)
  for (int p0 = 0; p0 < active; p0 += 4) {
    float4 v[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float *src = acc + min(p0 + j, active - 1) * step * part_acc_floats(D);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] = *reinterpret_cast<const float4 *>(src + (i >> 1) * 256 + (i & 1) * 128);  // group 2 g + i / 2, lane half i % 2
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float w = 0.f;
      if (p0 + j >= active) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int p = 0; p < kMaxParts; ++p)
        if (p == p0 + j && p < active) w = __builtin_amdgcn_exp2f(m[p] - top), sum = fmaf(w, l[p], sum);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o[4 * i] = fmaf(w, v[j][i].x, o[4 * i]), o[4 * i + 1] = fmaf(w, v[j][i].y, o[4 * i + 1]);
        o[4 * i + 2] = fmaf(w, v[j][i].z, o[4 * i + 2]), o[4 * i + 3] = fmaf(w, v[j][i].w, o[4 * i + 3]);
      }
    }
  }
  const int row = rb * kRowsPerWave + n;
  if (row >= a.sq) return;
  const float inv = 1.0f / sum;
  uint16_t *op = a.out + b * a.out_bs + hq * a.out_hs + (int64_t)row * a.out_ts + 16 * g;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<uint2 *>(op + 4 * i) = make_uint2(pack_bf16x2(o[4 * i] * inv, o[4 * i + 1] * inv), pack_bf16x2(o[4 * i + 2] * inv, o[4 * i + 3] * inv));
}

// Workgroups of the launch without a split, and what it may be split into: as many parts as fill the workgroup slots of
// every CU once, if its row blocks leave at least half of them empty and its page keys may be enough to be split at all.
inline void set_parts(PrefillArgs &a, int heads, const SplitRule &rule) {
  const int pairs = (a.sq + kRowsPerWave - 1) / kRowsPerWave * heads;
  const int64_t wgs = (int64_t)a.batch * (a.hq / heads) * ((pairs + 3) / 4);
  const int blocks = (int)((a.keys_bound + kBlockKeys - 1) / kBlockKeys);
  const int most = std::min(kMaxParts, (blocks + rule.min_part - 1) / rule.min_part);
  const int64_t from = 2 * wgs <= a.cus ? 7 * wgs / 16 : std::min<int64_t>(wgs, rule.wgs_per_cu * a.cus) / 2;
  a.split_from = (int)std::max<int64_t>(rule.min_split, 100 * from / rule.block_cost);
  a.part_min = rule.min_part;
  a.parts = blocks < a.split_from * (a.keys_known ? rule.known_percent : rule.table_percent) / 100 ? 1 : (int)std::max<int64_t>(1, std::min<int64_t>(rule.wgs_per_cu * a.cus / wgs, most));
  a.parts_one = (int)std::max<int64_t>(1, std::min<int64_t>(a.cus / wgs, most));
  a.by_parts = divisor(a.parts), a.by_parts_one = divisor(a.parts_one);
}

inline int64_t part_bytes(PrefillArgs a, int heads, const SplitRule &rule, int d) {
  set_parts(a, heads, rule);
  if (a.parts <= 1) return 0;
  return part_layout(a).slots * (part_acc_floats(d) + 2 * kRowsPerWave) * (int64_t)sizeof(float);
}

// Bytes of the scratch an expanded block-float-8 pass needs: K and V copies of batch * width blocks
// and their table.
inline int64_t expand_bytes(int batch, int width, int kv_heads, int block_size, int d) {
  const int64_t blocks = (int64_t)batch * width;
  return 2 * blocks * kv_heads * block_size * d * 2 + ((blocks * 4 + 255) & ~int64_t(255));
}

// Query heads of a workgroup of the plain loop, which takes whole row blocks of 4, 2 or 1 heads.
inline int heads_per_workgroup(const PrefillArgs &a) {
  const int g = a.hq / a.hkv;
  return g % 4 == 0 ? 4 : g % 2 == 0 ? 2 : 1;
}

// What a launch of `heads` query heads per head group is cut into for the most keys that it may see: its workgroups, the blocks of a part.
struct Cut {
  int64_t workgroups;  // of all parts
  int part, parts;
};
inline Cut cut(PrefillArgs a, int heads, const SplitRule &rule) {
  set_parts(a, heads, rule);
  const int pairs = (a.sq + kRowsPerWave - 1) / kRowsPerWave * heads, blocks = (int)((a.keys_bound + kBlockKeys - 1) / kBlockKeys);
  const int part = a.parts > 1 ? part_of_blocks(a, blocks) : blocks, parts = (blocks + part - 1) / part;
  return {(int64_t)a.batch * (a.hq / heads) * ((pairs + 3) / 4) * parts, part, parts};
}

// Query heads of a head group of the streaming loop, whose wavefronts may be of different row blocks wherever the heads end: four, or all of a KV
// head's where these are no multiple of four, but for a chunk of one row block that the plain loop's groups, a workgroup for every one or two heads, leave
// as short: each of those has a CU to itself (13 of 16 are taken at most), and its one or two wavefronts with rows wait for no others.  A split costs
// about what eleven blocks do.  us per pass, pairs / a workgroup per head, 40 / 8 of 128: 1 x 32 rows behind 512 tokens 15.8 / 15.3, 832 16.1 / 15.5,
// 2 x 32 behind 512, which then is not split, 16.6 / 15.5; 24 / 8, 3 x 32 behind 512 16.3 / 15.3; 10 / 2 of 64, 1 x 32 behind 512 12.3 / 11.3;
// beyond: 40 / 8, 1 x 32 behind 2432 18.9 / 21.8, 2 x 32 behind 640 16.7 / 18.0, 3 x 32 behind 512 15.7 / 16.8.
constexpr int kSplitBlocks = 11;
inline int head_group_size(const PrefillArgs &a, int d) {
  const int g = a.hq / a.hkv, fewer = heads_per_workgroup(a);
  if (g % 4 == 0) return 4;
  if (!a.pt || a.sq > kRowsPerWave || g == fewer) return g;
  const Cut pairs = cut(a, g, stream_split(d)), heads = cut(a, fewer, stream_split(d));
  const bool as_short = heads.part + (heads.parts > 1 ? kSplitBlocks : 0) <= pairs.part + kSplitBlocks;
  return pairs.parts > 1 && as_short && 16 * heads.workgroups <= 13 * a.cus ? fewer : g;
}

// Whether the workgroups of a KV head's pairs are spread over the XCDs: three quarters of the CUs or more have a part each, all of a KV head's, which ask
// for the same blocks at the same time, would be on one or two XCDs, and the caches are small enough for several XCDs to read the same.  (One row block has too
// few workgroups per KV head for that, and at head size 64 there was nothing in it.)  us per pass of 40 / 8 heads of 128, a KV head on one XCD / spread (before
// pairs, whole row blocks of single heads, five KV heads on an XCD): 1 x 96 rows behind 1600 tokens 23.1 / 21.1 (21.3), 1 x 128 behind 2432
// 26.7 / 24.6 (24.3), 1 x 256 behind 1216 28.9 / 26.3 (25.8), 2 x 96 behind 832 23.9 / 21.7 (22.8), 1 x 384 behind 1600 36.1 / 33.8
// (33.6); 28 / 4, 1 x 256 behind 2432 29.7 / 27.0 (27.0).  Fewer workgroups: 1 x 128 behind 832 20.4 / 20.9; more keys: 1 x 192 behind 5504
// 39.9 / 46.5, 2 x 96 behind 3200 30.1 / 31.5; head size 64: 1 x 256 behind 512 17.9 / 17.9.
constexpr int64_t kSpreadBytes = 14 << 20;
inline bool spreads_groups(const PrefillArgs &a, int heads, int d) {
  if (a.parts <= 1 || heads == heads_per_workgroup(a) || a.sq <= kRowsPerWave || d < 128 || 4 * a.batch * a.hkv * a.keys_bound * d > kSpreadBytes) return false;
  // (a caller's bound may be a few blocks beyond the chunk: parts that two workgroups of a CU would only just share count as not shared)
  const int64_t blocks = (a.keys_bound + kBlockKeys - 1) / kBlockKeys;
  if ((blocks + a.parts - 1) / a.parts >= kSharedPartBlocks + 2) return false;
  const int64_t part = (std::max<int64_t>((blocks + a.parts_one - 1) / a.parts_one, a.part_min) + 1) & ~1;
  const int64_t pairs = (a.sq + kRowsPerWave - 1) / kRowsPerWave * heads, workgroups = a.batch * (a.hq / heads) * ((pairs + 3) / 4) * ((blocks + part - 1) / part);
  return 4 * workgroups >= 3 * a.cus && workgroups <= a.cus;
}

// Whether the plain loop may split the keys of this launch: paged, each row sees all keys up to its own.
inline bool plain_splits(const PrefillArgs &a) { return a.pt != nullptr && a.window == 0 && a.mask == nullptr; }

// Bytes of scratch with which it does (0: it would not).
inline int64_t plain_part_bytes(const PrefillArgs &a, int d, bool bfp8) {
  return plain_splits(a) ? part_bytes(a, heads_per_workgroup(a), plain_split(d, bfp8), d) : 0;
}

}  // namespace
}  // namespace ttpa
